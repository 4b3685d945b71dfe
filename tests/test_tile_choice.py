"""Which tile a product of many rows takes (host code of the kernels' library, no GPU)."""

import ctypes

import pytest

from liyab_amd.csrc import build


@pytest.fixture(scope="module")
def choose():
    path = build.find_library()
    if path is None:
        pytest.skip("the kernels' library is not built")
    return ctypes.CDLL(path)._ZN5liyab16choose_gemm_tileEiii


@pytest.mark.parametrize("width", [512, 768, 1024, 1280, 1536, 1600, 2048])
def test_128_by_192_is_taken_for_a_single_round(choose, width):
    """Its second round overlaps nothing: 4 to 16 % slower there than the tiles it was taken for."""
    taken = 0
    for k, n in ((width, 3 * width), (width, width), (width, 4 * width), (4 * width, width)):
        for m in range(65, 8300, 13):
            if choose(m, n, k) == 21:
                taken += 1
                assert -(-m // 128) * -(-n // 192) <= 256, (m, n, k)
    assert taken > 0 or width == 1280


def test_256_by_256_leaves_192_by_128_what_it_takes_faster(choose):
    assert all(choose(m, 6144, 2048) == 9 for m in range(6148, 6551, 25)) and choose(7500, 6144, 2048) == 15
