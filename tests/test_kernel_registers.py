"""What the compiler says of kernels that are laid out to fit their registers (needs hipcc, no GPU)."""

import os
import re
import subprocess

import pytest

from liyab_amd.csrc import build


@pytest.mark.parametrize("source", ["attention_prefill_direct.hip", "sampling.hip", "gemm_skinny_ln.hip", "gemm_skinny.hip", "gemm_rows.hip", "grouped_product.hip", "gemm_mfma_waves.hip", "gemm_mfma_tile.hip", "gemm_mfma_dl.hip",
                                    "attention_mixed.hip", "attention_rows.hip"])
def test_no_kernel_spills(source, tmp_path):
    """A spilled register goes to memory and back in the walk over the keys, and counts among the loads that its waits count; in the sampler, whose threads
    hold a row, in every pass over it; in the norm's product, which is as short as the trips it waits for, in the middle of them. The kernels with rings in LDS wait for
    their loads by count: one to memory that is not theirs would be counted too. Of a tile of 256 x 256 a wave holds 128 sums a lane: a store loop that is not
    unrolled over them puts them all in memory, in every workgroup."""
    hipcc = build.hipcc_path()
    if hipcc is None:
        pytest.skip("hipcc was not found")
    r = subprocess.run([hipcc, *build.FLAGS, *build.FILE_FLAGS.get(source, []), "-I", build.CSRC, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                        os.path.join(build.CSRC, source), "-o", str(tmp_path / "kernels.o")], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.split(r"Function Name: ", r.stderr)[1:]
    assert kernels
    for k in kernels:
        spilled, scratch = (int(re.search(what + r": (\d+)", k)[1]) for what in ("VGPRs Spill", r"ScratchSize \[bytes/lane\]"))
        assert spilled == 0 and scratch == 0, f"{k.split()[0]}: {spilled} registers spilled, {scratch} bytes of scratch a lane"


def test_keys_go_to_lds_without_a_wait_between_them(tmp_path):
    """attention_rows.hip asks for 256 keys and values in loads that nobody counts: a wait for a register between two of them waits for all of them, a trip to memory each."""
    hipcc = build.hipcc_path()
    if hipcc is None:
        pytest.skip("hipcc was not found")
    source, out = "attention_rows.hip", tmp_path / "kernel.s"
    r = subprocess.run([hipcc, *build.FLAGS, *build.FILE_FLAGS.get(source, []), "-I", build.CSRC, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    blocks = re.split(r"(?m)^\.LBB\S*:|^\s+s_c?branch\S* .*$|^\s+s_barrier.*$", out.read_text())
    loads = [b for b in blocks if "global_load_lds" in b]
    assert len(loads) == 8
    assert not any("vmcnt" in b[:b.rindex("global_load_lds")] for b in loads)


def test_waves_parts_are_read_in_pieces_of_eight_bytes(tmp_path):
    """Decode attention merges its waves' parts from LDS, ten floats each: single floats, which an array that is known to be aligned to four bytes gets, make eight waves 2 to 10 % slower."""
    hipcc = build.hipcc_path()
    if hipcc is None:
        pytest.skip("hipcc was not found")
    source, out = "attention_decode.hip", tmp_path / "kernels.s"
    r = subprocess.run([hipcc, *build.FLAGS, *build.FILE_FLAGS.get(source, []), "-I", build.CSRC, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"(?ms)^_ZN5liyab23attention_decode_kernelI\S*Li8ELi4E\S*:.*?^\.Lfunc_end", out.read_text())  # (eight waves)
    assert kernels
    assert all(k.count("ds_read2_b64") > k.count("ds_read2_b32") / 4 for k in kernels), [(k.split(":")[0], k.count("ds_read2_b64"), k.count("ds_read2_b32")) for k in kernels]
