"""The small-tile GEMM fills an LDS slot again behind the barrier that ends the
step which read it.  What orders the reads before that barrier is the kernel's
own wait, not where the compiler happens to place one: checked in the assembly
of this file's kernels."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


def _kernels(listing):
    """name -> basic blocks (lists of instructions) of each gemm_mid_kernel."""
    out, name, block = {}, None, None
    for line in listing.splitlines():
        m = re.match(r"(_ZN\w*gemm_mid_kernel\w*):", line)
        if m:
            name, block = m.group(1), []
            out[name] = [block]
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and re.match(r"\.LBB\w+:", line):
            block = []
            out[name].append(block)
        elif name and re.match(r"\s+[a-z]", line):
            block.append(line.split(";")[0].strip())
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_reads_of_a_slot_complete_before_its_refill(tmp_path):
    out = tmp_path / "gemm_mid.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(out),
                    os.path.join(ROOT, "lite_ssm_amd", "csrc", "gemm_mid.hip")],
                   check=True, capture_output=True, timeout=300)
    kernels = _kernels(out.read_text())
    assert len(kernels) == 24                          # 4 formats, 2 types, 3 tiles
    for name, blocks in kernels.items():
        loops = [b for b in blocks if any(i.startswith("v_mfma") for i in b) and "s_barrier" in b]
        assert len(loops) == 1, name
        step = loops[0]
        reads = [k for k, i in enumerate(step) if i.startswith("ds_read")]
        dma = next(k for k, i in enumerate(step) if i.startswith("global_load_lds"))
        end = step.index("s_barrier")
        # a quarter of the step's reads (the slot's last sub-step) are the
        # oldest: issued before its first DMA, all others after
        assert 4 * sum(k < dma for k in reads) == len(reads) and max(reads) < end, name
        # LDS reads complete in order: with three quarters outstanding the
        # oldest are done.  This wait stands right before the barrier.
        waits = [i for i in step[max(reads):end] if i.startswith("s_waitcnt") and "lgkmcnt" in i and "vmcnt" in i]
        assert waits, f"{name}: no wait for the slot's reads before the barrier"
        assert 4 * int(re.search(r"lgkmcnt\((\d+)\)", waits[-1]).group(1)) <= 3 * len(reads), name
