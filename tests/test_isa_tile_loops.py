"""Register use of the 256-row GEMM tiles (CPU only: hipcc cross-compiles gfx950 device assembly).

The main loops of gemm_bf16.hip fill the 256 vector registers.  An epilogue that asks for more may
make the compiler spill an operand of every K-tile, with a wait for everything in flight at its
reload: the MX product with ReLU, 2048 x 1600 x 6400, took 84 us so and takes 59."""
import os
import re
import shutil
import subprocess
import tempfile

import pytest

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def main_loops(asm: str, kernel: str):
    """(kernel, lines) of the loop with the most matrix instructions of every instance of ``kernel``."""
    for m in re.finditer(rf"^(_ZN3dnn\d+{kernel}I\S+):\s.*?\n(.*?)s_endpgm", asm, re.S | re.M):
        body = m.group(2).split("\n")
        label = {ln.split(":")[0]: i for i, ln in enumerate(body) if ln.startswith(".LBB")}
        loops = [[]]
        for i, ln in enumerate(body):
            b = re.search(r"s_c?branch\S* (\.LBB\S+)", ln)
            if b and label.get(b.group(1), i) < i:
                loops.append(body[label[b.group(1)]:i])
        yield m.group(1), max(loops, key=lambda lp: sum("v_mfma" in ln for ln in lp))


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_no_spill_between_k_tiles():
    from distributed_neural_networks_amd.ops import build as b
    src = os.path.join(b.CSRC, "kernels", "gemm_bf16.hip")
    with tempfile.TemporaryDirectory() as d:
        out = os.path.join(d, "g.s")
        r = subprocess.run([HIPCC] + b._flags(src) + ["-S", "--cuda-device-only", src, "-o", out], capture_output=True,
                           text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        asm = open(out).read()
    for kernel, count in (("gemm_fp8_256_kernel", 16), ("gemm_bf16_256_kernel", 23)):
        loops = list(main_loops(asm, kernel))
        assert len(loops) == count and all(sum("v_mfma" in ln for ln in lp) >= 32 for _, lp in loops)
        assert [n for n, lp in loops if any("scratch_" in ln for ln in lp)] == []


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_paged_decode_spills():
    """Heads of 256 fill the registers: the row's own addresses and the pages beside them spilled 31 and took 10 % longer."""
    from distributed_neural_networks_amd.ops import build as b
    src = os.path.join(b.CSRC, "kernels", "paged_attention.hip")
    with tempfile.TemporaryDirectory() as d:
        r = subprocess.run([HIPCC] + b._flags(src) + ["-c", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", src,
                                                      "-o", os.path.join(d, "p.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    spilled = {m.group(1): int(m.group(2)) for m in
               re.finditer(r"Function Name: _ZN3dnn19paged_decode_kernelI(\S+?)EEE.*?VGPRs Spill: (\d+)", r.stderr, re.S)}
    assert len(spilled) == 13 and spilled.pop("Li256ELi256ELi4") <= 20 and not any(spilled.values())
