"""Order of the decode attention's probabilities through LDS, in the front end's IR (CPU
only: hipcc compiles for gfx950, nothing runs).

attention_stream.h stores the probabilities of grouped heads as 16-bit values and other
lanes of the wave read them in pairs.  The wave's LDS operations run in order, so what has
to hold is that the compiler keeps it: a wavefront fence on either side of the reads, and a
read type that may alias 16-bit stores (a vector)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_probabilities_are_fenced(tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.ll"
    src.write_text('#include "kernels/attention.hip"\n'
                   "void* keep[] = {(void*)&dnn::attn_decode_stream_kernel<128, 4, 1, true, 8, 4>};\n")
    r = subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-emit-llvm",
                        "-Xclang", "-disable-llvm-passes", "-I" + os.path.join(ROOT, "csrc"), "-Wno-unused-result",
                        "-o", str(out), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    name = "attn_decode_stream_kernelILi128ELi4ELi1ELb1ELi8ELi4E"
    text = out.read_text()
    body = re.search(r"^define [^\n]*" + name + r".*?^}", text, re.S | re.M).group(0)
    parts = re.split(r'fence syncscope\("wavefront"\) acq_rel', body)
    assert len(parts) == 3
    tags = re.findall(r"= load i32, ptr %\d+, align 2, !tbaa (!\d+)", parts[1])  # the pairs; the rest are locals
    assert len(tags) == 1 and not re.search(r"= load i32, ptr %\d+, align 2,", parts[0] + parts[2])
    node = re.search(r"^%s = !{(!\d+), \1, i64 0}$" % tags[0], text, re.M).group(1)
    assert re.search(r'^%s = !{!"omnipotent char"' % node, text, re.M)
