"""Lanes of a wave that exchange rows through LDS without a barrier: stores and loads of them stay in order (CPU only:
hipcc cross-compiles, nothing runs on a GPU).

A wave's LDS operations run in the order they are issued in, so a wavefront fence is all that the exchange needs, and
nothing less will do: without it the compiler may take a lane's load ahead of the stores in front of it, which are at
addresses of this lane's that it can show to be others.  The check reads the optimised LLVM IR of every kernel that
stages rows this way: between a store to LDS and a load, and between a load and the next store, there is a fence."""
import os
import re
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

from distributed_neural_networks_amd.ops import build

HIPCC = build._hipcc()


def _ir(name):
    src = os.path.join(build.CSRC, "kernels", name)
    with tempfile.TemporaryDirectory(prefix="dnn_ir_") as d:
        out = os.path.join(d, "ir.ll")
        r = subprocess.run([HIPCC, *build._flags(src), "--cuda-device-only", "-S", "-emit-llvm", "-o", out, src],
                           capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-2000:]
        with open(out) as f:
            return f.read()


def _unordered(body):
    """Lines that load from LDS behind a store to it, or store behind a load, with no fence in between."""
    last, bad = None, []
    for line in body.splitlines():
        if re.match(r"\s+fence ", line):
            last = None
        m = re.match(r"\s+(?:%\S+ = )?(load|store) .*ptr addrspace\(3\)", line)
        if m:
            if last not in (None, m.group(1)):
                bad.append(line.strip())
            last = m.group(1)
    return bad


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_rows_turned_to_fragments_by_other_lanes():
    files = {"gemm_lean.hip": "gemm_lean_kernel", "token_gate.hip": "token_gate_lean_kernel"}
    with ThreadPoolExecutor(2) as pool:
        irs = list(pool.map(_ir, files))
    for (name, kernel), ir in zip(files.items(), irs):
        found = re.findall(r"^define .*? @(\S*" + kernel + r"\S*)\(.*?\{\n(.*?)^\}", ir, re.M | re.S)
        assert len(found) >= 6, (name, [k for k, _ in found])
        for k, body in found:
            assert re.search(r"store .*ptr addrspace\(3\)", body) and re.search(r"load .*ptr addrspace\(3\)", body), k
            bad = _unordered(body)
            assert not bad, f"{name} {k}: {len(bad)} unordered, first: {bad[0]}"
