"""Build the in-tree HIP kernel library ``_dnn_hip`` for gfx950 with hipcc.

No torch cpp_extension (it hipifies sources); plain ``hipcc --offload-arch=gfx950``
per translation unit, incremental on mtimes, then one shared-object link into
the package directory so the built ``.so`` ships with the repo snapshot to the
GPU box.  Usage: ``python -m distributed_neural_networks_amd.ops.build [-j N] [--force]``.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import glob
import os
import subprocess
import sys
import sysconfig
from typing import List

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
CSRC = os.path.join(ROOT, "csrc")
PKG = os.path.join(ROOT, "distributed_neural_networks_amd")
BUILD = os.path.join(ROOT, "build", "hip")
ARCH = os.environ.get("DNN_OFFLOAD_ARCH", "gfx950")
EXT_SUFFIX = sysconfig.get_config_var("EXT_SUFFIX") or ".so"
TRANSFORMER_SRCS = ("norm_embed.hip", "attention.hip", "sampler.hip", "gemm_fp8.hip")
# ReLU/max-pool epilogues: no NaN-canonicalising v_max before every fmaxf of an MFMA result
# No SLP vectoriser where it packs scalar FP32 into cross-half v_pk_*_f32 (op_sel
# reads of a pair's other half) whose low result a 32-bit VALU op reads: under two
# workgroups per CU that read returned the pre-op value in lanes 48-63 (the
# one-shot GEMM's row statistics, csrc/kernels/gemm_oneshot.h; 100 -> 0
# mismatches in 10000 calls, profiles/r6_oneshot_race_root_cause.md).
NO_SLP = ["-fno-slp-vectorize"]
# No packed FP32 instructions anywhere (some v_pk_*_f32 forms returned wrong
# lanes, see above): explicit float2 / ext_vector code is split per element too.
NO_PACKED_FP32 = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
PER_FILE_FLAGS = {"cifar_fused.hip": ["-ffast-math"],
                  # fp32-accurate split path: keep IEEE rounding, only drop NaN canonicalisation in fmaxf
                  "cifar_x3.hip": ["-fno-honor-nans"],
                  "cifar_wino.hip": ["-fno-honor-nans"] + NO_SLP,
                  # flash / decode softmax maxima over MFMA results: no v_max canonicalise
                  # per score (52 -> 17 v_max per GPT-2 flash block); -inf masking is kept
                  "attention.hip": ["-fno-honor-nans"] + NO_SLP,
                  "paged_attention.hip": ["-fno-honor-nans"] + NO_SLP,
                  "latent_attention.hip": ["-fno-honor-nans"] + NO_SLP,
                  "recurrence.hip": NO_SLP,
                  "wkv.hip": NO_SLP,
                  "delta_rule.hip": NO_SLP,
                  "moe.hip": NO_SLP,
                  "gemm_skinny.hip": NO_SLP,
                  "gemm_lean.hip": NO_SLP,
                  "gemm_mid.hip": NO_SLP,
                  "gemm_mid_plain.hip": NO_SLP,
                  "gemm_mid_fp8.hip": NO_SLP,
                  "gemm_bf16.hip": NO_SLP}


def _hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.exists(c) or c == "hipcc"):
            return c
    raise RuntimeError("hipcc not found")


def sources(subset: str = "") -> List[str]:
    names = SUBSETS[subset][1]
    if names is not None:
        return [os.path.join(CSRC, n) if n.endswith(".cpp") else os.path.join(CSRC, "kernels", n) for n in names]
    return (sorted(glob.glob(os.path.join(CSRC, "kernels", "*.hip"))) + sorted(glob.glob(os.path.join(CSRC, "comm", "*.cpp")))
            + [os.path.join(CSRC, "bindings.cpp")])


def _flags(src: str) -> List[str]:
    f = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I" + CSRC, "-Wno-unused-result",
         "-Wno-unused-command-line-argument"] + NO_PACKED_FP32
    f += PER_FILE_FLAGS.get(os.path.basename(src), [])
    have_tf = all(os.path.exists(os.path.join(CSRC, "kernels", s)) for s in TRANSFORMER_SRCS)
    if have_tf:
        f.append("-DDNN_HAVE_TRANSFORMER")
    if os.path.basename(src).startswith("bindings"):
        import pybind11
        f += ["-x", "hip", "-I" + pybind11.get_include(), "-I" + sysconfig.get_paths()["include"]]
    return f


def _includes(src: str, seen: set = None) -> set:
    """``src`` and every in-tree header it includes, directly or not."""
    import re
    seen = set() if seen is None else seen
    if src in seen:
        return seen
    seen.add(src)
    with open(src) as f:
        names = re.findall(r'^\s*#\s*include\s+"([^"]+)"', f.read(), re.M)
    for n in names:
        for d in (os.path.dirname(src), CSRC):
            h = os.path.normpath(os.path.join(d, n))
            if os.path.exists(h):
                _includes(h, seen)
                break
    return seen


def _newest(src: str) -> float:
    return max(os.path.getmtime(f) for f in _includes(src))


def _obj(src: str, extra: List[str]) -> str:
    import hashlib
    tag = hashlib.sha1(" ".join(_flags(src) + extra).encode()).hexdigest()[:8]
    return os.path.join(BUILD, f"{os.path.basename(src)}.{tag}.o")


def _compile(src: str, force: bool, extra: List[str]) -> str:
    obj = _obj(src, extra)
    if not force and os.path.exists(obj) and os.path.getmtime(obj) >= _newest(src):
        return obj
    cmd = [_hipcc()] + _flags(src) + extra + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


# The full library, and the decoder subset: the kernels a paged decoder model
# runs (runtime/decoder.py), compiled without the other families' entry points,
# for a first use in a checkout that has no library yet (``ensure``).
SUBSETS = {"": ("_dnn_hip", None, []),
           "decoder": ("_dnn_decoder", ("gemm_bf16.hip", "gemm_mid.hip", "gemm_mid_plain.hip", "gemm_skinny.hip", "gemm_lean.hip", "sampler.hip", "gemm_f32.hip",
                                        "residual_rows.hip", "token_gate.hip", "paged_attention.hip",
                                        "qk_norm.hip", "recurrence.hip", "moe.hip", "token_shift.hip", "wkv.hip",
                                        "delta_rule.hip", "latent_attention.hip", "poly_norm.hip", "bindings_decoder.cpp"),
                       ["-DDNN_DECODER_ONLY"])}


def lib_path(subset: str = "") -> str:
    return os.path.join(PKG, SUBSETS[subset][0] + EXT_SUFFIX)


def stamp_path(lib: str) -> str:
    return lib[:-len(EXT_SUFFIX)] + ".build.json"


def build(force: bool = False, jobs: int = 0, verbose: bool = True, subset: str = "") -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs, lib, extra = sources(subset), lib_path(subset), SUBSETS[subset][2]
    jobs = jobs or min(len(srcs), int(os.environ.get("MAX_JOBS", "8")), os.cpu_count() or 4, 16)
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force, extra), srcs))
    newest = max(os.path.getmtime(o) for o in objs)
    if force or not os.path.exists(lib) or os.path.getmtime(lib) < newest:
        part = lib + ".part"  # moved into place whole: another process may be loading it
        cmd = [_hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}"] + objs + ["-o", part]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
        os.replace(part, lib)
    write_stamp(srcs, lib, extra)
    if verbose:
        print(f"[build] {lib} ({len(objs)} objects, arch {ARCH})", file=sys.stderr)
    return lib


def ensure(subset: str) -> None:
    """Compile ``subset`` unless a library that holds it is built from these sources."""
    from ._lib import verify_stamp
    for s in ("", subset):
        try:
            if os.path.exists(lib_path(s)):
                verify_stamp(lib_path(s))
                return
        except RuntimeError:
            pass
    build(subset=subset)


def source_digest(srcs: List[str] = None) -> dict:
    """sha256 of every source and header the library is built from."""
    import hashlib
    files = sorted(set().union(*(_includes(s) for s in (srcs or sources()))))
    return {os.path.relpath(f, ROOT): hashlib.sha256(open(f, "rb").read()).hexdigest() for f in files}


def write_stamp(srcs: List[str], lib: str, extra: List[str]) -> None:
    """Build provenance next to the .so: source hashes, per-file flags, the
    compiler, the library's own hash (``_lib.verify_stamp`` checks them at
    load, so a stale or foreign binary fails loudly instead of running)."""
    import hashlib
    import json
    import time
    r = subprocess.run([_hipcc(), "--version"], capture_output=True, text=True)
    stamp = {"arch": ARCH, "built_at": time.strftime("%Y-%m-%dT%H:%M:%S"),
             "hipcc": (r.stdout or r.stderr).strip().splitlines()[:2],
             "flags": {os.path.basename(s): _flags(s) + extra for s in srcs},
             "sources": source_digest(srcs),
             "library_sha256": hashlib.sha256(open(lib, "rb").read()).hexdigest()}
    with open(stamp_path(lib), "w") as f:
        json.dump(stamp, f, indent=1)


def main(argv=None) -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", "--jobs", type=int, default=0)
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--subset", default="", choices=sorted(SUBSETS))
    a = ap.parse_args(argv)
    build(a.force, a.jobs, subset=a.subset)
    return 0


if __name__ == "__main__":
    sys.exit(main())
