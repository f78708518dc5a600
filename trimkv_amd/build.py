"""Build the C-ABI libraries of HIP kernels in-tree for gfx950: libtrimkv_hip.so (the TRIM-KV cache path and its decoders),
libtrimkv_hybrid.so (what the hybrid decoders share, windowed attention), libtrimkv_mlstm.so and libtrimkv_moe.so (their
recurrent layers and routed experts).

and the extension module _step.so, the host side of decode steps (C++ against Python's and torch's headers).

Usage: ``python -m trimkv_amd.build [--changed] [hip|hybrid|mlstm|moe|step ...]`` (hipcc cross-compiles without a GPU; ``--changed``
recompiles only the sources whose object file is older than its inputs; no name: all of them).
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
LIB_PATH = os.path.join(HERE, "libtrimkv_hip.so")
STEP_PATH = os.path.join(HERE, "_step.so")
SOURCES = ["api.hip", "append.hip", "evict.hip", "attn_decode.hip", "attn_decode_append.hip", "attn_decode_pieces.hip", "attn_decode_append_pieces.hip", "attn_decode_append_gated.hip", "attn_decode_append_pieces_gated.hip", "pieces_plan.hip", "attn_prefill.hip", "gate.hip", "stream_probe.hip", "decoder_ops.hip", "linear_rows.hip", "linear_tiles.hip"]
HYBRID_SOURCES = ["hybrid_ops.hip", "window_attn.hip", "window_decode.hip", "linear_rows.hip", "linear_tiles.hip", "linear_f32_tiles.hip"]
LIBRARIES = {"hip": (LIB_PATH, SOURCES), "hybrid": (os.path.join(HERE, "libtrimkv_hybrid.so"), HYBRID_SOURCES),
             "mlstm": (os.path.join(HERE, "libtrimkv_mlstm.so"), ["mlstm.hip"]), "moe": (os.path.join(HERE, "libtrimkv_moe.so"), ["moe.hip"])}

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I" + INCLUDE, "-I" + CSRC,
    # packed fp32 VALU ops are kept out of every kernel in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-value",
]
# maxima of scores: without this every operand of fmaxf is first run through v_max_f32 to quiet a NaN that cannot be there
# (the decode kernel is scheduled worse with it: 246 against 185 us at 64 x 8 heads of 4096 rows)
EXTRA_FLAGS = {"window_attn.hip": ["-fno-honor-nans"]}


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def _stale(src: str, obj: str) -> bool:
    """An object is stale when its source, any header beside it or the public header is newer."""
    if not os.path.exists(obj):
        return True
    deps = [os.path.join(CSRC, src)] + [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    deps += [os.path.join(INCLUDE, f) for f in os.listdir(INCLUDE)]
    return any(os.path.getmtime(d) > os.path.getmtime(obj) for d in deps)


def _build_step(verbose: bool, only_changed: bool) -> None:
    src = os.path.join(CSRC, "step.cpp")
    if only_changed and not _stale("step.cpp", STEP_PATH):
        return
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    part = "%s.%d" % (STEP_PATH, os.getpid())
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, "-I" + INCLUDE, "-I" + inc,
          "-I" + os.path.join(inc, "torch", "csrc", "api", "include"), "-I" + sysconfig.get_paths()["include"], "-o", part, src,
          "-L" + lib, "-ltorch_python", "-ltorch_cpu", "-lc10", "-Wl,-rpath," + lib])
    os.replace(part, STEP_PATH)
    if verbose:
        print("built", STEP_PATH)


def build(verbose: bool = True, only_changed: bool = False, libraries=(*LIBRARIES, "step")) -> str:
    """Compile every source of the named libraries (or, with ``only_changed``, the ones whose object is older than its
    inputs) and link them."""
    if "step" in libraries:
        _build_step(verbose, only_changed)
        libraries = tuple(n for n in libraries if n != "step")
        if not libraries:
            return STEP_PATH
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    obj_of = lambda s: os.path.join(objdir, s.replace(".hip", ".o"))
    srcs = [s for name in libraries for s in LIBRARIES[name][1]]
    if only_changed:
        srcs = [s for s in srcs if _stale(s, obj_of(s))]

    def compile_one(src):
        return _run([hipcc] + HIPCC_FLAGS + EXTRA_FLAGS.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj_of(src)])

    srcs = list(dict.fromkeys(srcs))       # linear_rows.hip and linear_tiles.hip belong to two libraries
    if srcs:
        with ThreadPoolExecutor(max_workers=min(os.cpu_count() or 4, 8, len(srcs))) as ex:
            for src, out in zip(srcs, ex.map(compile_one, srcs)):
                if verbose and out.strip():
                    print("[%s]\n%s" % (src, out))
    for name in libraries:
        path, sources = LIBRARIES[name]
        part = "%s.%d" % (path, os.getpid())       # linked beside and renamed: nobody loads half a library
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", part] + [obj_of(s) for s in sources])
        os.replace(part, path)
        if verbose:
            print("built", path)
    return LIBRARIES[libraries[-1]][0]


def ensure(libraries) -> None:
    """Build those of the named libraries that are not there (``bin/trace_run`` in a fresh checkout: what its model needs)."""
    missing = tuple(n for n in libraries if not os.path.exists(STEP_PATH if n == "step" else LIBRARIES[n][0]))
    if missing:
        build(verbose=False, only_changed=True, libraries=missing)


if __name__ == "__main__":
    names = [a for a in sys.argv[1:] if not a.startswith("--")]
    build(only_changed="--changed" in sys.argv[1:], libraries=tuple(names) or (*LIBRARIES, "step"))
    sys.exit(0)
