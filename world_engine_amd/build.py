"""Build ``libwe_attn.so`` (HIP, gfx950) and its Python binding in-tree: ``python -m world_engine_amd.build``.

Every source is compiled to its own object, in parallel (the main attention kernel once per
element type / head dim family), and the objects are linked into the shared library.  The binding is host code: g++ against torch's headers."""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "_obj")
# (source, extra defines, object name)
_RING = [("attn_ring.hip", [f"-DWE_RING_PART={i}"], f"attn_ring_{name}.o")
         for i, name in enumerate(("bf16_128", "bf16_64", "f16_128", "f16_64", "short_bf16", "short_f16", "shared_bf16", "shared_f16"))]
_SHARED = [("rope_kv_store.hip", [], "rope_kv_store.o"),
           ("qkv_proj_store.hip", [], "qkv_proj_store.o"),
           ("linear_skinny.hip", [], "linear_skinny.o"),
           ("attn_ring_f32.hip", [], "attn_ring_f32.o"),
           ("attn_combine.hip", [], "attn_combine.o")]
# the product: libwe_attn.so
UNITS = _SHARED + _RING + [("device_state.hip", [], "device_state.o"), ("capi.hip", [], "capi.o")]
# the measurement library: the same kernels plus their clocked instantiations and the tile-stream
# probe (its own copies of the objects that hold state or differ; the rest are the product's)
PROBE_UNITS = _SHARED + [(src, defs + ["-DWE_WITH_PROBES"], "probe_" + obj) for src, defs, obj in _RING] + [
    ("device_state.hip", [], "probe_device_state.o"), ("capi.hip", [], "probe_capi_base.o"),
    ("probe_capi.hip", [], "probe_capi.o"), ("stream_probe.hip", [], "stream_probe.o")]
SOURCES = sorted({u[0] for u in UNITS + PROBE_UNITS} | {"bindings.cpp"})
OUT = os.path.join(HERE, "libwe_attn.so")
PROBE_OUT = os.path.join(HERE, "libwe_probe.so")
NATIVE_OUT = os.path.join(HERE, "_native.so")   # Python binding of libwe_attn.so (host code only)

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # keep fp32 arithmetic scalar: packed fp32 instructions are avoided on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = ("packed-fp32-ops", "Reserved registers on the clobber list", "warnings generated", "warning generated")
    lines = res.stderr.splitlines()
    err = "\n".join(l for l in lines if not any(n in l for n in noise))
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}): {' '.join(cmd)}\n{err}")
    return err


def _binding_command():
    """g++ line of the Python binding: torch's headers for the tensors, the library next to it."""
    import sysconfig
    from torch.utils import cpp_extension as ext
    import torch
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    inc = [*ext.include_paths(), sysconfig.get_paths()["include"], os.path.join(rocm, "include")]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-isystem{p}" for p in inc],
            os.path.join(CSRC, "bindings.cpp"), "-o", NATIVE_OUT, f"-L{HERE}", "-l:libwe_attn.so", *[f"-L{p}" for p in ext.library_paths()],
            "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", f"-L{os.path.join(rocm, 'lib')}", "-lamdhip64",
            "-Wl,-rpath,$ORIGIN", *[f"-Wl,-rpath,{p}" for p in ext.library_paths()]]


def build(verbose: bool = False, jobs: int = 8) -> str:
    """Compile every unit once, link ``libwe_attn.so`` and ``libwe_probe.so`` and build the Python binding
    ``_native.so`` on top; returns the product's path."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(OBJ_DIR, exist_ok=True)
    units = list({u[2]: u for u in UNITS + PROBE_UNITS}.values())   # one compile per object
    cmds = [[hipcc, *HIPCC_FLAGS, *defs, "-c", os.path.join(CSRC, src), "-o", os.path.join(OBJ_DIR, obj)]
            for src, defs, obj in units]
    with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(cmds)))) as pool:
        list(pool.map(lambda c: _run(c, verbose), cmds))
    for out, group in ((OUT, UNITS), (PROBE_OUT, PROBE_UNITS)):
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *[os.path.join(OBJ_DIR, u[2]) for u in group], "-o", out],
             verbose)
    _run(_binding_command(), verbose)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
