"""Build libxkv_hip.so (gfx950 only) from csrc/*.hip with hipcc - no torch headers involved - and the native host layer
_xkv_host.so from csrc/host.cpp with the host compiler."""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libxkv_hip.so")
HOST = os.path.join(HERE, "_xkv_host.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++20",
    # keep the compiler from forming packed-fp32 VALU ops from scalar float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-inline-asm",
]
# Per-file additions.  the recon_scores.hip, recon_heads_*.hip, recon_spec_*.hip and recon_duo_*.hip units: MFMA results must land in ordinary VGPRs (the RoPE / softmax VALU code reads
# them; with accumulation-register results every value costs a v_accvgpr_read), while the stationary B operands are
# pinned to accumulation registers by the source itself.
_VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
EXTRA_FLAGS = {
    "recon_scores.hip": _VGPR_FORM,
    "recon_heads_512.hip": _VGPR_FORM, "recon_heads_384.hip": _VGPR_FORM, "recon_heads_256.hip": _VGPR_FORM,
    "recon_duo_b.hip": _VGPR_FORM, "recon_duo_c.hip": _VGPR_FORM, "recon_spec_512.hip": _VGPR_FORM, "recon_spec_384.hip": _VGPR_FORM, "recon_spec_256.hip": _VGPR_FORM,
}


# The compiler the kernels were validated with.  latent_ring.hip, recon_scores / recon_duo / recon_spec / recon_heads issue loads in asm
# and track their completion by hand; that is correct for the register allocation this compiler produces and is re-checked
# by tests/test_gpu_ring_forms.py and the parity suite.  Another compiler builds, with a loud warning: run those tests on a
# GPU before trusting it.  (At run time the library refuses such a kernel outright if its build spills registers.)
VALIDATED_HIPCC = "roc-7.2.0 26014"


def _check_compiler() -> None:
    try:
        out = subprocess.run([HIPCC, "--version"], capture_output=True, text=True).stdout
    except OSError as e:   # pragma: no cover
        raise RuntimeError(f"cannot run {HIPCC}: {e}")
    if VALIDATED_HIPCC not in out:
        line = next((l for l in out.splitlines() if "clang version" in l), out.strip()[:120])
        sys.stderr.write(
            "\n*** kernel_collections_amd.build: hipcc is not the validated one (%s); found: %s\n"
            "*** the kernels that track their own loads (latent_ring, recon_scores, recon_duo, recon_spec, recon_heads) must be re-checked:\n"
            "***   python -m pytest tests/test_gpu_ring_forms.py tests/test_gpu_parity.py tests/test_gpu_peaked.py -m gpu\n\n"
            % (VALIDATED_HIPCC, line))


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    cmd = [HIPCC, *FLAGS, *EXTRA_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_host() -> None:
    """csrc/host.cpp, the native host layer: a plain CPython extension over the C++ tensor API (the libraries it names are
    those `import torch` has loaded)."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
           "-isystem", os.path.join(root, "include"), "-isystem", sysconfig.get_paths()["include"], "-isystem", "/opt/rocm/include",
           os.path.join(CSRC, "host.cpp"), "-o", HOST, "-L" + os.path.join(root, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10",
           "-lc10_hip", "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on host.cpp:\n{r.stderr}")


def build(verbose: bool = True) -> str:
    """Compile every kernel source and link the shared library, and build the native host layer; always recompiles."""
    _check_compiler()
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, srcs))
        host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    subprocess.check_call(cmd)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources")
    return LIB


if __name__ == "__main__":
    build()
