"""Builds libps_adam.so (the C-ABI HIP library) for gfx950 with hipcc and _binding.so (host code) with g++, in-tree."""
import contextlib
import os
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
LIB_PATH = os.path.join(PKG_DIR, "libps_adam.so")
SOURCES = [os.path.join(PKG_DIR, "csrc", "ps_adam.hip")]
BINDING_SOURCE = os.path.join(PKG_DIR, "csrc", "ps_binding.cpp")
BINDING_PATH = os.path.join(PKG_DIR, "_binding.so")
INCLUDE = os.path.join(ROOT, "include")

# -ffp-contract=off: fused multiply-adds are written out explicitly; the compiler must not add or remove any.
# -fhip-fp32-correctly-rounded-divide-sqrt: IEEE-rounded '/' and sqrtf (hipcc's default, stated on purpose).
# Denormals are kept: -fgpu-flush-denormals-to-zero is not given.
# packed-fp32 ops are switched off: the compiler otherwise pairs independent float ops into v_pk_* forms.
# Kernels whose first arguments are plain numbers or pointers get up to 14 words of them preloaded into scalar registers.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    "--offload-arch=gfx950",
    "-fPIC",
    "-shared",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-fast-math",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-mllvm",
    "-amdgpu-kernarg-preload-count=16",
    "-Wall",
    "-Wextra",
    "-Wno-unused-function",
]


def is_built():
    """Whether everything that build() makes is there."""
    return all(os.path.exists(path) for path in (LIB_PATH, BINDING_PATH))


def hipcc_path():
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP library cannot be built")


@contextlib.contextmanager
def _replacing(*targets):
    """Paths beside the targets to build into; they take the targets' places together, once all of them are built.  (A process
    that has an old file mapped keeps its own copy.)"""
    made = [f"{target}.{os.getpid()}.tmp" for target in targets]
    try:
        yield made
        for path, target in zip(made, targets):
            os.replace(path, target)
    finally:
        for path in made:
            if os.path.exists(path):
                os.remove(path)


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)


def _compile_hip(sources, out, verbose, extra_flags):
    _run([hipcc_path(), *HIPCC_FLAGS, *extra_flags, "-I", INCLUDE, *sources, "-o", out], verbose)


def compile_shared(sources, target, verbose=False, extra_flags=()):
    """hipcc the given sources into one shared library with this package's flags."""
    with _replacing(target) as (out,):
        _compile_hip(sources, out, verbose, extra_flags)
    return target


def built_for():
    """What a binding that is compiled now can be used with."""
    import torch

    return f"Python {sys.version_info[0]}.{sys.version_info[1]}, torch {torch.__version__}"


def _compile_binding(out, verbose):
    import sysconfig

    from torch.utils import cpp_extension

    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f'-DPS_BUILT_FOR="{built_for()}"']
    for path in [INCLUDE, sysconfig.get_paths()["include"], "/opt/rocm/include"]:
        cmd += ["-I", path]
    for path in cpp_extension.include_paths():
        cmd += ["-isystem", path]
    cmd += [BINDING_SOURCE, "-o", out]
    for path in cpp_extension.library_paths():
        cmd += ["-L", path]
    _run(cmd + ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"], verbose)


def build_binding(verbose=False):
    """Compile the Python side of the operator call, host code only, into patrickstar_amd/_binding.so (returned)."""
    with _replacing(BINDING_PATH) as (out,):
        _compile_binding(out, verbose)
    return BINDING_PATH


def build(verbose=False, extra_flags=()):
    """Compile the package's HIP sources into patrickstar_amd/libps_adam.so (returned), and the binding beside it.  Neither
    replaces what is there before both are compiled: the binding calls into the library it was built with."""
    with _replacing(BINDING_PATH, LIB_PATH) as (binding, library):
        _compile_binding(binding, verbose)
        _compile_hip(SOURCES, library, verbose, extra_flags)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
