"""Build recipe for the HIP kernel library: hipcc for gfx950, in-tree output.

`python -m popcorn_amd.build` compiles every `csrc/*.hip` to an object in
`popcorn_amd/_build/` (in parallel) and links `popcorn_amd/libpopcorn_amd.so`,
and `csrc/host.cpp`, the calls into it that do not pass through Python, to
`popcorn_amd/_native.<ABI tag>.so`, an extension module of the running Python and torch.
Both are always rebuilt: the call is the "does it build" check. Asked
to (`python -m popcorn_amd.build` and `__graft_entry__.build()` ask), it then
writes the `popcorn-amd` distribution metadata beside the package in a source
tree (setup.py's `egg_info`, as an editable install would), so Popcorn's
version gate sees the backend when the tree itself is on `sys.path`. setup.py's
own build step does not ask: an install writes its metadata itself.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE = Path(__file__).resolve().parent
CSRC = PACKAGE / "csrc"
BUILD = PACKAGE / "_build"
LIBRARY = PACKAGE / "libpopcorn_amd.so"
NATIVE = PACKAGE / f"_native{sysconfig.get_config_var('EXT_SUFFIX')}"  # no other Python finds it
INCLUDE = PACKAGE.parent / "include"

ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # The kernels reproduce torch's rounding sequence (separate products and
    # sums); contraction would fuse them. FMAs are written out where wanted.
    "-ffp-contract=off",
    # Packed fp32 VALU ops are kept out of every kernel.
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    f"-I{INCLUDE}",
]


def hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(found).exists():
        raise RuntimeError("hipcc not found; the popcorn_amd kernels need ROCm's hipcc")
    return found


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(source: Path) -> Path:
    obj = BUILD / (source.stem + ".o")
    cmd = [hipcc(), *FLAGS, "-c", str(source), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {source.name}:\n{proc.stderr}")
    return obj


def _compile_host() -> Path:
    """The extension module's object: host code only, against torch's and Python's headers."""
    import torch
    from torch.utils.cpp_extension import include_paths

    obj = BUILD / "host.o"
    cmd = [hipcc(), "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
           f'-DPK_TORCH_VERSION="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *(f"-isystem{p}" for p in (*include_paths("cuda"), sysconfig.get_paths()["include"])),
           "-c", str(CSRC / "host.cpp"), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on host.cpp:\n{proc.stderr}")
    return obj


def _link(output: Path, *args: str) -> None:
    tmp = output.with_suffix(".so.tmp")
    proc = subprocess.run([hipcc(), "-shared", "-fPIC", *args, "-o", str(tmp)], capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of {output.name} failed:\n{proc.stderr}")
    os.replace(tmp, output)


def _link_native(obj: Path) -> None:
    import torch

    # libpopcorn_amd.so is found beside the module; torch's libraries are loaded before it by `import torch`
    _link(NATIVE, str(obj), f"-L{PACKAGE}", f"-l:{LIBRARY.name}", "-Wl,-rpath,$ORIGIN",
          f"-L{Path(torch.__file__).parent / 'lib'}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip")


def build(verbose: bool = False, write_metadata: bool = False, native: bool = True) -> Path:
    """Compile all kernels and the host calls and link both libraries; returns the kernels' path.

    With `write_metadata`, also write the distribution metadata into the source tree (see
    `write_source_metadata`). With `native` False, host calls that cannot be built here (no torch headers,
    say) are left out with a message: every call then goes through Python.
    """
    BUILD.mkdir(exist_ok=True)
    srcs = sources()
    workers = min(len(srcs) + 1, int(os.environ.get("MAX_JOBS", "8")), 16) or 1
    with ThreadPoolExecutor(max_workers=workers) as pool:
        host = pool.submit(_compile_host)
        objects = list(pool.map(_compile, srcs))
    _link(LIBRARY, f"--offload-arch={ARCH}", *map(str, objects))
    for old in PACKAGE.glob("_native*.so"):  # of an earlier build, which the import must not take for this one
        old.unlink()
    try:
        _link_native(host.result())
    except Exception as e:
        if native:
            raise
        print(f"{NATIVE.name} cannot be built and is left out: {e}", file=sys.stderr)
    if verbose:
        print(f"built {LIBRARY} from {len(srcs)} sources{', and ' + NATIVE.name if NATIVE.exists() else ''}",
              file=sys.stderr)
    if write_metadata:
        write_source_metadata()
    return LIBRARY


def write_source_metadata() -> None:
    """Run setup.py's `egg_info` in a source tree (no-op for an installed package, which has its metadata)."""
    setup_py = PACKAGE.parent / "setup.py"
    if not setup_py.exists():
        return
    proc = subprocess.run([sys.executable, str(setup_py), "-q", "egg_info", "--egg-base", str(PACKAGE.parent)],
                          cwd=PACKAGE.parent, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"writing the popcorn-amd metadata failed:\n{proc.stderr}")


if __name__ == "__main__":
    build(verbose=True, write_metadata=True)
