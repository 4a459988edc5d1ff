"""Kernel-package layout of the ``kernels`` library's local loader, for ROCm.

The reference publishes TiledAttention as a Hugging Face kernel: ``build.toml`` drives a
Nix kernel-builder that compiles the CUDA backend and lays the package out under
``build/<variant>/tiledattention/``, next to a builder-generated ``_ops.py`` that the sync
script keeps (``scripts/sync_torch_ext_from_src.py:38-40``); ``example.py:15`` then loads it
with ``kernels.get_local_kernel(Path("build"), "tiledattention")``.

Here the native side is a C-ABI library plus gfx950 code objects (``tiledattention_amd/lib``),
not a torch extension, so the Nix builder has nothing to compile.  This module writes the
same layout from the already built files instead:

* ``<out>/<variant>/tiledattention/``: every ``*.py`` of the ``tiledattention`` package
  (copied as the reference's sync script copies ``src/tiledattention``), a generated
  ``_ops.py`` (the operator namespace handle and ``add_op_namespace_prefix``, the two names
  kernel-builder generates) and ``lib/`` with ``libtiledattn.so``, the C++ torch operator
  ``libtiledattn_torch.so`` and the ``.hsaco`` code
  objects, which ``tiledattention._lib.lib_dir`` finds next to the package;
* ``<variant>`` = ``torch<major><minor>-cxx11-rocm<major><minor>-<arch>-linux``, the build
  variant name for the running torch.

``load_local_kernel`` resolves and imports such a package the way ``get_local_kernel`` does
(``<repo>/<variant>/<name>`` or ``<repo>/build/<variant>/<name>``), for environments without
the ``kernels`` library.

Run: ``python -m tiledattention_amd.kernel_build [--out build]``.
"""

from __future__ import annotations

import argparse
import hashlib
import importlib.util
import platform
import shutil
import sys
from pathlib import Path
from types import ModuleType

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
PY_SRC = ROOT / "tiledattention"
LIB_SRC = HERE / "lib"
PACKAGE = "tiledattention"

_OPS_PY = '''"""Operator namespace of this kernel package (generated by tiledattention_amd.kernel_build).

``ops`` is ``torch.ops.tiledattention``; importing ``tiledattention.torch_op`` registers its
``sdpa_fwd`` operator there.
"""

import torch

ops = torch.ops.tiledattention


def add_op_namespace_prefix(op_name: str) -> str:
    """Prefix op_name with the namespace of this package's operators."""
    return f"tiledattention::{op_name}"
'''


def build_variant() -> str:
    """Build variant of the running torch: torch<maj><min>-cxx11-rocm<maj><min>-<arch>-linux."""
    import torch

    tv = torch.__version__.split("+")[0].split(".")
    hip = getattr(torch.version, "hip", None)
    if not hip:
        raise RuntimeError("this torch is not a ROCm build (torch.version.hip is unset)")
    hv = hip.split(".")
    abi = "cxx11" if getattr(torch._C, "_GLIBCXX_USE_CXX11_ABI", True) else "cxx98"
    return f"torch{tv[0]}{tv[1]}-{abi}-rocm{hv[0]}{hv[1]}-{platform.machine()}-linux"


def write_kernel_package(out: Path, variant: str | None = None) -> Path:
    """Lay the kernel package out under ``out/<variant>/tiledattention`` (replacing a previous
    one) and return that directory."""
    lib_files = (sorted(LIB_SRC.glob("libtiledattn.so")) + sorted(LIB_SRC.glob("libtiledattn_torch.so"))
                 + sorted(LIB_SRC.glob("_tiledattn_call.*.so")) + sorted(LIB_SRC.glob("*.hsaco")))
    if not any(f.name == "libtiledattn.so" for f in lib_files):
        raise FileNotFoundError(
            f"{LIB_SRC}/libtiledattn.so is missing: build it first (python -m tiledattention_amd.csrc.build)"
        )
    dst = Path(out) / (variant or build_variant()) / PACKAGE
    if dst.exists():
        shutil.rmtree(dst)
    for src in sorted(PY_SRC.rglob("*.py")):
        if "__pycache__" in src.parts:
            continue
        target = dst / src.relative_to(PY_SRC)
        target.parent.mkdir(parents=True, exist_ok=True)
        shutil.copy2(src, target)
    (dst / "_ops.py").write_text(_OPS_PY)
    (dst / "lib").mkdir()
    for f in lib_files:
        shutil.copy2(f, dst / "lib" / f.name)
    return dst


def load_local_kernel(repo_path: Path, package_name: str = PACKAGE) -> ModuleType:
    """Import the kernel package under ``repo_path/<variant>/<name>`` or
    ``repo_path/build/<variant>/<name>``, as ``kernels.get_local_kernel`` resolves it.  The
    module gets a name of its own (``<name>_<hash of the path>``), so it does not replace an
    imported ``tiledattention``."""
    variant = build_variant()
    for base in (Path(repo_path), Path(repo_path) / "build"):
        pkg = base / variant / package_name
        init = pkg / "__init__.py"
        if init.exists():
            name = f"{package_name}_{hashlib.sha1(str(pkg.resolve()).encode()).hexdigest()[:10]}"
            if name in sys.modules:
                return sys.modules[name]
            spec = importlib.util.spec_from_file_location(name, init, submodule_search_locations=[str(pkg)])
            module = importlib.util.module_from_spec(spec)
            sys.modules[name] = module
            try:
                spec.loader.exec_module(module)
            except BaseException:
                del sys.modules[name]
                raise
            return module
    raise FileNotFoundError(f"no {variant}/{package_name} under {repo_path} or {Path(repo_path) / 'build'}")


def main(argv: list[str] | None = None) -> int:
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--out", default=str(ROOT / "build"), help="root of the build variants")
    args = ap.parse_args(argv)
    print(write_kernel_package(Path(args.out)))
    return 0


if __name__ == "__main__":
    raise SystemExit(main())
