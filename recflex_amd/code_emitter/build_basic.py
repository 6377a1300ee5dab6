"""Locations and compiler settings shared by every emitted library, and the build of the
model-independent host library ``librecflex_host.so``.

Reference counterpart: ``RecFlex/code_emitter/build_basic.py:17-28`` (``BasicBuilder`` builds
``libsched_basic.so`` once and hands its include directory and path to the generated
CMakeLists).  Here the device side is header-only (``csrc/include/*.hip.h``), so only the CPU
text front end is a prebuilt library.
"""

import hashlib
import os
import shutil
import subprocess
import sys
import sysconfig
import warnings
from typing import List

import recflex_amd

GPU_ARCH = "gfx950"


class BasicBuilder:
    def __init__(self):
        self.package_dir = os.path.dirname(os.path.abspath(recflex_amd.__file__))
        self.csrc_dir = os.path.join(self.package_dir, "csrc")
        self.include = os.path.join(self.csrc_dir, "include")
        # include/recflex_hip.h sits at the repository root, beside the package
        self.abi_include = os.path.join(os.path.dirname(self.package_dir), "include")
        self.host_source = os.path.join(self.csrc_dir, "host", "recflex_host.cpp")
        self.strings_source = os.path.join(self.csrc_dir, "host", "recflex_strings.cpp")
        self.hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
        self.cxx = shutil.which("g++") or "g++"
        # gfx950 only; packed fp32 instructions are disabled on purpose
        self.hip_flags: List[str] = [
            f"--offload-arch={GPU_ARCH}", "-std=c++17", "-shared", "-fPIC",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
        ]
        # e.g. RECFLEX_HIP_EXTRA_FLAGS="-DRFX_PREFETCH_GROUPS=0" for an experiment
        self.hip_flags += os.environ.get("RECFLEX_HIP_EXTRA_FLAGS", "").split()
        self.host_flags: List[str] = ["-std=c++17", "-shared", "-fPIC", "-Wall", "-pthread"]

    def device_headers(self) -> List[str]:
        """The headers every emitted ``process.hip`` is built from."""
        names = sorted(n for n in os.listdir(self.include) if n.endswith(".h"))
        return [os.path.join(self.include, n) for n in names] + \
               [os.path.join(self.abi_include, "recflex_hip.h")]

    def host_lib_path(self, dirname: str = "build") -> str:
        return os.path.join(self.csrc_dir, dirname, "librecflex_host.so")

    def strings_build(self) -> List[str]:
        """What the reader of Python's own strings adds to the compiler's arguments; nothing where this
        interpreter's headers are not installed."""
        include = sysconfig.get_paths()["include"]
        if not os.path.exists(os.path.join(include, "Python.h")) or not os.path.exists(self.strings_source):
            return []
        return [self.strings_source, f"-I{include}"]

    def build(self, dirname: str = "build", force: bool = False) -> str:
        """Build ``librecflex_host.so`` if it is missing or was built from other sources, with other flags or
        for another interpreter's strings (or ``force``); returns its path."""
        lib = self.host_lib_path(dirname)
        strings = self.strings_build()
        sources = [self.host_source, self.strings_source, os.path.join(self.abi_include, "recflex_hip.h")]
        flags = [*self.host_flags, "-O3"]
        interpreter = [sys.implementation.cache_tag or "", *strings[1:]] if strings else []

        def compile_to(tmp):
            cmd = [self.cxx, *flags, f"-I{self.abi_include}", self.host_source, "-o", tmp]
            if strings:
                done = subprocess.run([*cmd, *strings], stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)
                if done.returncode == 0:
                    return
                warnings.warn("the reader of Python's strings does not compile, sample lines are joined first:\n"
                              + done.stderr[-2000:], RuntimeWarning, stacklevel=3)
            subprocess.run(cmd, check=True)

        try:
            return self._build_from(lib, sources, [*flags, *interpreter], force, compile_to)
        except (OSError, subprocess.SubprocessError) as e:      # no compiler, nowhere to write, ...
            if force or not os.path.exists(lib):
                raise
            warnings.warn(f"{lib} was built from other sources and could not be built again: {e}", RuntimeWarning,
                          stacklevel=2)
            return lib

    def _build_from(self, lib: str, sources: List[str], flags: List[str], force: bool, compile_to) -> str:
        """``lib``, made anew by ``compile_to(path)`` unless it is there, from these sources and flags."""
        if not force and os.path.exists(lib) and not all(map(os.path.exists, sources)):
            return lib                              # a package without its sources
        key = hashlib.sha256(" ".join(flags).encode())
        for path in filter(os.path.exists, sources):
            with open(path, "rb") as f:
                key.update(f.read())
        built_from = lib + ".from"                  # what the library beside it was built from
        current = ""
        if os.path.exists(lib) and os.path.exists(built_from):
            with open(built_from) as f:
                current = f.read()
        if force or current != key.hexdigest():
            os.makedirs(os.path.dirname(lib), exist_ok=True)
            tmp = lib + f".tmp{os.getpid()}"
            compile_to(tmp)
            os.replace(tmp, lib)
            with open(tmp, "w") as f:
                f.write(key.hexdigest())
            os.replace(tmp, built_from)
        return lib

    def mlp_lib_path(self, dirname: str = "build") -> str:
        return os.path.join(self.csrc_dir, dirname, "librecflex_mlp.so")

    def build_mlp(self, dirname: str = "build", force: bool = False) -> str:
        """Build ``librecflex_mlp.so`` (the kernels of ``RecomModel``'s MLP, model independent) if it is
        missing or was built from another source or with other flags (or ``force``); returns its path."""
        sources = [os.path.join(self.csrc_dir, "mlp", n) for n in ("recflex_mlp.hip", "recflex_mlp.h")]
        flags = [*self.hip_flags, "-O3"]
        return self._build_from(self.mlp_lib_path(dirname), sources, flags, force,
                                lambda tmp: subprocess.run([self.hipcc, *flags, sources[0], "-o", tmp], check=True))
