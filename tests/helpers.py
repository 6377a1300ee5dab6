"""Shared pieces of the parity tests: run a prebuilt model through the C ABI on the GPU and
compare with the CPU oracle."""

import ctypes
import os
import subprocess
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

from oracle import oracle  # noqa: E402  (the checker; tests are allowed to use it)

# tolerances of the path: fp32 tables within 1e-5 relative or 1e-6 absolute of the oracle;
# fp16 / int8 tables within 1e-3 relative (or 1e-6 absolute) of dequantise-then-fp32-sum
TOL = {"float": (1e-5, 1e-6), "half": (1e-3, 1e-6), "int8": (1e-3, 1e-6)}


def require_lib(name: str) -> str:
    """Path of a prebuilt model library; GPU tests fail loudly if it was not built in-tree."""
    from recflex_amd import prebuilt
    path = prebuilt.lib_path(name)
    if not os.path.exists(path):
        raise RuntimeError(f"{path} is missing: run `python -c 'import __graft_entry__ as g; g.build()'` "
                           "before the GPU tests (no CPU fallback exists)")
    return path


def oracle_output(wl, host_tables, indices, offsets):
    dims = [f.dim for f in wl.features]
    dts = [f.data_type for f in wl.features]
    return oracle.pooled_sum_c(host_tables, dims, dts, indices, offsets)


def check_against_oracle(wl, got: np.ndarray, want: np.ndarray):
    """Per feature column slab, with that feature's tolerance.  Returns a list of failures."""
    failures = []
    col = 0
    for f, spec in enumerate(wl.features):
        rtol, atol = TOL[spec.data_type]
        ok, max_abs, max_rel = oracle.within_tolerance(got[:, col:col + spec.dim],
                                                       want[:, col:col + spec.dim], rtol, atol)
        if not ok:
            failures.append((f, spec, max_abs, max_rel))
        col += spec.dim
    return failures


PART_COST = 35 * 1024           # rfx::kSplitPartCost


def build_tile_model(lib: str) -> ctypes.CDLL:
    """``tests/cpu/tile_sizes_model.cpp`` built as ``lib``: the binding's tile sizes on the CPU."""
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-shared", "-fPIC", "-ffp-contract=off",
                    f"-I{ROOT}/recflex_amd/csrc/include", os.path.join(ROOT, "tests", "cpu", "tile_sizes_model.cpp"),
                    "-o", lib], check=True)
    return ctypes.CDLL(lib)


def bind_tiles_on_cpu(model, cost, gran, batch, grid, tile_size) -> dict:
    """Part size, tiles per feature and the price of a round-by-round walk over them, as the binding
    chooses them and as its plain rule would (``rule``, ``rule_price``); ``counted``: the tiles the
    search counted, -1 where it was not due."""
    n = len(cost)
    cost, gran = np.asarray(cost, np.float32), np.asarray(gran, np.int32)
    tiles, rule_tiles, out = np.zeros(n, np.int32), np.zeros(n, np.int32), np.zeros(3, np.int64)
    longest, rule_longest = np.zeros(1, np.float32), np.zeros(1, np.float32)
    ptr = [a.ctypes.data_as(ctypes.c_void_p) for a in (cost, gran, tiles, longest, rule_tiles, rule_longest, out)]
    model.model_bind(n, batch, grid, tile_size, *ptr)
    price = [-(-int(t.sum()) // grid) * (float(l[0]) + PART_COST)
             for t, l in ((tiles, longest), (rule_tiles, rule_longest))]
    return dict(unit=int(out[0]), counted=int(out[1]), rule=int(out[2]), tiles=tiles, price=price[0],
                rule_price=price[1])
