"""What ``RecomModel`` does around its MLP kernels, as far as that needs no GPU."""

import os
import re
import shutil
import subprocess
import sys

import pytest
import torch
import torch.nn as nn

from helpers import ROOT
from recflex_amd import mlp as kernels
from recflex_amd import rec_modules
from recflex_amd.code_emitter.build_basic import BasicBuilder


class _Embed(nn.Module):
    """In ``FeatEmbed``'s place: hands its first argument on."""
    output_units = 12

    def __init__(self, device, **kwargs):
        super().__init__()
        self.device = device

    def forward(self, x, *rest):
        return x


@pytest.fixture
def no_library(monkeypatch, tmp_path):
    """A package without the built library, on a machine without the compiler."""
    def init(self):
        real_init(self)
        self.csrc_dir, self.hipcc = str(tmp_path / "csrc"), str(tmp_path / "no_hipcc")

    real_init = BasicBuilder.__init__
    monkeypatch.setattr(BasicBuilder, "__init__", init)
    monkeypatch.setattr(kernels, "_lib", None)
    monkeypatch.setattr(kernels, "_missing", False, raising=False)
    monkeypatch.setattr(rec_modules, "FeatEmbed", _Embed)


def test_model_without_the_mlp_library_runs_its_modules(no_library):
    with pytest.warns(RuntimeWarning, match="MLP kernels"):
        model = rec_modules.RecomModel([8, 4], torch.device("cpu"))
    x = torch.randn(3, 12)
    assert torch.equal(model(x, *[None] * 8), model.mlp(x))
    # asked for without a model: once, not on every call
    assert kernels._missing and kernels._lib is None


def test_mlp_library_follows_its_source(monkeypatch, tmp_path):
    """Built when it is missing, kept as long as source and flags are what it was built from."""
    builder = BasicBuilder()
    (tmp_path / "mlp").mkdir()
    for name in ("recflex_mlp.hip", "recflex_mlp.h"):
        shutil.copy(f"{builder.csrc_dir}/mlp/{name}", tmp_path / "mlp" / name)
    builder.csrc_dir = str(tmp_path)
    builds = []

    def compile_(cmd, check):
        builds.append(cmd)
        with open(cmd[-1], "w") as f:
            f.write("library %d" % len(builds))

    monkeypatch.setattr("subprocess.run", compile_)
    for source, flags, want in (("", [], 1), ("", [], 1), ("\n// edited\n", [], 2), ("", [], 2), ("", ["-DX"], 3)):
        with open(tmp_path / "mlp" / "recflex_mlp.hip", "a") as f:
            f.write(source)
        builder.hip_flags = builder.hip_flags + [x for x in flags if x not in builder.hip_flags]
        with open(builder.build_mlp()) as f:
            assert f.read() == "library %d" % want
    assert builder.build_mlp(force=True) and len(builds) == 4
    (tmp_path / "mlp" / "recflex_mlp.h").unlink()       # a package without its sources keeps its library
    assert builder.build_mlp() and len(builds) == 4


@pytest.mark.parametrize("name", ["torch._C._cuda_getCurrentRawStream", "torch._C._functorch.peek_interpreter_stack",
                                  "torch._C._len_torch_dispatch_stack", "torch._C._len_torch_function_stack",
                                  "torch.autograd.forward_ad._current_level",
                                  "torch.nn.modules.module._has_any_global_hook"])
def test_a_torch_without_a_private_name(name):
    """The public call, or the modules, take its place."""
    script = f'''
import torch, types
import torch.utils._python_dispatch, torch.overrides
del {name}
from recflex_amd import mlp, rec_modules
torch.cuda.current_stream = lambda device: types.SimpleNamespace(cuda_stream=77)
if "RawStream" in "{name}":
    assert mlp._KNOWS_OBSERVERS and rec_modules._stream_of(torch.device("cuda", 0)) == 77
else:
    assert rec_modules._RAW_STREAM is not None
    assert mlp.forward(None, None) is None
'''
    subprocess.run([sys.executable, "-c", script], check=True, cwd=ROOT, timeout=120)


@pytest.mark.parametrize("batch, units, pays", [
    (512, (4408, 1024, 256, 128), True), (512, (23980, 1024, 256, 128), True), (513, (64, 32, 16), False),
    (256, (4408, 8192, 512, 128), True), (257, (4408, 8192, 512, 128), False), (512, (4408, 8192, 128), False),
    (352, (4408, 2048, 512, 128), True), (416, (4408, 2048, 512, 128), False), (512, (512, 2048, 128), True),
    # a wide layer behind a narrow one
    (512, (4408, 512, 4096, 1024, 128), False)])
def test_where_the_mlp_kernels_pay(batch, units, pays):
    assert kernels._pays(batch, units) is pays


def _registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
    if not m:
        return range(0)
    return range(int(m[1]), int(m[2]) + 1) if m[1] else range(int(m[3]), int(m[3]) + 1)


def test_mlp_kernels_wait_before_matrix_instructions(tmp_path):
    """Two wait states lie between a vector instruction and a matrix instruction that reads its result; the
    compiler sees to it except behind an instruction written in inline assembly."""
    builder = BasicBuilder()
    if not os.path.exists(builder.hipcc):
        pytest.skip("no hipcc")
    listing = tmp_path / "mlp.s"
    flags = [f for f in builder.hip_flags if f not in ("-shared", "-fPIC")]
    subprocess.run([builder.hipcc, *flags, "-O3", "--offload-device-only", "-S",
                    f"{builder.csrc_dir}/mlp/recflex_mlp.hip", "-o", str(listing)], check=True, stderr=subprocess.DEVNULL)
    products, since = 0, {}             # wait states since a vector instruction wrote the register
    for line in listing.read_text().splitlines():
        op, _, rest = line.split(";")[0].strip().partition(" ")
        if op.endswith(":"):
            since = {}
        if not op or op.endswith(":") or op.startswith("."):
            continue
        operands = [o.strip() for o in rest.split(",")]
        if op.startswith("v_mfma"):
            products += 1
            for operand in operands[1:]:
                assert all(since.get(r, 2) >= 2 for r in _registers(operand)), line
        states = int(operands[0], 0) + 1 if op == "s_nop" else 1
        since = {r: n + states for r, n in since.items() if n + states < 2}
        if op.startswith("v_") and not op.startswith("v_mfma"):
            since.update(dict.fromkeys(_registers(operands[0]), 0))
    assert products > 0
