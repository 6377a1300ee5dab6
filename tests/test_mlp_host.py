"""What ``RecomModel`` does around its MLP kernels, as far as that needs no GPU."""

import pytest
import torch
import torch.nn as nn

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
