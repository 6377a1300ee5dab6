"""The kernels of ``RecomModel``'s MLP against the same layers in 64 bits, and the module they stand
in for wherever they step aside."""

import pytest
import torch
import torch.nn as nn

from recflex_amd import mlp as kernels

pytestmark = pytest.mark.gpu

# fp32 sums in one order or another of up to some hundred partial sums: errors of a few eps per layer in the 2-norm
REL = 1e-6
GRAD_REL = 1e-5


def build(units, device="cuda", seed=0):
    torch.manual_seed(seed)
    sizes = list(units) + [1]
    mods = []
    for i, (a, b) in enumerate(zip(sizes, sizes[1:])):
        mods += [nn.Linear(a, b), nn.Sigmoid() if i + 2 == len(sizes) else nn.ReLU()]
    return nn.Sequential(*mods).to(device)


def rel(got, want):
    return float((got.double().cpu() - want.double().cpu()).norm() / want.double().cpu().norm())


def hidden_of(mlp, x):
    out = []
    for m in mlp[:-2]:
        x = m(x)
        if isinstance(m, nn.ReLU):
            out.append(x.detach())
    return out


# edges of the tiles (32 and 64 rows, 64 units), of a chunk of K (128), of the tail (16 rows, 128 units,
# 1 024 inputs), odd unit counts where they are allowed, many layers, many splits of K
@pytest.mark.parametrize("units, batch", [
    ((4, 4, 1), 1), ((20, 36, 100, 8), 17), ((128, 64, 128), 16), ((132, 68, 127), 33),
    ((64, 1024, 3), 31), ((512, 1020, 128), 65), ((4408, 1024, 256, 128), 37),
    ((4408, 1024, 256, 128), 512), ((12, 8, 8, 8, 8, 8, 8, 8, 8), 5), ((23980, 64, 128), 3),
    ((1000, 200, 64, 16), 449),
])
def test_mlp_forward_and_gradients(units, batch):
    print("[case] mlp", units, batch, flush=True)
    mlp = build(units)
    exact = build(units).double()
    exact.load_state_dict({k: v.double() for k, v in mlp.state_dict().items()})
    x = torch.randn(batch, units[0], device="cuda", requires_grad=True)
    xd = x.detach().double().requires_grad_()
    want = exact(xd)
    with torch.no_grad():
        got = kernels.forward(mlp, x.detach())
    assert got is not None and got.shape == (batch, 1) and not got.requires_grad
    assert rel(got, want.detach()) < REL
    out = kernels.forward(mlp, x)
    assert torch.equal(out.detach(), got)
    weight = torch.linspace(0.5, 1.5, batch, device="cuda")[:, None]
    (out * weight).sum().backward()
    # the gradients, in 64 bits from the kernels' own activations (against another path's, a unit within
    # rounding of zero would be on for one and off for the other): stock fp32 products of up to 1 024
    # terms, a layer's error handed on to the next, some 1e-7 each
    ws, bs = [m.weight.detach() for m in mlp[::2]], [m.bias.detach() for m in mlp[::2]]
    out, hidden = kernels._run(x.detach(), ws, bs, True)
    acts = [x.detach().double()] + [h.double() for h in hidden]
    for want_h, got_h in zip(hidden_of(exact, xd.detach()), hidden):
        assert rel(got_h, want_h) < REL
    g = weight.double() * out.double() * (1 - out.double())
    for l in range(len(ws) - 1, -1, -1):
        assert rel(mlp[2 * l].weight.grad, g.t() @ acts[l]) < GRAD_REL
        assert rel(mlp[2 * l].bias.grad, g.sum(0)) < GRAD_REL
        g = g @ ws[l].double()
        if l:
            g = g * (acts[l] > 0)
    assert rel(x.grad, g) < GRAD_REL


def test_mlp_repeats_bits_and_passes_nan_on():
    mlp = build((256, 96, 32))
    x = torch.randn(70, 256, device="cuda")
    with torch.no_grad():
        first = kernels.forward(mlp, x)
        assert all(torch.equal(kernels.forward(mlp, x), first) for _ in range(3))
        x[5, 7], x[6, 9] = float("nan"), float("inf")
        got, want = kernels.forward(mlp, x), mlp(x)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and bool(torch.isnan(got[5]))
    assert torch.equal(got[7:], first[7:])


def test_mlp_second_derivatives():
    """Through the hidden layers' outputs too: the gradient's gradient equals the modules'."""
    units = (16, 12, 8, 4)
    mlp, stock = build(units), build(units)
    x = torch.randn(9, 16, device="cuda")
    got = []
    for net, run in ((mlp, lambda v: kernels.forward(mlp, v)), (stock, stock)):
        v = x.clone().requires_grad_()
        (g,) = torch.autograd.grad(run(v).sum(), v, create_graph=True)
        got.append(torch.autograd.grad((g * g).sum(), [v] + [p for p in net.parameters() if p.dim() == 2]))
    for a, b in zip(*got):
        assert torch.allclose(a, b, rtol=1e-3, atol=1e-7)


def test_mlp_graph_replays():
    mlp = build((200, 64, 32))
    x = torch.randn(50, 200, device="cuda")
    side = torch.cuda.Stream()
    with torch.no_grad():
        kernels.forward(mlp, x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = kernels.forward(mlp, x)
        for seed in range(3):
            torch.manual_seed(seed)
            x.copy_(torch.randn(50, 200, device="cuda"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, kernels.forward(mlp, x))


def test_mlp_steps_aside():
    """Whatever wants to see the layers gets them."""
    mlp = build((64, 32, 16))
    x = torch.randn(8, 64, device="cuda")
    assert kernels.forward(mlp, x) is not None
    handle = mlp[2].register_forward_hook(lambda *a: None)
    assert kernels.forward(mlp, x) is None
    handle.remove()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert kernels.forward(mlp, x) is None
    seen = []
    torch.func.vmap(lambda row: seen.append(kernels.forward(mlp, row[None])) or row)(x)
    assert seen == [None]
    with torch.autograd.forward_ad.dual_level():
        assert kernels.forward(mlp, x) is None
    for other in (build((64, 32, 16)).double(), build((62, 32, 16)), build((64, 16)), build((64, 32, 132)),
                  build((64, 1028, 16)), build((64, 32, 16), device="cpu")):
        v = torch.randn(8, other[0].in_features, device=other[0].weight.device, dtype=other[0].weight.dtype)
        assert kernels.forward(other, v) is None
    assert kernels.forward(mlp, x.t().contiguous().t()) is None
    assert kernels.forward(mlp, torch.randn(kernels.MAX_BATCH + 1, 64, device="cuda")) is None
    assert kernels.forward(mlp, x[:0]) is None
    mlp[0].bias = None
    assert kernels.forward(mlp, x) is None


def test_mlp_leaves_large_products_to_the_library():
    """Wide layers on many rows, where the library's products are the faster ones."""
    mlp = build((4096, 4096, 64, 16))
    x = torch.randn(512, 4096, device="cuda")
    with torch.no_grad():
        assert kernels.forward(mlp, x) is None
        got = kernels.forward(mlp, x[:kernels.ANY_WIDTH_BATCH])
        assert got is not None and rel(got, mlp.double()(x[:kernels.ANY_WIDTH_BATCH].double())) < REL


# tiny and huge inputs; long K and its remainders, tiles of 64 rows without splits
@pytest.mark.parametrize("units, batch, scale", [
    ((260, 96, 32), 70, 1e-36), ((260, 96, 32), 70, 1e-30), ((260, 96, 32), 70, 1e30), ((8196, 64, 16), 40, 1.),
    ((8224, 100, 16), 65, 1.), ((1000, 1024, 128), 1025, 1.), ((4408, 1024, 128), 512, 1e-30)])
def test_mlp_products_of_parts(units, batch, scale):
    print("[case] mlp", units, batch, scale, flush=True)
    mlp = build(units)
    for m in mlp[::2]:
        m.bias.data.zero_()
    x = torch.randn(batch, units[0], device="cuda") * scale
    ws, bs = [m.weight.detach() for m in mlp[::2]], [m.bias.detach() for m in mlp[::2]]
    hidden = kernels._run(x, ws, bs, True)[1][0]
    assert rel(hidden / scale, torch.relu(x.double() @ ws[0].double().t()) / scale) < REL


def first_hidden(x, w, b=None):
    """The first hidden layer of an MLP whose first weights are ``w``, as the kernels form it."""
    units = (w.shape[1], w.shape[0], 16)
    mlp = build(units)
    ws, bs = [m.weight.detach() for m in mlp[::2]], [m.bias.detach() for m in mlp[::2]]
    ws[0], bs[0] = w, torch.zeros(w.shape[0], device="cuda") if b is None else b
    return kernels._run(x, ws, bs, True)[1][0]


# with and without splits of K, tiles of 32 and of 64 rows
SHAPES = [(70, 260, 96), (33, 4408, 64), (512, 4408, 1024), (1025, 1000, 1024)]


@pytest.mark.parametrize("batch, inputs, units", SHAPES)
def test_mlp_single_products_are_fp32_products(batch, inputs, units):
    """One active input per row: every sum is one product.  Rounded to fp32 it is off by up to 2^-24 of itself; what is
    cut off ahead of that (parts of it, seven times by up to 2^-30, once by 2^-34) is less than an eighth of this."""
    print("[case] mlp single products", batch, inputs, units, flush=True)
    torch.manual_seed(1)
    at = torch.randint(0, inputs, (batch,), device="cuda")
    value, w = torch.randn(batch, device="cuda"), torch.randn(units, inputs, device="cuda")
    x = torch.zeros(batch, inputs, device="cuda").scatter_(1, at[:, None], value[:, None])
    want = torch.relu(value.double()[:, None] * w.double().t()[at])
    assert bool(((first_hidden(x, w) - want).abs() <= 2 ** -24 * (1 + 1 / 8) * want).all())


@pytest.mark.parametrize("inputs_scale, weights_scale", [(1e-34, 1e12), (1e-36, 1e20), (1e-37, 1e30), (1e20, 1e-36)])
def test_mlp_tiny_numbers_times_large_ones(inputs_scale, weights_scale):
    """Numbers whose parts would be subnormal, in products that are not."""
    print("[case] mlp", inputs_scale, weights_scale, flush=True)
    torch.manual_seed(2)
    x, w = torch.randn(70, 260, device="cuda") * inputs_scale, torch.randn(96, 260, device="cuda") * weights_scale
    scale = inputs_scale * weights_scale
    assert rel(first_hidden(x, w) / scale, torch.relu(x.double() @ w.double().t()) / scale) < REL


@pytest.mark.parametrize("batch, inputs, units", SHAPES)
def test_mlp_infinities_stay_infinities(batch, inputs, units):
    """Rows with an infinity of either sign, a NaN, numbers between the largest bf16 and the largest fp32."""
    print("[case] mlp infinities", batch, inputs, units, flush=True)
    torch.manual_seed(3)
    x, w = torch.randn(batch, inputs, device="cuda"), torch.randn(units, inputs, device="cuda") * 1e-3
    x[3, 5], x[7, inputs - 1], x[11, 0], x[13, 2] = float("inf"), -float("inf"), float("nan"), 3.4e38
    x[20, 1], x[20, 2] = float("inf"), -float("inf")
    got = first_hidden(x, w)
    want = torch.relu(x.double() @ w.double().t())
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
    for row in (3, 7):                  # infinite or, behind the ReLU, zero
        assert bool((torch.isposinf(got[row]) | (got[row] == 0)).all()) and bool(torch.isposinf(got[row]).any())
    finite = torch.isfinite(want)
    for row in (13, 0):
        assert bool(finite[row].all()) and rel(got[row], want[row]) < REL
    rest = finite.all(1)
    rest[13] = False
    assert rel(got[rest], want[rest]) < REL
