"""The MLP of ``RecomModel`` on the hand-written kernels of ``librecflex_mlp.so``
(``csrc/mlp/recflex_mlp.hip``): three launches for the default three hidden layers instead of the
eight of the same ``nn.Sequential`` run layer by layer.

``forward(mlp, x)`` returns ``None`` where the kernels don't apply, and the caller then runs the
modules: other layers than ``RecomModel`` builds, hooks on any of them, parameters that are not
plain fp32 tensors on the current device, sizes outside the kernels' range or where the modules
are the faster ones, no library and no compiler to build it, and whatever wants to see the single
operations (autocast, tracing, compiling, vmap and the other function transforms, forward-mode
derivatives, dispatch and function modes).
"""

import ctypes
import subprocess
import warnings
from typing import List, Optional, Sequence

import torch
import torch.nn as nn

# What wants to see the single operations, as far as torch has no public name for it.  In a torch
# without one of these the modules run.
try:
    from torch.nn.modules.module import _has_any_global_hook
    _transforms = torch._C._functorch.peek_interpreter_stack
    _dispatch_modes = torch._C._len_torch_dispatch_stack
    _function_modes = torch._C._len_torch_function_stack
    _KNOWS_OBSERVERS = isinstance(torch.autograd.forward_ad._current_level, int)
except (ImportError, AttributeError):
    _KNOWS_OBSERVERS = False

MAX_LAYERS = 8                      # RECFLEX_MLP_MAX_LAYERS
TAIL_MAX_UNITS = 128                # RECFLEX_MLP_TAIL_MAX_UNITS
TAIL_MAX_INPUTS = 1024              # RECFLEX_MLP_TAIL_MAX_INPUTS
# Where the kernels serve, against the modules (in us; both in a graph, where the library's launches cost
# least).  Up to 256 rows: the library's products take 1.1 to 5 times as long as these (except where there is as much
# to multiply as in 8192, 512, 128 units on 23 980 inputs, 256 rows, 103 GFLOP: 994 against 857).  Beyond, up to 512
# rows: 1024, 256, 128 units on 4 408 inputs, 384 / 512 rows 57 / 65 against 76 / 77, on 23 980 inputs 183 / 235 against
# 360 / 252, on 512 inputs 28 / 29 against 45 / 46; wider layers gain less or lose (4 408 inputs: 2048, 512, 128 units,
# 384 rows, 8 GFLOP, 96 to 104 against 97 to 101; 4096, 512, 128, 300 / 512 rows, 12 / 21 GFLOP, 149 / 191 against 144 /
# 185; 8192, 512, 128, 512 rows, 41 GFLOP, 364 against 324): beyond 8 GFLOP they are left to the modules (not without
# exceptions: 1536, 512, 128 on 23 980 inputs, 512 rows, 346 against 687).  Beyond 512 rows the modules serve: 1024,
# 256, 128 on 4 408 inputs, 700 / 1 024 / 2 048 rows 86 / 103 / 189 against 93 / 110 / 176, on 23 980 inputs 328 / 451 /
# 899 against 683 / 379 / 720.
MAX_BATCH = 512
ANY_WIDTH_BATCH = 256
NARROW_UNITS = 1024
WIDE_MAX_FLOPS = 8e9


def _pays(batch: int, units: Sequence[int]) -> bool:
    """``units``: of the input and of the hidden layers."""
    if batch > MAX_BATCH:
        return False
    return batch <= ANY_WIDTH_BATCH or max(units[1:]) <= NARROW_UNITS \
        or 2. * batch * sum(a * b for a, b in zip(units, units[1:])) <= WIDE_MAX_FLOPS


class _Args(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("out", ctypes.c_void_p), ("workspace", ctypes.c_void_p),
                ("stream", ctypes.c_void_p), ("batch", ctypes.c_int32), ("layers", ctypes.c_int32),
                ("units", ctypes.c_int32 * (MAX_LAYERS + 1)),
                ("weights", ctypes.c_void_p * (MAX_LAYERS + 1)),
                ("biases", ctypes.c_void_p * (MAX_LAYERS + 1)),
                ("hidden", ctypes.c_void_p * MAX_LAYERS)]


_lib = None
_missing = False                    # it could not be loaded, nor built: the modules run


def load_library() -> ctypes.CDLL:
    """The built library (built now if it is missing)."""
    global _lib
    if _lib is None:
        from .code_emitter.build_basic import BasicBuilder
        lib = ctypes.CDLL(BasicBuilder().build_mlp())
        lib.recflex_mlp_forward.restype = ctypes.c_int
        lib.recflex_mlp_forward.argtypes = [ctypes.POINTER(_Args)]
        lib.recflex_mlp_workspace_floats.restype = ctypes.c_int
        lib.recflex_mlp_workspace_floats.argtypes = [ctypes.POINTER(_Args), ctypes.POINTER(ctypes.c_int64)]
        _lib = lib
    return _lib


def try_load_library() -> bool:
    """Load the library, with a warning where that fails: the modules serve without it."""
    global _missing
    try:
        load_library()
        _missing = False
    except (OSError, subprocess.SubprocessError) as e:      # no file and no compiler, nowhere to write, ...
        _missing = True
        warnings.warn(f"the MLP kernels could not be loaded or built, RecomModel runs its layers one by one: {e}",
                      RuntimeWarning, stacklevel=3)
    return not _missing


def _hooked(m: nn.Module) -> bool:
    return bool(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                or "forward" in m.__dict__)


def _linears(mlp: nn.Module) -> Optional[List[nn.Linear]]:
    """The linear layers if ``mlp`` is what ``RecomModel`` builds and nobody listens in."""
    if type(mlp) is not nn.Sequential or _hooked(mlp) or _has_any_global_hook():
        return None
    mods = list(mlp._modules.values())
    if len(mods) < 6 or len(mods) % 2:
        return None
    for i, m in enumerate(mods):
        want = nn.Linear if i % 2 == 0 else (nn.Sigmoid if i + 1 == len(mods) else nn.ReLU)
        if type(m) is not want or _hooked(m):
            return None
    return mods[::2]


def _plain(t, shape, x) -> bool:
    return type(t) in (nn.Parameter, torch.Tensor) and t.dtype is torch.float32 and t.shape == shape \
        and t.device == x.device and t.is_contiguous()


def _observed() -> bool:
    """Something wants to see every operation."""
    return torch.is_autocast_enabled("cuda") or torch.jit.is_tracing() or torch.compiler.is_compiling() \
        or _transforms() is not None or torch.autograd.forward_ad._current_level >= 0 \
        or _dispatch_modes() > 0 or _function_modes() > 0


def _run(x: torch.Tensor, weights, biases, keep_hidden: bool):
    """(output [M, 1], the layers' outputs after their ReLU -- all of them, or what the kernels need)"""
    lib = load_library()
    layers, batch = len(weights) - 1, x.shape[0]
    units = [x.shape[1]] + [w.shape[0] for w in weights[:-1]]
    a = _Args(x=x.data_ptr(), batch=batch, layers=layers,
              stream=torch.cuda.current_stream(x.device).cuda_stream)
    a.units[:layers + 1] = units
    a.weights[:layers + 1] = [w.data_ptr() for w in weights]
    a.biases[:layers + 1] = [b.data_ptr() for b in biases]
    floats = ctypes.c_int64(0)
    rc = lib.recflex_mlp_workspace_floats(ctypes.byref(a), ctypes.byref(floats))
    if rc != 0:
        raise RuntimeError(f"recflex_mlp_workspace_floats: hipError_t {rc}")
    out = x.new_empty((batch, 1))
    hidden = [x.new_empty((batch, n)) for n in (units[1:] if keep_hidden else units[1:-2])]
    workspace = x.new_empty(floats.value)
    a.out, a.workspace = out.data_ptr(), workspace.data_ptr()
    a.hidden[:len(hidden)] = [h.data_ptr() for h in hidden]
    rc = lib.recflex_mlp_forward(ctypes.byref(a))
    if rc != 0:
        raise RuntimeError(f"recflex_mlp_forward: hipError_t {rc}")
    return out, hidden


class _Mlp(torch.autograd.Function):
    """Outputs: the MLP's and every hidden layer's (so that second derivatives find their way)."""

    @staticmethod
    def forward(ctx, x, *params):
        weights, biases = params[0::2], params[1::2]
        out, hidden = _run(x, weights, biases, True)
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(x, *weights, *hidden, out)
        return (out, *hidden)

    @staticmethod
    def backward(ctx, g_out, *g_hidden):
        n = len(g_hidden)
        x, weights = ctx.saved_tensors[0], ctx.saved_tensors[1:n + 2]
        acts, out = (x, *ctx.saved_tensors[n + 2:2 * n + 2]), ctx.saved_tensors[-1]
        grads = [None] * (1 + 2 * len(weights))
        g = g_out                                # of the output of layer l, after its activation
        for l in range(n, -1, -1):
            if l < n and g_hidden[l] is not None:
                g = g_hidden[l] if g is None else g + g_hidden[l]
            if g is None:
                continue
            g = torch.ops.aten.sigmoid_backward(g, out) if l == n \
                else torch.ops.aten.threshold_backward(g, acts[l + 1], 0)
            if ctx.needs_input_grad[1 + 2 * l]:
                grads[1 + 2 * l] = g.t().mm(acts[l])
            if ctx.needs_input_grad[2 + 2 * l]:
                grads[2 + 2 * l] = g.sum(0)
            if any(ctx.needs_input_grad[:1 + 2 * l]):
                g = g.mm(weights[l])
            else:
                break
        if ctx.needs_input_grad[0]:
            grads[0] = g
        return tuple(grads)


def forward(mlp: nn.Module, x: torch.Tensor) -> Optional[torch.Tensor]:
    if not _KNOWS_OBSERVERS:
        return None
    linears = _linears(mlp)
    if linears is None or _observed():
        return None
    if type(x) is not torch.Tensor or x.dim() != 2:
        return None
    batch, fan_in = x.shape
    if not 0 < batch <= MAX_BATCH or x.dtype is not torch.float32 or not x.is_cuda or not x.is_contiguous() \
            or x.data_ptr() % 16 or x.device.index != torch.cuda.current_device():
        return None
    params, units = [], [fan_in]
    hidden = len(linears) - 1
    if hidden > MAX_LAYERS or linears[-1].weight.shape[0] != 1:
        return None
    for l, m in enumerate(linears):
        w, b = m.weight, m.bias
        if b is None or w.dim() != 2 or not _plain(w, (w.shape[0], fan_in), x) or not _plain(b, w.shape[:1], x) \
                or (l < hidden and (fan_in % 4 or w.data_ptr() % 16)):
            return None
        params += [w, b]
        fan_in = w.shape[0]
        units.append(fan_in)
    if units[-2] > TAIL_MAX_UNITS or units[-3] > TAIL_MAX_INPUTS or not _pays(batch, units[:-1]):
        return None
    if _lib is None and (_missing or not try_load_library()):
        return None
    if torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in params)):
        return _Mlp.apply(x, *params)[0]
    return _run(x, params[0::2], params[1::2], False)[0]
