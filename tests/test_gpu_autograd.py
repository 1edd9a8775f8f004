"""GPU tests of the autograd Function / nn.Module surface against the reference path on the CPU."""
import pytest
import torch

import nanoplm_amd as npa
from nanoplm_amd.workloads import make_workload
from oracle import dwconv_ref as O

from gpu_util import assert_act_close, assert_red_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_function_backward_matches_reference_autograd_fp32():
    wl = make_workload(1, with_dy=True)
    y_r, dx_r, dw_r, db_r = O.ref_dwconv_varlen_grads(wl.x, wl.cu_seqlens, wl.weight, wl.bias, wl.dy, torch.float64)
    x = wl.x.to(DEV).requires_grad_(True)
    w = wl.weight.to(DEV).requires_grad_(True)
    b = wl.bias.to(DEV).requires_grad_(True)
    y = npa.VarlenDWConv1dFunction.apply(x, wl.cu_seqlens.to(DEV), w, b)
    y.backward(wl.dy.to(DEV))
    assert_act_close(y, y_r, torch.float32, "y")
    assert_act_close(x.grad, dx_r, torch.float32, "dx")
    assert_red_close(w.grad, dw_r, "dw")
    assert_red_close(b.grad, db_r, "db")


def test_module_under_autocast_with_fp32_parameters():
    """bf16 activations with fp32 master parameters, as under torch.autocast in the training loop
    (src/nanoplm/pretraining/pure_pipeline.py:717-722); gradients come back in the parameters' dtype."""
    wl = make_workload(5, T=5000, C=512)
    conv = npa.VarlenDWConv1d(512, 7).to(DEV)
    with torch.no_grad():
        conv.weight.copy_(wl.weight.float())
        conv.bias.copy_(wl.bias.float())
    x = wl.x.to(DEV).requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = conv(x, wl.cu_seqlens.to(DEV))
    assert y.dtype == torch.bfloat16
    y.backward(wl.dy.to(DEV))
    assert conv.weight.grad.dtype == torch.float32 and x.grad.dtype == torch.bfloat16
    y_r, dx_r, dw_r, db_r = O.ref_dwconv_varlen_grads(wl.x, wl.cu_seqlens, wl.weight, wl.bias, wl.dy, torch.float64)
    assert_act_close(y, y_r, torch.bfloat16, "y")
    assert_act_close(x.grad, dx_r, torch.bfloat16, "dx")
    assert_red_close(conv.weight.grad, dw_r, "dw")
    assert_red_close(conv.bias.grad, db_r, "db")


def test_bf16_parameters_get_bf16_gradients_and_frozen_inputs_get_none():
    wl = make_workload(5, T=3000, C=256)
    x = wl.x.to(DEV)                                   # no grad wanted for x
    w = wl.weight.to(DEV).requires_grad_(True)
    b = wl.bias.to(DEV).requires_grad_(True)
    y = npa.varlen_dwconv(x, wl.cu_seqlens.to(DEV), w, b)
    y.backward(wl.dy.to(DEV))
    assert w.grad.dtype == torch.bfloat16 and b.grad.dtype == torch.bfloat16
    _, _, dw_r, db_r = O.ref_dwconv_varlen_grads(wl.x, wl.cu_seqlens, wl.weight, wl.bias, wl.dy, torch.float64)
    # one bf16 rounding of the fp32 result
    assert bool(((w.grad.double().cpu() - dw_r).abs() <= dw_r.abs() * 2.0 ** -8 + 1e-3).all())
    assert bool(((b.grad.double().cpu() - db_r).abs() <= db_r.abs() * 2.0 ** -8 + 1e-3).all())
    # only dx requested
    x2 = wl.x.to(DEV).requires_grad_(True)
    y2 = npa.varlen_dwconv(x2, wl.cu_seqlens.to(DEV), w.detach(), b.detach())
    y2.backward(wl.dy.to(DEV))
    assert x2.grad is not None


def test_non_contiguous_inputs_are_accepted():
    wl = make_workload(5, T=2000, C=256)
    xt = wl.x.to(DEV).t().contiguous().t()             # [T, C] view with transposed strides
    assert not xt.is_contiguous()
    y = npa.varlen_dwconv_fwd(xt, wl.cu_seqlens.to(DEV), wl.weight.to(DEV), wl.bias.to(DEV))
    y0 = npa.varlen_dwconv_fwd(wl.x.to(DEV), wl.cu_seqlens.to(DEV), wl.weight.to(DEV), wl.bias.to(DEV))
    assert torch.equal(y, y0)


def test_runs_on_a_side_stream():
    wl = make_workload(5, T=4000, C=256).to(DEV)
    y0 = npa.varlen_dwconv_fwd(wl.x, wl.cu_seqlens, wl.weight, wl.bias)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y1 = npa.varlen_dwconv_fwd(wl.x, wl.cu_seqlens, wl.weight, wl.bias)
        dx1, dw1, db1 = npa.varlen_dwconv_bwd(wl.x, wl.dy, wl.cu_seqlens, wl.weight)
    s.synchronize()
    dx0, dw0, db0 = npa.varlen_dwconv_bwd(wl.x, wl.dy, wl.cu_seqlens, wl.weight)
    torch.cuda.synchronize()
    assert torch.equal(y0, y1) and torch.equal(dx0, dx1) and torch.equal(dw0, dw1) and torch.equal(db0, db1)


def test_registered_custom_ops_pass_opcheck_and_compile_without_graph_breaks():
    """torch.compile(dynamic=False) is how the reference runs its model
    (src/nanoplm/pretraining/pure_pipeline.py:519-524); the conv must trace as one opaque op and accept
    the static collator's fixed-length cu_seqlens (collator.py:430-450)."""
    from nanoplm_amd.workloads import static_packed_cu

    wl = make_workload(2, T=3000, C=256, with_dy=True)
    F, W = 4096, 512
    cu = static_packed_cu(wl.cu_seqlens, F, W, cu_len=64).to(DEV)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(F, 256, generator=g).bfloat16().to(DEV)
    dy = torch.randn(F, 256, generator=g).bfloat16().to(DEV)
    torch.library.opcheck(npa.varlen_dwconv_fwd_op, (x, cu, wl.weight.to(DEV), wl.bias.to(DEV)),
                          test_utils=("test_schema", "test_faketensor"))
    torch.library.opcheck(npa.varlen_dwconv_bwd_op, (x, dy, cu, wl.weight.to(DEV)),
                          test_utils=("test_schema", "test_faketensor"))

    conv = npa.VarlenDWConv1d(256, 7).to(DEV).to(torch.bfloat16)
    with torch.no_grad():
        conv.weight.copy_(wl.weight.to(DEV))
        conv.bias.copy_(wl.bias.to(DEV))

    def run(mod):
        xin = x.clone().requires_grad_(True)
        for p in conv.parameters():
            p.grad = None
        y = mod(xin, cu)
        (y.float() * dy.float()).sum().backward()
        return y.detach(), xin.grad, conv.weight.grad.clone(), conv.bias.grad.clone()

    y0, dx0, dw0, db0 = run(conv)
    compiled = torch.compile(conv, backend="aot_eager", fullgraph=True, dynamic=False)
    y1, dx1, dw1, db1 = run(compiled)
    assert torch.equal(y0, y1) and torch.equal(dx0, dx1) and torch.equal(dw0, dw1) and torch.equal(db0, db1)
    # and against the oracle on the real (unpadded) part
    T = wl.T
    cu_host = cu.cpu()
    y64 = O.c_oracle_fwd(x.cpu(), cu_host, wl.weight, wl.bias)
    assert_act_close(y1, y64, torch.bfloat16, "compiled y")
    assert T < F


def test_forward_and_backward_replay_correctly_from_a_hip_graph():
    """The op allocates nothing, reads cu_seqlens on the device and never synchronises, so a training
    step that contains it can be captured (reference: torch.compile + static shapes,
    pure_pipeline.py:519-529). Replay several times with new contents in the static buffers, with eager
    work and synchronisation between replays, and compare every replay with the eager result."""
    torch.manual_seed(1)
    lens = torch.tensor([100, 3, 512, 1, 408])
    cu = torch.zeros(6, dtype=torch.int32)
    cu[1:] = torch.cumsum(lens, 0)
    cu = cu.to(DEV)
    T, C, K = int(lens.sum()), 1024, 7
    w = (torch.randn(C, K, device=DEV) * K ** -0.5).bfloat16()
    b = (torch.randn(C, device=DEV) * 0.02).bfloat16()
    sx = torch.zeros(T, C, device=DEV, dtype=torch.bfloat16)
    sdy = torch.zeros_like(sx)
    ws = torch.empty(npa.bwd_workspace_bytes(T, C, K, torch.bfloat16), dtype=torch.uint8, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                      # warm-up outside capture
        npa.varlen_dwconv_fwd(sx, cu, w, b, residual=True)
        npa.varlen_dwconv_bwd(sx, sdy, cu, w, residual=True, workspace=ws)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gy = npa.varlen_dwconv_fwd(sx, cu, w, b, residual=True)
        gdx, gdw, gdb = npa.varlen_dwconv_bwd(sx, sdy, cu, w, residual=True, workspace=ws)
    for it in range(4):
        x = torch.randn(T, C, device=DEV).bfloat16()
        dy = torch.randn(T, C, device=DEV).bfloat16()
        sx.copy_(x)
        sdy.copy_(dy)
        graph.replay()
        torch.cuda.synchronize()
        ey = npa.varlen_dwconv_fwd(x, cu, w, b, residual=True)
        edx, edw, edb = npa.varlen_dwconv_bwd(x, dy, cu, w, residual=True)
        torch.cuda.synchronize()
        assert torch.equal(gy, ey) and torch.equal(gdx, edx), f"replay {it}"
        assert torch.equal(gdw, edw) and torch.equal(gdb, edb), f"replay {it}"


def test_the_integration_guides_ctypes_binding_runs_as_written():
    """The reference-side binding a maintainer would paste (the first Python block of the integration guide: a ctypes
    load of the shared object and an autograd Function over the two plain entry points) is executed as it stands, with
    only the library's file name replaced by its path, and gives this package's own results bit for bit."""
    import os
    import re
    from nanoplm_amd import _lib
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    guide = open(os.path.join(root, "INTEGRATION.md")).read()
    block = re.search(r"```python\n(import ctypes, torch\n.*?)```", guide, re.S).group(1)
    assert 'ctypes.CDLL("libnplm_dwconv.so")' in block
    ns = {}
    exec(block.replace('"libnplm_dwconv.so"', repr(_lib.LIB_PATH)), ns)
    fn = ns["VarlenDWConv1dFunction"]
    for cfg, kw in ((1, {}), (5, dict(T=5000, C=512))):
        wl = make_workload(cfg, with_dy=True, **kw)
        d = wl.to(DEV)
        x = d.x.clone().requires_grad_(True)
        w = d.weight.clone().requires_grad_(True)
        b = d.bias.clone().requires_grad_(True)
        y = fn.apply(x, d.cu_seqlens, w, b)
        y.backward(d.dy)
        assert torch.equal(y, npa.varlen_dwconv_fwd(d.x, d.cu_seqlens, d.weight, d.bias))
        dx, dw, db = npa.varlen_dwconv_bwd(d.x, d.dy, d.cu_seqlens, d.weight)
        assert torch.equal(x.grad, dx) and torch.equal(w.grad, dw.to(w.dtype)) and torch.equal(b.grad, db.to(b.dtype))


# ---- native nodes ---------------------------------------------------------------------------------
def _door(form, act, par, bias, residual):
    """(call through the public door, the same call as a Python Function, its tensors) for T=600 rows of 512 channels, 7 taps."""
    C, K = 512, 7
    g = torch.Generator().manual_seed(7)
    rnd = lambda *s, dt: torch.randn(*s, generator=g).to(dt).to(DEV)
    cu = torch.tensor([0, 3, 3, 200, 600], dtype=torch.int32, device=DEV)
    x = rnd(600, 2 * C if form == "gated" else C, dt=act)
    w, b = rnd(C, K, dt=par), rnd(C, dt=par) if bias else None
    if form == "ln":
        lw, lb = rnd(C, dt=par), rnd(C, dt=par) if bias else None
        return (lambda x, lw, lb, w, b: npa.ln_varlen_dwconv_compilable(x, cu, lw, lb, w, b, residual=residual),
                lambda x, lw, lb, w, b: npa.ln_varlen_dwconv(x, cu, lw, lb, w, b, residual=residual), [x, lw, lb, w, b])
    public, function = ((npa.gated_varlen_dwconv, npa.GatedVarlenDWConv1dFunction) if form == "gated" else
                        (npa.varlen_dwconv, npa.VarlenDWConv1dFunction))
    return (lambda x, w, b: public(x, cu, w, b, residual), lambda x, w, b: function.apply(x, cu, w, b, residual), [x, w, b])


@pytest.mark.parametrize("form", ["plain", "gated", "ln"])
@pytest.mark.parametrize("act,par", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("bias,residual,frozen", [(True, False, ()), (False, True, ()), (True, True, (0,)), (True, False, (-1, -2))])
def test_native_nodes_give_the_bits_of_the_python_functions(form, act, par, bias, residual, frozen):
    door, function, args = _door(form, act, par, bias, residual)
    frozen = [args[i] for i in frozen]
    leaves = [None if t is None else t.clone().requires_grad_(all(t is not f for f in frozen)) for t in args]
    wanted = [t for t in leaves if t is not None and t.requires_grad]
    y, y1 = door(*leaves), function(*leaves)
    assert "Backward" not in type(y.grad_fn).__name__ and "Backward" in type(y1.grad_fn).__name__
    dy = torch.randn(y.shape, device=DEV).to(y.dtype)
    got, want = torch.autograd.grad(y, wanted, dy), torch.autograd.grad(y1, wanted, dy)
    assert torch.equal(y, y1) and y.dtype == y1.dtype
    for a, c, t in zip(got, want, wanted):
        assert a.dtype == c.dtype == t.dtype and torch.equal(a, c)
    with torch.no_grad():
        y0 = door(*leaves)
    assert torch.equal(y0, y1) and not y0.requires_grad


@pytest.mark.parametrize("form", ["plain", "gated", "ln"])
def test_native_nodes_leave_other_forms_of_call_to_the_python_route(form):
    """Strided and unaligned tensors, mixed parameter dtypes, saved-tensor hooks, dy that is no dense tensor, transforms, forward mode."""
    bf16, f32 = torch.bfloat16, torch.float32
    door, function, args = _door(form, bf16, bf16, True, False)
    y = function(*args)
    x, rest = args[0], args[1:]
    wide = torch.empty(600, 2 * x.shape[1], dtype=bf16, device=DEV)
    wide[:, :x.shape[1]] = x
    assert torch.equal(door(wide[:, :x.shape[1]], *rest), y)
    odd = torch.empty(x.numel() + 1, dtype=bf16, device=DEV)[1:].view(x.shape).copy_(x)
    torch.testing.assert_close(door(odd, *rest), function(odd, *rest), rtol=0, atol=0)
    mixed = [x] + rest[:-1] + [rest[-1].to(f32)]
    assert torch.equal(door(*mixed), function(*mixed))
    xg = x.clone().requires_grad_()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.clone(), lambda t: t):
        yg = door(xg, *rest)
    assert any(t is xg or t.data_ptr() == xg.data_ptr() for t in packed)
    dy = torch.ones(1, dtype=bf16, device=DEV).expand(y.shape)
    got = torch.autograd.grad(yg, xg, dy)[0]
    assert torch.equal(got, torch.autograd.grad(function(xg, *rest), xg, dy.contiguous())[0])
    batch = lambda: torch.func.vmap(lambda x: door(x, *rest))(x[None].expand(2, *x.shape))
    if form == "ln":                                         # (a registered op, which vmap takes apart)
        assert torch.equal(batch(), y[None].expand(2, *y.shape))
    else:
        pytest.raises(RuntimeError, batch)                   # (a Function without a rule for it)
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level(), pytest.raises(Exception):
        door(fwd.make_dual(xg, x), *rest)
    with pytest.raises(RuntimeError):                        # not differentiable twice
        g = torch.autograd.grad(door(xg, *rest).float().sum(), xg, create_graph=True)[0]
        torch.autograd.grad(g.float().sum(), xg)


@pytest.mark.parametrize("form", ["plain", "gated", "ln"])
def test_native_nodes_take_what_saved_tensor_hooks_give_back(form):
    """Hooks may hand back other strides than were saved (made dense by the Python route), or another size (refused by it). An incoming
    gradient that is not aligned goes the same way where the kernels want it aligned."""
    door, function, args = _door(form, torch.bfloat16, torch.bfloat16, True, False)
    dy = torch.randn(args[0].shape[0], 512, device=DEV).to(torch.bfloat16)

    def grads(call, unpack, dy=dy):
        leaves = [t.clone().requires_grad_() for t in args]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            y = call(*leaves)
        return torch.autograd.grad(y, leaves, dy)

    def strided(t):
        wide = torch.empty(*t.shape, 2, dtype=t.dtype, device=t.device)
        wide[..., 0] = t
        return wide[..., 0]

    for a, c in zip(grads(door, strided), grads(function, lambda t: t)):
        assert torch.equal(a, c)
    odd = torch.empty(dy.numel() + 1, dtype=dy.dtype, device=DEV)[1:].view(dy.shape).copy_(dy)
    for a, c in zip(grads(door, lambda t: t, odd), grads(function, lambda t: t, odd)):
        torch.testing.assert_close(a, c, rtol=0, atol=0)
    with pytest.raises((ValueError, RuntimeError)):
        grads(door, lambda t: t[:300] if t.shape[0] == 600 else t)


class _Wrapper(torch.Tensor):
    """A tensor that holds another one and hands every operation on to it."""
    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, strides=inner.stride(), dtype=inner.dtype, device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        from torch.utils._pytree import tree_map_only
        out = func(*tree_map_only(cls, lambda t: t.inner, args), **tree_map_only(cls, lambda t: t.inner, kwargs or {}))
        return tree_map_only(torch.Tensor, cls, out)


def test_native_prenorm_node_takes_gradients_and_tensors_of_every_kind():
    """What reached the registered ops of the pre-norm door reaches them still: incoming gradients that are a batch of gradients, wrap
    another tensor, are known to be zero or are negated as they are read, negated inputs and weights, and a backward that a mode watches."""
    from torch.utils._python_dispatch import TorchDispatchMode

    door, function, args = _door("ln", torch.bfloat16, torch.bfloat16, True, False)
    leaves = [t.clone().requires_grad_() for t in args]
    dy = torch.randn(args[0].shape, device=DEV).bfloat16()
    grads = lambda d, **kw: torch.autograd.grad(door(*leaves), leaves, d, **kw)
    want, want2 = grads(dy), grads(-2 * dy)
    same = lambda got, ref: all(torch.equal(a, c) for a, c in zip(got, ref))
    assert same(want, torch.autograd.grad(function(*leaves), leaves, dy))
    batch = grads(torch.stack([dy, -2 * dy]), is_grads_batched=True)
    assert same([t[0] for t in batch], want) and same([t[1] for t in batch], want2)
    y = door(*leaves)
    batch = torch.func.vmap(lambda d: torch.autograd.grad(y, leaves[0], d, retain_graph=True)[0])(torch.stack([dy, -2 * dy]))
    assert torch.equal(batch[0], want[0]) and torch.equal(batch[1], want2[0])
    assert same([t.inner for t in grads(_Wrapper(dy))], want)
    assert all(not bool(t.any()) for t in grads(torch._efficientzerotensor(dy.shape, dtype=dy.dtype, device=DEV)))
    assert same(grads(torch._neg_view(dy)), grads(-dy))
    for i in range(len(args)):
        neg = [torch._neg_view(t) if j == i else t for j, t in enumerate(args)]
        assert torch.equal(door(*neg), door(*[-t if j == i else t for j, t in enumerate(args)]))
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    y = door(*leaves)
    with Watch():
        got = torch.autograd.grad(y, leaves, dy)
    assert same(got, want) and any("ln_dwconv_bwd" in f for f in seen)


@pytest.mark.filterwarnings("ignore:Error detected in")
@pytest.mark.parametrize("form,name", [("plain", "varlen_dwconv"), ("gated", "gated_dwconv"), ("ln", "ln_dwconv")])
def test_profiles_and_messages_name_the_native_nodes(form, name):
    """A profile lists an eager call and its backward by the names of the registered ops; autograd's messages name the function."""
    door, _, args = _door(form, torch.bfloat16, torch.bfloat16, True, False)
    leaves = [t.clone().requires_grad_() for t in args]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as p:
        y = door(*leaves)
        torch.autograd.grad(y, leaves, torch.ones_like(y))
    keys = {e.key for e in p.key_averages()}
    assert {f"nanoplm_amd::{name}_fwd", f"nanoplm_amd::{name}_bwd"} <= keys
    with pytest.raises(RuntimeError, match="VarlenDWConv1d.* returned nan"), torch.autograd.set_detect_anomaly(True):
        y = door(*leaves)
        torch.autograd.grad(y, leaves, torch.full_like(y, float("nan")))


@pytest.mark.parametrize("form", ["gated", "ln"])
def test_native_nodes_leave_calls_without_a_fused_kernel_before_they_begin(form):
    """Rows that the fused kernels are not built for: no output is allocated for a call that the Python route takes."""
    from nanoplm_amd import _lib
    C, K = (24, 7) if form == "gated" else (24, 11)
    x = torch.randn(64, 2 * C if form == "gated" else C, device=DEV)
    cu = torch.tensor([0, 64], dtype=torch.int32, device=DEV)
    w, v = torch.randn(C, K, device=DEV), torch.randn(C, device=DEV)
    node = _lib.load_node()
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = count()
    assert (node.gated_dwconv(x, cu, w, v, False) if form == "gated" else node.ln_dwconv(x, cu, v, None, w, v, 1e-5, False)) is None
    assert count() == before


def _kernel_door(form, K):
    """The door with kernels of K taps (on the matrix cores where they exist) on 4500 rows of 512 channels; its tensors, x first."""
    C, T = 512, 4500
    g = torch.Generator().manual_seed(K)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).bfloat16().to(DEV)
    cu = torch.tensor([0, 1000, 1001, 2500, T], dtype=torch.int32, device=DEV)
    x, w, b = rnd(T, 2 * C if form == "gated" else C), rnd(C, K, scale=K ** -0.5), rnd(C)
    if form == "ln":
        return lambda x, lw, lb, w, b: npa.ln_varlen_dwconv_compilable(x, cu, lw, lb, w, b, residual=True), [x, rnd(C), rnd(C), w, b]
    f = npa.gated_varlen_dwconv if form == "gated" else npa.varlen_dwconv
    return lambda x, w, b: f(x, cu, w, b, True), [x, w, b]


_NODE_CASES = [("plain", 7), ("plain", 31), ("gated", 7), ("gated", 31), ("ln", 7)]


def _step(door, leaves, dy):
    y = door(*leaves)
    return (y.detach(), *torch.autograd.grad(y, leaves, dy))


@pytest.mark.parametrize("form,K", _NODE_CASES)
def test_native_nodes_on_a_side_stream_and_from_several_threads(form, K):
    """Forwards on streams of their own (the engine runs their backwards there), temporaries freed and reused meanwhile; then two threads."""
    import threading
    door, args = _kernel_door(form, K)
    g = torch.Generator(device=DEV).manual_seed(3)
    calls = []
    for _ in range(6):
        leaves = [torch.empty_like(args[0]).normal_(generator=g)] + [t.clone() for t in args[1:]]
        leaves = [t.requires_grad_() for t in leaves]
        calls.append((leaves, torch.empty(args[0].shape[0], 512, dtype=torch.bfloat16, device=DEV).normal_(generator=g)))
    want = [_step(door, *c) for c in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    got = []
    for i, c in enumerate(calls):
        with torch.cuda.stream(streams[i % 3]):
            got.append(_step(door, *c))
    torch.cuda.synchronize()
    assert all(torch.equal(a, r) for gs, ws in zip(got, want) for a, r in zip(gs, ws))
    out = [None] * len(calls)

    def work(k):
        with torch.cuda.stream(streams[k]):
            for i in range(k, len(calls), 2):
                out[i] = _step(door, *calls[i])

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(torch.equal(a, r) for gs, ws in zip(out, want) for a, r in zip(gs, ws))


@pytest.mark.parametrize("form,K", _NODE_CASES)
def test_native_nodes_replay_from_a_hip_graph_and_run_under_checkpointing(form, K):
    """A captured forward and backward of the door, replayed on new contents with eager work and synchronization between the replays; and
    the same step under activation checkpointing, reentrant and not."""
    from torch.utils.checkpoint import checkpoint
    door, args = _kernel_door(form, K)
    leaves = [t.clone().requires_grad_() for t in args]
    dy = torch.randn(args[0].shape[0], 512, device=DEV).bfloat16()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(door, leaves, dy)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _step(door, leaves, dy)
    for it in range(4):
        with torch.no_grad():
            leaves[0].normal_()
            dy.normal_()
        graph.replay()
        torch.cuda.synchronize()
        eager = _step(door, leaves, dy)
        torch.cuda.synchronize()
        assert all(torch.equal(a, r) for a, r in zip(captured, eager)), f"replay {it}"
    for reentrant in (False, True):
        y = checkpoint(door, *leaves, use_reentrant=reentrant)
        for t in leaves:
            t.grad = None
        y.backward(dy)
        assert torch.equal(y, eager[0]) and all(torch.equal(t.grad, r) for t, r in zip(leaves, eager[1:]))
