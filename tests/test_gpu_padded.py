"""Padded-batch door of the op ([B, L, C] + attention mask, the reference's SDPA-path layout,
modeling.py:505-544) and the flat_weight parameterisation, on the GPU against the oracle."""
import pytest
import torch

import nanoplm_amd as npa
from oracle import dwconv_ref as O
from tests.gpu_util import assert_act_close, assert_red_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _padded_case(lens, L, C, K, dt, seed):
    g = torch.Generator().manual_seed(seed)
    B = len(lens)
    x = torch.randn(B, L, C, generator=g).to(dt)
    mask = torch.zeros(B, L, dtype=torch.bool)
    for b, n in enumerate(lens):
        mask[b, :n] = True
    w = (torch.randn(C, K, generator=g) * K ** -0.5).to(dt)
    bias = (torch.randn(C, generator=g) * 0.02).to(dt)
    return x, mask, w, bias


def _oracle_on_real_rows(x, mask, w, bias, residual=False):
    idx, cu, _ = npa.unpad_input(mask)
    B, L, C = x.shape
    return idx, O.c_oracle_fwd(x.reshape(B * L, C)[idx], cu, w, bias, residual=residual)


@pytest.mark.parametrize("residual", [False, True])
def test_right_padded_batch_in_place(residual):
    lens = [37, 128, 0, 1, 90, 128, 5]
    x, mask, w, bias = _padded_case(lens, 128, 1024, 7, torch.bfloat16, seed=1)
    idx, y64 = _oracle_on_real_rows(x, mask, w, bias, residual)
    xd, md, wd, bd = x.to(DEV), mask.to(DEV), w.to(DEV), bias.to(DEV)
    y = npa.padded_dwconv(xd, md, wd, bd, residual=residual)
    assert y.shape == x.shape
    assert_act_close(y.reshape(-1, 1024)[idx.to(DEV)], y64, x.dtype, "padded y (real rows)")
    assert torch.isfinite(y.float()).all()
    # padding positions depend on pad rows only: change every real token, pads stay bit-identical
    x2 = xd.clone()
    x2[md] = 7.0
    y2 = npa.padded_dwconv(x2, md, wd, bd, residual=residual)
    assert torch.equal(y[~md], y2[~md])


@pytest.mark.parametrize("dt", [torch.bool, torch.uint8, torch.int32, torch.int64, torch.float32])
@pytest.mark.parametrize("B,L", [(1, 1), (33, 63), (31, 65), (32, 128), (5, 129), (3, 640), (6, 1024), (2, 1025), (2, 8192), (1, 8193),
                                 (2, 9000), (1, 1 << 17), (1, (1 << 17) + 1), (65537, 2), (0, 8), (4, 0)])
def test_boundaries_in_one_launch_equal_the_elementwise_ones(B, L, dt):
    """Row lengths around those at which more threads share a row (128, 1024, 8192) and their passes of eight loads, numbers
    of rows around those of a block, the longest row of the one launch, rows that are a slice of a wider tensor and
    transposed ones (which take the elementwise operations), against the boundaries formed on the CPU; not every row is
    right-padded."""
    from nanoplm_amd.padded import _flat_cu_seqlens
    wide = (torch.rand(B, L + 3, generator=torch.Generator().manual_seed(B * L)) > 0.3).to(dt)
    x = torch.zeros(1, device=DEV)
    d = wide.to(DEV)
    assert torch.equal(_flat_cu_seqlens(d[:, 1:L + 1], x).cpu(), npa.right_padded_cu_seqlens(wide[:, 1:L + 1]))
    assert torch.equal(_flat_cu_seqlens(d.t(), x).cpu(), npa.right_padded_cu_seqlens(wide.t()))


def test_boundaries_of_a_bool_mask_that_is_a_view_of_bytes():
    """A bool counts as one whatever its byte holds if that is not zero (what torch's sum does); a uint8 counts as its value."""
    from nanoplm_amd.padded import _flat_cu_seqlens
    x = torch.zeros(1, device=DEV)
    raw = torch.zeros(4, 300, dtype=torch.uint8)
    raw[0, :2], raw[1, :300], raw[3, :7] = 255, 2, torch.arange(1, 8, dtype=torch.uint8)
    assert _flat_cu_seqlens(raw.to(DEV).view(torch.bool), x).tolist() == [0, 2, 300, 600, 600, 600, 900, 907, 1200]
    assert _flat_cu_seqlens(raw.to(DEV), x).tolist() == [0, 510, 300, 900, 600, 600, 900, 928, 1200]


def test_traced_door_follows_the_mask_of_the_replay():
    """torch.jit.trace of the padded door with one mask, replayed with another, gives what the eager call gives."""
    x, first, w, bias = _padded_case([37, 128, 0, 1], 128, 512, 7, torch.bfloat16, seed=4)
    second = _padded_case([5, 0, 128, 90], 128, 512, 7, torch.bfloat16, seed=4)[1]
    xd, wd, bd, m1, m2 = (t.to(DEV) for t in (x, w, bias, first, second))
    traced = torch.jit.trace(lambda xx, mm: npa.padded_dwconv(xx, mm, wd, bd), (xd, m1))
    for m in (m1, m2, m1):
        assert torch.equal(traced(xd, m), npa.padded_dwconv(xd, m, wd, bd))


def test_arbitrary_mask_goes_through_gather_and_scatter():
    g = torch.Generator().manual_seed(2)
    B, L, C = 5, 64, 256
    x = torch.randn(B, L, C, generator=g)
    mask = torch.rand(B, L, generator=g) > 0.3          # holes anywhere (left padding included)
    mask[2] = False
    w = torch.randn(C, 5, generator=g) * 5 ** -0.5
    bias = torch.randn(C, generator=g) * 0.02
    idx, y64 = _oracle_on_real_rows(x, mask, w, bias)
    y = npa.padded_dwconv(x.to(DEV), mask.to(DEV), w.to(DEV), bias.to(DEV), assume_right_padded=False)
    assert_act_close(y.reshape(-1, C)[idx.to(DEV)], y64, x.dtype, "gathered y")
    assert float(y[~mask.to(DEV)].abs().sum()) == 0.0


def test_padded_module_gradients_match_the_packed_op():
    """Loss on real tokens only (what masked-LM labels give): dw/db/dx of the in-place padded route
    equal those of the packed route on the gathered rows."""
    lens = [50, 128, 3, 77]
    x, mask, w, bias = _padded_case(lens, 128, 256, 7, torch.float32, seed=3)
    idx, cu, _ = npa.unpad_input(mask)
    conv = npa.VarlenDWConv1d(256, 7, device=DEV)
    with torch.no_grad():
        conv.weight.copy_(w)
        conv.bias.copy_(bias)
    xd = x.to(DEV).requires_grad_(True)
    md = mask.to(DEV)
    gy = torch.randn(int(mask.sum()), 256, device=DEV)
    y = conv.forward_padded(xd, md)
    (y[md] * gy).sum().backward()
    dw_p, db_p, dx_p = conv.weight.grad.clone(), conv.bias.grad.clone(), xd.grad.clone()
    conv.zero_grad()
    xr = x.reshape(-1, 256)[idx].to(DEV).requires_grad_(True)
    (conv(xr, cu.to(DEV)) * gy).sum().backward()
    torch.testing.assert_close(dw_p, conv.weight.grad, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(db_p, conv.bias.grad, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(dx_p[md], xr.grad, rtol=1e-5, atol=1e-5)
    assert float(dx_p[~md].abs().sum()) == 0.0


def test_flat_weight_module_trains_like_the_2d_one():
    torch.manual_seed(4)
    lens = torch.tensor([30, 2, 200, 24])
    cu = torch.zeros(5, dtype=torch.int32)
    cu[1:] = torch.cumsum(lens, 0)
    cu = cu.to(DEV)
    a = npa.VarlenDWConv1d(128, 7, residual=True, device=DEV)
    b = npa.VarlenDWConv1d(128, 7, residual=True, flat_weight=True, device=DEV)
    with torch.no_grad():
        b.weight_flat.copy_(a.weight.reshape(-1))
        b.bias.copy_(a.bias)
    x = torch.randn(256, 128, device=DEV)
    gy = torch.randn(256, 128, device=DEV)
    a(x, cu).backward(gy)
    b(x, cu).backward(gy)
    assert torch.equal(b.weight_flat.grad.view(128, 7), a.weight.grad)
    assert torch.equal(b.bias.grad, a.bias.grad)
    # zero-initialised residual block is the identity
    z = npa.VarlenDWConv1d(128, 7, residual=True, init="zero", device=DEV)
    assert torch.equal(z(x, cu), x)


def test_padded_door_compiles_without_graph_breaks():
    """forward_padded inside a compiled model (torch.compile(dynamic=False), pure_pipeline.py:519-524): the call
    reaches the registered custom ops, so fullgraph=True holds, forward and backward."""
    lens = [37, 128, 0, 1, 90, 128, 5]
    x, mask, w, bias = _padded_case(lens, 128, 1024, 7, torch.bfloat16, seed=3)
    conv = npa.VarlenDWConv1d(1024, 7, residual=True, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        conv.weight.copy_(w.to(DEV))
        conv.bias.copy_(bias.to(DEV))
    xd, md = x.to(DEV), mask.to(DEV)

    class Door(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.conv = conv

        def forward(self, xx, mm):
            return self.conv.forward_padded(xx, mm)

    def run(mod):
        conv.zero_grad()
        xin = xd.clone().requires_grad_(True)
        y = mod(xin, md)
        y.float().square().sum().backward()
        return y.detach(), xin.grad, conv.weight.grad.clone(), conv.bias.grad.clone()

    door = Door()
    eager = run(door)
    torch._dynamo.reset()
    compiled = run(torch.compile(door, backend="aot_eager", fullgraph=True, dynamic=False))
    for a, b in zip(eager, compiled):
        assert torch.equal(a, b)
