"""The kernels of 11 to 31 taps on the matrix cores (bf16 activations and weights) against the oracle and the vector kernels."""
import pytest
import torch

import nanoplm_amd as npa
from nanoplm_amd import _lib
from nanoplm_amd.workloads import cu_from_lengths
from oracle import dwconv_ref as O

from gpu_util import assert_act_close, assert_red_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# sequences shorter than four rows, than the halo and than a tile, empty ones, tile edges, and tiles without a boundary
LENS = [1, 2, 3, 8, 0, 1, 150, 0, 5, 7, 6, 1, 64, 63, 65, 2, 300, 4, 15, 16, 17, 30, 31, 32, 33, 700, 1, 1, 1, 29, 0, 0, 45,
        1200, 14]
MFMA = dict(algo=4)


def _case(lens, C, K, seed):
    g = torch.Generator().manual_seed(seed)
    cu = cu_from_lengths(torch.tensor(lens))
    T = int(cu[-1])
    return (torch.randn(T, C, generator=g).bfloat16(), cu, (torch.randn(C, K, generator=g) * K ** -0.5).bfloat16(),
            torch.randn(C, generator=g).bfloat16(), torch.randn(T, C, generator=g).bfloat16())


# (the K that run on 11, 15, 21 and 31 taps; whole, partial and several column blocks; one, few and many tiles a block; a last
# tile of 1, 63 and 64 rows)
CASES = [(11, LENS, 264, 1), (13, LENS, 256, 0), (15, LENS * 4, 512, 2), (17, [700], 1000, 0), (21, LENS, 264, 1),
         (25, LENS[::-1], 2056, 5), (29, [64, 1], 256, 0), (31, LENS * 4, 256, 1), (31, [127], 320, 0), (31, [1] * 130, 256, 0),
         (31, LENS, 2056, 0)]


@pytest.mark.parametrize("K,lens,C,nbt", CASES)
def test_forward_on_the_matrix_cores_matches_the_oracle(K, lens, C, nbt):
    """To one bf16 rounding of the oracle's y; the same bits again after a call that left NaN in every LDS byte it used, and
    from the weights zero-padded to the planned size."""
    print(f"[case] K={K} C={C} nbt={nbt}", flush=True)
    x, cu, w, b, _ = _case(lens, C, K, C + K + nbt)
    xd, cud, wd, bd = x.to(DEV), cu.to(DEV), w.to(DEV), b.to(DEV)
    tn = _lib.Tuning(nbt=nbt, **MFMA)
    y64 = O.c_oracle_fwd(x, cu, w, b)
    y = npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=tn)
    assert_act_close(y, y64, torch.bfloat16, "y")
    assert_act_close(npa.varlen_dwconv_fwd(xd, cud, wd, bd, residual=True, tuning=tn), y64 + x.double(), torch.bfloat16, "y + x")
    npa.varlen_dwconv_fwd(torch.full_like(xd, float("nan")), cud, wd, bd, tuning=tn)
    assert torch.equal(npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=tn), y)
    off = ((15 if K <= 15 else 31) - K) // 2
    wide = torch.nn.functional.pad(wd, (off, off)).contiguous()
    assert torch.equal(npa.varlen_dwconv_fwd(xd, cud, wide, bd, tuning=tn), y)


@pytest.mark.parametrize("K", [15, 21, 31])
@pytest.mark.parametrize("step", [63, 95, 191])
def test_one_to_three_sequences_a_tile_with_a_boundary_at_every_row_of_it(K, step):
    """Sequences of `step` rows begin at every row of the 64-row tiles and the 32-row groups in turn: the sweeps over single sequences."""
    print(f"[case] K={K} step={step}", flush=True)
    x, cu, w, b, dy = _case([step] * 65 + [7], 264, K, K + step)
    xd, cud, wd, bd, dyd = x.to(DEV), cu.to(DEV), w.to(DEV), b.to(DEV), dy.to(DEV)
    tn = _lib.Tuning(**MFMA)
    assert_act_close(npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=tn), O.c_oracle_fwd(x, cu, w, b), torch.bfloat16, "y")
    dx64, dw64, db64 = O.c_oracle_bwd(x, dy, cu, w)
    dx, dw, db = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=tn)
    assert_act_close(dx, dx64, torch.bfloat16, "dx")
    assert_red_close(dw, dw64, "dw")
    assert_red_close(db, db64, "db")


def _plant_non_finite(t, cu):
    for i in range(0, cu.numel() - 1, 5):
        if cu[i + 1] - cu[i] < 10:
            t[cu[i]:cu[i + 1], i % 7::7] = float("inf") if i % 2 else float("nan")


@pytest.mark.parametrize("K", [11, 31])
def test_forward_non_finite_rows_stay_in_their_sequence(K):
    x, cu, w, b, _ = _case(LENS * 2, 512, K, K)
    _plant_non_finite(x, cu)
    xd, cud, wd, bd = x.to(DEV), cu.to(DEV), w.to(DEV), b.to(DEV)
    y1 = npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=_lib.Tuning(algo=1))
    y4 = npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=_lib.Tuning(**MFMA))
    assert not bool(torch.isfinite(y1).all())
    torch.testing.assert_close(y4, y1, rtol=2.0 ** -7, atol=1e-5, equal_nan=True)      # (two roundings of one sum)


@pytest.mark.parametrize("T,C,K,wdt,served", [(4096, 256, 31, torch.bfloat16, True), (4095, 256, 31, torch.bfloat16, False),
                                              (4096, 248, 31, torch.bfloat16, False), (4096, 260, 31, torch.bfloat16, False),
                                              (4096, 256, 31, torch.float32, False), (4096, 256, 9, torch.bfloat16, False),
                                              (4096, 264, 11, torch.bfloat16, True)])
def test_which_forward_calls_the_matrix_cores_serve(T, C, K, wdt, served):
    x, cu, w, b, _ = _case([T], C, K, T + C)
    xd, cud, wd = x.to(DEV), cu.to(DEV), w.to(DEV).to(wdt)
    y = npa.varlen_dwconv_fwd(xd, cud, wd, None)
    y1 = npa.varlen_dwconv_fwd(xd, cud, wd, None, tuning=_lib.Tuning(algo=1))
    if served:
        assert torch.equal(y, npa.varlen_dwconv_fwd(xd, cud, wd, None, tuning=_lib.Tuning(**MFMA)))
    else:
        assert torch.equal(y, y1)
        if T >= 4096:
            with pytest.raises(RuntimeError):
                npa.varlen_dwconv_fwd(xd, cud, wd, None, tuning=_lib.Tuning(**MFMA))
    torch.testing.assert_close(y, y1, rtol=2.0 ** -7, atol=1e-5)                          # (two roundings of one sum)


@pytest.mark.parametrize("K,lens,C,nbt", CASES)
def test_backward_on_the_matrix_cores_matches_the_oracle(K, lens, C, nbt):
    """dx to one bf16 rounding, dw and db to the reductions' tolerance; the same bits again after a call that left NaN in LDS."""
    print(f"[case] K={K} C={C} nbt={nbt}", flush=True)
    x, cu, w, _, dy = _case(lens, C, K, C + K + nbt)
    xd, cud, wd, dyd = x.to(DEV), cu.to(DEV), w.to(DEV), dy.to(DEV)
    tn = _lib.Tuning(nbt=nbt, **MFMA)
    dx64, dw64, db64 = O.c_oracle_bwd(x, dy, cu, w)
    got = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=tn)
    assert_act_close(got[0], dx64, torch.bfloat16, "dx")
    assert_red_close(got[1], dw64, "dw")
    assert_red_close(got[2], db64, "db")
    dxr, dwr, dbr = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, residual=True, tuning=tn)
    assert_act_close(dxr, dx64 + dy.double(), torch.bfloat16, "dx + dy")
    assert torch.equal(dwr, got[1]) and torch.equal(dbr, got[2])
    nan = torch.full_like(xd, float("nan"))
    npa.varlen_dwconv_bwd(nan, nan, cud, wd, tuning=tn)
    again = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=tn)
    assert all(torch.equal(a, c) for a, c in zip(again, got))


@pytest.mark.parametrize("K", [15, 31])
@pytest.mark.parametrize("which", ["x", "dy"])
def test_backward_non_finite_rows_stay_in_their_sequence(K, which):
    x, cu, w, _, dy = _case(LENS * 2, 512, K, K)
    _plant_non_finite(x if which == "x" else dy, cu)
    xd, cud, wd, dyd = x.to(DEV), cu.to(DEV), w.to(DEV), dy.to(DEV)
    dx1, dw1, db1 = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=_lib.Tuning(algo=1))
    dx4, dw4, db4 = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=_lib.Tuning(**MFMA))
    assert not bool(torch.isfinite(dw1).all())
    torch.testing.assert_close(dx4, dx1, rtol=2.0 ** -7, atol=1e-5, equal_nan=True)
    for got, ref in ((dw4, dw1), (db4, db1)):                                             # assert_red_close's bar
        torch.testing.assert_close(got, ref, rtol=0, atol=1e-5 * float(ref[torch.isfinite(ref)].abs().max()), equal_nan=True)


@pytest.mark.parametrize("T,n,K,wdt,served", [(4096, 128, 31, torch.bfloat16, True), (4096, 129, 31, torch.bfloat16, False),
                                              (4095, 1, 31, torch.bfloat16, False), (4096, 1, 31, torch.float32, False),
                                              (4096, 64, 15, torch.bfloat16, True), (4096, 65, 15, torch.bfloat16, False),
                                              (4096, 8, 21, torch.bfloat16, True), (4096, 9, 21, torch.bfloat16, False),
                                              (4096, 8, 11, torch.bfloat16, True), (4096, 9, 11, torch.bfloat16, False)])
def test_which_backward_calls_the_matrix_cores_serve(T, n, K, wdt, served):
    x, cu, w, _, dy = _case([T // n] * (n - 1) + [T - T // n * (n - 1)], 256, K, T + n)
    xd, cud, wd, dyd = x.to(DEV), cu.to(DEV), w.to(DEV).to(wdt), dy.to(DEV)
    got = npa.varlen_dwconv_bwd(xd, dyd, cud, wd)
    want = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=_lib.Tuning(algo=4 if served else 3))
    assert all(torch.equal(a, c) for a, c in zip(got, want))
    assert torch.equal(npa.varlen_dwconv_bwd(xd, dyd, cud, wd, need_dw=False)[0],
                       npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=_lib.Tuning(algo=1))[0])


# (rows of 128-byte lines or not; outputs below and above the sizes from which the others take over: forward 200 MiB, backward 270)
@pytest.mark.parametrize("bwd,T,C,K,offset,served", [
    (False, 105984, 1000, 15, 0, False), (False, 104000, 1000, 15, 0, True), (False, 102400, 1024, 11, 0, True), (False, 105984, 1000, 21, 0, True),
    (False, 180224, 584, 11, 0, True), (False, 102400, 1024, 11, 16, False), (False, 16384, 1000, 31, 0, True), (False, 15700, 1000, 31, 0, True),
    (True, 141824, 1000, 15, 0, False), (True, 141000, 1000, 15, 0, True), (True, 138240, 1024, 15, 0, True), (True, 141824, 1000, 31, 0, True),
    (True, 141824, 1000, 21, 0, True), (True, 138240, 1024, 15, 8, False)])
def test_which_rows_of_partial_cache_lines_the_matrix_cores_serve(bwd, T, C, K, offset, served):
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(T)
    x, dy = (torch.empty(T, C, device=DEV, dtype=torch.bfloat16).normal_(generator=g) for _ in range(2))
    w = torch.empty(C, K, device=DEV, dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g)
    cu = cu_from_lengths(torch.tensor([T])).to(DEV)
    out = torch.empty(T * C + offset, device=DEV, dtype=torch.bfloat16)[offset:].view(T, C)       # (allocations begin on a line)
    st = torch.cuda.current_stream().cuda_stream
    if not bwd:
        _lib.check(lib.nplm_dwconv_fwd(x.data_ptr(), cu.data_ptr(), w.data_ptr(), None, out.data_ptr(), T, C, K, 1, _lib.BF16, _lib.BF16, st), "fwd")
        assert torch.equal(out, npa.varlen_dwconv_fwd(x, cu, w, None, tuning=_lib.Tuning(algo=4 if served else 2)))
        return
    ws = torch.empty(int(lib.nplm_dwconv_bwd_workspace_bytes(T, C, K, _lib.BF16)), dtype=torch.uint8, device=DEV)
    dw, db = torch.empty(C, K, device=DEV), torch.empty(C, device=DEV)
    _lib.check(lib.nplm_dwconv_bwd(x.data_ptr(), dy.data_ptr(), cu.data_ptr(), w.data_ptr(), out.data_ptr(), dw.data_ptr(), db.data_ptr(),
                                   ws.data_ptr(), ws.numel(), T, C, K, 1, _lib.BF16, _lib.BF16, st), "bwd")
    want = npa.varlen_dwconv_bwd(x, dy, cu, w, tuning=_lib.Tuning(algo=4 if served else 3))
    assert all(torch.equal(a, c) for a, c in zip((out, dw, db), want))


def _gated_algo(bwd, T, C, K, S):
    """4: matrix cores, 3: role-split."""
    return _lib.load().nplm_dwconv_debug_gated_algo(bwd, T, C, K, S, _lib.BF16, _lib.BF16)


@pytest.mark.parametrize("K,lens,C,algo", [
    (31, LENS * 2, 512, 4), (29, LENS[::-1] * 2, 520, 4), (25, [4096], 1000, 4), (31, [4095, 1, 63], 648, 4), (31, LENS * 4, 2056, 3), (31, LENS * 4, 2048, 4),
    (31, [1] * 4160, 512, 4), (31, [4095], 512, 4), (31, [16500] + [1] * 200, 512, 3),
    # both sides of the lines: 16384 rows, five to 63 rows a sequence in more than four tiles a block
    (31, [100] * 163 + [84], 512, 4), (31, [100] * 163 + [85], 512, 3), (31, [16] * 160, 2560, 4), (31, [16] * 210, 2560, 3), (31, [64] * 52, 2560, 4)])
def test_gated_backward_of_31_taps_matches_the_oracle(K, lens, C, algo):
    """dz comes from the matrix cores and dw from waves of 8 rows that leave out the products across a boundary (with short sequences in
    long batches, or in wide rows, from the role-split kernel): whole, partial and several column blocks, rows of one sequence and of
    many in a wave, and the same bits after a call that left NaN in LDS."""
    print(f"[case] gated K={K} C={C}", flush=True)
    _, cu, w, b, dy = _case(lens, C, K, C + K)
    assert _gated_algo(1, dy.shape[0], C, K, len(lens)) == algo
    z = torch.randn(dy.shape[0], 2 * C, generator=torch.Generator().manual_seed(C)).bfloat16()
    zd, cud, wd, dyd = z.to(DEV), cu.to(DEV), w.to(DEV), dy.to(DEV)
    for res in (False, True):
        _, dz64, dw64, db64 = O.ref_gated_dwconv_grads(z, cu, w, b, dy, torch.float64, res)
        got = npa.gated_dwconv_bwd(zd, dyd, cud, wd, residual=res)
        assert_act_close(got[0], dz64, torch.bfloat16, "dz")
        assert_red_close(got[1], dw64, "dw")
        assert_red_close(got[2], db64, "db")
    npa.gated_dwconv_bwd(torch.full_like(zd, float("nan")), torch.full_like(dyd, float("nan")), cud, wd, residual=True)
    again = npa.gated_dwconv_bwd(zd, dyd, cud, wd, residual=True)
    assert all(torch.equal(a, c) for a, c in zip(again, got))


@pytest.mark.parametrize("which", ["z", "dy"])
def test_gated_backward_non_finite_rows_stay_in_their_sequence(which):
    """Rows of one-row sequences reach the centre tap (and, from dy, db) only; rows of other sequences keep their dz."""
    C, K, lens = 512, 31, [40, 1, 700, 1, 213, 64, 1, 33, 1, 1500, 1, 1700]
    _, cu, w, _, dy = _case(lens, C, K, 3)
    z = torch.randn(dy.shape[0], 2 * C, generator=torch.Generator().manual_seed(5)).bfloat16()
    bad = torch.zeros(dy.shape[0], dtype=torch.bool)
    for i, n in enumerate(lens):
        if n == 1:
            bad[cu[i]] = True
    cud, wd = cu.to(DEV), w.to(DEV)
    dz0, dw0, db0 = npa.gated_dwconv_bwd(z.to(DEV), dy.to(DEV), cud, wd)
    t = z if which == "z" else dy
    t[bad, ::3] = float("inf")
    dz, dw, db = npa.gated_dwconv_bwd(z.to(DEV), dy.to(DEV), cud, wd)
    assert torch.equal(dz[~bad.to(DEV)], dz0[~bad.to(DEV)])
    hit = torch.zeros(C, K, dtype=torch.bool, device=DEV)
    hit[0::3 if which == "dy" else 1, K // 2] = True
    if which == "z":                                                  # (u's columns 0, 3, ...; g's from where C leaves off)
        hit[:, K // 2] = ((torch.arange(C) % 3 == 0) | ((torch.arange(C) + C) % 3 == 0)).to(DEV)
    assert not bool(torch.isfinite(dw[hit]).any()) and bool(torch.isfinite(dw[~hit]).all())
    torch.testing.assert_close(dw[~hit], dw0[~hit], rtol=0, atol=1e-5 * float(dw0.abs().max()))
    keep = torch.ones(C, dtype=torch.bool, device=DEV)
    if which == "dy":
        keep[0::3] = False
    assert not bool(torch.isfinite(db[~keep]).any())
    torch.testing.assert_close(db[keep], db0[keep], rtol=0, atol=1e-5 * float(db0.abs().max()))


@pytest.mark.parametrize("K", [11, 15, 21, 31])
@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_what_non_finite_rows_do_not_feed_keeps_its_bits(K, seed):
    """Inf and NaN in single rows (in front of, between and behind boundaries, in tiles without one) and in whole short sequences:
    every y, dx, dw and db that no such value belongs to has the bits of the call without them, the others are not finite."""
    x, cu, w, b, dy = _case(LENS[seed:] + LENS * 2, 512, K, 31 * K + seed)
    T, P = x.shape[0], (K - 1) // 2
    seq = torch.searchsorted(cu.long(), torch.arange(T), right=True)
    bad = torch.zeros(T, 512, dtype=torch.bool)
    g = torch.Generator().manual_seed(seed)
    bad[torch.randint(T, (40,), generator=g), torch.randint(512, (40,), generator=g)] = True
    for i in range(0, cu.numel() - 1, 7):
        if cu[i + 1] - cu[i] < 10:
            bad[cu[i]:cu[i + 1], i % 5::5] = True
    value = torch.where(torch.arange(512) % 3 == 0, float("nan"), float("inf")).bfloat16().expand(T, 512)
    reach, tap = torch.zeros_like(bad), torch.zeros(512, K, dtype=torch.bool)      # outputs a bad row belongs to; (x[t], dy[t + P - k])
    for k in range(K):
        d = k - P
        o, i = slice(max(0, -d), T - max(0, d)), slice(max(0, d), T - max(0, -d))
        reach[o] |= bad[i] & (seq[o] == seq[i])[:, None]
    cud, wd, bd = cu.to(DEV), w.to(DEV), b.to(DEV)
    tn = _lib.Tuning(**MFMA)
    same = lambda got, ref, hit: torch.equal(got[~hit], ref[~hit]) and not bool(torch.isfinite(got[hit]).any())
    xb, dyb = torch.where(bad, value, x), torch.where(bad, value, dy)
    for res in (False, True):
        y0, y = (npa.varlen_dwconv_fwd(t.to(DEV), cud, wd, bd, residual=res, tuning=tn) for t in (x, xb))
        assert same(y, y0, reach.to(DEV))
        dx0, dw0, db0 = npa.varlen_dwconv_bwd(x.to(DEV), dy.to(DEV), cud, wd, residual=res, tuning=tn)
        for which in ("x", "dy"):
            dx, dw, db = npa.varlen_dwconv_bwd((xb if which == "x" else x).to(DEV), (dyb if which == "dy" else dy).to(DEV), cud, wd,
                                               residual=res, tuning=tn)
            tap.zero_()
            for k in range(K):              # dw[k] sums dy[t] * x[t + k - P]
                d = k - P
                o, i = slice(max(0, -d), T - max(0, d)), slice(max(0, d), T - max(0, -d))
                tap[:, k] = (bad[i if which == "x" else o] & (seq[o] == seq[i])[:, None]).any(0)
            assert same(dw, dw0, tap.to(DEV))
            assert torch.equal(dx, dx0) if which == "x" else same(dx, dx0, reach.to(DEV))
            assert torch.equal(db, db0) if which == "x" else same(db, db0, bad.any(0).to(DEV))


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_what_non_finite_rows_do_not_feed_keeps_its_bits_gated(seed):
    C, K, lens = 512, 31, LENS + [1500, 3, 40, 1, 1, 700]
    _, cu, w, _, dy = _case(lens, C, K, 100 + seed)
    T = dy.shape[0]
    assert T >= 4096
    g = torch.Generator().manual_seed(seed)
    z = torch.randn(T, 2 * C, generator=g).bfloat16()
    bad = torch.zeros(T, C, dtype=torch.bool)
    bad[torch.randint(T, (30,), generator=g), torch.randint(C, (30,), generator=g)] = True
    seq = torch.searchsorted(cu.long(), torch.arange(T), right=True)
    reach, tap = torch.zeros_like(bad), torch.zeros(C, K, dtype=torch.bool)
    for k in range(K):
        d = k - K // 2
        o, i = slice(max(0, -d), T - max(0, d)), slice(max(0, d), T - max(0, -d))
        reach[o] |= bad[i] & (seq[o] == seq[i])[:, None]
        tap[:, k] = (bad[o] & (seq[o] == seq[i])[:, None]).any(0)
    cud, wd = cu.to(DEV), w.to(DEV)
    dz0, dw0, db0 = npa.gated_dwconv_bwd(z.to(DEV), dy.to(DEV), cud, wd)
    dz, dw, db = npa.gated_dwconv_bwd(z.to(DEV), dy.masked_fill(bad, float("inf")).to(DEV), cud, wd)
    for half in (slice(0, C), slice(C, None)):
        keep = ~reach.to(DEV)
        assert torch.equal(dz[:, half][keep], dz0[:, half][keep])
    assert not bool(torch.isfinite(dz[:, :C][reach.to(DEV)]).any())
    assert torch.equal(dw[~tap.to(DEV)], dw0[~tap.to(DEV)]) and not bool(torch.isfinite(dw[tap.to(DEV)]).any())
    col = bad.any(0).to(DEV)
    assert torch.equal(db[~col], db0[~col]) and not bool(torch.isfinite(db[col]).any())


@pytest.mark.parametrize("K", [11, 15, 21, 31])
def test_a_non_finite_weight_meets_the_rows_of_its_tap_only(K):
    """Weights of Inf and NaN at one tap of every fifth channel, sequences of one row and a few among them: outputs whose sequence
    has no row at that tap are those of a zero weight, bit for bit. Forward, dx and the gated dz."""
    lens = [1] * 300 + LENS + [1, 2, 3, 1, 4, 1, 1, 5] * 40 + [500, 1, 1, 900, 2, 460]
    C = 512
    x, cu, w, b, dy = _case(lens, C, K, K)
    T = x.shape[0]
    assert T >= 4096
    odd = w.clone()
    for c in range(0, C, 5):
        odd[c, c // 5 % K] = float("nan") if c % 2 else float("inf")
    seq = torch.searchsorted(cu.long(), torch.arange(T), right=True)
    fwd, bwd = torch.zeros(T, C, dtype=torch.bool), torch.zeros(T, C, dtype=torch.bool)      # outputs that such a weight belongs to
    for k in range(K):
        d = k - K // 2
        o, i = slice(max(0, -d), T - max(0, d)), slice(max(0, d), T - max(0, -d))
        both = (seq[o] == seq[i])[:, None] & ~torch.isfinite(odd[:, k])
        fwd[o] |= both              # y[t] takes w[k] from x[t + d], dx[t + d] takes it from dy[t]
        bwd[i] |= both
    zeros = torch.where(torch.isfinite(odd), odd, 0.0)
    xd, dyd, cud, od, zd, bd, fwd, bwd = (t.to(DEV) for t in (x, dy, cu, odd, zeros, b, fwd, bwd))
    tn = _lib.Tuning(**MFMA)
    g = torch.randn(T, 2 * C, generator=torch.Generator().manual_seed(K)).bfloat16().to(DEV)
    for res in (False, True):
        y, y0 = (npa.varlen_dwconv_fwd(xd, cud, v, bd, residual=res, tuning=tn) for v in (od, zd))
        (dx, dw, db), (dx0, dw0, db0) = (npa.varlen_dwconv_bwd(xd, dyd, cud, v, residual=res, tuning=tn) for v in (od, zd))
        for got, want, hit in ((y, y0, fwd), (dx, dx0, bwd)):
            assert torch.equal(got[~hit], want[~hit]) and not bool(torch.isfinite(got[hit]).any())
        assert torch.equal(dw, dw0) and torch.equal(db, db0)
        if K == 31:
            dz, dz0 = (npa.gated_dwconv_bwd(g, dyd, cud, v, residual=res)[0] for v in (od, zd))
            assert torch.equal(dz[:, :C][~bwd], dz0[:, :C][~bwd]) and torch.equal(dz[:, C:][~bwd], dz0[:, C:][~bwd])
            assert not bool(torch.isfinite(dz[:, :C][bwd]).any())


@pytest.mark.parametrize("K,C", [(15, 512), (31, 264)])
@pytest.mark.parametrize("seq_len,nbt", [(64, 0), (96, 24), (17, 10), (512, 7)])
def test_equal_length_sequences_on_rotating_tile_slots(K, C, seq_len, nbt):
    """Boundaries at a fixed period of tiles, grids whose last round is partial, empty sequences behind the last row."""
    T = 2700
    x, cu, w, b, dy = _case([seq_len] * (T // seq_len) + [T % seq_len] + [0] * 300, C, K, K + seq_len)
    xd, cud, wd, dyd = x.to(DEV), cu.to(DEV), w.to(DEV), dy.to(DEV)
    tn = _lib.Tuning(nbt=nbt, **MFMA)
    assert_act_close(npa.varlen_dwconv_fwd(xd, cud, wd, b.to(DEV), tuning=tn), O.c_oracle_fwd(x, cu, w, b), torch.bfloat16, "y")
    dx64, dw64, db64 = O.c_oracle_bwd(x, dy, cu, w)
    dx, dw, db = npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=tn)
    assert_act_close(dx, dx64, torch.bfloat16, "dx")
    assert_red_close(dw, dw64, "dw")
    assert_red_close(db, db64, "db")


def test_empty_sequences_do_not_change_the_bits():
    """In front of the rows, between sequences and behind them, thousands at a time: the kernels mark the same starts."""
    x, cu, w, b, dy = _case(LENS * 2, 512, 31, 8)
    lens = []
    for i, n in enumerate(LENS * 2):
        lens += [n] + [0] * (3000 if i in (0, 7, 40) else i % 3)
    many = cu_from_lengths(torch.tensor([0] * 5000 + lens + [0] * 20000))
    xd, wd, bd, dyd, tn = x.to(DEV), w.to(DEV), b.to(DEV), dy.to(DEV), _lib.Tuning(**MFMA)
    assert torch.equal(npa.varlen_dwconv_fwd(xd, cu.to(DEV), wd, bd, tuning=tn), npa.varlen_dwconv_fwd(xd, many.to(DEV), wd, bd, tuning=tn))
    one, two = (npa.varlen_dwconv_bwd(xd, dyd, c.to(DEV), wd, tuning=tn) for c in (cu, many))
    assert all(torch.equal(a, c) for a, c in zip(one, two))


def test_rows_beyond_2_and_4_gib_offsets():
    """1.1 M rows x 4 KiB: row offsets cross 2^31 and 2^32 bytes. Whole sequences cut out of the batch give the same y and dx alone:
    their first row is a multiple of four, which is what the order of a row's sums goes by."""
    T, C, K = 1_100_000, 2048, 31
    g = torch.Generator().manual_seed(78)
    lens = 4 * torch.randint(5, 129, (T // 200,), generator=g)
    lens = lens[torch.cumsum(lens, 0) <= T]
    cu = cu_from_lengths(torch.cat([lens, torch.tensor([T - int(lens.sum())])])).to(DEV)
    x, dy = (torch.randn(T, C, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    w = (torch.randn(C, K, device=DEV) * K ** -0.5).bfloat16()
    tn = _lib.Tuning(**MFMA)
    y = npa.varlen_dwconv_fwd(x, cu, w, None)
    dx, _, db = npa.varlen_dwconv_bwd(x, dy, cu, w)
    cul = cu.tolist()
    S = len(cul) - 1
    assert cul[S // 2] * C * 2 > 2 ** 31 and cul[S - 40] * C * 2 > 2 ** 32
    for first in (0, S // 2 - 20, S - 40):
        s, e = cul[first], cul[first + 40]
        sub = (cu[first:first + 41] - s).contiguous()
        assert torch.equal(y[s:e], npa.varlen_dwconv_fwd(x[s:e], sub, w, None, tuning=tn)), f"rows {s}..{e}"
        assert torch.equal(dx[s:e], npa.varlen_dwconv_bwd(x[s:e], dy[s:e], sub, w, tuning=tn)[0]), f"rows {s}..{e}"
    torch.testing.assert_close(db, dy.float().sum(0), rtol=2e-5, atol=0.05)


@pytest.mark.parametrize("K", [11, 31])
def test_share_of_outputs_that_are_not_correctly_rounded(K):
    """fp32 sums of K exact products are off by up to K 2^-24 of the products' absolute sum, about sqrt(K) times an output, and land on
    the other side of a rounding boundary of bf16 (one every 2^-8 of the value) once in about 2^8 * sqrt(K) * sqrt(K) 2^-24 outputs, with errors that
    add at random: 1.7e-4 at 11 taps, 4.7e-4 at 31 as a bound; not more than a few times the share of the vector kernels."""
    x, cu, w, b, dy = _case([5000, 300, 12000, 64] + LENS, 512, K, K)
    xd, dyd, cud, wd, bd = (t.to(DEV) for t in (x, dy, cu, w, b))
    want = (O.c_oracle_fwd(x, cu, w, b).bfloat16(), O.c_oracle_bwd(x, dy, cu, w)[0].bfloat16())
    for name, f, ref in (("y", lambda t: npa.varlen_dwconv_fwd(xd, cud, wd, bd, tuning=t), want[0]),
                         ("dx", lambda t: npa.varlen_dwconv_bwd(xd, dyd, cud, wd, tuning=t)[0], want[1])):
        share = [float((f(_lib.Tuning(algo=a)).cpu() != ref).double().mean()) for a in (4, 1)]
        print(f"[share] K={K} {name}: matrix cores {share[0]:.2e}, vector {share[1]:.2e}", flush=True)
        assert share[0] <= K * 2.0 ** -16 and share[0] <= 2 * share[1] + 2e-6


# (built as 15 and 31 taps; whole, partial and several column blocks; one run a block, and with C=8200 two; runs that end inside a
# step; a boundary at every row of the 32-row groups, one to many in a group; some calls that the role-split kernel keeps)
@pytest.mark.parametrize("K,lens,C,algo", [
    (31, LENS * 2, 512, 4), (29, LENS[::-1] * 2, 520, 4), (25, [4096], 1000, 4), (31, [95] * 44, 520, 4), (31, [191] * 22, 8200, 4),
    (15, LENS * 2, 776, 3), (13, [63] * 66, 1160, 3), (21, [4095, 1], 512, 4), (11, [2500, 1, 1700], 520, 4), (31, [1] * 4100, 512, 4),
    (15, [17] * 260, 512, 3), (15, [17] * 120, 512, 4), (13, [63] * 32, 1160, 3), (11, [1] * 1900, 512, 4),
    (15, LENS[:30], 776, 4), (13, [63] * 32, 1000, 4), (15, [63] * 10 + [1500, 2, 3, 1700, 1, 700], 776, 4), (15, [3] * 600, 1160, 4),
    (21, [95] * 21, 2048, 4), (17, [31] * 60, 1544, 4)])
def test_gated_forward_on_the_matrix_cores_matches_the_oracle(K, lens, C, algo):
    """To one bf16 rounding of the oracle's y: the three bf16 terms add up to the fp32 h. The same bits again after a call that left NaN
    in the LDS; rows in front of and behind y keep theirs."""
    print(f"[case] gated forward K={K} C={C}", flush=True)
    _, cu, w, b, dy = _case(lens, C, K, C + K)
    T = dy.shape[0]
    assert _gated_algo(0, T, C, K, len(lens)) == algo
    z = torch.randn(T, 2 * C, generator=torch.Generator().manual_seed(C)).bfloat16()
    zd, cud, wd, bd = z.to(DEV), cu.to(DEV), w.to(DEV), b.to(DEV)
    lib = _lib.load()
    for res in (False, True):
        y64 = O.ref_gated_dwconv_grads(z, cu, w, b, None, torch.float64, res)
        y = npa.gated_dwconv_fwd(zd, cud, wd, bd, residual=res)
        assert_act_close(y, y64, torch.bfloat16, "y")
        npa.gated_dwconv_fwd(torch.full_like(zd, float("nan")), cud, wd, bd, residual=res)
        room = torch.full((T + 4, C), 7.0, dtype=torch.bfloat16, device=DEV)
        _lib.check(lib.nplm_dwconv_gated_fwd(zd.data_ptr(), cud.data_ptr(), wd.data_ptr(), bd.data_ptr(), room[2:].data_ptr(), T, C, K,
                                             len(lens), _lib.BF16, _lib.BF16, _lib.RESIDUAL if res else 0,
                                             torch.cuda.current_stream().cuda_stream), "gated_fwd")
        assert torch.equal(room[2:T + 2], y) and bool((room[:2] == 7).all()) and bool((room[T + 2:] == 7).all())


@pytest.mark.parametrize("K", [15, 31])
@pytest.mark.parametrize("where", ["u", "gate", "weight"])
def test_gated_forward_non_finite_values_reach_the_rows_of_their_taps_only(K, where):
    """Against the vector ALU's kernel (which takes the same weights in fp32): the same outputs are not finite, in the same way, and
    the others differ by a rounding; rows of other sequences keep the bits of a clean call."""
    C, lens = 512, [40, 1, 700, 1, 213, 64, 1, 33, 2, 1500, 1, 1700]
    _, cu, w, b, dy = _case(lens, C, K, 3)
    z = torch.randn(dy.shape[0], 2 * C, generator=torch.Generator().manual_seed(5)).bfloat16()
    cud, bd = cu.to(DEV), b.to(DEV)
    clean = npa.gated_dwconv_fwd(z.to(DEV), cud, w.to(DEV), bd)
    hit = torch.zeros(dy.shape[0], dtype=torch.bool)
    if where == "weight":
        w[5::7, K // 2 - 3], w[6::7, K // 2] = float("inf"), float("nan")
    else:
        off = 0 if where == "u" else C
        for i, n in enumerate(lens):
            if n <= 2:
                hit[cu[i]:cu[i + 1]] = True
                z[cu[i], off + i % 7:off + C:7] = float("nan") if i % 2 else float("inf")
        z[1700:1701, off:off + C:5] = -float("inf")          # inside a long sequence
        hit[1055:2555] = True
    y = npa.gated_dwconv_fwd(z.to(DEV), cud, w.to(DEV), bd)
    want = npa.gated_dwconv_fwd(z.to(DEV), cud, w.to(DEV).float(), bd.float())
    assert not bool(torch.isfinite(want).all())
    torch.testing.assert_close(y, want, rtol=2.0 ** -7, atol=1e-5, equal_nan=True)
    if where != "weight":
        assert torch.equal(y[~hit.to(DEV)], clean[~hit.to(DEV)])


@pytest.mark.parametrize("K", [15, 31])
@pytest.mark.parametrize("what,h_exp,w_exp", [("small h", -100, 90), ("large h", 123, -90), ("small weights", 60, -103)])
@pytest.mark.parametrize("residual", [False, True])
def test_gated_forward_keeps_the_range_of_fp32(K, what, h_exp, w_exp, residual):
    """|h| from 2^-100 to 2^-135 and from 2^123 down, weights from 2^-103 to 2^-133, by channel; every seventh channel ordinary. A bf16
    term ends at 2^-133, fp32 does not. Boundaries in most windows and in none. To one bf16 rounding of y, the fp32 sums' noise and the last
    bits of a subnormal h or product; non-finite values among them reach what they reach on the vector ALU (which takes the same weights
    in fp32)."""
    C, lens = 520, LENS[:25] + [700, 1, 300]
    _, cu, w, _, dy = _case(lens, C, K, K)
    T = dy.shape[0]
    g = torch.Generator().manual_seed(K)
    ch = torch.arange(C, dtype=torch.float64)
    usual = ch % 7 == 3
    size = torch.where(usual, 1.0, 2.0 ** (h_exp - (0 if what == "small weights" else ch % 27)))
    z = torch.cat([torch.randn(T, C, generator=g) * size, torch.randn(T, C, generator=g)], 1).bfloat16()
    w = (w.double() * torch.where(usual, 1.0, 2.0 ** (w_exp - (ch % 27 if what == "small weights" else 0)))[:, None]).bfloat16()
    cud, wd = cu.to(DEV), w.to(DEV)
    ref, mass = (O.ref_gated_dwconv_grads(a, cu, b, None, None, torch.float64, residual)
                 for a, b in ((z.double(), w.double()), (z.double().abs(), w.double().abs())))
    y = npa.gated_dwconv_fwd(z.to(DEV), cud, wd, None, residual=residual).cpu().double()
    # (gate_mul() is off by up to 4 roundings, K sums by one each; an h or a product below 2^-126 by 2^-149)
    bound = ref.abs() * 2.0 ** -8 + (K + 8) * 2.0 ** -23 * mass + (w.double().abs().sum(1) + K) * 2.0 ** -148 + 2.0 ** -134
    assert bool(((y - ref).abs() <= bound).all()), float(((y - ref).abs() / bound).max())
    for where in ("z", "w"):
        zo, wo = z.clone(), w.clone()
        if where == "z":
            zo[500, 5::11], zo[2, 1::13], zo[900, 2::17] = float("inf"), float("nan"), -float("inf")
        else:
            wo[5::11, 2], wo[4::13, K // 2], wo[2::17, K - 1] = float("inf"), float("nan"), -float("inf")
        got = npa.gated_dwconv_fwd(zo.to(DEV), cud, wo.to(DEV), None, residual=residual)
        want = npa.gated_dwconv_fwd(zo.to(DEV), cud, wo.to(DEV).float(), None, residual=residual)
        fin = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), fin) and not bool(fin.all())
        torch.testing.assert_close(got[~fin], want[~fin], rtol=0, atol=0, equal_nan=True)
        if where == "z":
            assert bool(((got.cpu().double() - ref).abs() <= bound)[fin.cpu()].all())


@pytest.mark.parametrize("K", [15, 21, 31])
@pytest.mark.parametrize("C", [512, 520])
def test_gated_calls_of_fewer_rows_than_a_tile_or_a_halo(K, C):
    """One sequence, and a boundary behind every third row; forward, and (31 taps on the matrix cores) backward. Rows around the outputs keep
    their values."""
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    for T in (1, 2, 15, 16, 31, 63, 64, 65, 129):
        for lens in ([T], [3] * (T // 3) + [T % 3]):
            _, cu, w, b, dy = _case(lens, C, K, C + K + T)
            z = torch.randn(T, 2 * C, generator=torch.Generator().manual_seed(T)).bfloat16()
            assert _gated_algo(0, T, C, K, len(lens)) == 4 and _gated_algo(1, T, C, K, len(lens)) == (4 if K == 31 else 3)
            y64, dz64, dw64, db64 = O.ref_gated_dwconv_grads(z, cu, w, b, dy, torch.float64)
            zd, cud, wd, bd, dyd = (t.to(DEV) for t in (z, cu, w, b, dy))
            y, dz = (torch.full((T + 4, n), 7.0, dtype=torch.bfloat16, device=DEV) for n in (C, 2 * C))
            dw, db = torch.full((C + 2, K), 7.0, device=DEV), torch.full((C + 2,), 7.0, device=DEV)
            ws = torch.empty(int(lib.nplm_dwconv_gated_bwd_workspace_bytes(T, C, K, _lib.BF16)), dtype=torch.uint8, device=DEV)
            sizes = (T, C, K, len(lens), _lib.BF16, _lib.BF16, 0, st)
            _lib.check(lib.nplm_dwconv_gated_fwd(zd.data_ptr(), cud.data_ptr(), wd.data_ptr(), bd.data_ptr(), y[2:].data_ptr(), *sizes), "fwd")
            _lib.check(lib.nplm_dwconv_gated_bwd(zd.data_ptr(), dyd.data_ptr(), cud.data_ptr(), wd.data_ptr(), dz[2:].data_ptr(), dw[1:].data_ptr(),
                                                 db[1:].data_ptr(), ws.data_ptr(), ws.numel(), *sizes), "bwd")
            assert_act_close(y[2:-2], y64, torch.bfloat16, f"y T={T}")
            assert_act_close(dz[2:-2], dz64, torch.bfloat16, f"dz T={T}")
            assert_red_close(dw[1:-1], dw64, f"dw T={T}")
            assert_red_close(db[1:-1], db64, f"db T={T}")
            for t, n in ((y, 2), (dz, 2), (dw, 1), (db, 1)):
                assert bool((t[:n] == 7).all()) and bool((t[-n:] == 7).all())


# runs of the gated forward: T, C -> steps a run, runs and slots: (16347, 2176) 9, 29 on 15 (a slot without a run in the last round), the last run
# cut inside a step; (65500, 768) 13, 79 on 42; (131072, 2048) 16, 128 on 16
@pytest.mark.parametrize("K,T,C", [(15, 16347, 2176), (31, 16347, 2176), (31, 65500, 768), (31, 131072, 2048)])
def test_gated_forward_in_several_runs_a_block(K, T, C):
    """Boundaries at a run's first rows, in front of and behind them (a run of 9 steps begins every 576 rows, of 13 every 832, of 16 every 1024);
    a few channels of every column block against the oracle, all against the role-split kernel (which takes the same weights in fp32)."""
    run = {16347: 576, 65500: 832, 131072: 1024}[T]
    starts = sorted({run * i + d for i in range(1, T // run + 1) for d in ((0,), (1,), (-1,), (0, 3), (-2, 2), (15,), (-15, 31))[i % 7] if i % 3})
    cu = torch.tensor([0] + [t for t in starts if t < T] + [T], dtype=torch.int32)
    S = cu.numel() - 1
    assert _gated_algo(0, T, C, K, S) == 4
    g = torch.Generator(device=DEV).manual_seed(T)
    z = torch.empty(T, 2 * C, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(C, K, device=DEV, dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g)
    b = torch.empty(C, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    y = npa.gated_dwconv_fwd(z, cu.to(DEV), w, b)
    torch.testing.assert_close(y, npa.gated_dwconv_fwd(z, cu.to(DEV), w.float(), b.float()), rtol=2.0 ** -7, atol=1e-5)
    ch = torch.arange(37, C, 128, device=DEV)
    want = O.ref_gated_dwconv_grads(z[:, torch.cat([ch, ch + C])].cpu(), cu, w[ch].cpu(), b[ch].cpu(), None, torch.float64)
    assert_act_close(y[:, ch], want, torch.bfloat16, "y")


def test_gated_forward_rows_beyond_2_and_4_gib_offsets():
    """1.2 M rows of z of 4 KiB: whole sequences cut out of the batch give the same y alone (their first row is a multiple of four, which is
    what the order of a row's sums goes by)."""
    T, C, K = 1_200_000, 1024, 31
    g = torch.Generator().manual_seed(79)
    lens = 4 * torch.randint(5, 129, (T // 200,), generator=g)
    lens = lens[torch.cumsum(lens, 0) <= T]
    cu = cu_from_lengths(torch.cat([lens, torch.tensor([T - int(lens.sum())])])).to(DEV)
    z = torch.randn(T, 2 * C, device=DEV, dtype=torch.bfloat16)
    w = (torch.randn(C, K, device=DEV) * K ** -0.5).bfloat16()
    cul = cu.tolist()
    S = len(cul) - 1
    assert _gated_algo(0, T, C, K, S) == 4
    y = npa.gated_dwconv_fwd(z, cu, w, None, residual=True)
    assert cul[S // 2] * C * 4 > 2 ** 31 and cul[S - 40] * C * 4 > 2 ** 32
    for first in (0, S // 2 - 20, S - 40):
        s, e = cul[first], cul[first + 40]
        sub = (cu[first:first + 41] - s).contiguous()
        assert _gated_algo(0, e - s, C, K, 40) == 4
        assert torch.equal(y[s:e], npa.gated_dwconv_fwd(z[s:e], sub, w, None, residual=True)), f"rows {s}..{e}"


@pytest.mark.parametrize("K,Kx,lens,same", [(11, 15, [17] * 120, True), (11, 15, [200] * 12, True), (21, 31, [300] * 10, True),
                                            (21, 31, [20] * 300, False), (17, 31, [20] * 300, False)])
def test_gated_taps_padded_to_the_planned_size(K, Kx, lens, same):
    """The same bits where both sizes take the same kernels; 17 to 21 taps and 31 part where short sequences keep the smaller one on the
    role-split kernel, and in the backward: there to the two roundings of one sum."""
    C = 512
    _, cu, w, b, dy = _case(lens, C, K, K)
    z = torch.randn(dy.shape[0], 2 * C, generator=torch.Generator().manual_seed(K)).bfloat16().to(DEV)
    wide = torch.nn.functional.pad(w, ((Kx - K) // 2,) * 2).contiguous().to(DEV)
    cu, w, b, dy = (t.to(DEV) for t in (cu, w, b, dy))
    assert (_gated_algo(0, dy.shape[0], C, K, len(lens)) == _gated_algo(0, dy.shape[0], C, Kx, len(lens))) == same
    y, yx = npa.gated_dwconv_fwd(z, cu, w, b), npa.gated_dwconv_fwd(z, cu, wide, b)
    assert torch.equal(y, yx) or not same
    torch.testing.assert_close(y, yx, rtol=2.0 ** -7, atol=1e-5)
    bwd = [npa.gated_dwconv_bwd(z, dy, cu, v) for v in (w, wide)]
    equal = _gated_algo(1, dy.shape[0], C, K, len(lens)) == _gated_algo(1, dy.shape[0], C, Kx, len(lens))
    assert equal == (Kx == 15)
    assert torch.equal(bwd[0][0], bwd[1][0]) or not equal
    torch.testing.assert_close(bwd[0][0], bwd[1][0], rtol=2.0 ** -7, atol=1e-5)
