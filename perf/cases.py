"""The work that users of nanoplm_amd have it do, as cases that can be timed.

A case is one call of a public door of the library - ``VarlenDWConv1d`` called on packed rows, ``forward_gated``,
``forward_prenorm``, ``forward_padded`` - either alone (``train`` false: inference, no gradients) or with the gradients of
everything a training step needs (``train`` true). Sizes are those of the repository's five benchmark configurations, of
the default widths of the model the conv sits in (hidden 768 and 1024, intermediate 1152 and 2048) and generic ragged ones.

Fields: ``form`` plain | gated | ln | padded; ``T`` packed rows; ``C`` channels; ``K`` kernel size; ``act`` / ``par`` the
dtypes of activations and parameters (bf16 | fp32; they differ under autocast); ``mix`` the length distribution;
``residual``; ``static`` whether cu_seqlens is the static collator's fixed-length tensor; ``train``.
"""
import math

import torch
from torch import nn

import nanoplm_amd as npa
from nanoplm_amd.workloads import cu_from_lengths, draw_lengths, static_packed_cu

DEV = "cuda"
_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp32": 4}
# length distributions of nanoplm_amd.workloads, by what the packed batch holds
_MIX = {"short": "n8_u20_128", "usual": "u20_512", "skewed": "lognormal", "stress": "stress"}


def _case(name, form, T, C, K, act, par, mix, train, residual=False, static=False):
    return dict(name=name, form=form, T=T, C=C, K=K, act=act, par=par, mix=mix, train=train, residual=residual, static=static)


def listed():
    return [
        # one small batch through a narrow layer: the latency of a call (configuration 1's shape)
        _case("single_call_small", "plain", 776, 64, 3, "fp32", "fp32", "short", False),
        # a small micro-batch of a fine-tuning loop, forward and backward: launches and host work of a training step
        _case("train_small", "plain", 2048, 768, 7, "bf16", "bf16", "usual", True, residual=True),
        # embedding a padded batch of 32 proteins of up to 512 residues at hidden 768
        _case("embed_padded", "padded", 32 * 512, 768, 7, "bf16", "bf16", "usual", False, residual=True),
        # inference on one packed batch (configuration 2)
        _case("forward_packed", "plain", 32768, 1024, 7, "bf16", "bf16", "usual", False),
        # the headline training step (configuration 3)
        _case("train_headline", "plain", 131072, 1024, 7, "bf16", "bf16", "usual", True),
        # many sequences shorter than the kernel's radius (configuration 5)
        _case("train_stress", "plain", 65536, 1024, 7, "bf16", "bf16", "stress", True),
        # the intermediate width with the long kernel (configuration 4)
        _case("train_wide_k31", "plain", 131072, 2048, 31, "bf16", "bf16", "skewed", True),
        # the same conv inside the SwiGLU MLP, gate product fused in
        _case("train_gated_k31", "gated", 131072, 2048, 31, "bf16", "bf16", "skewed", True),
        # the MLP conv at the default intermediate width under autocast: bf16 activations, fp32 parameters
        _case("train_gated_autocast", "gated", 65536, 1152, 7, "bf16", "fp32", "usual", True),
        # pre-norm fused in, on the fp32 residual stream that autocast leaves, hidden 768
        _case("train_prenorm_fp32", "ln", 65536, 768, 7, "fp32", "fp32", "usual", True, residual=True),
        # pre-norm fused in, all bf16, hidden 1024
        _case("train_prenorm_bf16", "ln", 131072, 1024, 7, "bf16", "bf16", "usual", True, residual=True),
        # a ragged batch of the static-shape collator with a kernel size between the built ones, autocast dtypes
        _case("train_ragged_k11", "plain", 50021, 1000, 11, "bf16", "fp32", "usual", True, static=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["plain", "plain", "plain", "plain", "gated", "gated", "ln", "ln", "padded"])
    T = _log(rng, 600, 131072)
    act, par = rng.choice([("bf16", "bf16"), ("bf16", "bf16"), ("bf16", "fp32"), ("fp32", "fp32")])
    mix = rng.choice(["usual", "usual", "skewed", "stress", "short"])
    train = rng.random() < 0.65
    residual = rng.random() < 0.5
    static = form != "padded" and rng.random() < 0.25
    if form == "ln":            # the pre-norm door: hidden widths, the kernel sizes it is built for
        C, K = rng.choice([512, 640, 768, 896, 1000, 1024]), rng.choice([3, 5, 7, 7, 9])
    elif form == "gated":       # the MLP: intermediate widths
        C, K = rng.choice([768, 1024, 1152, 1536, 2048]), rng.choice([3, 5, 7, 9, 15, 31])
        residual = False
    elif form == "padded":
        C, K = rng.choice([512, 768, 1024]), rng.choice([3, 7, 9])
        T = max(2, T // 512) * 512
        train, mix = False, "usual"
    else:
        C, K = rng.choice([64, 320, 512, 768, 1000, 1024, 1152, 2048]), rng.choice([3, 5, 7, 7, 9, 11, 15, 21, 31])
    size = _BYTES[act] * (2 if form == "gated" else 1)
    T = min(T, 131072 * 2048 * 4 // (C * size))          # no larger than the largest listed case
    if form == "padded":
        T = T // 512 * 512
    return {k: v for k, v in _case("", form, T, C, K, act, par, mix, train, residual, static).items() if k != "name"}


def prepare(case, seed):
    c = dict(case)
    T, C, K, act, par = c["T"], c["C"], c["K"], _DT[c["act"]], _DT[c["par"]]
    cpu = torch.Generator().manual_seed(seed)
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape, dtype, std=1.0):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)

    s = dict(case=c)
    if c["form"] == "padded":   # right-padded batch [B, L, C] with its attention mask
        B, L = T // 512, 512
        lens = torch.randint(20, L + 1, (B,), generator=cpu)
        s["mask"] = (torch.arange(L)[None, :] < lens[:, None]).to(torch.int64).to(DEV)
    elif c["static"]:           # the last tenth of the rows is padding; entries up to a fixed length follow
        real = cu_from_lengths(draw_lengths(_MIX[c["mix"]], T - T // 10, cpu))
        s["cu"] = static_packed_cu(real, T, 512, cu_len=real.numel() + T // 5120 + 16).to(DEV)
    else:
        s["cu"] = cu_from_lengths(draw_lengths(_MIX[c["mix"]], T, cpu)).to(DEV)
    conv = npa.VarlenDWConv1d(C, K, residual=c["residual"], device=DEV, dtype=par)
    with torch.no_grad():
        conv.weight.normal_(0.0, K ** -0.5, generator=g)
        conv.bias.normal_(0.0, 0.02, generator=g)
    params = [conv.weight, conv.bias]
    if c["form"] == "ln":
        norm = nn.LayerNorm(C, device=DEV, dtype=par)
        with torch.no_grad():
            norm.weight.normal_(1.0, 0.1, generator=g)
            norm.bias.normal_(0.0, 0.1, generator=g)
        s["norm"] = norm
        params += [norm.weight, norm.bias]
    width = 2 * C if c["form"] == "gated" else C
    shape = (T // 512, 512, C) if c["form"] == "padded" else (T, width)
    x = normal(*shape, dtype=act).requires_grad_(c["train"])
    s.update(conv=conv, x=x, wanted=[x] + params)
    if c["train"]:
        s["dy"] = normal(T, C, dtype=act)
    return s


def _forward(s):
    form, conv = s["case"]["form"], s["conv"]
    if form == "padded":
        return conv.forward_padded(s["x"], s["mask"])
    if form == "gated":
        return conv.forward_gated(s["x"], s["cu"])
    if form == "ln":
        return conv.forward_prenorm(s["x"], s["cu"], s["norm"])
    return conv(s["x"], s["cu"])


def run(s):
    if not s["case"]["train"]:
        with torch.no_grad():
            return _forward(s)
    y = _forward(s)
    return (y.detach(), *torch.autograd.grad(y, s["wanted"], s["dy"]))


def exact(case, seed):
    """The same outputs from plain torch in float64: one shifted product per tap, products across a boundary dropped."""
    s = prepare(case, seed)
    x, conv, K, res = s["x"], s["conv"], case["K"], case["residual"]
    leaves = [t.detach().double().requires_grad_(case["train"]) for t in s["wanted"]]
    X, W, B = leaves[0].reshape(-1, x.shape[-1]), leaves[1], leaves[2]
    T, P = X.shape[0], (K - 1) // 2
    rows = torch.arange(T, device=DEV)
    if case["form"] == "padded":
        row_in = torch.arange(512, device=DEV)[None, :]
        seq = 2 * torch.arange(T // 512, device=DEV)[:, None] + (row_in >= s["mask"].sum(1)[:, None])
        seq = seq.reshape(-1)
    else:
        seq = torch.searchsorted(s["cu"].long(), rows, right=True)
    if case["form"] == "ln":
        mean = X.mean(1, keepdim=True)
        h = (X - mean) * torch.rsqrt((X - mean).pow(2).mean(1, keepdim=True) + s["norm"].eps) * leaves[3] + leaves[4]
    elif case["form"] == "gated":
        h = X[:, :case["C"]] * X[:, case["C"]:] * torch.sigmoid(X[:, case["C"]:])
    else:
        h = X
    valid = [None] * K
    y = torch.zeros_like(h.detach())

    def spans(d):               # output rows and input rows of the tap d rows away
        return slice(max(0, -d), T - max(0, d)), slice(max(0, d), T - max(0, -d))

    hd, wd = h.detach(), W.detach()
    for k in range(K):
        if abs(k - P) >= T:
            continue
        o, i = spans(k - P)
        valid[k] = (seq[o] == seq[i])[:, None]
        y[o] += torch.where(valid[k], hd[i] * wd[:, k], 0.0)
    y += B.detach()
    if res:
        y += X.detach()
    if not case["train"]:
        return y.reshape(*x.shape[:-1], case["C"])
    dy = s["dy"].double()
    dh, dw = torch.zeros_like(hd), torch.zeros_like(wd)
    for k in range(K):
        if valid[k] is None:
            continue
        o, i = spans(k - P)
        g = torch.where(valid[k], dy[o], 0.0)
        dh[i] += g * wd[:, k]
        dw[:, k] = (g * hd[i]).sum(0)
    dx, rest = dh, []
    if case["form"] in ("ln", "gated"):
        inner = [leaves[0]] + leaves[3:]
        dx, *rest = torch.autograd.grad(h, inner, dh)
    if res:
        dx = dx + dy
    return (y, dx, dw, dy.sum(0), *rest)


def work(case):
    """Bytes: every input read once and every output written once, in each direction (the backward reads x again). Operations:
    two per tap and element forward, four backward (dx and dw), one for db, and the gate's or the norm's few."""
    c = case
    T, C, K, e, ep = c["T"], c["C"], c["K"], _BYTES[c["act"]], _BYTES[c["par"]]
    n = T * C
    x = 2 * n if c["form"] == "gated" else n
    per = 3 + (1 if c["form"] == "ln" else 0)       # parameter rows: taps counted apart
    small = C * (K + per) * ep
    nbytes = (x + n) * e + small
    extra = {"gated": 6, "ln": 8}.get(c["form"], 0) + (1 if c["residual"] else 0)
    flops = (2 * K + extra) * n
    if c["train"]:
        nbytes += (2 * x + n) * e + 2 * small
        flops += (4 * K + 1 + 2 * extra) * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Against the same composition in float64 the outputs differ by 1.7e-3 (2-norm) and 3.9e-3 (largest difference) where a
    result is rounded to bf16, by 2e-7 and 8e-7 where everything is fp32 (sums over up to 16384 rows; they grow with the
    rows)."""
    if "bf16" in (case["act"], case["par"]):
        return {"rel": 7e-3, "max": 1.6e-2}
    return {"rel": 2e-6, "max": 1e-5}
