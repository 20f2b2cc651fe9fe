"""The calls that a training program makes of this library, as timed cases: the fused SwiGLU MLP with LoRA (forward,
training step, a checkpoint's recompute), the grouped projections around attention, a single MX linear, the unfused MLP
and the quantizer, from a few hundred tokens to a whole 16 x 8896 batch.

listed() names the cases, draw() makes more of the same ranges, prepare() makes what a program holds before the call,
run() is one pass through the public entry points, work() counts what a pass cannot do without, exact() is the same
result in float64 from plain torch, and tolerance() is what another correct implementation at these precisions would
differ by.
"""
import contextlib
import io
import math
import os
import sys
import types

import torch

_PKG = os.path.join(os.getcwd(), "train-model-template_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_GRADS = ("mlp_step", "mlp_recompute", "unfused_step")


def listed():
    return [
        # evaluation of a short prompt with the adapters on: forward alone, the smallest call (launches and latency)
        dict(name="mlp_forward_256", kind="mlp_forward", T=256, K=1024, N=3584, r=16, outliers=False),
        # a short, ragged micro-batch at the larger adapter rank, with outlier channels in x and dy
        dict(name="mlp_step_1000_r32", kind="mlp_step", T=1000, K=2048, N=6144, r=32, outliers=True),
        # the training step of the small model's layer
        dict(name="mlp_step_4096", kind="mlp_step", T=4096, K=1024, N=3584, r=16, outliers=False),
        # the last layer of a checkpointed segment: forward for the graph only, then backward, one 8896-token sequence
        dict(name="mlp_recompute_8896", kind="mlp_recompute", T=8896, K=2048, N=6144, r=16, outliers=False),
        # the headline shape of bench.py
        dict(name="mlp_step_10752", kind="mlp_step", T=10752, K=2048, N=6144, r=16, outliers=False),
        # one layer of the full training batch, 16 sequences of 8896 tokens
        dict(name="mlp_step_142336", kind="mlp_step", T=142336, K=2048, N=6144, r=16, outliers=False),
        # the MLP without a shared gate|up copy (gate and up as grouped linears, SwiGLU, down)
        dict(name="unfused_step_2688", kind="unfused_step", T=2688, K=1024, N=3584, r=16, outliers=False),
        # q|k|v and o_proj with the residual add, small layer and ragged token count
        dict(name="attn_step_1500", kind="attn_step", T=1500, K=1024, N=1024, nkv=256, r=16, outliers=False),
        # the same at the bench's attention shape
        dict(name="attn_step_10752", kind="attn_step", T=10752, K=2048, N=2048, nkv=512, r=16, outliers=False),
        # linear-attention projections: qkv|z grouped with two thin gates, out_proj with the residual add
        dict(name="delta_step_4096", kind="delta_step", T=4096, K=2048, N=2048, r=16, outliers=False),
        # one frozen MX linear called by itself, without an adapter
        dict(name="linear_step_4096", kind="linear_step", T=4096, K=2048, N=2048, outliers=False),
        # the row quantizer alone, on the headline activation
        dict(name="quantize_10752", kind="quantize", T=10752, K=2048, outliers=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp_forward", "mlp_step", "mlp_step", "mlp_step", "mlp_recompute", "unfused_step", "attn_step",
                       "attn_step", "delta_step", "linear_step", "quantize"])
    c = dict(kind=kind, T=_log_int(rng, 256, {"unfused_step": 10752, "mlp_recompute": 20000}.get(kind, 40000)),
             outliers=rng.random() < 0.3)
    if kind in ("mlp_forward", "mlp_step", "mlp_recompute", "unfused_step"):
        c["K"], c["N"] = rng.choice([(1024, 3584), (2048, 6144), (128 * rng.randint(6, 16), 128 * rng.randint(12, 48))])
        c["r"] = 16 if kind == "unfused_step" else rng.choice([16, 16, 32])
    elif kind == "attn_step":
        c["K"] = 128 * rng.choice([8, 12, 16])
        c["N"], c["nkv"], c["r"] = rng.choice([c["K"], 2 * c["K"]]), 128 * rng.randint(2, 4), 16
    elif kind == "delta_step":
        c["K"] = 128 * rng.choice([8, 12, 16])
        c["N"], c["r"] = c["K"], 16
    elif kind == "linear_step":
        c["K"], c["N"] = 128 * rng.randint(4, 16), 128 * rng.randint(4, 48)
    else:
        c["K"] = 128 * rng.randint(4, 48)
    return c


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, k):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + k)


def _randn(seed, k, *shape, std=1.0):
    return torch.randn(*shape, generator=_gen(seed, k), device="cuda") * std


def _act(case, seed, k, cols, std=1.0):
    """Activations or upstream gradients [T, cols] in bf16; with outliers, a thousandth of the channels 100 times as
    large and heavier tails, as the residual stream of a trained model has them."""
    t = _randn(seed, k, case["T"], cols, std=std)
    if case["outliers"]:
        t = t * torch.exp(0.5 * _randn(seed, k + 500, case["T"], 1))
        ch = torch.randperm(cols, generator=_gen(seed, k + 600), device="cuda")[:max(1, cols // 1000)]
        t[:, ch] *= 100.0
    return t.to(torch.bfloat16)


_ALPHA = 32.0


def _linears(case):
    """(name, outputs, inputs, has an adapter) of the case's frozen linears, in the order of their gradients."""
    K, N = case["K"], case.get("N")
    kind = case["kind"]
    if kind == "attn_step":
        return [("q_proj", N, K, True), ("k_proj", case["nkv"], K, True), ("v_proj", case["nkv"], K, True),
                ("o_proj", K, N, True)]
    if kind == "delta_step":
        return [("in_proj_qkv", 3 * N, K, True), ("in_proj_z", N, K, True), ("in_proj_b", 16, K, False),
                ("in_proj_a", 16, K, False), ("out_proj", K, N, True)]
    if kind == "linear_step":
        return [("out_proj", N, K, False)]
    if kind == "quantize":
        return []
    return [("gate_proj", N, K, True), ("up_proj", N, K, True), ("down_proj", K, N, True)]


def _weights(case, seed):
    """name -> (W bf16, A fp32, B fp32), A and B None without an adapter."""
    out = {}
    for i, (name, n, k, lora) in enumerate(_linears(case)):
        W = _randn(seed, 10 * i + 1, n, k, std=0.02).to(torch.bfloat16)
        A = _randn(seed, 10 * i + 2, case["r"], k, std=0.02) if lora else None
        B = _randn(seed, 10 * i + 3, n, case["r"], std=0.02) if lora else None
        out[name] = (W, A, B)
    return out


def _inputs(case, seed):
    """The activations and upstream gradients of a pass."""
    K, N, kind = case["K"], case.get("N"), case["kind"]
    d = dict(x=_act(case, seed, 101, K))
    if kind in _GRADS:
        d["dy"] = _act(case, seed, 102, K, 1e-2)
    elif kind == "attn_step":
        d.update(resid=_act(case, seed, 103, K), mid=_act(case, seed, 104, N), dq=_act(case, seed, 105, N, 1e-2),
                 dk=_act(case, seed, 106, case["nkv"], 1e-2), dv=_act(case, seed, 107, case["nkv"], 1e-2),
                 dout=_act(case, seed, 108, K, 1e-2))
    elif kind == "delta_step":
        d.update(resid=_act(case, seed, 103, K), mid=_act(case, seed, 104, N), dqkv=_act(case, seed, 105, 3 * N, 1e-2),
                 dz=_act(case, seed, 106, N, 1e-2), db=_act(case, seed, 107, 16, 1e-2),
                 da=_act(case, seed, 109, 16, 1e-2), dout=_act(case, seed, 108, K, 1e-2))
    elif kind == "linear_step":
        d["dy"] = _act(case, seed, 102, N, 1e-2)
    return d


def prepare(case, seed):
    s = types.SimpleNamespace(kind=case["kind"], **_inputs(case, seed))
    if s.kind == "quantize":
        return s
    import mxfp8
    import workloads
    with torch.device("cuda"):
        block = torch.nn.Module()
        for name, (W, A, B) in _weights(case, seed).items():
            lin = torch.nn.Linear(W.shape[1], W.shape[0], bias=False, dtype=torch.bfloat16)
            lin.weight.data.copy_(W)
            lin.weight.requires_grad_(False)
            setattr(block, name, lin if A is None else workloads.LoraLinear(lin, A, B, _ALPHA))
        block.act_fn = torch.nn.SiLU()
        s.model = torch.nn.Module()
        s.model.layers = torch.nn.ModuleList([block])
    s.root = torch.nn.Module()
    s.root.model = s.model
    s.block = block
    keep = mxfp8.FUSE_GU
    mxfp8.FUSE_GU = keep and s.kind != "unfused_step"
    try:
        with contextlib.redirect_stdout(io.StringIO()):
            mxfp8.enable_mxfp8(s.root)
    finally:
        mxfp8.FUSE_GU = keep
    s.params = [p for p in s.root.parameters() if p.requires_grad]
    return s


def _param_grads(s, names):
    out = []
    for n in names:
        m = getattr(s.block, n)
        out += [m.lora_A["default"].weight.grad, m.lora_B["default"].weight.grad]
    return out


def run(s):
    import mxfp8
    if s.kind == "quantize":
        q, sc = mxfp8.mx_quant(s.x)
        return q.view(torch.uint8), sc.view(torch.uint8)
    import fused_linear
    import fused_mlp
    import shared_prefix
    fused_linear.new_step()
    for p in s.params:
        p.grad = None
    b = s.block
    if s.kind == "mlp_forward":
        with torch.no_grad():
            return fused_mlp.mlp(b, s.x)
    x = s.x.detach().requires_grad_(True)
    if s.kind == "linear_step":
        y = b.out_proj(x)
        y.backward(s.dy)
        return y.detach(), x.grad
    if s.kind in _GRADS:
        y = shared_prefix._mlp(b, x, need_out=s.kind != "mlp_recompute")
        y.backward(s.dy)
        grads = [x.grad] + _param_grads(s, ("gate_proj", "up_proj", "down_proj"))
        return grads if s.kind == "mlp_recompute" else [y.detach()] + grads
    mid = s.mid.detach().requires_grad_(True)
    if s.kind == "attn_step":
        names, last, dys = ("q_proj", "k_proj", "v_proj"), "o_proj", [s.dq, s.dk, s.dv]
    else:
        names, last = ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a"), "out_proj"
        dys = [s.dqkv, s.dz, s.db, s.da]
    outs = fused_linear.group_linear(x, [getattr(b, n) for n in names])
    (o,) = fused_linear.group_linear(mid, [getattr(b, last)], defer=True)
    out = fused_linear.residual_add(s.resid, o)
    torch.autograd.backward([out, *outs], [s.dout, *dys])
    lora = [n for n in (*names, last) if hasattr(getattr(b, n), "lora_A")]
    return [out.detach()] + [t.detach() for t in outs] + [x.grad, mid.grad] + _param_grads(s, lora)


# ------------------------------------------------------------------------------------------------ work
def work(case):
    """Bytes: activations, gradients, weights (one byte a code and one scale a 32-block, both axes in a step) and LoRA
    parameters read once, results written once.  Flops: the frozen products and the rank-r ones."""
    T, K, kind = case["T"], case["K"], case["kind"]
    if kind == "quantize":
        return {"bytes": T * K * 3 + T * K // 32, "flops": 0}
    back = kind != "mlp_forward"
    fwd_down = 0 if kind == "mlp_recompute" else 1
    by = fl = 0.0
    for name, n, k, lora in _linears(case):
        mx = n > 64
        passes = (fwd_down if name == "down_proj" else 1) + (1 if back else 0)
        by += n * k * (33 / 32 * passes if mx else 2)
        fl += 2.0 * T * n * k * passes
        if lora:
            r = case["r"]
            by += (n + k) * r * 4 * (2 if back else 1)
            fl += 2.0 * T * (n + k) * r * (3 if back else 1)
    if kind == "attn_step":
        rows = 4 * K + 4 * case["N"] + 4 * case["nkv"]  # x, resid, out, dout; mid, q, dq, dmid; k, v, dk, dv
        rows += K  # dx
    elif kind == "delta_step":
        rows = 5 * K + 2 * case["N"] + 2 * (4 * case["N"] + 32)
    elif kind == "linear_step":
        rows = 2 * K + 2 * case["N"]
    else:
        rows = {"mlp_forward": 2, "mlp_recompute": 3}.get(kind, 4) * K
    return {"bytes": by + 2.0 * T * rows, "flops": fl}


# ------------------------------------------------------------------------------------------------ float64
def _mx(t):
    """The values that an MXFP8 operand of t [rows, cols] holds, in float64: blocks of 32 along the columns, a power of
    two scale with ceil(log2(amax / 448)), E4M3 codes rounded to nearest even."""
    rows, cols = t.shape
    b = t.double().reshape(rows, cols // 32, 32)
    m, e = torch.frexp(b.abs().amax(-1, keepdim=True) / 448.0)
    e = (e - (m == 0.5).int()).clamp(-127, 127)
    v = torch.ldexp(b, -e).float().to(torch.float8_e4m3fn).double()
    return torch.ldexp(v, e).reshape(rows, cols)


def _bf(t):
    return t.to(torch.bfloat16).double()


_ROWS = 16384  # rows of a float64 chunk


def _chunks(T):
    return [slice(i, min(T, i + _ROWS)) for i in range(0, T, _ROWS)]


def _cat(parts):
    return torch.cat(parts) if len(parts) > 1 else parts[0]


def _exact_mlp(case, W, d):
    kind, back = case["kind"], case["kind"] != "mlp_forward"
    s = _ALPHA / case["r"]
    (Wg, Ag, Bg), (Wu, Au, Bu), (Wd, Ad, Bd) = ((w.double(), _bf(a), _bf(b)) for w, a, b in W.values())
    fg, fu, fd = _mx(Wg), _mx(Wu), _mx(Wd)
    tg, tu, td = _mx(Wg.t().contiguous()), _mx(Wu.t().contiguous()), _mx(Wd.t().contiguous())
    ys, dxs, g6 = [], [], [torch.zeros_like(t) for t in (Ag, Bg, Au, Bu, Ad, Bd)]
    for c in _chunks(case["T"]):
        x = d["x"][c].double()
        xq = _mx(x)
        ag, au = x @ Ag.t(), x @ Au.t()
        g, u = xq @ fg.t() + s * ag @ Bg.t(), xq @ fu.t() + s * au @ Bu.t()
        sig = torch.sigmoid(g)
        h = g * sig * u
        hd = h @ Ad.t()
        if kind != "mlp_recompute":
            ys.append(_mx(h) @ fd.t() + s * hd @ Bd.t())
        if not back:
            continue
        dy = d["dy"][c].double()
        dh_lo = s * dy @ Bd
        g6[5] += s * dy.t() @ hd
        g6[4] += dh_lo.t() @ h
        dh = _mx(dy) @ td.t() + dh_lo @ Ad
        du, dg = dh * g * sig, dh * u * sig * (1 + g * (1 - sig))
        dag, dau = s * dg @ Bg, s * du @ Bu
        g6[0] += dag.t() @ x
        g6[1] += s * dg.t() @ ag
        g6[2] += dau.t() @ x
        g6[3] += s * du.t() @ au
        dxs.append(_mx(dg) @ tg.t() + _mx(du) @ tu.t() + dag @ Ag + dau @ Au)
    if not back:
        return _cat(ys)
    return ([] if kind == "mlp_recompute" else [_cat(ys)]) + [_cat(dxs)] + g6


def _exact_group(W, s, x, dys, resid=None):
    """Outputs, dx and [dA, dB, ...] of linears on one input; resid is added to the (single) output."""
    outs, dx, grads = [], 0.0, []
    xd, xq = x.double(), _mx(x)
    for (w, A, B), dy in zip(W, dys):
        dyd, wd = dy.double(), w.double()
        if w.shape[0] <= 64:
            outs.append(xd @ wd.t())
            dx = dx + dyd @ wd
            continue
        y = xq @ _mx(wd).t()
        dx = dx + _mx(dyd) @ _mx(wd.t().contiguous()).t()
        if A is not None:
            a, b = _bf(A), _bf(B)
            xa, dxa = xd @ a.t(), s * dyd @ b
            y = y + s * xa @ b.t()
            dx = dx + dxa @ a
            grads += [dxa.t() @ xd, s * dyd.t() @ xa]
        outs.append(y)
    if resid is not None:
        outs[0] = outs[0] + resid.double()
    return outs, dx, grads


def exact(case, seed):
    kind, d, W = case["kind"], _inputs(case, seed), _weights(case, seed)
    if kind == "quantize":
        return None  # codes and scales are compared bit for bit
    if kind.startswith("mlp") or kind == "unfused_step":
        return _exact_mlp(case, W, d)
    s, w = _ALPHA / case.get("r", 1), list(W.values())
    if kind == "linear_step":
        outs, dx, _ = _exact_group(w, s, d["x"], [d["dy"]])
        return outs[0], dx
    dys = [d[k] for k in (("dq", "dk", "dv") if kind == "attn_step" else ("dqkv", "dz", "db", "da"))]
    outs, dx, grads = _exact_group(w[:-1], s, d["x"], dys)
    (out,), dmid, glast = _exact_group(w[-1:], s, d["mid"], [d["dout"]], d["resid"])
    return [out] + outs + [dx, dmid] + grads + glast


def tolerance(case):
    """Bytes of the quantizer are exact.  A grouped or single linear returns bf16 sums of bf16-rounded terms: measured
    1.6e-3 to 2.4e-3 from exact(), four times that here.  In the MLP, a last-bit change of gate, up or dh moves codes
    of h, dg and du across an E4M3 step: measured 1.7e-2 to 2.0e-2 from exact() for y and dx."""
    kind = case["kind"]
    return "exact" if kind == "quantize" else {"rel": 0.01} if kind in ("attn_step", "delta_step", "linear_step") else {
        "rel": 0.02}
