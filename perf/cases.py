"""Performance cases of the SolveDelta layer through its public entry points.

Kinds of case (a case is a dict of plain values):

  op       ``solvedelta_native`` / ``solvedelta_masked_native``: forward with all
           gradients (``train``) or forward alone with the final state (prefill);
  decode   ``solvedelta_native`` at T = 1, one step of a batch of streams;
  mixer    the whole mixer layer, forward and all gradients, FP32 parameters
           under bf16 autocast;
  frontend conv4 + SiLU on the projection's q / k / v columns (under valid / reset
           masks if ``masked``) and the decay gate, forward and gradients;
  readout  the sigmoid-gated RMSNorm, forward and gradients.

Inputs follow the benchmark's distributions: u, h, v ~ N(0,1); q, k normalised per
head; raw gates ~ N(0,1); log-decay = -softplus(N(0,1)); gamma 0.9; masks with
10 % invalid tokens and 1 % resets.
"""
import math

import torch
import torch.nn.functional as F
import torch.utils.checkpoint

from solvedelta_amd import solvedelta_native
from solvedelta_amd.masks import solvedelta_masked_native
from solvedelta_amd.mixer import (RMSNormGated, SolveDelta, SolveDeltaMixerConfig, conv4_silu,
                                  conv4_silu_masked, kda_decay_gate)
from solvedelta_amd.state import SolveDeltaState

BF16 = torch.bfloat16


def _op(name, B, T, H, r, V, train=True, masked=False, state=True):
    return {"name": name, "kind": "op", "B": B, "T": T, "H": H, "r": r, "V": V, "train": train,
            "masked": masked, "state": state}


def listed():
    return [
        # one layer of a training step at the benchmark's shape
        _op("train", 4, 2048, 8, 128, 128),
        # the same at a small per-GPU batch (the reference's published shape)
        _op("train_short", 1, 1024, 8, 128, 128),
        # a small model's layer: launches and latency count
        _op("train_small", 2, 128, 4, 64, 64, state=False),
        # training on padded and packed rows
        _op("train_masked", 4, 2048, 8, 128, 128, masked=True, state=False),
        # a prompt of odd length continued from a cached state, no gradients
        _op("prefill", 2, 3001, 16, 128, 128, train=False),
        # heads of 256 channels: training, the largest case
        _op("wide_train", 4, 2048, 8, 256, 256),
        # a prompt of odd length with heads wider than 128, from a cached state
        _op("wide_prefill", 1, 1333, 12, 192, 160, train=False),
        # one generated token for each of 64 streams
        {"name": "decode", "kind": "decode", "B": 64, "H": 8, "r": 128, "V": 128},
        # the whole layer of a model of hidden size 1024 in a training step
        {"name": "mixer_train", "kind": "mixer", "B": 1, "T": 1024, "hidden": 1024, "H": 8,
         "r": 128, "V": 128},
        # the operator's operands: short convolution and decay gate, training
        {"name": "frontend_train", "kind": "frontend", "B": 3, "T": 1777, "H": 8, "r": 128,
         "V": 128, "masked": False},
        # the same on padded and packed rows
        {"name": "frontend_masked", "kind": "frontend", "B": 4, "T": 2048, "H": 8, "r": 128,
         "V": 128, "masked": True},
        # the gated norm behind the operator, training
        {"name": "readout_train", "kind": "readout", "B": 4, "T": 2048, "H": 8, "V": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A head width: a multiple of 16 three times out of four, else any."""
    w = rng.randint(lo, hi)
    return min(hi, (w + 15) // 16 * 16) if rng.random() < 0.75 else w


def draw(rng):
    kind = rng.choice(["op", "op", "op", "wide", "decode", "mixer", "frontend", "readout"])
    B, H = rng.choice([1, 1, 2, 3, 4, 6, 8]), rng.choice([1, 2, 4, 5, 8, 12, 16])
    if kind in ("op", "wide"):
        lo, hi = (129, 256) if kind == "wide" else (32, 128)
        T = min(_log(rng, 16, 4096), 65536 // (B * H))
        train = rng.random() < 0.6
        c = _op("", B, T, H, _width(rng, lo, hi), _width(rng, lo, hi), train,
                rng.random() < 0.25, rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "decode":
        return {"kind": kind, "B": _log(rng, 1, 256), "H": H, "r": _width(rng, 32, 128),
                "V": _width(rng, 32, 128)}
    if kind == "mixer":
        r = rng.choice([64, 96, 128])
        T = min(_log(rng, 64, 2048), 4096 // B)
        return {"kind": kind, "B": B, "T": T, "hidden": rng.choice([256, 512, 768, 1024]),
                "H": min(H, 8), "r": r, "V": r}
    T = min(_log(rng, 16, 4096), 65536 // (B * H))
    if kind == "frontend":
        return {"kind": kind, "B": B, "T": T, "H": H, "r": _width(rng, 32, 128),
                "V": _width(rng, 32, 128), "masked": rng.random() < 0.5}
    return {"kind": kind, "B": B, "T": T, "H": H, "V": _width(rng, 32, 256)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _normal(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return g, lambda *s: torch.randn(*s, generator=g, device="cuda")


def _masks(g, B, T):
    u = lambda: torch.rand(B, T, generator=g, device="cuda")
    return u() >= 0.1, u() < 0.01


def _operands(n, B, T, H, r, V):
    bf = lambda x: x.to(BF16)
    return [bf(n(B, T, H, r)), bf(n(B, T, H, r)), bf(F.normalize(n(B, T, H, r), dim=-1)),
            bf(F.normalize(n(B, T, H, 1, r), dim=-1)), bf(n(B, T, H, 1, V)),
            -F.softplus(n(B, T, H, r)), bf(n(B, T, H, 1, r)), bf(n(B, T, H, 1, V)),
            torch.full((B, T, H), 0.9, device="cuda")]


OPERANDS = ("u", "h", "q", "k", "v", "log_decay", "erase", "write", "gamma")


def prepare(case, seed):
    kind, B, H = case["kind"], case["B"], case["H"]
    g, n = _normal(seed)
    s = {"case": case}
    if kind in ("op", "decode"):
        T, r, V = case.get("T", 1), case["r"], case["V"]
        s["args"] = _operands(n, B, T, H, r, V)
        s["masks"] = _masks(g, B, T) if case.get("masked") else None
        s["state"] = None
        if kind == "decode" or case["state"]:
            s["state"] = SolveDeltaState(0.02 * n(B, H, r, r), 0.02 * n(B, H, r, V))
        if case.get("train"):
            s["dout"] = n(B, T, H, V).to(BF16)
            s["leaves"] = list(s["args"]) + list(s["state"] or ())
            for x in s["leaves"]:
                x.requires_grad_()
    elif kind == "mixer":
        T, r, V = case["T"], case["r"], case["V"]
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            s["layer"] = SolveDelta(SolveDeltaMixerConfig(
                hidden_size=case["hidden"], num_heads=H, head_k_dim=r, head_v_dim=V)).cuda()
        s["x"] = n(B, T, case["hidden"]).requires_grad_()
        s["dout"] = n(B, T, case["hidden"]).to(BF16)
    elif kind == "frontend":
        T, r, V = case["T"], case["r"], case["V"]
        D = 2 * H * r + H * V
        # the q / k / v columns of the packed projection
        proj = n(B, T, D + 3 * H * r + H * V).to(BF16)
        s["x"] = proj[..., :D].detach().requires_grad_()
        s["w"] = (0.5 * n(D, 4)).requires_grad_()
        s["raw"] = n(B, T, H, r).to(BF16).requires_grad_()
        s["rate"] = torch.log(1 + 15 * torch.rand(H, generator=g, device="cuda")).requires_grad_()
        s["bias"] = (n(H, r) - 4).requires_grad_()
        s["masks"] = _masks(g, B, T) if case["masked"] else None
        s["dy"], s["dg"] = n(B, T, D).to(BF16), n(B, T, H, r)
    else:
        T, V = case["T"], case["V"]
        s["norm"] = RMSNormGated(V).cuda()
        with torch.no_grad():
            s["norm"].weight.copy_(1 + 0.1 * n(V))
        s["x"], s["gate"] = (n(B, T, H, V).to(BF16).requires_grad_() for _ in range(2))
        s["dy"] = n(B, T, H, V).to(BF16)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_op(s):
    train = s["case"].get("train", False)
    kw = dict(initial_state=s["state"], return_final_state=s["state"] is not None)
    with torch.set_grad_enabled(train):
        if s["masks"] is None:
            out, st = solvedelta_native(*s["args"], **kw)
        else:
            out, st = solvedelta_masked_native(*s["args"], *s["masks"], **kw)
    res = {"out": out}
    if st is not None:
        res.update(C=st.predictor, S=st.S)
    if train:
        grads = torch.autograd.grad(out, s["leaves"], s["dout"])
        res.update({"d_" + k: x for k, x in zip(OPERANDS + ("C0", "S0"), grads)})
    return res


def _run_mixer(s):
    layer = s["layer"]
    names, params = zip(*layer.named_parameters())
    with torch.autocast("cuda", dtype=BF16):
        out = layer(s["x"])
    grads = torch.autograd.grad(out, (s["x"],) + params, s["dout"])
    return {"out": out, **{"d_" + k: x for k, x in zip(("x",) + names, grads)}}


def _run_frontend(s):
    if s["masks"] is None:
        y, _ = conv4_silu(s["x"], s["w"])
    else:
        y, _ = conv4_silu_masked(s["x"], s["w"], *s["masks"])
    g = kda_decay_gate(s["raw"], s["rate"], s["bias"])
    dx, dw, draw, drate, dbias = torch.autograd.grad(
        (y, g), (s["x"], s["w"], s["raw"], s["rate"], s["bias"]), (s["dy"], s["dg"]))
    return {"y": y, "log_decay": g, "d_x": dx, "d_w": dw, "d_raw": draw, "d_rate": drate,
            "d_bias": dbias}


def _run_readout(s):
    y = s["norm"](s["x"], s["gate"])
    dx, dg, dw = torch.autograd.grad(y, (s["x"], s["gate"], s["norm"].weight), s["dy"])
    return {"y": y, "d_x": dx, "d_gate": dg, "d_weight": dw}


def run(state):
    kind = state["case"]["kind"]
    if kind in ("op", "decode"):
        return _run_op(state)
    return {"mixer": _run_mixer, "frontend": _run_frontend, "readout": _run_readout}[kind](state)


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------
def _op_work(B, T, H, r, V, train, state, masked):
    n = B * T * H
    operands = n * (5 * 2 * r + 2 * 2 * V + 4 * r + 4) + (2 * B * T if masked else 0)
    states = B * H * (r * r + r * V) * 4 if state else 0
    out = n * V * 2
    # per token: C u, C^T k, S^T e, S^T chi and the two rank-one updates
    flops = n * 6 * (r * r + r * V)
    if not train:
        return operands + 2 * states + out, flops
    # the backward reads the output's cotangent and writes every operand's gradient
    return 2 * (operands + out) + 3 * states, 3 * flops


def work(case):
    kind, B, H, T, V = case["kind"], case["B"], case["H"], case.get("T", 1), case["V"]
    if kind in ("op", "decode"):
        b, f = _op_work(B, T, H, case["r"], V, case.get("train", False),
                        case.get("state", True), case.get("masked", False))
    elif kind == "mixer":
        r, hidden, n = case["r"], case["hidden"], B * T
        cols = 5 * H * r + 2 * H * V + H + 2 * V
        weights = hidden * cols + V * (H * r + H * V) + H * V * hidden
        f = 6 * n * weights + _op_work(B, T, H, r, V, True, False, False)[1]
        b = 8 * weights + n * hidden * (4 + 2 + 2 + 4)
    elif kind == "frontend":
        n, D, K = B * T, 2 * H * case["r"] + H * V, H * case["r"]
        b = n * (D * 2 * 4 + K * (2 + 4 + 4 + 2)) + (2 * n if case["masked"] else 0)
        f = n * (30 * D + 20 * K)
    else:
        n = B * T * H * V
        b, f = n * 2 * 6, n * 30
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    # bf16 outputs round at 2e-3 of their norm; gradients follow 16-bit token panels
    if case["kind"] == "op":
        return {"rel": 1.6e-2 if case["train"] else 8e-3}
    return {"rel": {"decode": 8e-3, "mixer": 3e-2, "frontend": 8e-3, "readout": 8e-3}[case["kind"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits, token by token
# ---------------------------------------------------------------------------
def _recur(u, h, q, k, v, g, erase, write, gamma, valid, reset, C, S):
    """Tokens one after the other; u, q, k normalised, gates in [0, 1]; [B,T,H,...] operands."""
    outs = []
    for t in range(u.shape[1]):
        if valid is not None:
            ok = valid[:, t, None, None, None]
            keep = ~(reset[:, t, None, None, None] & ok)
            C, S = C * keep, S * keep
        ut, kt = u[:, t], k[:, t]
        D = g[:, t].exp()
        delta = gamma[:, t, :, None] * (h[:, t] - (C @ ut[..., None])[..., 0])
        C1 = C * D[..., None, :] + delta[..., :, None] * ut[..., None, :]
        phi = 0.625 * delta / torch.sqrt(
            0.625 ** 2 + (ut * ut).sum(-1, keepdim=True) * (delta * delta).sum(-1, keepdim=True))
        den = 1 + (phi * ut).sum(-1, keepdim=True)
        d = kt + (kt[..., None, :] @ C1)[..., 0, :]
        b = erase[:, t] * kt
        e = b - phi * ((ut * b).sum(-1, keepdim=True) / den)
        chi = q[:, t] - phi * ((ut * q[:, t]).sum(-1, keepdim=True) / den)
        S1 = D[..., :, None] * S
        z = write[:, t] * v[:, t] - (e[..., None, :] @ S1)[..., 0, :]
        S1 = S1 + d[..., :, None] * z[..., None, :]
        o = (chi[..., None, :] @ S1)[..., 0, :]
        if valid is not None:
            o, C1, S1 = o * ok[..., 0], torch.where(ok, C1, C), torch.where(ok, S1, S)
        C, S = C1, S1
        outs.append(o)
    return torch.stack(outs, 1), C, S


def _exact_op(args, masks, state):
    """64-bit operator: (out, C, S), with the tokens' states recomputed in pieces in the backward."""
    u, h, q, k, v, g, er, wr, gamma = args
    unit = lambda x: F.normalize(x, dim=-1)
    flat = [unit(u), h, unit(q), unit(k[:, :, :, 0]), v[:, :, :, 0], g, torch.sigmoid(er[:, :, :, 0]),
            torch.sigmoid(wr[:, :, :, 0]), gamma]
    B, T, H, r = u.shape
    if state is None:
        C, S = (torch.zeros(B, H, r, w, dtype=torch.float64, device=u.device)
                for w in (r, v.shape[-1]))
    else:
        C, S = state
    outs = []
    for t in range(0, T, 64):
        piece = [x[:, t:t + 64] for x in flat]
        m = (None, None) if masks is None else [x[:, t:t + 64] for x in masks]
        if torch.is_grad_enabled():
            o, C, S = torch.utils.checkpoint.checkpoint(_recur, *piece, *m, C, S,
                                                        use_reentrant=False)
        else:
            o, C, S = _recur(*piece, *m, C, S)
        outs.append(o)
    return torch.cat(outs, 1), C, S


def _wide(x):
    return x.detach().double().requires_grad_()


def _conv(x, w, masks):
    """y_t = silu(sum_j w[3 - j] x(j-th last valid token since the last reset)), 0 on invalid tokens."""
    if masks is None:
        p = F.pad(x, (0, 0, 3, 0))
        return F.silu(sum(p[:, j:j + x.shape[1]] * w[:, j] for j in range(4)))
    rows = []
    for xb, ok, rs in zip(x, *masks):
        at = ok.nonzero()[:, 0]
        xv, n = xb[at], len(at)
        start = torch.where(rs[at], torch.arange(n, device=x.device), 0).cummax(0).values if n else at
        pos = torch.arange(n, device=x.device) - start
        p = F.pad(xv, (0, 0, 3, 0))
        a = sum(p[3 - j:3 - j + n] * w[:, 3 - j] * (pos >= j)[:, None] for j in range(4))
        rows.append(torch.zeros_like(xb).index_copy(0, at, F.silu(a)))
    return torch.stack(rows)


def _decay(raw, rate, bias):
    return -torch.exp(rate)[:, None] * F.softplus(raw + bias)


def _norm(x, gate, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w * torch.sigmoid(gate)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("op", "decode"):
        train = case.get("train", False)
        args = [_wide(x) for x in s["args"]]
        state = None if s["state"] is None else [_wide(x) for x in s["state"]]
        with torch.set_grad_enabled(train):
            out, C, S = _exact_op(args, s["masks"], state)
        res = {"out": out}
        if state is not None:
            res.update(C=C, S=S)
        if train:
            grads = torch.autograd.grad(out, args + (state or []), s["dout"].double(),
                                        allow_unused=True, materialize_grads=True)
            res.update({"d_" + k: x for k, x in zip(OPERANDS + ("C0", "S0"), grads)})
        return {k: x.detach() for k, x in res.items()}
    if kind == "frontend":
        x, w, raw, rate, bias = (_wide(s[k]) for k in ("x", "w", "raw", "rate", "bias"))
        y, g = _conv(x, w, s["masks"]), _decay(raw, rate, bias)
        grads = torch.autograd.grad((y, g), (x, w, raw, rate, bias),
                                    (s["dy"].double(), s["dg"].double()))
        names = ("d_x", "d_w", "d_raw", "d_rate", "d_bias")
        return {"y": y.detach(), "log_decay": g.detach(), **dict(zip(names, grads))}
    if kind == "readout":
        x, gate, w = _wide(s["x"]), _wide(s["gate"]), _wide(s["norm"].weight)
        y = _norm(x, gate, w, s["norm"].eps)
        dx, dg, dw = torch.autograd.grad(y, (x, gate, w), s["dy"].double())
        return {"y": y.detach(), "d_x": dx, "d_gate": dg, "d_weight": dw}
    return _exact_mixer(s)


def _exact_mixer(s):
    layer, case = s["layer"], s["case"]
    B, T, H, r, V = (case[k] for k in ("B", "T", "H", "r", "V"))
    p = {k: _wide(x) for k, x in layer.named_parameters()}
    x = _wide(s["x"])
    sizes = (H * r, H * r, H * V, H * r, H * r, H * r, H * V, H, V, V)
    proj = F.linear(x, p["in_proj.weight"])[..., :sum(sizes)].split(sizes, dim=-1)
    q, k, v = _conv(torch.cat(proj[:3], -1), p["conv_weight"], None).split(sizes[:3], dim=-1)
    u, h, er, wr, geo, dec, gate = proj[3:]
    heads = lambda y, w: y.reshape(B, T, H, w)
    edits = lambda y, w: y.reshape(B, T, H, 1, w)
    g = _decay(heads(F.linear(dec, p["decay_proj.weight"]), r), p["associative_log_rate"],
               p["associative_decay_bias"])
    gamma = torch.sigmoid(geo + p["geometry_write_bias"])
    gate = F.linear(gate, p["output_gate_proj.weight"], p["output_gate_proj.bias"])
    o, _, _ = _exact_op([heads(u, r), heads(h, r), heads(q, r), edits(k, r), edits(v, V), g,
                         edits(er, r), edits(wr, V), gamma], None, None)
    y = _norm(o, heads(gate, V), p["output_norm.weight"], layer.output_norm.eps)
    out = F.linear(y.reshape(B, T, H * V), p["output_proj.weight"])
    grads = torch.autograd.grad(out, (x, *p.values()), s["dout"].double())
    return {"out": out.detach(), **{"d_" + n: gr for n, gr in zip(("x", *p), grads)}}
