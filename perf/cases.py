"""Performance cases of the carrier framework: what a training, prefill or serving program has it do.

The kinds of case, each over the range that `draw` spans:

    scan    the associative scan with bf16 operands (`assoc_scan(mm=bfloat16)`), plain and delta write rules, heads of
            64 and 128, one window of 64 tokens to a context of 8192, 1 to 16 sequences of 2 to 12 heads, with and
            without a carried state; a training step (outputs, final state, every gradient), or forward only
    exact   the same scan with fp32 operands (`assoc_scan`), which the carriers with a few wide heads (d / 4 and d / 2)
            and every kernel=False carrier run on
    diag    the complex diagonal scan (`scan_hip`) of the forget-gated carrier, training step
    layer   one whole AssocCarrier layer under bf16 autocast: norm, projections, scan, output norm and projection,
            forward and backward with every parameter's gradient
    lm      `LM.forward_carried`: a long sequence read in windows with the state carried, the last window's logits
    decode  `GreedyDecoder`: a prefilled state loaded, then greedy tokens one step at a time

A training program captures its step in a HIP graph and replays it (a step is some tens of launches); `graph` cases do
the same in `prepare` and replay in `run`. The others call the entry point eagerly.
"""
import math

import torch
import torch.nn.functional as F

from pragnosia_amd.assoc import AssocCarrier, assoc_scan
from pragnosia_amd.decode import GreedyDecoder
from pragnosia_amd.model import LM
from pragnosia_amd.scan import scan_hip

DEV = "cuda"


def listed():
    return [
        # a sequence chunk arriving at a stream's carried state, one user: latency
        {"name": "scan_plain_window", "kind": "scan", "rule": "plain", "B": 1, "H": 12, "T": 100, "D": 64, "S0": True,
         "grad": False, "graph": False},
        # the benchmark's shape: training at short context, many sequences
        {"name": "scan_plain_step", "kind": "scan", "rule": "plain", "B": 16, "H": 12, "T": 512, "D": 64, "S0": False,
         "grad": True, "graph": True},
        # the delta carrier in a d704 model's training micro-batch (4 sequences of 2048)
        {"name": "scan_delta_step", "kind": "scan", "rule": "delta", "B": 4, "H": 11, "T": 2048, "D": 64, "S0": False,
         "grad": True, "graph": True},
        # 128-wide heads, a ragged length and a carried state
        {"name": "scan_delta_wide", "kind": "scan", "rule": "delta", "B": 3, "H": 6, "T": 1000, "D": 128, "S0": True,
         "grad": True, "graph": True},
        # four wide heads of a d704 model, fp32, the same micro-batch
        {"name": "exact_plain_wide", "kind": "exact", "rule": "plain", "B": 4, "H": 4, "T": 2048, "D": 176,
         "S0": False, "grad": True},
        # four wide heads of a d768 model under the delta rule, ragged, carried state
        {"name": "exact_delta_wide", "kind": "exact", "rule": "delta", "B": 2, "H": 4, "T": 1000, "D": 192,
         "S0": True, "grad": True},
        # the diagonal scan at the benchmark's shape, and in a d704 model's micro-batch
        {"name": "diag_step", "kind": "diag", "B": 16, "T": 512, "D": 768, "h0": False, "graph": True},
        {"name": "diag_context", "kind": "diag", "B": 4, "T": 2048, "D": 704, "h0": True, "graph": True},
        # one carrier layer's training step in the d704 model's micro-batch
        {"name": "layer_train", "kind": "layer", "d": 704, "head_dim": 64, "rule": "plain", "B": 4, "T": 2048},
        # reading a long document: 16 windows of 512 (four layers: rounding grows with each)
        {"name": "lm_carried", "kind": "lm", "rule": "delta", "d": 768, "layers": 4, "B": 2, "T": 8192,
         "window": 512, "amp": True},
        # generation for one user and for a batch, the 92M-parameter model
        {"name": "decode_one", "kind": "decode", "rule": "plain", "d": 768, "layers": 12, "B": 1, "n": 33},
        {"name": "decode_batch", "kind": "decode", "rule": "plain", "d": 768, "layers": 12, "B": 32, "n": 17},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan"] * 5 + ["exact"] * 4 + ["diag"] * 3 + ["layer"] * 2 + ["lm", "decode"])
    if kind == "scan":
        D = rng.choice([64, 64, 128])
        H = rng.choice([4, 6, 8, 11, 12]) if D == 64 else rng.choice([2, 3, 4, 5, 6])
        B, T = _log(rng, 1, 16), _log(rng, 64, 8192)
        T = max(64, min(T, (12 << 20) // (B * H * D)))
        if rng.random() < 0.5:
            T = 64 * max(1, T // 64)
        grad = rng.random() < 0.75
        return {"kind": kind, "rule": rng.choice(["plain", "delta"]), "B": B, "H": H, "T": T, "D": D,
                "S0": rng.random() < 0.5, "grad": grad, "graph": grad}
    if kind == "exact":
        D = rng.choice([64, 96, 128, 176, 176, 192, 192, 352])
        H = max(1, rng.choice([704, 768]) // D)
        B, T = _log(rng, 1, 8), _log(rng, 64, 2048)
        T = max(64, min(T, (5 << 20) // (B * H * D)))
        if D == 352:
            T = min(T, 512)
        return {"kind": kind, "rule": rng.choice(["plain", "delta"]), "B": B, "H": H, "T": T, "D": D,
                "S0": rng.random() < 0.5, "grad": rng.random() < 0.75}
    if kind == "diag":
        D = rng.choice([250, 256, 384, 512, 704, 768, 1000, 1024])
        B, T = _log(rng, 1, 16), _log(rng, 64, 8192)
        T = max(64, min(T, (6 << 20) // (B * D)))
        return {"kind": kind, "B": B, "T": T, "D": D, "h0": rng.random() < 0.5, "graph": rng.random() < 0.75}
    if kind == "layer":
        hd = rng.choice([64, 64, 128])
        d = rng.choice([256, 384, 512, 704, 768]) // hd * hd
        B, T = _log(rng, 1, 16), _log(rng, 128, 4096)
        T = max(128, min(T, (6 << 20) // (B * d)))
        # plain rule: under the delta rule theta's gradient cancels to within a few percent of what bf16 resolves (6%
        # off 64 bits at T 4096), so no tolerance could tell a right one from a wrong one; `scan` and `lm` hold that rule
        return {"kind": kind, "d": d, "head_dim": hd, "rule": "plain", "B": B, "T": T}
    if kind == "lm":
        T = _log(rng, 1024, 8192)
        return {"kind": kind, "rule": rng.choice(["plain", "delta"]), "d": rng.choice([512, 768]),
                "layers": rng.randint(2, 4), "B": rng.choice([1, 2]), "T": T, "window": rng.choice([256, 512]),
                "amp": rng.random() < 0.75}
    return {"kind": kind, "rule": rng.choice(["plain", "delta"]), "d": rng.choice([512, 768]),
            "layers": rng.randint(2, 12), "B": _log(rng, 1, 32), "n": 17}


# ------------------------------------------------------------------------------------------------------------------
# inputs

VOCAB, CTX = 8192, 512


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _scan_inputs(case, seed, dtype):
    """What a carrier hands the scan: unit q, k and v per head, k gated under the plain rule, decays with per-head
    timescales from about ten tokens to ten thousand, write strengths around one half; a state of the scale a window
    leaves behind; gradients of unit scale."""
    g = _gen(seed)
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    q, k, v = (F.normalize(_randn(g, B, H, T, D), dim=-1) for _ in range(3))
    if case["rule"] == "plain":
        k = k * torch.sigmoid(_randn(g, B, H, T, 1))
    scale = torch.logspace(-1, -4, H, device=DEV).view(1, H, 1)
    la = -F.softplus(_randn(g, B, H, T)) / 0.69 * scale
    beta = torch.sigmoid(_randn(g, B, H, T)) if case["rule"] == "delta" else None
    S0 = 0.1 * _randn(g, B, H, D, D) if case["S0"] else None
    x = {"q": q.to(dtype), "k": k.to(dtype), "v": v.to(dtype), "la": la, "beta": beta, "S0": S0}
    do, dS = _randn(g, B, H, T, D).to(dtype), _randn(g, B, H, D, D)
    return {n: t for n, t in x.items() if t is not None}, do, dS


def _diag_inputs(case, seed):
    """What the forget-gated carrier hands the diagonal scan: |lambda| from its gate and timescales, angles per
    channel over [0, pi], inputs normalised by sqrt(1 - |lambda|^2)."""
    g = _gen(seed)
    B, T, D = case["B"], case["T"], case["D"]
    nu = torch.logspace(-3, math.log10(0.3), D, device=DEV)
    lm = -8.0 * torch.sigmoid(_randn(g, B, T, D)) * nu
    an = torch.linspace(0.0, math.pi, D, device=DEV).expand(B, T, D).contiguous()
    u = _randn(g, B, T, D) * torch.sqrt((1 - torch.exp(2 * lm)).clamp_min(1e-6))
    x = {"u": u, "lm": lm, "an": an}
    if case["h0"]:
        x["h0r"], x["h0i"] = _randn(g, B, D), _randn(g, B, D)
    return x, _randn(g, B, T, D), _randn(g, B, D), _randn(g, B, D)


def _layer_parts(case, seed):
    g = _gen(seed)
    with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
        torch.manual_seed(seed)
        torch.cuda.manual_seed(seed)
        with torch.device(DEV):
            m = AssocCarrier(case["d"], delta=case["rule"] == "delta", head_dim=case["head_dim"])
        m.apply(LM._init)
    x = _randn(g, case["B"], case["T"], case["d"])
    return m, x, _randn(g, case["B"], case["T"], case["d"])


def _lm(case, seed):
    with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
        torch.manual_seed(seed)
        torch.cuda.manual_seed(seed)
        with torch.device(DEV):
            m = LM(vocab=VOCAB, d=case["d"], layers=case["layers"], mlp_mult=4, ctx=case.get("window", CTX),
                   mixer="dspin" if case["rule"] == "delta" else "aspin")
    return m.eval()


def _decode_inputs(case, seed, m):
    g = _gen(seed + 1)
    H = m.mix[0].h
    states = [(0.1 * _randn(g, case["B"], H, 64, 64), 300) for _ in range(case["layers"])]
    return states, 300, _randn(g, case["B"], VOCAB)


# ------------------------------------------------------------------------------------------------------------------
# the passes

def _capture(step):
    """The step as a training program captures it: run a few times on a side stream, then recorded once."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def _scan_step(case, x, do, dS):
    mm = torch.bfloat16 if case["kind"] == "scan" else None
    names = list(x)

    def step():
        if not case["grad"]:
            with torch.no_grad():
                return assoc_scan(x["q"], x["k"], x["v"], x["la"], x.get("S0"), mm=mm, beta=x.get("beta"))
        o, S = assoc_scan(x["q"], x["k"], x["v"], x["la"], x.get("S0"), mm=mm, beta=x.get("beta"))
        grads = torch.autograd.grad([o, S], [x[n] for n in names], [do, dS])
        return (o.detach(), S.detach()) + grads

    return step


def _diag_step(x, gy, gr, gi):
    names = list(x)

    def step():
        y, (hr, hi) = scan_hip(x["u"], x["lm"], x["an"], (x["h0r"], x["h0i"]) if "h0r" in x else None)
        grads = torch.autograd.grad([y, hr, hi], [x[n] for n in names], [gy, gr, gi])
        return (y.detach(), hr.detach(), hi.detach()) + grads

    return step


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("scan", "exact"):
        x, do, dS = _scan_inputs(case, seed, torch.bfloat16 if kind == "scan" else torch.float32)
        if case["grad"]:
            for t in x.values():
                t.requires_grad_(True)
        step = _scan_step(case, x, do, dS)
    elif kind == "diag":
        x, gy, gr, gi = _diag_inputs(case, seed)
        for t in x.values():
            t.requires_grad_(True)
        step = _diag_step(x, gy, gr, gi)
    elif kind == "layer":
        m, x, target = _layer_parts(case, seed)
        x.requires_grad_(True)
        params = list(m.parameters())

        def step():  # the gradient of |y - target|^2 / 2
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y, (S, _) = m(x)
            y0 = y.detach()
            return (y0, S.detach()) + torch.autograd.grad(y, [x] + params, y0 - target)

    elif kind == "lm":
        m = _lm(case, seed)
        ids = torch.randint(0, VOCAB, (case["B"], case["T"]), generator=_gen(seed + 1), device=DEV)

        def step():
            with torch.autocast("cuda", dtype=torch.bfloat16, enabled=case["amp"]):
                return m.forward_carried(ids, case["window"])

        return {"step": step, "graph": None}
    else:
        m = _lm(case, seed)
        states, pw, lg = _decode_inputs(case, seed, m)
        dec, n = GreedyDecoder(m, case["B"], steps_per_graph=8, record_logits=True), case["n"]

        def step():
            dec.start(states, pw, lg, n)
            dec.replay(n)
            return dec.logits(n), [st[0] for st in dec.st]

        return {"step": step, "graph": None}
    if case.get("graph", kind == "layer"):
        graph, out = _capture(step)
        return {"graph": graph, "out": out, "step": step}  # the step holds the tensors that the graph reads
    return {"graph": None, "step": step}


def run(state):
    if state["graph"] is None:
        return state["step"]()
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without

def _scan_work(B, H, T, D, delta, S0, grad, es):
    """Bytes: inputs read once, outputs written once. Flops: the chunked form's dense products at 64 tokens a chunk (a
    head-token: forward 4 D (64 + D), backward 2.5 times that; the delta rule about twice the plain one's)."""
    n, s, gates = B * H * T * D * es, B * H * D * D * 4, B * H * T * 4 * (2 if delta else 1)
    by = 4 * n + gates + s * (2 if S0 else 1)
    fl = B * H * T * 4.0 * D * (64 + D) * (2 if delta else 1)
    if grad:
        by += 7 * n + 2 * gates + s * (2 if S0 else 1)
        fl *= 3.5
    return by, fl


def work(case):
    kind = case["kind"]
    if kind in ("scan", "exact"):
        by, fl = _scan_work(case["B"], case["H"], case["T"], case["D"], case["rule"] == "delta", case["S0"],
                            case["grad"], 2 if kind == "scan" else 4)
        return {"bytes": by, "flops": fl}
    if kind == "diag":
        n = case["B"] * case["T"] * case["D"]
        return {"bytes": 48 * n, "flops": 40.0 * n}
    d, B = case["d"], case["B"]
    delta = case["rule"] == "delta"
    if kind == "layer":
        H, n = d // case["head_dim"], B * case["T"]
        _, fl = _scan_work(B, H, case["T"], case["head_dim"], delta, False, True, 2)
        return {"bytes": 4 * n * d * 4 + 4 * d * d * 4 * 2, "flops": fl + 3 * 2.0 * n * 4 * d * d}
    if kind == "lm":
        n = B * case["T"]
        _, fl = _scan_work(B, d // 64, case["T"], 64, delta, False, False, 4)
        last = B * (case["T"] - case["window"] * ((case["T"] - 1) // case["window"]))
        weights = 4 * (12 * d * d * case["layers"] + VOCAB * d)
        return {"bytes": weights + 4 * n * d + 4 * last * VOCAB,
                "flops": case["layers"] * (fl + 24.0 * n * d * d) + 2.0 * last * VOCAB * d}
    steps, H = case["n"] - 1, d // 64
    per = 4 * (12 * d * d * case["layers"] + VOCAB * d) + 2 * 4 * B * H * 4096 * case["layers"] + 4 * B * VOCAB
    return {"bytes": steps * per, "flops": steps * 2.0 * B * (12 * d * d * case["layers"] + VOCAB * d)}


# ------------------------------------------------------------------------------------------------------------------
# how far another correct implementation at the same precision may be

def tolerance(case):
    kind = case["kind"]
    if kind == "scan":  # bf16 operands, intermediates and outputs
        return {"rel": 2e-2, "max": 0.5}
    if kind == "exact":  # fp32 throughout, sums over the key width and the context
        return {"rel": 3e-5, "max": 1.5e-3}
    if kind == "diag":  # fp32 throughout, sums over the context
        return {"rel": 4e-5, "max": 2e-3}
    if kind == "layer":  # bf16 autocast
        return {"rel": 3e-2, "max": 0.9}
    if kind == "lm":  # bf16 through all layers
        return {"rel": 3e-2, "max": 0.9}
    return {"rel": 1e-3, "max": 2e-2}  # fp32 decode, rounding fed back through the steps


# ------------------------------------------------------------------------------------------------------------------
# the same in 64 bits, plain torch

def _scan64(q, k, v, la, beta, S0, C=64):
    """The chunked scan in fp64: within a chunk the decayed scores, across chunks the carried state."""
    B, H, T, D = q.shape
    S = torch.zeros(B, H, D, v.shape[-1], dtype=torch.float64, device=q.device) if S0 is None else S0
    outs = []
    for s in range(0, T, C):
        qc, kc, vc, L = q[:, :, s:s + C], k[:, :, s:s + C], v[:, :, s:s + C], la[:, :, s:s + C].cumsum(-1)
        n = L.shape[-1]
        tri = torch.ones(n, n, dtype=torch.bool, device=q.device).tril()
        dec = torch.exp((L.unsqueeze(-1) - L.unsqueeze(-2)).masked_fill(~tri, -math.inf))
        eL = torch.exp(L).unsqueeze(-1)
        u = vc
        if beta is not None:
            b = beta[:, :, s:s + C]
            N = (kc @ kc.transpose(-1, -2) * dec).tril(-1) * b.unsqueeze(-2)
            N = N + torch.eye(n, dtype=torch.float64, device=q.device)
            r = torch.linalg.solve_triangular(N, vc - eL * (kc @ S), upper=False, unitriangular=True)
            u = r * b.unsqueeze(-1)
        outs.append(eL * (qc @ S) + (qc @ kc.transpose(-1, -2) * dec) @ u)
        w = torch.exp(L[..., -1:] - L).unsqueeze(-1)
        S = torch.exp(L[..., -1:]).unsqueeze(-1) * S + (kc * w).transpose(-1, -2) @ u
    return torch.cat(outs, 2), S


def _rot64(x, theta, pos):
    a = pos.view(1, 1, -1, 1) * theta.view(1, theta.shape[0], 1, -1)
    c, s = torch.cos(a), torch.sin(a)
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * c - o * s, e * s + o * c), -1).flatten(-2)


def _rms64(o, w):
    return o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + torch.finfo(torch.float32).eps) * w


def _carrier64(P, x, delta, state=None):
    """One carrier layer in fp64 from its parameters P (name -> fp64 tensor); state (S, p0) of a previous window."""
    B, T, d = x.shape
    H = P["A"].shape[0]
    z = F.layer_norm(x, (d,), P["ln.weight"], P["ln.bias"], 1e-5)
    q, k, v = (F.normalize((z @ P[n + ".weight"].t()).view(B, T, H, d // H).transpose(1, 2), dim=-1) for n in "qkv")
    la = (-F.softplus(z @ P["wa.weight"].t() + P["wa.bias"]) * torch.exp(P["A"])).transpose(1, 2)
    beta = None
    if delta:
        beta = torch.sigmoid(z @ P["wb.weight"].t() + P["wb.bias"]).transpose(1, 2)
    else:
        k = k * torch.sigmoid(z @ P["wi.weight"].t() + P["wi.bias"]).transpose(1, 2).unsqueeze(-1)
    pos = torch.arange(T, device=x.device, dtype=torch.float64)
    q, k = _rot64(q, P["theta"], pos), _rot64(k, P["theta"], pos)
    S0 = None
    if state is not None:
        S0, p0 = state
        back = torch.full((S0.shape[-1],), -float(p0), device=x.device, dtype=torch.float64)
        S0 = _rot64(S0.transpose(-1, -2), P["theta"], back).transpose(-1, -2)
    o, S = _scan64(q, k, v, la, beta, S0)
    o = _rms64(o, P["on.weight"]).transpose(1, 2).reshape(B, T, d)
    return x + (o @ P["o.weight"].t()) * torch.sigmoid(P["gate"]), (S, T)


def _mlp64(P, x):
    h = F.layer_norm(x, (x.shape[-1],), P["n.weight"], P["n.bias"], 1e-5)
    return x + F.gelu(h @ P["a.weight"].t() + P["a.bias"]) @ P["b.weight"].t() + P["b.bias"]


def _params64(m):
    return {n: p.detach().double() for n, p in m.named_parameters()}


def _part(P, prefix):
    return {n[len(prefix):]: t for n, t in P.items() if n.startswith(prefix)}


def _window64(case, P, h, states):
    for i in range(case["layers"]):
        h, states[i] = _carrier64(_part(P, "mix.%d." % i), h, case["rule"] == "delta", states[i])
        h = _mlp64(_part(P, "mlp.%d." % i), h)
    return h


def _head64(P, h):
    return F.layer_norm(h, (h.shape[-1],), P["n.weight"], P["n.bias"], 1e-5) @ P["e.weight"].t()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("scan", "exact"):
        x, do, dS = _scan_inputs(case, seed, torch.bfloat16 if kind == "scan" else torch.float32)
        x = {n: t.double().requires_grad_(case["grad"]) for n, t in x.items()}
        o, S = _scan64(x["q"], x["k"], x["v"], x["la"], x.get("beta"), x.get("S0"))
        if not case["grad"]:
            return o, S
        grads = torch.autograd.grad([o, S], list(x.values()), [do.double(), dS.double()])
        return (o.detach(), S.detach()) + grads
    if kind == "diag":
        x, gy, gr, gi = _diag_inputs(case, seed)
        x = {n: t.double().requires_grad_(True) for n, t in x.items()}
        lam = torch.polar(torch.exp(x["lm"]), x["an"]).unbind(1)
        h = torch.complex(x["h0r"], x["h0i"]) if "h0r" in x else torch.zeros_like(lam[0])
        hs = []
        for lt, ut in zip(lam, x["u"].unbind(1)):
            h = lt * h + ut
            hs.append(h.real)
        y = torch.stack(hs, 1)
        grads = torch.autograd.grad([y, h.real, h.imag], list(x.values()), [gy.double(), gr.double(), gi.double()])
        return (y.detach(), h.real.detach(), h.imag.detach()) + grads
    if kind == "layer":
        m, x, target = _layer_parts(case, seed)
        P = {n: t.requires_grad_(True) for n, t in _params64(m).items()}
        x = x.double().requires_grad_(True)
        y, (S, _) = _carrier64(P, x, case["rule"] == "delta")
        y0 = y.detach()
        grads = torch.autograd.grad(y, [x] + list(P.values()), y0 - target.double())
        return (y0, S.detach()) + grads
    with torch.no_grad():
        m = _lm(case, seed)
        P = _params64(m)
        states = [None] * case["layers"]
        if kind == "lm":
            ids = torch.randint(0, VOCAB, (case["B"], case["T"]), generator=_gen(seed + 1), device=DEV)
            for s in range(0, case["T"], case["window"]):
                x = ids[:, s:s + case["window"]]
                h = _window64(case, P, P["e.weight"][x] + P["p.weight"][:x.shape[1]], states)
            return _head64(P, h)
        given, pw, lg = _decode_inputs(case, seed, m)
        states = [(S.double(), p0) for S, p0 in given]
        lgs, lg = [lg.double()], lg.double()
        for step in range(case["n"] - 1):
            h = (P["e.weight"][lg.argmax(-1)] + P["p.weight"][(pw + step) % CTX]).unsqueeze(1)
            lg = _head64(P, _window64(case, P, h, states))[:, 0]
            lgs.append(lg)
        return torch.stack(lgs, 1), [S for S, _ in states]
