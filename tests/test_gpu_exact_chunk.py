"""GPU parity of the exact scan's chunked form (fp32 operands on the fp32 matrix cores, `aspin_exact` from
EXACT_CHUNK_MIN_T tokens) at the sizes where its tiles end: chunks of 64 tokens, key and value tiles of 64 in blocks of
16, 16-byte or 4-byte loads.

Tolerance: every output is a sum of fp32 products along at most T + Dk + Dv <= 1000 terms, so a relative error of a few
times sqrt(1000) eps = 1.9e-6; 2e-5 in the maximum norm over the result's largest value leaves a factor of ten."""
import pytest
import torch
import torch.nn.functional as F

from oracle import aspin as O

pytestmark = pytest.mark.gpu

TOL = 2e-5


@pytest.fixture(autouse=True)
def _chunked(monkeypatch):
    """Every size that the chunked form takes runs in it, also where token by token is the faster one."""
    from pragnosia_amd import ops
    monkeypatch.setattr(ops, "exact_chunk_pays", lambda *a: True)


def _inputs(B, H, T, Dk, Dv, delta, seed, s0, steep=False):
    g = torch.Generator().manual_seed(seed)
    q, v = torch.randn(B, H, T, Dk, generator=g), torch.randn(B, H, T, Dv, generator=g)
    k = F.normalize(torch.randn(B, H, T, Dk, generator=g), dim=-1)
    la = -torch.rand(B, H, T, generator=g) * 20 if steep else F.logsigmoid(torch.randn(B, H, T, generator=g) + 3.0)
    x = {"q": q, "k": k, "v": v, "la": la}
    if delta:
        x["beta"] = torch.sigmoid(torch.randn(B, H, T, generator=g))
    if s0:
        x["S0"] = torch.randn(B, H, Dk, Dv, generator=g) * 0.1
    return x, torch.randn(B, H, T, Dv, generator=g), torch.randn(B, H, Dk, Dv, generator=g)


def _check(x, wo, wS, place=lambda t: t.cuda()):
    from pragnosia_amd.assoc import assoc_scan
    r = {n: t.double().requires_grad_(True) for n, t in x.items()}
    yr, Sr = O.assoc_scan(r["q"], r["k"], r["v"], r["la"], r.get("S0"), chunk=16, beta=r.get("beta"))
    gr = torch.autograd.grad([yr, Sr], list(r.values()), [wo.double(), wS.double()])
    d = {n: place(t).requires_grad_(True) for n, t in x.items()}
    y, S = assoc_scan(d["q"], d["k"], d["v"], d["la"], d.get("S0"), beta=d.get("beta"))
    gd = torch.autograd.grad([y, S], list(d.values()), [wo.cuda(), wS.cuda()])
    errs = {}
    for n, a, b in zip(["o", "S"] + ["d" + n for n in x], [y, S, *gd], [yr, Sr, *gr]):
        errs[n] = ((a.detach().double().cpu() - b).abs().max() / b.abs().max()).item()
    assert max(errs.values()) < TOL, errs


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("B,H,T,Dk,Dv,s0", [
    (1, 1, 32, 16, 16, False),     # half a chunk, one tile
    (1, 2, 63, 64, 64, True), (1, 2, 64, 64, 64, True), (1, 1, 65, 64, 64, False),   # a chunk's edges
    (2, 1, 200, 17, 33, True),     # rows that start off 16 bytes: 4-byte loads, partial blocks both ways
    (1, 1, 129, 100, 20, True),    # 16-byte loads, partial blocks
    (1, 2, 97, 4, 130, True),      # less than one key block; value tiles past 128
    (3, 3, 128, 80, 144, True),    # two key tiles a wave, three value tiles; groups past a multiple of 8
    (1, 1, 70, 192, 176, True), (1, 1, 40, 256, 16, False), (1, 1, 66, 320, 48, True), (1, 1, 90, 384, 24, True),
])
def test_chunked_exact_scan_matches_oracle(delta, B, H, T, Dk, Dv, s0):
    _check(*_inputs(B, H, T, Dk, Dv, delta, seed=T + Dk, s0=s0))


def test_chunked_plain_rule_keys_past_384():
    _check(*_inputs(1, 1, 50, 400, 24, False, seed=7, s0=True))


@pytest.mark.parametrize("delta", [False, True])
def test_chunked_steep_decays_and_resets(delta):
    """Log-decays down to -20 a token, and -inf (a reset: the state is dropped, no NaN)."""
    x, wo, wS = _inputs(1, 2, 150, 32, 32, delta, seed=11, s0=True, steep=True)
    _check(x, wo, wS)
    from pragnosia_amd.assoc import assoc_scan
    dev = {n: t.cuda() for n, t in x.items()}
    dev["la"][:, :, 100] = -float("inf")
    y, S = assoc_scan(dev["q"], dev["k"], dev["v"], dev["la"], dev["S0"], beta=dev.get("beta"))
    cut = {n: t[:, :, 100:] for n, t in dev.items() if n != "S0"}
    cut["la"] = cut["la"].clone()
    cut["la"][:, :, 0] = 0.0   # no state to decay
    y2, S2 = assoc_scan(cut["q"], cut["k"], cut["v"], cut["la"], None, beta=cut.get("beta"))
    assert (y[:, :, 100:] - y2).abs().max() < TOL * y2.abs().max() and (S - S2).abs().max() < TOL * S2.abs().max()


@pytest.mark.parametrize("delta", [False, True])
def test_chunked_off_16_byte_addresses(delta):
    """Contiguous operands that start 4 bytes past a 16-byte address take the 4-byte loads."""
    def shifted(t):
        buf = torch.empty(t.numel() + 1, device="cuda")
        buf[1:] = t.reshape(-1).cuda()
        return buf[1:].view(t.shape).detach()
    _check(*_inputs(1, 2, 100, 64, 48, delta, seed=13, s0=True), place=shifted)


@pytest.mark.parametrize("delta,name", [(r, n) for r in (False, True) for n in "q k v la beta S0 do dS".split()
                                        if r or n != "beta"])
def test_chunked_non_finite_values_stay_where_the_recurrence_takes_them(delta, name, monkeypatch):
    """An infinity or a NaN in one place of one operand: every output that is finite token by token is finite here, and
    the same, and no other one is (ragged rows and tiles; tokens at a chunk's start, inside blocks and at the end)."""
    from pragnosia_amd import ops
    B, H, T, Dk, Dv = 1, 2, 150, 34, 70
    x, do, dS = _inputs(B, H, T, Dk, Dv, delta, seed=17, s0=True)

    def run(a, min_t):
        monkeypatch.setattr(ops, "EXACT_CHUNK_MIN_T", min_t)
        args = (a["q"], a["k"], a["v"], a["la"], a.get("beta"))
        o, S, ckpt, resid = ops.aspin_exact(*args, a["S0"], True)
        return o, S, *ops.aspin_exact_bwd(*args, ckpt, resid if resid.numel() else None, a["do"], a["dS"])

    for val in (float("inf"), float("nan")):
        for s in (64, 90, 149) if name not in ("S0", "dS") else (3,):
            a = {n: t.clone().cuda() for n, t in {**x, "do": do, "dS": dS}.items()}
            a[name][(0, 1, s) if name in ("la", "beta") else (0, 1, s, 7)] = val
            for n, got, want in zip("o S dq dk dv dla dbeta dS0".split(), run(a, 32), run(a, 1 << 30)):
                fine = want.isfinite()
                assert torch.equal(got.isfinite(), fine), (val, s, n, (got.isfinite() != fine).nonzero()[:4])
                assert not fine.any() or (got - want)[fine].abs().max() < TOL * want[fine].abs().max(), (val, s, n)


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("B,H,T,Dk,Dv,mib", [(1, 2, 12000, 48, 32, 1), (3, 5, 4400, 32, 64, 4),
                                             (20, 9, 130, 64, 64, 1)])
def test_chunked_without_a_backward_bounds_its_scratch(delta, B, H, T, Dk, Dv, mib, monkeypatch):
    """Without gradients the states, scores and inverses are scratch of a piece of the sequences (or of a group of
    heads) at a time: the same outputs bit for bit, and no more memory than the bound (or 16 chunks of a head, a piece's
    least) beside the outputs. The allocator may hand out up to 1 MiB more than asked for, in five arrays; whole, the
    scratch is 8 MiB and more."""
    from pragnosia_amd import ops
    x, _, _ = _inputs(B, H, T, Dk, Dv, delta, seed=19, s0=True)
    a = [x[n].cuda() if n in x else None for n in ("q", "k", "v", "la", "beta", "S0")]
    o, S, _, _ = ops.aspin_exact(*a, True)
    monkeypatch.setattr(ops, "EXACT_SCRATCH_BYTES", mib << 20)
    heads, chunks = ops._exact_pieces(B * H, T, Dk, Dv, delta)
    assert heads < B * H or 64 * chunks < T
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    o2, S2, _, _ = ops.aspin_exact(*a, False)
    peak = torch.cuda.max_memory_allocated() - before
    assert torch.equal(o, o2) and torch.equal(S, S2)
    per = 4 * (Dk * Dv + 64 * 66 + (2 * 64 * 64 + 64 * (2 * Dv + (Dk + 15) // 16 * 16) if delta else 0))
    assert peak <= max(mib << 20, 16 * per) + 4 * (o.numel() + S.numel()) + (5 << 20), peak
