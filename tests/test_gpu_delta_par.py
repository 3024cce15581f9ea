"""GPU: the chunk-parallel form of the delta scan (`pragnosia_aspin_delta_par_fwd` / `_bwd`) against the
one-workgroup-a-scan kernels, which the oracle comparisons of test_gpu_delta.py hold. The two perform the same
operations on the same rounded operands and sum in the same order, so at head dim 128 (the same two-kernel backward)
everything is equal bit for bit; at head dim 64 the other backward is one fused kernel that rounds where this one does
but sums the decay and strength gradients in another order: outputs and states equal, gradients to bf16 rounding (2^-8)
of their largest value."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _inputs(B, H, T, D, s0, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    q, k = (F.normalize(r(B, H, T, D), dim=-1).bfloat16().cuda() for _ in range(2))
    v = r(B, H, T, D).bfloat16().cuda()
    la, be = F.logsigmoid(r(B, H, T) + 3).cuda(), torch.sigmoid(r(B, H, T)).cuda()
    S0 = (0.1 * r(B, H, D, D)).cuda() if s0 else None
    return (q, k, v, la, be, S0), r(B, H, T, D).bfloat16().cuda(), r(B, H, D, D).cuda()


def _both(x, do, dS, monkeypatch):
    from pragnosia_amd import ops
    res = []
    for par in (False, True):
        monkeypatch.setattr(ops, "delta_parallel", lambda *a, par=par: par)
        o, S, sent, W, X = ops.aspin_delta(*x, True)
        res.append((o, S, sent, W, X) + ops.aspin_delta_bwd(*x[:5], sent, W, X, do, dS))
    return res


# one chunk and its edges; lengths around a turn of the copying waves' register sets (6 at 64, 4 at 128); heads past a
# multiple of 8 (grid padding) and past one round of workgroups
@pytest.mark.parametrize("B,H,T,D,s0", [
    (1, 1, 1, 64, False), (1, 3, 63, 64, True), (1, 1, 64, 64, True), (2, 1, 65, 64, True), (1, 2, 320, 64, False),
    (3, 3, 384, 64, True), (1, 2, 385, 64, True), (1, 1, 833, 64, True), (7, 10, 130, 64, True),
    (1, 1, 17, 128, True), (1, 3, 64, 128, False), (3, 3, 200, 128, True), (1, 2, 256, 128, True),
    (1, 1, 321, 128, True), (2, 17, 130, 128, True),
])
def test_matches_one_workgroup_per_scan(B, H, T, D, s0, monkeypatch):
    x, do, dS = _inputs(B, H, T, D, s0, seed=T + D)
    a, b = _both(x, do, dS, monkeypatch)
    names = "o S sent W X dq dk dv dla dbeta dS0".split()
    for i, (n, p, q) in enumerate(zip(names, a, b)):
        if i < 5 or D == 128:
            assert torch.equal(p, q), n
        else:
            assert (p.float() - q.float()).abs().max() <= 2.0 ** -8 * p.float().abs().max(), n


@pytest.mark.parametrize("maps", [False, True])
@pytest.mark.parametrize("B,H,T,window,s0", [(1, 2, 200, 64, True), (2, 5, 448, 128, False), (1, 1, 1000, 192, True),
                                             (1, 3, 768, 256, True)])
def test_windows_match_the_window_loop(B, H, T, window, s0, maps, monkeypatch):
    """Carried windows, in one walk and as the windows' affine maps, against one call a window with the state rebased
    between (ragged last window and chunk): the state is rotated in fp32 every way, by the rebase kernel there, in the
    walk or the maps' chain here; the maps come from the same bf16 operands as the window's own pass."""
    from pragnosia_amd import ops
    monkeypatch.setattr(ops, "delta_window_maps", lambda *a: maps)
    x, _, _ = _inputs(B, H, T, 64, s0, seed=T)
    theta = (torch.rand(H, 32, generator=torch.Generator().manual_seed(1)) * 0.1).cuda()
    o, S = ops.aspin_delta_windows(*x, theta, window)
    st, outs = x[5], []
    for s in range(0, T, window):
        if s:
            st = ops.aspin_rebase(st, theta, None, float(window))
        ow, st, _, _, _ = ops.aspin_delta(*(t[:, :, s:s + window] for t in x[:5]), st, False)
        outs.append(ow)
    ref = torch.cat(outs, 2).float()
    assert (o.float() - ref).abs().max() <= 2.0 ** -7 * ref.abs().max()
    assert (S - st).abs().max() <= 2.0 ** -8 * st.abs().max()


def test_fused_forward_keeps_states_on_chip():
    """The scan that keeps nothing for its backward takes no memory beside o and S either, at a size whose plain forward
    runs chunk-parallel and writes 22 MiB of states, W and X (the allocator may hand out up to 1 MiB more than asked
    for, in two arrays), and gives the plain forward's outputs."""
    from pragnosia_amd import ops
    x, _, _ = _inputs(2, 12, 2560, 64, True, seed=3)
    assert ops.delta_parallel(24, 40, 64, False)
    o, S, _, _, _ = ops.aspin_delta(*x, True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    of, Sf = ops.aspin_delta_fused(*x)
    peak = torch.cuda.max_memory_allocated() - before
    assert torch.equal(o, of) and torch.equal(S, Sf)
    assert peak <= 2 * o.numel() + 4 * S.numel() + (2 << 20), peak
