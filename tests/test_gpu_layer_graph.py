"""GPU: one carrier layer's training step captured in a HIP graph, at the widths of the models trained on it."""
import pytest
import torch

from test_gpu_training import _memset_nodes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,head_dim,delta,T", [(384, 128, False, 400), (704, 64, False, 400), (768, 64, True, 400),
                                                (704, 176, False, 2048), (352, 176, True, 1000)])
def test_layer_step_records_no_memset(d, head_dim, delta, T):
    """The step's graph holds no memset node (a reduction of the d x d gated weight to the scalar gate's gradient would
    record one from d 384 on, and of the rotation's over 2048 positions to its frequencies' one each for q and k), and
    its replays, with eager steps and synchronisations between them, give the eager step's gradients: the gate's to fp32
    rounding of sums of d^2 terms, which cancel to some hundredths, the others to fp32 sums in another order."""
    from pragnosia_amd.assoc import AssocCarrier
    torch.manual_seed(d)
    with torch.device("cuda"):
        m = AssocCarrier(d, head_dim=head_dim, delta=delta)
    m.need_sent = False
    x, t = torch.zeros(4, T, d, device="cuda"), torch.randn(4, T, d, device="cuda")
    params = [p for n, p in m.named_parameters()]

    def step():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, _ = m(x)
        return torch.autograd.grad(y, params, t, allow_unused=True)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        out = step()
    assert _memset_nodes(graph) == 0
    gate = [n for n, _ in m.named_parameters()].index("gate")
    for _ in range(6):
        x.normal_()
        graph.replay()
        got = [None if o is None else o.clone() for o in out]
        torch.cuda.synchronize()
        eager = step()
        for (n, _), a, b in zip(m.named_parameters(), got, eager):
            assert (a is None) == (b is None) and (a is None or n == "gate" or (a - b).norm() <= 1e-4 * b.norm()), n
        got, want = got[gate], eager[gate]
        assert want.abs() > 0 and (got - want).abs() <= 1e-4 * want.abs() + 1e-3, (got.item(), want.item())


@pytest.mark.parametrize("d,B,T", [(704, 4, 2048), (256, 3, 1999)])
def test_diagonal_layer_step_records_no_memset(d, B, T):
    """SpinCarrier: the timescales, frequencies and the gate are broadcast over all tokens, and their gradients' sums
    record no memset. The replays give the eager step's gradients to the order of fp32 sums; the gate's, a sum
    that autograd rounds to the product's type, to one step of bf16 (2^-7)."""
    from pragnosia_amd.spin import SpinCarrier
    torch.manual_seed(d)
    with torch.device("cuda"):
        m = SpinCarrier(d, gated="rf")
        x, t = torch.zeros(B, T, d), torch.randn(B, T, d)
    params = list(m.parameters())

    def step():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, _ = m(x)
        return torch.autograd.grad(y, params, t)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        out = step()
    assert _memset_nodes(graph) == 0
    for _ in range(6):
        x.normal_()
        graph.replay()
        got = [o.clone() for o in out]
        torch.cuda.synchronize()
        for (n, _), a, b in zip(m.named_parameters(), got, step()):
            assert (a - b).norm() <= (2.0 ** -7 if n == "gate" else 1e-5) * b.norm(), n


@pytest.mark.parametrize("d,head_dim,delta,B,T", [(128, 64, False, 1, 1536), (128, 64, True, 3, 517),
                                                  (704, 64, False, 2, 300), (256, 128, True, 2, 2100)])
def test_padded_projection_equals_unpadded(d, head_dim, delta, B, T, monkeypatch):
    """A training step whose projection is padded for aligned rows gives the unpadded one's output, state and gradients:
    the padded columns are read by nothing and their gradient is zero. The weight gradients differ by the unpadded
    form's rounding to bf16 (2^-9 of each value), everything else by the order of sums in other GEMM tiles, at bf16."""
    from pragnosia_amd import assoc
    torch.manual_seed(d + T)
    with torch.device("cuda"):
        m = assoc.AssocCarrier(d, head_dim=head_dim, delta=delta)
        x, t = torch.randn(B, T, d, requires_grad=True), torch.randn(B, T, d)
    assert assoc._proj_padding(3 * d + 2 * m.h, B * T, True) > 0

    def step():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, (S, _) = m(x)
        return y.detach(), S.detach(), *torch.autograd.grad(y, [x, *m.parameters()], t, allow_unused=True)

    padded = step()
    monkeypatch.setattr(assoc, "PROJ_ALIGN", 1)
    for n, a, b in zip(["y", "S", "x", *dict(m.named_parameters())], padded, step()):
        assert (a is None) == (b is None), n
        if a is not None:
            assert (a - b).norm() <= 2.0 ** -8 * b.norm(), (n, ((a - b).norm() / b.norm()).item())
