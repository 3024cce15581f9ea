"""GPU: a language model's training step captured at a size whose embedding gradient torch would form by sorting."""
import pytest
import torch

from test_gpu_training import _memset_nodes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixer", ["aspin", "dspin"])
def test_step_past_3072_tokens_records_no_memset(mixer):
    """The captured step of 4 x 800 tokens holds no memset node (and so none of the sort's kernels, whose state one
    would clear); its replays on new batches, with eager steps between them, give the eager step's gradients to the
    order of fp32 sums. An eager step's embedding is torch's."""
    from pragnosia_amd.model import Embedding, LM
    torch.manual_seed(5)
    with torch.device("cuda"):
        m = LM(vocab=1000, d=128, layers=1, mlp_mult=2, ctx=800, mixer=mixer)
    xs = torch.randint(0, 1000, (4, 801), device="cuda")
    assert xs[:, :800].numel() >= Embedding.SORTED_FROM
    assert "Embedding" in type(m.e(xs[:, :800]).grad_fn).__name__
    for p in m.parameters():
        p.grad = torch.zeros_like(p)

    def micro():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            h = m.trunk(xs[:, :800])
        m.loss(h.float(), xs[:, 1:]).backward()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            micro()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        micro()
    assert _memset_nodes(graph) == 0
    for _ in range(4):
        xs.random_(0, 1000)
        grads = []
        for run in (graph.replay, micro):
            for p in m.parameters():
                p.grad.zero_()
            run()
            torch.cuda.synchronize()
            grads.append([p.grad.clone() for p in m.parameters()])
        for (n, _), a, b in zip(m.named_parameters(), *grads):
            assert (a - b).norm() <= 1e-4 * b.norm(), n


def test_traced_trunk_past_3072_tokens():
    """A compiled trunk, which a caller may capture, takes the indexed form in one graph and gives the eager step's
    gradient to the bf16 rounding of the autocast step (as the compiled trunk's other gradients: 1e-2)."""
    from pragnosia_amd.model import LM
    torch.manual_seed(6)
    with torch.device("cuda"):
        m = LM(vocab=1000, d=128, layers=1, mlp_mult=2, ctx=800, mixer="aspin")
    xs, t = torch.randint(0, 1000, (4, 800), device="cuda"), torch.randn(4, 800, 128, device="cuda")
    grads = []
    for trunk in (torch.compile(m.trunk, backend="aot_eager", fullgraph=True), m.trunk):
        m.zero_grad()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            h = trunk(xs)
        h.float().backward(t)
        grads.append(m.e.weight.grad.clone())
    assert (grads[0] - grads[1]).norm() <= 1e-2 * grads[1].norm()
