"""The language model's embedding on the CPU: the indexed form against torch's, and when it is taken."""
import pytest
import torch
import torch.nn.functional as F

from pragnosia_amd import model


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2.0 ** -20), (torch.float64, 1e-12),
                                       (torch.bfloat16, 2.0 ** -8)])
def test_indexed_form_is_the_embedding(dtype, tol):
    """Rows looked up once, often and never: the values are F.embedding's; the gradient is within the sums' rounding (at
    most 70 terms in fp32, under 2^-20 of the largest) and one rounding to the table's type of the fp64 gradient."""
    g = torch.Generator().manual_seed(0)
    W = torch.randn(50, 8, generator=g, dtype=torch.float64).to(dtype).requires_grad_()
    x = torch.randint(0, 40, (4, 90), generator=g)
    x[0, :30] = 7
    for ids in (x, x.int(), x.t(), x[1, 3]):
        y = model._rows(W, ids)
        assert y.dtype == dtype and torch.equal(y, F.embedding(ids, W))
        gy = torch.randn(y.shape, generator=g, dtype=torch.float64).to(dtype)
        got, = torch.autograd.grad(y, W, gy)
        W64 = W.detach().double().requires_grad_()
        want, = torch.autograd.grad(F.embedding(ids, W64), W64, gy.double())
        assert got.dtype == dtype and (got.double() - want).abs().max() <= tol * want.abs().max()
        assert not got[40:].any()


def test_taken_only_in_a_capture():
    """On the CPU it is nn.Embedding, with the module's own state and the same initial draw."""
    torch.manual_seed(0)
    m = model.Embedding(20, 4)
    torch.manual_seed(0)
    want = torch.nn.Embedding(20, 4)
    assert list(m.state_dict()) == ["weight"] and torch.equal(m.weight, want.weight)
    x = torch.randint(0, 20, (2, 4000))
    y = m(x)
    assert torch.equal(y, want(x)) and "Embedding" in type(y.grad_fn).__name__
