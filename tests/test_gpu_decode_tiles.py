"""The decode step's dense layers where a workgroup takes two column tiles (a partial last group, a ragged last tile, a
partial row block) and the one-wave GEMV with operands left out, against fp64 torch; the step tail's argmax at its
edges.

Tolerance: sums of K fp32 products in any order, each within K 2^-24 of the sum of magnitudes at the worst and about
sqrt(K) 2^-24 as rounding errors go: 1e-5 of the largest output holds both at these K with inputs of unit size."""
import pytest
import torch
import torch.nn.functional as F

from pragnosia_amd import ops

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b).abs().max() / b.abs().max()).item()


def _rand(seed):
    g = torch.Generator("cuda").manual_seed(seed)
    return lambda *s: torch.randn(*s, device="cuda", generator=g)


# 145 tiles in 73 groups, 193 in 97 (an odd count and a ragged tile), 512 tiles at one row block, one tile more than two
@pytest.mark.parametrize("B,K,N", [(32, 768, 2316), (47, 768, 2316), (17, 768, 3081), (9, 768, 8192), (48, 512, 2056),
                                   (33, 1024, 4100)])
@pytest.mark.parametrize("mode", [0, 1])
def test_two_tiles_a_workgroup(B, K, N, mode):
    r = _rand(B + N)
    x, W, nw, nb, bias, resid = r(B, K) + 0.5, r(N, K) * 0.05, 1 + 0.1 * r(K), r(K), r(N), r(B, N)
    if mode == 1:
        Wt, csum, b = ops.decode_gemm_ln(W, nw, nb, bias)
        y = torch.ops.pragnosia.decode_gemm(x, Wt, N, 1, csum, 1e-5, b, None, 1, resid)
        z = F.layer_norm(x.double(), (K,), nw.double(), nb.double(), 1e-5)
    else:
        y = torch.ops.pragnosia.decode_gemm(x, ops.decode_gemm_tile(W), N, 0, None, 0.0, bias, None, 1, resid)
        z = x.double()
    want = F.gelu(z @ W.double().t() + bias.double()) + resid.double()
    assert _rel(y, want) < 1e-5


@pytest.mark.parametrize("B,K,N", [(32, 3072, 776), (20, 3072, 769), (48, 2048, 500)])
def test_two_tiles_accumulating(B, K, N):
    r = _rand(B + N)
    x, W, bias, resid = r(B, K), r(N, K) * 0.05, r(N), r(B, N)
    y = resid.clone()
    torch.ops.pragnosia.decode_gemm_acc_(x, ops.decode_gemm_tile(W), 0, 0.0, bias, None, y)
    assert _rel(y, x.double() @ W.double().t() + bias.double() + resid.double()) < 1e-5


@pytest.mark.parametrize("given", ["none", "norm_bias", "bias", "scale", "resid"])
@pytest.mark.parametrize("B,K,N", [(1, 256, 5), (2, 768, 2316), (3, 1024, 130), (4, 2048, 33)])
def test_gemv_with_operands_left_out(given, B, K, N):
    r = _rand(B + K + N)
    x, W, nw = r(B, K), r(N, K) * 0.05, 1 + 0.1 * r(K)
    nb = r(K) if given == "norm_bias" else None
    bias = r(N) if given == "bias" else None
    scale = torch.rand(1, device="cuda") + 0.5 if given == "scale" else None
    resid = r(B, N) if given == "resid" else None
    d = lambda t, z: z if t is None else t.double()
    for ln in (True, False):
        if (ln and K > 1024) or (not ln and nb is not None):  # a LayerNorm'd row is at most 1024 wide
            continue
        y = torch.ops.pragnosia.decode_gemv(x, W, nw if ln else None, nb if ln else None, 1e-5, bias, scale, 0, resid)
        z = F.layer_norm(x.double(), (K,), nw.double(), None if nb is None else nb.double(), 1e-5) if ln else x.double()
        assert _rel(y, z @ W.double().t() * d(scale, 1.0) + d(bias, 0.0) + d(resid, 0.0)) < 1e-5


@pytest.mark.parametrize("V", [1, 5, 63, 64, 1023, 1025, 8193])
def test_decode_tail_argmax_edges(V):
    """The tail's argmax by ordered keys is torch's: waves and threads without a logit, the maximum in every kind of
    place, all values negative, -inf throughout, equal zeros of both signs, infinities, NaN of either sign."""
    from pragnosia_amd.ops import decode_tail
    g = torch.Generator(device="cuda").manual_seed(V)
    lg = torch.randn(10, V, device="cuda", generator=g)
    lg[0, 0] = lg[1, V - 1] = lg[2, V // 2] = 9.0
    lg[3] = -lg[3].abs() - 1.0
    lg[4] = -float("inf")
    lg[5] = -0.0
    lg[5, V // 2:] = 0.0
    lg[6, V // 3] = float("inf")
    lg[7, V // 2] = -float("nan")
    lg[7, V - 1] = float("nan")
    lg[8] = float("nan")
    lg[9] = 1e-42  # below the normal range
    B, d = lg.shape[0], 40
    emb, pemb = torch.randn(V, d, device="cuda", generator=g), torch.randn(7, d, device="cuda", generator=g)
    ctr, pos = torch.tensor([0, -1], device="cuda"), torch.tensor([3, -1], device="cuda")
    out = torch.zeros(1, B, dtype=torch.long, device="cuda")
    tok, h = torch.zeros(B, 1, dtype=torch.long, device="cuda"), torch.zeros(B, d, device="cuda")
    decode_tail(lg, emb, pemb, ctr[0], ctr[1], pos[0], pos[1], out, tok, h, None, None)
    # torch's rule from its parts: the first NaN if there is one, else the first index of the maximum
    ref = lg.cpu()
    best = torch.where(ref.isnan().any(1, keepdim=True), ref.isnan(), ref == ref.amax(1, keepdim=True))
    want = best.int().argmax(1).cuda()
    assert torch.equal(out[0], want) and torch.equal(tok.view(-1), want)
    assert torch.equal(h, emb[want] + pemb[4])
