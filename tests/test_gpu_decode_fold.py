"""Folding a model's dense layers for the batched decode step in one launch, against the one-layer folds."""
import pytest
import torch

from pragnosia_amd import PragnosiaError, ops

pytestmark = pytest.mark.gpu

# rows per block, K: the carrier projection's five blocks, ragged last tiles, one row, one 16-wide step, a tall head
LAYERS = [([768, 768, 768, 12, 12], 768), ([64], 128), ([5, 3, 40], 256), ([1], 16), ([17, 2], 48), ([4097], 128)]


def _layers(seed, dtype=torch.float32, shift=0):
    g = torch.Generator("cuda").manual_seed(seed)

    def t(*s):
        n = torch.Size(s).numel()
        return torch.randn(n + shift, generator=g, device="cuda")[shift:].view(s).to(dtype)

    src = []
    for rows, K in LAYERS:
        ws, N = [t(n, K) for n in rows], sum(rows)
        src += [(ws, 1 + t(K), t(K), t(N)), (ws, 1 + t(K), t(K), None), (ws, 1 + t(16), None, None),
                (ws, None, None, None)]
    return src


def _dests(src):
    e = lambda n: torch.full((n,), float("nan"), device="cuda")
    out = []
    for ws, cs, lb, bias in src:
        N, K = sum(w.shape[0] for w in ws), ws[0].shape[1]
        out.append((e((N + 15) // 16 * 16 * K), e(N) if lb is not None else None, e(N) if lb is not None else None))
    return out


# shift 1: sources that are not 16-byte aligned; bf16: converted first
@pytest.mark.parametrize("dtype,shift", [(torch.float32, 0), (torch.float32, 1), (torch.bfloat16, 0)])
def test_fold_matches_the_single_layer_folds(dtype, shift):
    src = _layers(3, dtype, shift)
    dst = _dests(src)
    fold = ops.DecodeFold(src, dst)
    fold.run(src)
    for turn in range(2):  # the second time with other sources of the same shapes
        for (ws, cs, lb, bias), (Wt, csum, bout) in zip(src, dst):
            W = torch.cat(ws).float()
            if lb is None:
                assert torch.equal(Wt, ops.decode_gemm_tile(W, None if cs is None else cs.float()))
                continue
            want = ops.decode_gemm_ln(W, cs.float(), lb.float(), None if bias is None else bias.float())
            assert torch.equal(Wt, want[0])
            # both sum in fp64 and round once: half an fp32 unit of the value each, and the sums' own 2^-53 K terms
            for got, ref, mag in ((csum, want[1], (W * cs.float()).abs().sum(1)),
                                  (bout, want[2], (W * lb.float()).abs().sum(1))):
                assert ((got - ref).abs() <= 2.0**-23 * ref.abs() + 1e-12 * mag).all()
        src = _layers(4, dtype, shift)
        fold.run(src)


def test_fold_refuses_other_shapes():
    src = _layers(3)
    fold = ops.DecodeFold(src, _dests(src))
    ws, cs, lb, bias = src[0]
    for bad in ((ws[:-1], cs, lb, bias), (ws, cs[:-4], lb, bias), (ws, cs, None, bias), (ws, cs, lb, bias[:-1]),
                ([ws[0][:-1]] + ws[1:], cs, lb, bias), ([w.cpu() for w in ws], cs, lb, bias)):
        with pytest.raises(PragnosiaError):
            fold.run([bad] + src[1:])
    with pytest.raises(PragnosiaError):
        fold.run(src[1:])
