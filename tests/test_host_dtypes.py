"""Every tensor whose address an op hands to the library has a dtype that the op states, not torch's default one: the
kernels take a buffer's element size for granted, so one in a narrower default would be written past its end. On the
CPU, with the library replaced by one that accepts every call and float64 (which no call below passes on) as the
default."""
import pytest
import torch

from pragnosia_amd import ops


class _Library:
    def __getattr__(self, name):
        sizes = name.endswith(("_bytes", "_partials"))
        return lambda *a: 6144 if sizes else 0


@pytest.fixture
def handed(monkeypatch):
    seen = []
    monkeypatch.setattr(ops, "_require_gpu", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda t: None)
    monkeypatch.setattr(ops, "lib", lambda: _Library())
    monkeypatch.setattr(ops, "_ptr", lambda t: seen.append(None if t is None else t.dtype))
    torch.set_default_dtype(torch.float64)
    yield seen
    torch.set_default_dtype(torch.float32)


def f(*s):
    return torch.zeros(*s, dtype=torch.float32)


def b(*s):
    return torch.zeros(*s, dtype=torch.bfloat16)


def exact(delta):
    x = (f(1, 2, 70, 20), f(1, 2, 70, 20), f(1, 2, 70, 24), f(1, 2, 70), f(1, 2, 70) if delta else None)
    o, S, ckpt, resid = ops.aspin_exact(*x, None, True)
    ops.aspin_exact_bwd(*x, ckpt, resid, o, None)


def diag():
    x = (f(2, 5, 8), f(2, 5, 8), f(2, 5, 8), f(2, 8), f(2, 8))
    y, hr, hi, im = ops.diag_scan(*x)
    ops.diag_scan_bwd(y, None, None, x[1], x[2], y, im, x[3], x[4])


def prep():
    p, s = b(2, 10, 3, 64), b(2, 3, 10, 64)
    ops.aspin_prep_bwd(p, p, p, f(2, 10, 3), f(3, 32), torch.arange(10), s, s, s)


def prep_proj():
    s = b(2, 3, 10, 64)
    ops.aspin_prep_proj_bwd(b(2, 10, 582), 3, f(3), f(3), None, None, f(3), 0.0, False, f(3, 32), torch.arange(10), s,
                            s, s, f(2, 3, 10), None)


def delta():
    x = (b(1, 2, 400, 64), b(1, 2, 400, 64), b(1, 2, 400, 64), f(1, 2, 400), f(1, 2, 400))
    o, S, sent, W, X = ops.aspin_delta(*x, None, True)
    ops.aspin_delta_bwd(*x, sent, W, X, o, None)
    ops.aspin_delta_windows(*x, None, f(2, 32), 128)


@pytest.mark.parametrize("call", [lambda: exact(False), lambda: exact(True), diag, prep, prep_proj, delta],
                         ids=["exact", "exact_delta", "diag", "prep", "prep_proj", "delta"])
def test_buffers_do_not_take_the_default_dtype(handed, call):
    call()
    assert handed and torch.float64 not in handed, handed


@pytest.mark.parametrize("pos", [[301, 1027], [301, torch.tensor(1027.0, dtype=torch.float32)]])
def test_decode_positions_keep_fp32(pos):
    """A position handed to the decoder as a number reaches its fp32 buffer unrounded under a 16-bit default."""
    from pragnosia_amd.decode import GreedyDecoder
    dec = GreedyDecoder.__new__(GreedyDecoder)
    dec.fused, dec.p0s, dec.st = True, f(2), [(f(1, 2, 2),), (f(1, 2, 2),)]
    torch.set_default_dtype(torch.bfloat16)
    try:
        dec._load_states([(f(1, 2, 2) + 1, p) for p in pos])
        states = GreedyDecoder._static_states(dec, [(f(1, 2, 2), 301)])
    finally:
        torch.set_default_dtype(torch.float32)
    assert dec.p0s.tolist() == [301.0, 1027.0] and states[0][1].item() == 301.0
    assert all((st[0] == 1).all() for st in dec.st)
