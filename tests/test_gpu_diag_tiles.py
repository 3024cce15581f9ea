"""GPU parity of the complex diagonal scan at each channel-tile width that its dispatch picks (64, 32, 16 or 8 channels
a workgroup, by how many 64-channel tiles there are), with ragged channels and lengths around a time block's end.

Tolerance: fp32 sums along at most 1100 tokens of contributions that decay; 1e-5 in the maximum norm over the result's
largest value (the oracle comparison of the other shapes measures 1e-6 to 3e-6)."""
import pytest
import torch

from oracle import diag as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,D", [
    (20, 70, 449),     # 160 tiles: 64 channels
    (8, 150, 577),     # 80 tiles: 32 channels, 128-token blocks
    (5, 257, 513),     # 45 tiles: 16 channels, 256-token blocks
    (1, 513, 65), (2, 1024, 129), (1, 1100, 7), (1, 300, 64),   # 8 channels, 512-token blocks
    (1, 65, 40), (1, 129, 40),   # the lengths at which narrower tiles begin
])
def test_channel_tiles_match_oracle(B, T, D):
    from pragnosia_amd.scan import scan_hip
    g = torch.Generator().manual_seed(T + D)
    r = lambda *s: torch.randn(*s, generator=g)
    x = [r(B, T, D), -torch.rand(B, T, D, generator=g) * 0.2, r(B, T, D), r(B, D), r(B, D)]
    gy, gr, gi = r(B, T, D), r(B, D), r(B, D)

    def run(fn, place):
        a = [place(t).requires_grad_(True) for t in x]
        y, (hr, hi) = fn(a[0], a[1], a[2], (a[3], a[4]))
        return [y, hr, hi, *torch.autograd.grad([y, hr, hi], a, [place(gy), place(gr), place(gi)])]

    for name, a, b in zip("y hr hi du dlogmag dang dh0r dh0i".split(), run(scan_hip, lambda t: t.cuda()),
                          run(O.recurrence, lambda t: t.double())):
        err = ((a.detach().double().cpu() - b).abs().max() / b.abs().max()).item()
        assert err < 1e-5, (name, err)
