"""Host-side choice of the plain forward's segment length (pure Python, no device)."""
from pragnosia_amd.ops import COMPUTE_UNITS, seg_chunks


def test_full_machine_keeps_one_workgroup_per_head():
    # 192 heads of 8 chunks already cover most compute units; so do 256 or more heads at any length
    assert seg_chunks(192, 8, range(1, 9)) == 8
    for heads in (256, 512, 4096):
        for NC in (1, 8, 64):
            assert seg_chunks(heads, NC, range(1, NC + 1)) == NC


def test_few_heads_over_many_chunks_split():
    # 24 heads of 128 chunks; one round of segments over the compute units, each walking 13 chunks
    P = seg_chunks(24, 128, range(1, 129))
    nseg = -(-128 // P)
    assert P == 13 and 24 * nseg <= COMPUTE_UNITS < 24 * (nseg + 1)
    # windowed carrying: only divisors of the window's chunk count are offered; the largest that fits is taken
    assert seg_chunks(24, 128, [1, 2, 4, 8]) == 8
    # never below two chunks, never when the walk saved is smaller than the sums' overhead
    assert seg_chunks(2, 64, range(1, 65)) == 2
    assert seg_chunks(96, 16, range(1, 17)) == 16


def test_single_chunk_and_single_candidate():
    assert seg_chunks(1, 1, [1]) == 1
    assert seg_chunks(4, 3, []) == 3


def test_backward_splits_sooner():
    # the backward's chunk step is heavier, so 96 heads of 16 chunks split for it (measured 41.8 -> 36.8 us) but
    # not for the forward (22.6 us sequential vs 26 segmented); 128 heads of 8 chunks split for neither
    assert seg_chunks(96, 16, range(1, 17), "bwd") == 8
    assert seg_chunks(96, 16, range(1, 17), "fwd") == 16
    assert seg_chunks(128, 8, range(1, 9), "bwd") == 8
    assert seg_chunks(192, 8, range(1, 9), "bwd") == 8


def test_exact_chunked_is_what_the_library_takes(monkeypatch):
    """The exact scan runs in chunked form only where the library's chunked entry points take the sizes; the rest stays
    with the token-by-token form, which takes more sequences."""
    import torch

    from pragnosia_amd import ops
    from pragnosia_amd._lib import lib
    from pragnosia_amd.ops import exact_chunked
    monkeypatch.setattr(ops, "exact_chunk_pays", lambda *a: True)
    cases = [(1, 32, 1, 1), (4, 2048, 176, 176), (1, 1 << 20, 352, 352), ((1 << 24) - 1, 32, 1, 1), (1 << 24, 32, 1, 1),
             (1, (1 << 28) - 1, 16, 16), (1, 1 << 28, 16, 16), (1 << 20, 65536, 64, 64), (1 << 20, 16384, 4, 4),
             ((1 << 24) - 1, 64, 8, 4096), (2, 100, 400, 16), (2, 100, 4097, 16), (2, 100, 16, 4097)]
    for delta in (False, True):
        for heads, T, Dk, Dv in cases:
            takes = lib().pragnosia_aspin_exact_chunk_bwd_workspace_bytes(heads, 1, T, Dk, Dv, int(delta)) >= 0
            assert exact_chunked(torch.float32, heads, T, Dk, Dv, delta) == takes, (heads, T, Dk, Dv, delta)
    assert not exact_chunked(torch.float32, 4, 31, 64, 64, False)
    assert not exact_chunked(torch.float64, 4, 64, 64, 64, False)


def test_carried_windows_take_the_faster_form():
    """The delta rule's carried windows: maps for long sequences of few heads, one walk for the rest."""
    from pragnosia_amd.ops import delta_window_maps
    for heads, T, window in ((4, 131072, 2048), (12, 32768, 1024), (12, 8192, 512), (24, 32768, 1024), (4, 4096, 256)):
        assert delta_window_maps(heads, T, window), (heads, T, window)
    for heads, T, window in ((24, 8192, 512), (12, 32768, 64), (12, 2048, 512), (96, 16384, 2048), (48, 32768, 2048),
                             (4, 1024, 4096), (1, 64, 64)):
        assert not delta_window_maps(heads, T, window), (heads, T, window)


def test_projection_padding_by_alignment_and_tokens():
    """Zero rows for a training step's projection: to a multiple of 64, from fewer tokens the further off alignment its
    rows are, never in fp32 where they are 16-byte aligned."""
    from pragnosia_amd.assoc import _proj_padding
    for width, least in ((2134, 512), (1164, 1536), (1940, 1536), (2328, 4096), (776, 4096)):
        assert _proj_padding(width, least - 1, True) == 0
        pad = _proj_padding(width, least, True)
        assert pad == -width % 64 and (width + pad) % 64 == 0
    assert _proj_padding(2304, 1 << 20, True) == 0
    assert _proj_padding(2134, 4096, False) == 42 and _proj_padding(2134, 4095, False) == 0
    assert _proj_padding(1164, 1 << 20, False) == 0


def test_delta_form_by_heads_and_chunks():
    """The chunk-parallel delta form at head dim 128: forward from six chunks where the states are wanted, else from more
    chunks the more heads there are, backward from eight; at 64 from four and five."""
    from pragnosia_amd.ops import delta_parallel
    for heads, least in ((1, 6), (12, 6), (13, 10), (18, 10), (19, 14), (32, 14)):
        assert delta_parallel(heads, least, 128, False, False)
        assert not delta_parallel(heads, least - 1, 128, False, False)
        assert delta_parallel(heads, 6, 128, False) and not delta_parallel(heads, 5, 128, False)
    assert not delta_parallel(33, 1000, 128, False) and not delta_parallel(25, 1000, 128, True)
    assert delta_parallel(24, 8, 128, True) and not delta_parallel(24, 7, 128, True)
    assert delta_parallel(64, 4, 64, False) and not delta_parallel(64, 3, 64, False)
    assert delta_parallel(96, 16, 64, False) and not delta_parallel(96, 15, 64, False)
    assert delta_parallel(64, 5, 64, True) and not delta_parallel(65, 100, 64, True)


def test_exact_form_by_heads_tokens_and_width():
    """The exact scan's chunked form where its products cost less than the token-by-token steps: wide heads, few heads over
    many tokens, and most training steps; not many narrow heads over few tokens."""
    from pragnosia_amd.ops import exact_chunk_pays
    #  heads, T, Dk, Dv, delta, grad
    for case in ((4, 32, 176, 176, False, False), (4096, 32, 16, 200, True, True), (12, 64, 64, 64, False, False),
                 (12, 32, 64, 64, True, True), (4096, 64, 64, 64, False, True), (1024, 256, 32, 32, False, False),
                 (12, 64, 64, 64, True, False), (1, 256, 8, 8, True, False)):
        assert exact_chunk_pays(*case), case
    for case in ((4096, 64, 8, 8, False, False), (4096, 64, 8, 8, False, True), (12, 32, 64, 64, True, False),
                 (1024, 64, 32, 32, True, False), (4096, 256, 16, 16, True, True), (1024, 32, 64, 64, False, False)):
        assert not exact_chunk_pays(*case), case
