"""The fused scan launch at the edges of its cut into segments and of its walk
over the segments before: one or two sub-chunks a segment, every remainder of
the records loaded ahead, more segments than one look at the flags covers."""
import numpy as np
import pytest
import torch

import test_gpu_scan as scan
import test_zz_no_alloc as no_alloc
from cases import rel_l2

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("B,T,H,N,theta,state,skip", [
    (1, 65, 2, 128, True, True, True),      # two segments of one sub-chunk
    (1, 63, 2, 64, True, True, False),      # one ragged segment, nothing published
    (1, 640, 3, 128, True, True, True),     # ten sub-chunks: segments of one
    (1, 641, 3, 128, True, True, True),     # eleven: segments of two
    (2, 300, 3, 64, False, False, True),    # five segments of one, no angles
    (64, 512, 1, 64, True, True, False),    # a grid of exactly 512 sub-chunks
    (65, 512, 1, 128, True, True, False),   # and past it
    (1, 770, 3, 64, True, False, True),     # walks of 1 .. 6 records, three ahead
    (1, 9000, 1, 64, True, True, True),     # 71 segments
    (1, 8900, 1, 128, True, False, False),  # 70 segments
])
def test_segments_and_walks(B, T, H, N, theta, state, skip):
    scan.test_fused_launch_matches_the_three_launches_and_f64(B, T, H, N, theta, state, skip)


@gpu
@pytest.mark.parametrize("B,T,H,N,R,dtype", [
    (1, 1024, 2, 64, 1, "f32"), (1, 1025, 2, 64, 1, "f32"),     # 32 and 33 sub-chunks
    (1, 1024, 1, 128, 4, "f32"), (1, 1032, 1, 64, 4, "f32"),    # 128 and 129
    (1, 64, 3, 128, 2, "f32"), (1, 4100, 1, 64, 4, "f32"),      # 4, and past 512
    (1, 512, 2, 128, 4, "bf16"), (1, 530, 2, 64, 4, "bf16"),    # 32 and 34
    (2, 1000, 2, 128, 2, "bf16"), (1, 31, 2, 64, 2, "bf16"),    # ragged, and one
])
def test_three_launch_segments_against_f64(B, T, H, N, R, dtype):
    scan.test_segments_against_f64(B, T, H, N, R, dtype, 64)


@gpu
@pytest.mark.parametrize("B,T,H,N,R,dtype", [
    (2, 600, 12, 128, 4, torch.float32),    # 58 MB of records in segments of 16 tokens
    (2, 700, 12, 128, 1, torch.float32),    # 34 MB in segments of 32
    (4, 1000, 8, 128, 2, torch.bfloat16),   # 33 MB in segments of 32
    (1, 1000, 4, 64, 4, torch.float32),     # short ones fit
])
def test_no_alloc_cuts_as_the_workspace_scan(B, T, H, N, R, dtype):
    """Where short segments' records exceed the static scratch both calls take
    the next longer ones that fit: equal bit for bit, as everywhere."""
    inp = no_alloc._inputs(77, B=B, L=T, H=H, N=N, R=R, dtype=dtype)
    ref = no_alloc._call(inp, no_alloc=False)
    got = no_alloc._call(inp, no_alloc=True)
    assert 0 < ref[4] <= 32 << 20
    for r, g in zip(ref[:4], got[:4]):
        assert torch.equal(r, g)


def test_records_of_short_segments_stay_within_the_scratch():
    """Sizes only: no shape whose 64-token segments fit the static scratch asks
    for more (and so for another cut than m3_scan_no_alloc's)."""
    import ctypes as C
    from mamba3 import _lib
    L = _lib.lib()
    for dt, R, N, BH, T in [(d, r, n, bh, t) for d in (_lib.M3_F32, _lib.M3_BF16) for r in (1, 2, 4)
                            for n in (64, 128) for bh in (1, 6, 24, 48, 64) for t in (64, 200, 600, 1000, 4096)]:
        need = L.m3_scan_workspace_bytes(C.byref(_lib.ScanInputsC(
            BH, T, 1, 64, N, R, dt, None, None, None, None, None, None, None, None, None, 64, 1,
            None, 0)))
        # a segment's U and S, its decay and its angle totals
        record = 2 * 64 * N * (4 if dt == _lib.M3_F32 else 2) + 4 + 3 * (N // 2) * 4
        if BH * ((T + 63) // 64) * record + 6 * 256 <= 32 << 20:
            assert need <= 32 << 20, (dt, R, N, BH, T)


@gpu
@pytest.mark.parametrize("B,T,H,N,R,dtype", [(2, 600, 3, 128, 4, torch.float32),
                                             (2, 600, 3, 64, 1, torch.bfloat16)])
def test_a_smaller_workspace_takes_longer_segments(B, T, H, N, R, dtype, monkeypatch):
    """A workspace 30 % short, which what longer segments need still fits, runs
    the chunk-parallel kernels (f32: three launches) to the same result."""
    from mamba3 import _lib
    L = _lib.lib()

    class Short:
        def __getattr__(self, k):
            f = getattr(L, k)
            return (lambda a: f(a) * 7 // 10) if k == "m3_scan_workspace_bytes" else f

    def call():
        n = L.m3_launch_count()
        return (*no_alloc._call(inp, no_alloc=False), L.m3_launch_count() - n)

    inp = no_alloc._inputs(78, B=B, L=T, H=H, N=N, R=R, dtype=dtype)
    full = call()
    monkeypatch.setattr(_lib, "_lib", Short())
    short = call()
    assert short[4] < full[4] and short[5] == full[5] == (3 if dtype == torch.float32 else 1)
    tol = 2 * (scan.BF16_TOL if dtype == torch.bfloat16 else scan.F32_TOL)   # each within the bar of f64
    for r, g in zip(full[:3], short[:3]):
        assert rel_l2(np.asarray(g.float().cpu()), np.asarray(r.float().cpu())) <= tol
