"""The fused scan launch at the edges of its cut into segments and of its walk
over the segments before: one or two sub-chunks a segment, every remainder of
the records loaded ahead, more segments than one look at the flags covers."""
import numpy as np
import pytest
import torch

import test_gpu_scan as scan
import test_zz_no_alloc as no_alloc
from cases import rel_l2

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("B,T,H,N,R,dtype", [
    (1, 1024, 2, 64, 1, "f32"), (1, 1025, 2, 64, 1, "f32"),     # 32 and 33 sub-chunks
    (1, 1024, 1, 128, 4, "f32"), (1, 1032, 1, 64, 4, "f32"),    # 128 and 129
    (1, 64, 3, 128, 2, "f32"), (1, 4100, 1, 64, 4, "f32"),      # 4, and past 512
    (1, 512, 2, 128, 4, "bf16"), (1, 530, 2, 64, 4, "bf16"),    # 32 and 34
    (2, 1000, 2, 128, 2, "bf16"), (1, 31, 2, 64, 2, "bf16"),    # ragged, and one
])
def test_three_launch_segments_against_f64(B, T, H, N, R, dtype):
    scan.test_segments_against_f64(B, T, H, N, R, dtype, 64)


def test_no_alloc_takes_longer_segments_where_the_short_ones_do_not_fit():
    """24 sequences of 600 f32 tokens at rank 4 and d_state 128: 58 MB in
    segments of 16 tokens, under the static scratch in segments of 64."""
    inp = no_alloc._inputs(77, B=2, L=600, H=12, N=128, R=4, dtype=torch.float32)
    ref = no_alloc._call(inp, no_alloc=False)
    got = no_alloc._call(inp, no_alloc=True)
    assert ref[4] > 32 << 20
    for r, g in zip(ref[:3], got[:3]):
        # both within F32_TOL of the f64 recurrence
        assert rel_l2(np.asarray(g.float().cpu()), np.asarray(r.float().cpu())) <= 2 * scan.F32_TOL


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
