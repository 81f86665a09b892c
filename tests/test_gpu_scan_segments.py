"""The fused scan launch at the edges of its cut into segments and of its walk
over the segments before: one or two sub-chunks a segment, every remainder of
the records loaded ahead, more segments than one look at the flags covers."""
import pytest

import test_gpu_scan as scan

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
