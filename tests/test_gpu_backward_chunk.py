"""The backward's chunk kernels past the shapes of test_gpu_backward.py: window
lengths at the edges of a 32-row chunk, every rank and d_state, a dy off the
4-byte grid, and gradients that repeat bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import host
from cases import rel_l2
from test_gpu_backward import BF16_TOL, F32_TOL, NAMES, _run

pytestmark = pytest.mark.gpu

EDGES = [(2, T, 3, 64, N, R, True, True, True, dt)
         for N, R in ((64, 1), (64, 2), (64, 4), (128, 1), (128, 2), (128, 4))
         for T, dt in ((32 // R, "f32"), (32 // R + 1, "bf16"), (3 * 32 // R - 1, "f32"),
                       (4 * 32 // R + 1, "f32"), (5 * 32 // R + 3, "bf16"))]


@pytest.mark.parametrize("case", EDGES, ids=[repr(c[1:]) for c in EDGES])
def test_chunk_edges_against_f64(case):
    g, ref = _run(case)
    tol = BF16_TOL if case[-1] == "bf16" else F32_TOL
    for k in NAMES:
        assert rel_l2(host(getattr(g, k)), ref[k]) <= tol, (k, rel_l2(host(getattr(g, k)), ref[k]))
        if k in ("dt", "lam", "a_log", "h0", "last_u0", "angle0", "d_skip"):   # f32 whatever the storage
            assert rel_l2(host(getattr(g, k)), ref[k]) <= F32_TOL, k


def _grads(dy_of, T=150, N=128, R=1):
    from mamba3.ssm import ScanInputs, mamba3_scan_backward
    g = torch.Generator(device="cuda").manual_seed(7)
    B, H, P = 2, 3, 64
    r = lambda *s: torch.randn(s, device="cuda", generator=g)
    si = ScanInputs(r(B, T, H, P, R).bfloat16(), (r(B, T, H, N, R) / 11).bfloat16(),
                    (r(B, T, H, N, R) / 11).bfloat16(), torch.rand(B, T, H, device="cuda", generator=g) * 0.1,
                    torch.rand(H, device="cuda", generator=g) * 2.7, torch.sigmoid(r(B, T, H)))
    si = si.with_theta((torch.rand(B, T, H, N // 2, device="cuda", generator=g) * 3).bfloat16()).with_skip(r(H))
    return mamba3_scan_backward(si, dy_of(r(B, T, H, P, R).bfloat16()))


@pytest.mark.parametrize("N,R", [(128, 1), (64, 2), (128, 4)])
def test_gradients_repeat_bit_for_bit(N, R):
    a, b = _grads(lambda t: t, N=N, R=R), _grads(lambda t: t, N=N, R=R)
    for k in ("x", "b", "c", "dt", "lam", "a_log", "theta", "d_skip"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k


def test_dy_off_the_dword_grid():
    """A bf16 dy that starts two bytes past a 4-byte boundary gives the same bytes."""
    def shifted(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        v = buf[1:].view(t.shape)
        v.copy_(t)
        assert v.data_ptr() % 4 == 2 and v.is_contiguous()
        return v
    a, b = _grads(lambda t: t), _grads(shifted)
    for k in ("x", "b", "c", "dt", "lam", "a_log", "theta", "d_skip"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k


@pytest.mark.parametrize("scale", [1.0, 300.0, 3e5])
def test_wide_angles_against_f64(scale):
    """In-chunk angles of a few turns, of hundreds and past the range of the
    short reduction; theta's own magnitude multiplies an angle's f32 rounding,
    2^-24 of up to scale * 0.1 * 32 a chunk, in every product it rotates."""
    import oracle
    from cases import baseline_inputs
    from gpu_util import dev
    from mamba3.ssm import ScanInputs, mamba3_scan_backward
    rng = np.random.default_rng(int(scale) % 977)
    B, T, H, P, N = 1, 64, 2, 64, 64
    inp = baseline_inputs(rng, B, T, H, P, N, 1, theta=True, theta_per_head=False)
    inp["theta"] = (inp["theta"] * np.float32(scale)).astype(np.float32)
    dy = rng.standard_normal((B, T, H, P, 1)).astype(np.float32)
    si = ScanInputs(dev(inp["x"]), dev(inp["b"]), dev(inp["c"]), dev(inp["dt"]), dev(inp["a_log"]),
                    dev(inp["lam"])).with_theta(dev(inp["theta"]))
    g = mamba3_scan_backward(si, dev(dy))
    ref = oracle.scan_backward_f64(inp["x"], inp["b"], inp["c"], inp["dt"], inp["a_log"], inp["lam"], dy,
                                   inp["theta"], None, None, None, None, None, None, None)
    tol = max(F32_TOL, 8 * 2.0 ** -24 * scale * 0.1 * 64)
    if tol > 0.1:       # the angles hold no f32 digits: only finite
        assert all(np.isfinite(host(getattr(g, k))).all() for k in ("x", "b", "c", "theta"))
        return
    for k in ("x", "b", "c", "lam"):
        assert rel_l2(host(getattr(g, k)), ref[k]) <= tol, (k, rel_l2(host(getattr(g, k)), ref[k]))
