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


def _former_bytes(BH, T, N, R):
    """The workspace of 64-row chunks, which bf16 storage at d_state 64 had."""
    up = lambda v: (v + 255) // 256 * 256
    nck = -(-T // (64 // R))
    pairs, tok = BH * nck * (N // 2) * 4, BH * T * 4
    return (2 * up(BH * nck * 64 * N * 4) + 3 * up(BH * nck * 4) + up(BH * T * (N // 2) * 4) + 2 * up(pairs)
            + 3 * up(tok) + up(BH * (N // 32) * 4) + up(BH * (N // 2) * 4) + up(BH * 64 * R * 4)
            + up(BH * N * R * 4))


@pytest.mark.parametrize("B,T,H,R", [(1, 1, 1, 1), (1, 33, 1, 1), (2, 64, 3, 1), (5, 65, 13, 1), (1, 1000, 2, 1),
                                     (2, 150, 3, 2), (3, 40, 5, 4)])
def test_a_workspace_of_64_row_chunks_still_runs(B, T, H, R):
    """Half the records: the chunks in two windows, the same gradients (those
    summed over chunks to f32 rounding); a byte less than the least is refused."""
    import ctypes as C
    from mamba3 import _lib
    L = _lib.lib()
    P = N = 64
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(s, device="cuda", generator=g)
    bf = lambda t: t.bfloat16()
    x, b, c, th = bf(r(B, T, H, P, R)), bf(r(B, T, H, N, R) / 8), bf(r(B, T, H, N, R) / 8), bf(r(B, T, H, N // 2))
    dt, lam, a_log, skip = r(B, T, H).abs() * 0.05, torch.sigmoid(r(B, T, H)), r(H).abs(), r(H)
    st = (r(B, H, P, N), r(B, H, P, N), r(B, H, N // 2))
    dy, dh, dang, dlu = bf(r(B, T, H, P, R)), r(B, H, P, N), r(B, H, N // 2), r(B, H, P, N)
    st_c = _lib.SsmStateC(*[t.data_ptr() for t in st])

    def call(size):
        ins = _lib.ScanInputsC(B, T, H, P, N, R, _lib.M3_BF16, *[t.data_ptr() for t in (x, b, c, dt, a_log, lam, th,
                               skip)], C.pointer(st_c), 64, 0, None, 0)
        full = int(L.m3_scan_backward_workspace_bytes(C.byref(ins)))
        ws = torch.full((max(full, size or 0),), 255, dtype=torch.uint8, device="cuda")   # NaN wherever unwritten
        ins.workspace, ins.workspace_bytes = ws.data_ptr(), size or full
        out = [torch.full_like(t, float("nan")) for t in (x, b, c, dt, lam, a_log, th, skip, *st)]
        gc = _lib.ScanGradsC(dy.data_ptr(), dh.data_ptr(), dang.data_ptr(), *[t.data_ptr() for t in out], dlu.data_ptr())
        n = L.m3_launch_count()
        status = L.m3_scan_backward(C.byref(ins), C.byref(gc), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return status, out, L.m3_launch_count() - n, full

    former = _former_bytes(B * H, T, N, R)
    ok, whole, n, full = call(None)
    ok2, two, n2, _ = call(former)
    assert ok == ok2 == _lib.M3_OK
    assert n2 == (n + 2 if former < full else n) and (former < full or T <= 32 // R)
    for i, (e, t) in enumerate(zip(whole, two)):
        if i in (5, 7):   # a_log, d_skip
            assert rel_l2(host(t), host(e)) <= F32_TOL, i
        else:
            assert torch.equal(t, e), i
    if T > 32 // R:
        assert call(former // 2)[0] == _lib.M3_ERR_ARGUMENT


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


@pytest.mark.parametrize("a_log", [40.0, 85.0, 100.0])
@pytest.mark.parametrize("P,N,R,dtype", [(64, 64, 1, "f32"), (64, 128, 2, "bf16"), (16, 16, 1, "f32")])
def test_decays_that_end_a_state_at_once(P, N, R, dtype, a_log):
    """exp(a_log) dt from 1e16 to past f32's range: every token forgets all
    before it, and the gradients of x, b, c, lambda and theta are those of the
    token itself (theta's, zero without a past, small against b's)."""
    import oracle
    from cases import baseline_inputs
    from gpu_util import dev
    from mamba3.ssm import ScanInputs, mamba3_scan_backward
    rng = np.random.default_rng(int(a_log) + N)
    B, T, H = 1, 70, 2
    inp = baseline_inputs(rng, B, T, H, P, N, R, theta=True, theta_per_head=False, dtype=dtype)
    inp["a_log"] = np.full((H,), a_log, np.float32)
    ty = torch.bfloat16 if dtype == "bf16" else torch.float32
    dy = dev(rng.standard_normal((B, T, H, P, R)), ty)
    si = ScanInputs(dev(inp["x"], ty), dev(inp["b"], ty), dev(inp["c"], ty), dev(inp["dt"]), dev(inp["a_log"]),
                    dev(inp["lam"])).with_theta(dev(inp["theta"], ty))
    g = mamba3_scan_backward(si, dy)
    ref = oracle.scan_backward_f64(inp["x"], inp["b"], inp["c"], inp["dt"], np.minimum(inp["a_log"], 60),
                                   inp["lam"], host(dy), inp["theta"], None, None, None, None, None, None, None)
    for k in ("x", "b", "c", "lam"):
        tol = F32_TOL if dtype == "f32" or k == "lam" else BF16_TOL
        assert rel_l2(host(getattr(g, k)), ref[k]) <= tol, (k, rel_l2(host(getattr(g, k)), ref[k]))
    assert np.abs(host(g.theta)).max() <= 1e-4 * np.abs(ref["b"]).max()
    assert a_log > 90 or np.isfinite(host(g.a_log)).all() and np.isfinite(host(g.dt)).all()


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


@pytest.mark.parametrize("N,R", [(64, 1), (128, 1), (64, 4)])
@pytest.mark.parametrize("lo,hi", [(200, 900), (1 << 15, 1 << 17)])
def test_exact_angles_past_the_short_reduction(N, R, lo, hi):
    """Angles that f32 holds exactly, whole numbers of radians below 2^24 (dt =
    1/16, theta whole multiples of 16), on both sides of 2^13 within a chunk,
    where the sine's short reduction hands over to the library's, and far past
    it: no angle is rounded, so the gradients hold F32_TOL as those of small
    angles do.  A sine past its range or a wrong hand-over would be off by its
    whole size."""
    import oracle
    from cases import baseline_inputs
    from gpu_util import dev
    from mamba3.ssm import ScanInputs, mamba3_scan_backward
    rng = np.random.default_rng(lo + N + R)
    B, T, H, P = 1, 70, 2, 64
    inp = baseline_inputs(rng, B, T, H, P, N, R, theta=True, theta_per_head=False)
    inp["dt"] = np.full((B, T, H), 1 / 16, np.float32)
    turn = rng.integers(lo, hi, (B, T, H, N // 2)) * rng.choice([-1, 1], (1, 1, H, N // 2))
    turn[..., 0] = 256      # exactly 2^13 at the 32nd token
    inp["theta"] = (16 * turn).astype(np.float32)
    phi = np.cumsum(turn, 1)
    assert np.abs(phi).max() < 1 << 24
    if lo < 1000:
        first = np.abs(phi[:, : 32 // R])
        assert R == 4 or (first.min() < 8192 < first.max())
    dy = rng.standard_normal((B, T, H, P, R)).astype(np.float32)
    si = ScanInputs(dev(inp["x"]), dev(inp["b"]), dev(inp["c"]), dev(inp["dt"]), dev(inp["a_log"]),
                    dev(inp["lam"])).with_theta(dev(inp["theta"]))
    g = mamba3_scan_backward(si, dev(dy))
    ref = oracle.scan_backward_f64(inp["x"], inp["b"], inp["c"], inp["dt"], inp["a_log"], inp["lam"], dy,
                                   inp["theta"], None, None, None, None, None, None, None)
    for k in ("x", "b", "c", "lam", "theta"):
        assert rel_l2(host(getattr(g, k)), ref[k]) <= F32_TOL, (k, rel_l2(host(getattr(g, k)), ref[k]))
