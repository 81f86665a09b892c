"""Small heads (head_dim <= 32, d_state <= 64) on zero-padded copies through
the chunk kernels: the forward and the backward against the f64 oracles at the
smallest and largest padded sizes, ragged windows, every option, and the
kernels the call took (its launch count); a workspace too small for the padded
copies runs the kernels of before.

Bars as in test_gpu_scan.py and test_gpu_backward.py: rel-L2 <= 1e-5 for f32
storage, <= 1e-2 for bf16.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from cases import baseline_inputs, rel_l2
from gpu_util import dev, host, oracle_scan, run_scan
from test_gpu_backward import BF16_TOL, F32_TOL, NAMES, _run

# B, T, H, P, N, R, theta, skip, state, dtype
CASES = [
    (2, 128, 3, 3, 6, 1, True, True, True, "f32"),       # the shortest window, far from a tile
    (1, 129, 2, 32, 64, 1, True, True, True, "f32"),     # the largest head, one token over
    (1, 200, 2, 16, 16, 1, True, True, True, "bf16"),
    (1, 131, 2, 1, 2, 1, True, False, False, "f32"),     # one column, one pair
    (2, 150, 1, 17, 5, 1, False, True, True, "f32"),     # odd d_state, real dynamics
    (1, 70, 3, 5, 1, 2, False, False, True, "f32"),      # d_state 1
    (1, 33, 2, 32, 32, 4, True, True, True, "bf16"),     # rank 4
    (1, 75, 2, 8, 64, 2, True, True, True, "bf16"),      # rank 2
]
SHORT = [(2, 8, 2, 16, 16, 1, True, True, True, "f32"), (1, 7, 2, 16, 16, 1, True, True, True, "f32")]


def _launches(fn):
    from mamba3 import _lib
    before = _lib.lib().m3_launch_count()
    out = fn()
    return out, _lib.lib().m3_launch_count() - before


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[repr(c) for c in CASES])
def test_forward_against_f64(case):
    B, T, H, P, N, R, theta, skip, state, dtype = case
    rng = np.random.default_rng(B * T + P * N + R)
    inp = baseline_inputs(rng, B, T, H, P, N, R, theta=theta, dtype=dtype, theta_per_head=False,
                          state=state)
    d_skip = rng.uniform(-1, 1, H).astype(np.float32) if skip else None
    st = (inp["h0"], inp["last_u0"], inp.get("angle0")) if state else None
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    (y, h, lu, ang), n = _launches(lambda: run_scan(inp, dtype=tdt, theta=theta, skip=d_skip,
                                                    state=st))
    assert n == 5   # the copies, the three chunk launches, the copies back
    y64, h64, lu64, ang64 = oracle_scan(inp, theta=theta, skip=d_skip, state=st)
    assert rel_l2(y, y64) <= (BF16_TOL if dtype == "bf16" else F32_TOL)
    # the state is f32 whatever the storage
    assert rel_l2(h, h64) <= F32_TOL and rel_l2(lu, lu64) <= F32_TOL
    if theta:
        d = np.abs(ang - ang64)
        assert np.max(np.minimum(d, 2 * np.pi - d)) <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + SHORT, ids=[repr(c) for c in CASES + SHORT])
def test_backward_against_f64_reverse_mode(case):
    (g, ref), n = _launches(lambda: _run(case))
    theta = case[6]
    # from 8 tokens on: the copies, the chunk kernels and the outgoing last_u's
    # two, the copies back; below, the token walk and the head sums
    assert n == (2 if case[1] < 8 else (9 if theta else 8))
    tol = BF16_TOL if case[-1] == "bf16" else F32_TOL
    checked = 0
    for k in NAMES:
        mine = getattr(g, k)
        if mine is None or ref.get(k) is None:
            continue
        assert rel_l2(host(mine), ref[k]) <= tol, (k, rel_l2(host(mine), ref[k]))
        checked += 1
    assert checked >= 6


def _query(B, T, H, P, N, R, dtype):
    from mamba3 import _lib
    cin = _lib.ScanInputsC(B, T, H, P, N, R, dtype, None, None, None, None, None, None, None, None,
                           None, 64, 1, None, 0)
    L = _lib.lib()
    return (int(L.m3_scan_workspace_bytes(C.byref(cin))),
            int(L.m3_scan_backward_workspace_bytes(C.byref(cin))))


def test_workspace_queries_at_the_edges():
    """Padded copies are asked for at head_dim <= 32, d_state <= 64 and rank 1,
    2 or 4; the forward from 128 rows and up to 512 sequences."""
    from mamba3 import _lib
    f32, bf16 = _lib.M3_F32, _lib.M3_BF16
    assert _query(2, 128, 4, 16, 16, 1, f32)[0] > 0 and _query(2, 127, 4, 16, 16, 1, f32)[0] == 0
    assert _query(2, 32, 4, 16, 16, 4, bf16)[0] > 0 and _query(2, 31, 4, 16, 16, 4, bf16)[0] == 0
    assert _query(64, 128, 8, 16, 16, 1, f32)[0] > 0 and _query(64, 128, 9, 16, 16, 1, f32)[0] == 0
    for P, N, R in ((33, 16, 1), (16, 65, 1), (16, 16, 3)):
        assert _query(2, 256, 4, P, N, R, f32)[0] == 0
    # the widened forward's copies are f32; the backward keeps the storage type
    assert _query(2, 256, 4, 16, 16, 1, bf16)[0] == _query(2, 256, 4, 16, 16, 1, f32)[0]
    assert _query(2, 256, 4, 16, 16, 1, bf16)[1] < _query(2, 256, 4, 16, 16, 1, f32)[1]


def test_workspace_queries_are_bounded():
    """Large calls run part by part: neither query passes 512 MiB where the
    padded copies are asked for, whatever the batch and the heads."""
    from mamba3 import _lib
    for dt in (_lib.M3_F32, _lib.M3_BF16):
        for B, T, H, P, N, R in ((256, 2048, 4, 16, 16, 1), (64, 4096, 16, 16, 16, 1), (512, 8192, 4, 16, 16, 1),
                                 (1, 40000, 8, 32, 64, 1), (3, 9000, 9, 8, 64, 4), (128, 512, 4, 16, 16, 1)):
            fw, bw = _query(B, T, H, P, N, R, dt)
            assert 0 < bw <= 512 << 20, (B, T, H, bw)
            assert (0 < fw <= 512 << 20) if B * H <= 512 else fw == 0, (B, T, H, fw)
            one = _query(1, T, 1, P, N, R, dt)[0]   # a sequence, or windows of it, within the static scratch
            assert 0 < one <= 32 << 20, (T, one)


def test_a_long_sequence_keeps_the_backward_copies():
    """One sequence is the backward's least part, past 512 MiB too: the query
    goes on growing with its length (the token walk's asks for some 90 bytes a
    token), and neither the batch nor the heads add to it."""
    from mamba3 import _lib
    for R, dt, T in ((1, _lib.M3_F32, 170000), (4, _lib.M3_F32, 47000), (4, _lib.M3_BF16, 70000)):
        one = _query(1, T, 1, 16, 16, R, dt)[1]
        assert one > 512 << 20 and one < 4000 * R * T, (R, T, one)
        gathered = 16 * (T + 64)   # dt, lambda and their gradients, where the heads are apart
        assert one <= _query(2, T, 3, 16, 16, R, dt)[1] <= one + gathered + 4096, (R, T)


@pytest.mark.gpu
def test_a_long_sequence_backward_is_its_padded_call():
    """Past 512 MiB of copies: the gradients of sequences of 47,000 tokens, two
    heads of them, against the call on heads of 64 that the zeros are written
    into here, one head at a time.  Zeros add nothing and the kernels are the
    same: bit for bit."""
    from mamba3.ssm import ScanInputs, mamba3_scan_backward
    T, H, P, N, R = 47000, 2, 16, 16, 4
    g = torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(s, device="cuda", generator=g)
    u = lambda *s: torch.rand(s, device="cuda", generator=g)
    x, b, c, dy = r(1, T, H, P, R), r(1, T, H, N, R) / 4, r(1, T, H, N, R) / 4, r(1, T, H, P, R)
    dt, a_log, lam, theta = u(1, T, H) * 0.1, u(H) * 2.7, u(1, T, H), u(1, T, H, N // 2) * 3

    def grown(t, n):
        out = t.new_zeros(*t.shape[:3], n, *t.shape[4:])
        out[:, :, :, :t.shape[3]] = t
        return out

    def call(hs, p, n):
        pick = lambda t: t[:, :, hs].contiguous()
        # a pair's two elements stand in the halves of d_state
        both = lambda t: torch.cat([grown(t[:, :, :, :N // 2], n // 2), grown(t[:, :, :, N // 2:], n // 2)], dim=3)
        si = ScanInputs(grown(pick(x), p), both(pick(b)), both(pick(c)), pick(dt), a_log[hs].contiguous(),
                        pick(lam)).with_theta(grown(pick(theta), n // 2))
        return mamba3_scan_backward(si, grown(pick(dy), p))

    got = call(slice(0, H), P, N)
    for h in range(H):
        want = call(slice(h, h + 1), 64, 64)
        assert torch.equal(got.x[:, :, h], want.x[:, :, 0, :P]), h
        assert torch.equal(got.theta[:, :, h], want.theta[:, :, 0, :N // 2]), h
        pairs = [*range(N // 2), *range(32, 32 + N // 2)]
        for name in ("b", "c"):
            assert torch.equal(getattr(got, name)[:, :, h], getattr(want, name)[:, :, 0, pairs]), (name, h)
        for name in ("dt", "lam"):
            assert torch.equal(getattr(got, name)[:, :, h], getattr(want, name)[:, :, 0]), (name, h)
        assert torch.equal(got.a_log[h], want.a_log[0]), h


# more rows than 512 MiB of copies hold: parts of the batch, the last one short;
# parts of the heads of one entry, forward and backward, with every option
LARGE = [(64, 1000, 8, 16, 16, 1, "f32"), (63, 1000, 8, 16, 16, 1, "bf16"), (1, 25000, 21, 8, 16, 1, "f32"),
         (2, 5000, 31, 6, 12, 4, "bf16")]


@pytest.mark.gpu
@pytest.mark.parametrize("case", LARGE, ids=[repr(c) for c in LARGE])
def test_parts_equal_calls_of_their_own(case):
    """Each batch entry's and head's outputs and gradients against a call on
    that sequence alone (whose segments are cut for one sequence: to f32
    rounding, and the rounding of bf16 storage), the heads' sums against the
    sum of those calls."""
    from mamba3.ssm import ScanInputs, SsmState, mamba3_scan, mamba3_scan_backward
    B, T, H, P, N, R, dtype = case
    ty = torch.bfloat16 if dtype == "bf16" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(B * T)
    r = lambda *s: torch.randn(s, device="cuda", generator=g)
    u = lambda *s: torch.rand(s, device="cuda", generator=g)
    x, b, c = r(B, T, H, P, R).to(ty), (r(B, T, H, N, R) / N ** 0.5).to(ty), (r(B, T, H, N, R) / N ** 0.5).to(ty)
    dt, a_log, lam, theta, skip = u(B, T, H) * 0.1, u(H) * 2.7, u(B, T, H), (u(B, T, H, N // 2) * 3).to(ty), r(H)
    st = (r(B, H, P, N) * 0.1, r(B, H, P, N) * 0.1, u(B, H, N // 2) * 3)
    dy, dh, dang, dlu = r(B, T, H, P, R).to(ty), r(B, H, P, N), r(B, H, N // 2), r(B, H, P, N)

    def call(bs, hs):
        pick = lambda t: t[bs][:, :, hs].contiguous()
        seq = lambda t: t[bs][:, hs].contiguous()
        si = ScanInputs(pick(x), pick(b), pick(c), pick(dt), a_log[hs].contiguous(), pick(lam))
        si = si.with_theta(pick(theta)).with_skip(skip[hs].contiguous()).with_state(
            SsmState(*[seq(t) for t in st]))
        out = mamba3_scan(si)
        gr = mamba3_scan_backward(si, pick(dy), seq(dh), seq(dang), seq(dlu))
        return out, gr

    all_b, all_h = slice(None), slice(None)
    (out, gr), n = _launches(lambda: call(all_b, all_h))
    assert n >= 10 + 18, "one part would be 5 and 9 launches"
    tol = 2 * (BF16_TOL if dtype == "bf16" else F32_TOL)
    picks = [(bb, hh) for bb in sorted({0, 1 % B, B // 2, B - 1}) for hh in sorted({0, H // 2, H - 1})]
    for bb, hh in picks:
        bs, hs = slice(bb, bb + 1), slice(hh, hh + 1)
        o1, g1 = call(bs, hs)
        near = lambda a, e, t: rel_l2(host(a), host(e)) <= t
        assert near(out.y[bs][:, :, hs], o1.y, tol), (bb, hh)
        assert near(out.state.h[bs, hs], o1.state.h, 2 * F32_TOL), (bb, hh)
        assert near(out.state.last_u[bs, hs], o1.state.last_u, 2 * F32_TOL), (bb, hh)
        for k in ("x", "b", "c", "theta"):
            assert near(getattr(gr, k)[bs][:, :, hs], getattr(g1, k), tol), (bb, hh, k)
        for k in ("dt", "lam"):
            assert near(getattr(gr, k)[bs][:, :, hs], getattr(g1, k), 2 * F32_TOL), (bb, hh, k)
        for k in ("h0", "last_u0", "angle0"):
            assert near(getattr(gr, k)[bs, hs], getattr(g1, k), 2 * F32_TOL), (bb, hh, k)
    for hh in (0, H - 1):
        each = [call(slice(bb, bb + 1), slice(hh, hh + 1))[1] for bb in range(B)]
        for k in ("a_log", "d_skip"):
            e = np.array([float(getattr(t, k)[0]) for t in each], np.float64)
            # f32 sums of terms that cancel: against the terms' own size
            assert abs(float(getattr(gr, k)[hh]) - e.sum()) <= 2 * F32_TOL * np.sqrt((e * e).sum()), (hh, k)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(1, 20100, 1, 16, 16, 1, True, "f32"), (1, 45001, 2, 8, 6, 1, True, "f32"),
                                  (2, 7100, 1, 32, 64, 4, True, "bf16"), (1, 30000, 1, 5, 7, 1, False, "f32")], ids=repr)
@pytest.mark.parametrize("state", [True, False])
def test_windows_of_a_long_sequence_against_f64(case, state):
    """A sequence whose copies exceed the static scratch runs in windows, the
    state of one entering the next: y at the usual bars, the final state with
    the angle's own error besides: every wrap takes f32's 2 pi, 1.75e-7 over, and
    every token rounds by 2^-24 pi at most, in random order (one workgroup over
    the whole sequence is off by as much)."""
    B, T, H, P, N, R, theta, dtype = case
    rng = np.random.default_rng(T + P)
    inp = baseline_inputs(rng, B, T, H, P, N, R, theta=theta, dtype=dtype, theta_per_head=False, state=True)
    st = (inp["h0"], inp["last_u0"], inp.get("angle0")) if state else None
    skip = rng.uniform(-1, 1, H).astype(np.float32)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    (y, h, lu, ang), n = _launches(lambda: run_scan(inp, dtype=tdt, theta=theta, skip=skip, state=st))
    assert n >= 2 * 5 * B * H
    y64, h64, lu64, ang64 = oracle_scan(inp, theta=theta, skip=skip, state=st)
    assert rel_l2(y, y64) <= (BF16_TOL if dtype == "bf16" else F32_TOL)
    turn = 0.0
    if theta:
        wraps = np.abs((inp["dt"][..., None].astype(np.float64) * inp["theta"]).sum(1)).max() / (2 * np.pi)
        turn = wraps * (float(np.float32(2 * np.pi)) - 2 * np.pi) + 2.0 ** -24 * np.pi * np.sqrt(T)
    assert rel_l2(h, h64) <= F32_TOL + turn and rel_l2(lu, lu64) <= F32_TOL + turn
    if theta:
        d = np.abs(ang - ang64)
        assert np.max(np.minimum(d, 2 * np.pi - d)) <= 1e-4 + turn
    # without the final state the same y
    y2 = run_scan(inp, dtype=tdt, theta=theta, skip=skip, state=st, want_state=False)[0]
    assert np.array_equal(y, y2)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(4, 512, 4, 16, 16, 1, "f32"), (64, 512, 4, 16, 16, 1, "f32"),
                                  (5, 4000, 9, 32, 64, 1, "bf16"), (2, 3000, 3, 7, 12, 4, "f32"),
                                  (1, 31000, 2, 16, 16, 1, "f32"), (2, 15000, 1, 8, 32, 4, "bf16")], ids=repr)
def test_no_alloc_equals_the_workspace_scan(case):
    """m3_scan_no_alloc's parts, within the static scratch, against m3_scan's,
    within its workspace: one part, parts of the batch, parts of the heads, and
    a sequence the scratch does not hold (windows of it in both), bit for bit."""
    import test_zz_no_alloc as no_alloc
    B, T, H, P, N, R, dtype = case
    inp = no_alloc._inputs(B + T, B, T, H, N, R, torch.bfloat16 if dtype == "bf16" else torch.float32)
    cut = lambda t: t[..., :P, :].contiguous()
    h0, u0, a0 = inp["state"]
    inp.update(P=P, x=cut(inp["x"]), state=(cut(h0), cut(u0), a0))
    (ref, n_ref), (got, n_got) = (_launches(lambda: no_alloc._call(inp, no_alloc=k)) for k in (False, True))
    assert (ref[4] > 0) == (n_ref > 1) == (n_got > 1)
    assert (n_got > n_ref) == (ref[4] > 32 << 20)
    for name, r, g in zip(("y", "h", "last_u", "angle"), ref[:4], got[:4]):
        assert torch.equal(r, g), name


@pytest.mark.gpu
def test_a_smaller_workspace_runs_the_kernels_of_before():
    from mamba3 import _lib
    L = _lib.lib()
    B, T, H, P, N = 1, 160, 2, 16, 16
    rng = np.random.default_rng(5)
    inp = baseline_inputs(rng, B, T, H, P, N, 1, theta=True, theta_per_head=False)
    t = {k: dev(v) for k, v in inp.items() if v is not None}
    cin = _lib.ScanInputsC(B, T, H, P, N, 1, _lib.M3_F32, t["x"].data_ptr(), t["b"].data_ptr(),
                           t["c"].data_ptr(), t["dt"].data_ptr(), t["a_log"].data_ptr(),
                           t["lam"].data_ptr(), t["theta"].data_ptr(), None, None, 64, 0, None, 0)
    fw, bw = (int(q(C.byref(cin))) for q in (L.m3_scan_workspace_bytes,
                                            L.m3_scan_backward_workspace_bytes))
    ws = torch.empty(max(fw, bw), dtype=torch.uint8, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    outs = []
    for size, launches in ((fw, 5), (fw - 1, 1)):
        cin.workspace, cin.workspace_bytes = ws.data_ptr(), size
        y = torch.empty_like(t["x"])
        cout = _lib.ScanOutputC(y.data_ptr(), _lib.SsmStateC())
        _, n = _launches(lambda: _lib.check(L.m3_scan(C.byref(cin), C.byref(cout), stream)))
        assert n == launches
        outs.append(host(y))
    assert rel_l2(outs[0], outs[1]) <= F32_TOL
    dy = dev(rng.standard_normal((B, T, H, P, 1)).astype(np.float32))
    grads = []
    for size, launches in ((bw, 7), (bw - 1, 2)):
        cin.workspace, cin.workspace_bytes = ws.data_ptr(), size
        g = {k: torch.empty_like(t[k]) for k in ("x", "b", "c", "dt", "lam", "a_log", "theta")}
        gc = _lib.ScanGradsC(dy.data_ptr(), None, None,
                             *[g[k].data_ptr() for k in ("x", "b", "c", "dt", "lam", "a_log",
                                                         "theta")], None, None, None, None)
        _, n = _launches(lambda: _lib.check(L.m3_scan_backward(C.byref(cin), C.byref(gc), stream)))
        assert n == launches
        grads.append({k: host(v) for k, v in g.items()})
    for k in grads[0]:
        assert rel_l2(grads[0][k], grads[1][k]) <= F32_TOL, k
