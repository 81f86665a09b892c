"""The product of a handful of rows (few_rows.hip) against f64 at the edges of
its tiles and of its dispatch: 1 to 16 rows at any width, to 32 under 4096
columns, to 64 where x's re-reads stay small; column counts that leave partial
16- and 32-column tiles, K of one 64-block, of fewer blocks than waves and of a
ragged split.

Bar: f32 sums of exact bf16 products, scaled in f32, one rounding to bf16:
each output within 2^-8 of its value (half an ulp) plus K 2^-24 of the sum of
the products' magnitudes (the order of the f32 sum).
"""
import numpy as np
import pytest
import torch

import mixer_oracle as mo
from test_gpu_mixer import host, t_bf16, t_f32

gpu = pytest.mark.gpu

CASES = [
    # m, k, n, int8, residual
    (1, 64, 16, True, True), (1, 192, 20, False, False), (3, 1536, 1000, True, True),
    (4, 768, 5400, True, False), (5, 512, 4100, True, True), (16, 1536, 4096, False, True),
    (16, 320, 300, True, True), (17, 1024, 516, True, True), (31, 768, 768, False, False),
    (32, 512, 4092, True, True), (32, 512, 4640, True, True), (33, 768, 5400, True, False),
    (64, 768, 4100, True, True), (49, 64, 6192, False, True),
    # both sides of the lines from 4096 columns on
    (4, 2816, 4096, True, True), (4, 2880, 4096, True, True), (1, 64, 32772, True, False),
    (16, 1024, 4096, True, True), (16, 1088, 4096, True, True), (5, 1536, 4608, True, False),
    (31, 2048, 4608, True, True), (32, 2048, 4608, True, True), (17, 448, 16388, True, False),
    (33, 64, 8192, True, True), (33, 64, 8196, True, True),
]


@gpu
@pytest.mark.parametrize("m,k,n,int8,resid", CASES)
def test_few_rows_against_f64(m, k, n, int8, resid):
    from mamba3.nn import Linear
    rng = np.random.default_rng(m * k + n)
    x = mo.bf16(rng.normal(0, 1, (m, k)))
    w = rng.normal(0, 0.02, (k, n)).astype(np.float32)
    lin = Linear(t_f32(w), int8_weights=int8)
    if int8:
        c, s = mo.quantize_int8_columns(w)
        w_eff = c.astype(np.float64) * s
    else:
        w_eff = mo.bf16(w)
    r = mo.bf16(rng.normal(0, 1, (m, n))) if resid else 0.0
    ref = x @ w_eff + r
    # a guard row after the output: nothing is written past it
    buf = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device="cuda")
    out = buf[:m]
    if resid:
        out.copy_(t_bf16(r))
    y = lin.apply(t_bf16(x), residual=out if resid else None, out=out)
    torch.cuda.synchronize()
    got = host(y)
    bound = 2.0 ** -8 * np.abs(ref) + k * 2.0 ** -24 * (np.abs(x) @ np.abs(w_eff) + np.abs(r))
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)
    assert torch.all(buf[m] == 7.0)


@gpu
def test_few_rows_repeat_bit_for_bit():
    from mamba3.nn import Linear
    rng = np.random.default_rng(2)
    lin = Linear(t_f32(rng.normal(0, 0.02, (1536, 10800)).astype(np.float32)), int8_weights=True)
    x = t_bf16(mo.bf16(rng.normal(0, 1, (6, 1536))))
    a, b = lin.apply(x), lin.apply(x)
    assert torch.equal(a, b)
    # a row's result does not depend on the rows beside it
    assert torch.equal(lin.apply(x[2:5].contiguous())[1], lin.apply(x[3:4].contiguous())[0])


@gpu
@pytest.mark.parametrize("m,k,n,int8,gain", [(1, 64, 16, True, True), (1, 1536, 1540, True, True),
                                             (4, 768, 5400, True, False), (3, 320, 4100, False, True),
                                             (4, 2560, 516, True, True), (2, 512, 1000, True, True)])
def test_normed_few_rows_against_f64(m, k, n, int8, gain):
    """m3_norm_linear_nt: the operand bf16(x gain) is off by 2^-9 of each
    product, the output by 2^-9 of itself, the f32 sum as above."""
    from mamba3.nn import Linear, RmsNorm
    rng = np.random.default_rng(m + k + n)
    x = mo.bf16(rng.normal(0, 3, (m, k)))
    x[0, : k // 2] = 0.0
    g = rng.uniform(-1.5, 1.5, k).astype(np.float32)
    w = rng.normal(0, 0.02, (k, n)).astype(np.float32)
    lin = Linear(t_f32(w), int8_weights=int8)
    norm = RmsNorm(k, torch.device("cuda"), weight=gain)
    if gain:
        norm.weight.copy_(t_f32(g))
    if int8:
        c, s = mo.quantize_int8_columns(w)
        w_eff = c.astype(np.float64) * s
    else:
        w_eff = mo.bf16(w)
    normed = mo.rms_norm(x, g if gain else None, 1e-5)
    ref = normed @ w_eff
    from mamba3 import _lib
    before = _lib.lib().m3_launch_count()
    y = lin.apply_normed(t_bf16(x), norm)
    torch.cuda.synchronize()
    assert _lib.lib().m3_launch_count() - before == 1
    got = host(y)
    bound = 2.0 ** -8 * np.abs(ref) + (2.0 ** -9 + (k + 4) * 2.0 ** -24) * (np.abs(normed) @ np.abs(w_eff))
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)
    # no further off than the two calls: both operands hold k independent
    # roundings, whose norms differ by a few k^-1/2 (shorter rows say nothing)
    if k < 500:
        return
    two = host(lin.apply(norm.apply(t_bf16(x))))
    err = lambda a: np.linalg.norm(a - ref) / np.linalg.norm(ref)
    assert err(got) <= 1.2 * err(two) + 1e-4


@gpu
@pytest.mark.parametrize("m,k", [(1, 25536), (2, 12736), (3, 8512), (4, 6336)])
def test_normed_rows_at_the_edge_of_their_lds(m, k):
    """The largest k whose m operand rows fit, against f64 in one launch, and
    64 more, which runs as the two calls, equal to them."""
    from mamba3 import _lib
    from mamba3.nn import Linear, RmsNorm
    rng = np.random.default_rng(k)
    n = 20
    for kk, launches in ((k, 1), (k + 64, 2)):
        w = rng.normal(0, 0.02, (kk, n)).astype(np.float32)
        lin, norm = Linear(t_f32(w)), RmsNorm(kk, torch.device("cuda"))
        x = mo.bf16(rng.normal(0, 1, (m, kk)))
        xt = t_bf16(x)
        before = _lib.lib().m3_launch_count()
        y = lin.apply_normed(xt, norm)
        assert _lib.lib().m3_launch_count() - before == launches
        two = lin.apply(norm.apply(xt))
        if launches == 2:
            assert torch.equal(y, two)
        normed, w_eff = mo.rms_norm(x, np.ones(kk, np.float32), 1e-5), mo.bf16(w)
        ref = normed @ w_eff
        bound = 2.0 ** -8 * np.abs(ref) + (2.0 ** -9 + (kk + 4) * 2.0 ** -24) * (np.abs(normed) @ np.abs(w_eff))
        assert np.all(np.abs(host(y) - ref) <= bound)


def test_normed_product_refuses_before_device_work():
    """Past each limit M3_ERR_UNSUPPORTED, from the shapes alone."""
    from mamba3 import _lib
    L = _lib.lib()
    for m, k, n in [(5, 64, 16), (4, 6400, 16), (1, 96, 16), (1, 64, 12), (1, 64, 18), (1, 16384, 1 << 16)]:
        st = L.m3_norm_linear_nt(m, k, n, 4096, 4096, 1e-5, 4096, 4096, None, 4096, None)
        assert st == _lib.M3_ERR_UNSUPPORTED, (m, k, n)
        assert b"normed product covers" in L.m3_last_error()


@gpu
def test_normed_rows_past_the_kernel_run_as_two_calls():
    from mamba3 import _lib
    from mamba3.nn import Linear, RmsNorm
    lin = Linear(t_f32(np.random.default_rng(1).normal(0, 0.02, (128, 64)).astype(np.float32)))
    norm = RmsNorm(128, torch.device("cuda"))
    x = torch.randn(5, 1, 128, device="cuda").bfloat16()
    before = _lib.lib().m3_launch_count()
    y = lin.apply_normed(x, norm)
    assert _lib.lib().m3_launch_count() - before == 2 and y.shape == (5, 1, 64)
    assert torch.equal(y, lin.apply(norm.apply(x)))
