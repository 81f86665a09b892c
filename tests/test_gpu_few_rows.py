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

pytestmark = pytest.mark.gpu

CASES = [
    # m, k, n, int8, residual
    (1, 64, 16, True, True), (1, 192, 20, False, False), (3, 1536, 1000, True, True),
    (4, 768, 5400, True, False), (5, 512, 4100, True, True), (16, 1536, 4096, False, True),
    (16, 320, 300, True, True), (17, 1024, 516, True, True), (31, 768, 768, False, False),
    (32, 512, 4092, True, True), (32, 512, 4640, True, True), (33, 768, 5400, True, False),
    (64, 768, 4100, True, True), (49, 64, 6192, False, True),
]


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


def test_few_rows_repeat_bit_for_bit():
    from mamba3.nn import Linear
    rng = np.random.default_rng(2)
    lin = Linear(t_f32(rng.normal(0, 0.02, (1536, 10800)).astype(np.float32)), int8_weights=True)
    x = t_bf16(mo.bf16(rng.normal(0, 1, (6, 1536))))
    a, b = lin.apply(x), lin.apply(x)
    assert torch.equal(a, b)
    # a row's result does not depend on the rows beside it
    assert torch.equal(lin.apply(x[2:5].contiguous())[1], lin.apply(x[3:4].contiguous())[0])
