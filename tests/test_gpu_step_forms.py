"""The forms of the decode step (threads a workgroup, early loads) by the number
of (batch, head) workgroups, d_state and rank: at both sides of each line of the
dispatch, with rows that do not fill a form's passes, the results equal those of
the one-launch form over layers (StateCache.step_all, 256 threads at every size)
bit for bit; the fused mixer step equals the composed calls bit for bit.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

STEP_CASES = [
    # B, H, P, N, R, factored, dtype, rotational
    (1, 1, 64, 128, 1, False, torch.float32, True),
    (16, 16, 50, 128, 1, False, torch.float32, True),      # 256: the last of the widest form
    (257, 1, 50, 128, 1, True, torch.bfloat16, True),      # 257
    (5, 3, 70, 256, 2, False, torch.bfloat16, True),       # one row a wave
    (5, 3, 33, 4, 2, True, torch.float32, True),           # one lane a row
    (3, 7, 64, 128, 4, False, torch.float32, False),       # rank 4: never the widest
    (4, 65, 64, 64, 4, True, torch.bfloat16, True),
    (64, 12, 9, 64, 1, False, torch.float32, True),        # 768
    (769, 1, 50, 64, 1, False, torch.float32, True),       # 769
    (97, 8, 64, 32, 1, False, torch.bfloat16, True),       # 776, d_state under 64
    (97, 8, 64, 128, 1, True, torch.float32, False),
    (97, 8, 63, 64, 1, False, torch.float32, True),        # rows short of 512 threads' two passes
    (65, 4, 15, 64, 1, False, torch.float32, True),        # and of any form past 256
    (3, 5, 16, 64, 8, True, torch.bfloat16, True),         # rank 8, factored and not
    (3, 5, 16, 64, 8, False, torch.bfloat16, True),
]


@pytest.mark.parametrize("B,H,P,N,R,factored,dtype,rot", STEP_CASES)
def test_step_forms_agree_bit_for_bit(B, H, P, N, R, factored, dtype, rot):
    from mamba3 import StateCache
    g = torch.Generator(device=DEV).manual_seed(B * H + P + N + R)
    make = lambda: StateCache(1, B, H, P, N, rot, DEV, init_std=0.1,
                              generator=torch.Generator(device=DEV).manual_seed(3),
                              factored=factored, rank=R, dtype=dtype)
    a, b = make(), make()
    rand = lambda *s: torch.randn(s, device=DEV, generator=g)
    for step in range(2):
        t = (rand(B, H, P, R).to(dtype), (rand(B, H, N, R) / N ** 0.5).to(dtype),
             (rand(B, H, N, R) / N ** 0.5).to(dtype), rand(B, H).abs() * 0.05,
             torch.sigmoid(rand(B, H)), rand(H).abs(),
             rand(B, H, N // 2).to(dtype) if rot else None, rand(H))
        ya, (yb,) = a.step_layer(0, *t), b.step_all([t])
        torch.cuda.synchronize()
        assert torch.equal(ya, yb), step
        for k in ("h", "last_u", "x_prev", "b_prev", "angle"):
            if getattr(a, k) is not None:
                assert torch.equal(getattr(a, k), getattr(b, k)), (step, k)


@pytest.mark.parametrize("B", [1, 64, 65, 128, 129, 192, 193, 383, 384])
@pytest.mark.parametrize("N,R,conv,factored", [(128, 1, False, False), (128, 1, True, False),
                                               (64, 1, False, False), (128, 1, False, True),
                                               (32, 2, True, True), (128, 4, False, False)])
def test_fused_mixer_forms_equal_the_composed_calls(B, N, R, conv, factored):
    from mamba3 import SsmConfig, SsmMode
    from mamba3.mixer import Mamba3Mixer
    g = torch.Generator(device=DEV).manual_seed(B + N + R)
    H, P = 4, 40 if R == 1 else 16
    mixer = Mamba3Mixer(SsmConfig(d_model=32, n_heads=H, head_dim=P, d_state=N, n_groups=H,
                                  mode=SsmMode(R), conv_kernel=4 if conv else None),
                        device=DEV, gen=g, int8_weights=True)
    cache = mixer.empty_cache(B, DEV, factored=factored)
    st = cache.ssm
    st.h.normal_(0.0, 0.1, generator=g)
    for t in (st.x_prev, st.b_prev) if factored else (st.last_u,):
        t.copy_(torch.randn(t.shape, device=DEV, generator=g) * 0.1)
    st.angle.uniform_(-3.0, 3.0, generator=g)
    if conv:
        cache.conv.copy_(torch.randn(cache.conv.shape, device=DEV, generator=g))
    fused, composed = cache.clone(), cache.clone()
    for step in range(2):
        x = torch.randn(B, 1, 32, device=DEV, generator=g).to(torch.bfloat16)
        mixer._fused_step_ok = None
        ya = mixer.step_(x, fused)
        assert mixer._fused_step_ok
        mixer._fused_step_ok = False
        yb = mixer.step_(x, composed)
        torch.cuda.synchronize()
        assert torch.equal(ya, yb), step
        for k in ("h", "last_u", "x_prev", "b_prev", "angle"):
            p, q = getattr(fused.ssm, k, None), getattr(composed.ssm, k, None)
            if p is not None:
                assert torch.equal(p, q), (step, k)
        if conv:
            assert torch.equal(fused.conv, composed.conv)
