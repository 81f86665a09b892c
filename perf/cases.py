"""The timed workloads of this framework: the scan, its training step, the decode
step, the mixer and the language model, each through its public entry points.

Sizes are those of the benchmark configurations (bench.py), of the reference's own
example and benchmark models (a 31.7 M-parameter language model with 16 heads of 64
and d_state 64 trained at batch 4 x 512; a small one with 4 heads of 16 and d_state
16), and of the default SsmConfig.  `listed()` names them, `draw(rng)` gives others
of the same ranges, `exact(case, seed)` restates each path in 64 bits with plain
torch.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "mamba-trainer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda:0"
_TYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
VOCAB = 32000


# ------------------------------------------------------------------ the cases
def _scan(kind, batch, seq, heads, head_dim, d_state, rank, dtype, theta=True, skip=True,
          carried=False):
    return dict(kind=kind, batch=batch, seq=seq, heads=heads, head_dim=head_dim, d_state=d_state,
                rank=rank, dtype=dtype, theta=theta, skip=skip, carried=carried)


def _step(batch, heads, layers, d_state=128, rank=1, factored=False):
    return dict(kind="step", batch=batch, heads=heads, layers=layers, head_dim=64,
                d_state=d_state, rank=rank, factored=factored)


def _model(kind, batch, seq, d_model, heads, d_state, conv, layers=1, factored=False):
    return dict(kind=kind, batch=batch, seq=seq, d_model=d_model, heads=heads, head_dim=64,
                d_state=d_state, conv=conv, layers=layers, factored=factored)


def listed():
    return [
        # A short f32 window of a small model, real dynamics: the smallest scan
        # call, where launches and latency count.
        dict(_scan("scan", 2, 512, 4, 64, 64, 1, "f32", theta=False, skip=False),
             name="scan_f32_512"),
        # The headline scan: one layer of a d_model-768 model, batch 8 x 2048.
        dict(_scan("scan", 8, 2048, 12, 64, 128, 1, "bf16", skip=False), name="scan_bf16_2048"),
        # The rank-4 (MIMO) layer at 4096 tokens.
        dict(_scan("scan", 4, 4096, 24, 64, 128, 4, "bf16", skip=False), name="scan_mimo4_4096"),
        # A ragged window continuing from a carried state, on the default
        # SsmConfig's 24 heads and d_state 64: chunked prefill in serving.
        dict(_scan("scan", 3, 777, 24, 64, 64, 1, "bf16", carried=True), name="scan_window_777"),
        # Forward and backward of the headline layer: the training step's scan.
        dict(_scan("train", 8, 2048, 12, 64, 128, 1, "bf16"), name="train_bf16_2048"),
        # The same for the 31.7 M-parameter model, trained in f32.
        dict(_scan("train", 4, 512, 16, 64, 64, 1, "f32"), name="train_f32_512"),
        # The same for the small example model (4 heads of 16, d_state 16).
        dict(_scan("train", 4, 512, 4, 16, 16, 1, "f32"), name="train_f32_small"),
        # One decode token over the f32 cache at batch 256 (four layers of it).
        dict(_step(256, 24, 4), name="step_256"),
        # One mixer layer of the d_model-768 model over a whole prefill batch.
        dict(_model("mixer", 16, 2048, 768, 12, 128, False), name="mixer_prefill"),
        # One decode step of the default mixer (convolution) at batch 256.
        dict(_model("mixer_step", 256, 1, 1536, 24, 128, True), name="mixer_step_256"),
        # A prompt through the language model, ragged: time to first token.
        dict(_model("lm_prefill", 2, 509, 768, 12, 128, False, layers=4), name="lm_prefill_509"),
        # Interactive generation: one token of one sequence, the captured step.
        dict(_model("lm_decode", 1, 1, 1536, 24, 128, False, layers=4), name="lm_decode_1"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (d_model, heads, d_state) of the models named above.
_SHAPES = [(512, 16, 64), (768, 12, 128), (768, 24, 64), (1536, 24, 128)]


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "train", "train", "train", "step", "mixer",
                       "mixer_step", "lm_prefill", "lm_decode", "lm_decode"])
    if kind in ("scan", "train"):
        if rng.random() < 0.2:
            # heads of a small model: short windows
            p = rng.choice([16, 32])
            return _scan(kind, _log(rng, 1, 8), _log(rng, 33, 400), rng.choice([2, 4, 8]), p,
                         rng.choice([16, 32]), 1, rng.choice(["f32", "bf16"]),
                         theta=rng.random() < 0.8, skip=rng.random() < 0.5)
        rank = rng.choice([1, 1, 1, 2, 4])
        dtype = rng.choice(["bf16", "bf16", "f32"])
        n = rng.choice([64, 128])
        heads = rng.choice([4, 8, 12, 16, 24])
        batch, seq = _log(rng, 1, 12), _log(rng, 64, 4096)
        # no more work than the listed rank-4 scan or bf16 training step
        most = 8 * 2048 * 12 / (rank if kind == "train" else 1)
        if dtype == "f32":
            most /= 4
        while batch * seq * heads > most:
            if batch > 1:
                batch = (batch + 1) // 2
            else:
                seq = seq * 2 // 3
        return _scan(kind, batch, seq, heads, 64, n, rank, dtype, theta=rng.random() < 0.8,
                     skip=rng.random() < 0.6, carried=rng.random() < 0.4)
    if kind == "step":
        return _step(_log(rng, 1, 256), rng.choice([8, 12, 16, 24]), rng.choice([1, 2, 4]),
                     d_state=rng.choice([64, 128]), rank=rng.choice([1, 1, 2, 4]),
                     factored=rng.random() < 0.4)
    d_model, heads, d_state = rng.choice(_SHAPES)
    conv, factored = rng.random() < 0.5, rng.random() < 0.4
    if kind == "mixer":
        seq = _log(rng, 100, 2048)
        return _model(kind, min(_log(rng, 1, 16), max(1, 12000 // seq)), seq, d_model, heads,
                      d_state, conv)
    if kind == "mixer_step":
        return _model(kind, _log(rng, 1, 256), 1, d_model, heads, d_state, conv,
                      factored=factored)
    if kind == "lm_prefill":
        seq = _log(rng, 32, 1024)
        return _model(kind, min(_log(rng, 1, 4), max(1, 1024 // seq)), seq, d_model, heads,
                      d_state, conv, layers=rng.choice([2, 4]))
    return _model(kind, _log(rng, 1, 64), 1, d_model, heads, d_state, conv,
                  layers=rng.choice([2, 4]), factored=factored)


# ------------------------------------------------------------------ the inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _scan_inputs(case, seed):
    """x ~ N(0, 1); B, C ~ N(0, 1) / sqrt(d_state); dt = softplus(N(-3, 1)) in
    [1e-3, 0.1]; lambda = sigmoid(N(0, 1)); A in U(1, 16); theta ~ U(0, pi)."""
    g = _gen(seed)
    B, T, H, P, N, R = (case[k] for k in ("batch", "seq", "heads", "head_dim", "d_state", "rank"))
    ty = _TYPES[case["dtype"]]
    normal = lambda *s: torch.randn(s, device=DEV, generator=g)
    uniform = lambda *s: torch.rand(s, device=DEV, generator=g)
    v = {
        "x": normal(B, T, H, P, R).to(ty),
        "b": (normal(B, T, H, N, R) / math.sqrt(N)).to(ty),
        "c": (normal(B, T, H, N, R) / math.sqrt(N)).to(ty),
        "dt": torch.nn.functional.softplus(normal(B, T, H) - 3.0).clamp(1e-3, 0.1),
        "a_log": uniform(H) * math.log(16.0),
        "lam": torch.sigmoid(normal(B, T, H)),
        "theta": (uniform(B, T, H, N // 2) * math.pi).to(ty) if case["theta"] else None,
        "skip": normal(H) if case["skip"] else None,
    }
    if case["carried"]:
        v["h"] = normal(B, H, P, N) * 0.1
        v["last_u"] = normal(B, H, P, N) * 0.1
        v["angle"] = (uniform(B, H, N // 2) * 2 - 1) * math.pi if case["theta"] else None
    if case["kind"] == "train":
        v["dy"] = normal(B, T, H, P, R).to(ty)
    return v


def _step_inputs(case, seed):
    g = _gen(seed)
    B, H, P, N, R, L = (case[k] for k in ("batch", "heads", "head_dim", "d_state", "rank",
                                          "layers"))
    normal = lambda *s: torch.randn(s, device=DEV, generator=g)
    uniform = lambda *s: torch.rand(s, device=DEV, generator=g)
    tokens = []
    for _ in range(L):
        tokens.append({
            "x": normal(B, H, P, R), "b": normal(B, H, N, R) / math.sqrt(N),
            "c": normal(B, H, N, R) / math.sqrt(N),
            "dt": torch.nn.functional.softplus(normal(B, H) - 3.0).clamp(1e-3, 0.1),
            "lam": torch.sigmoid(normal(B, H)), "a_log": uniform(H) * math.log(16.0),
            "theta": uniform(B, H, N // 2) * math.pi, "skip": torch.ones(H, device=DEV)})
    state = {"h": normal(L, B, H, P, N).mul_(0.1),
             "angle": (uniform(L, B, H, N // 2) * 2 - 1) * math.pi}
    if case["factored"]:
        state["x_prev"] = normal(L, B, H, P, R)
        state["b_prev"] = normal(L, B, H, N, R) / math.sqrt(N)
    else:
        state["last_u"] = normal(L, B, H, P, N).mul_(0.1)
    return tokens, state


def _ssm_config(case):
    from mamba3 import SsmConfig
    return SsmConfig(d_model=case["d_model"], n_heads=case["heads"], head_dim=case["head_dim"],
                     d_state=case["d_state"], n_groups=case["heads"],
                     conv_kernel=4 if case["conv"] else None)


def _mixer_params(case, g, pre=""):
    """The reference's initial distributions, with small random biases and gains
    as after some training."""
    D, H, P, N = case["d_model"], case["heads"], case["head_dim"], case["d_state"]
    inner = H * P
    width = 2 * inner + 2 * H * N + 2 * H + H * (N // 2)
    normal = lambda *s: torch.randn(s, device=DEV, generator=g)
    uniform = lambda *s: torch.rand(s, device=DEV, generator=g)
    dt = torch.exp(math.log(1e-3) + uniform(H) * math.log(100.0)).clamp_min(1e-4)
    p = {
        "in_proj.weight": normal(D, width) * 0.02,
        "out_proj.weight": normal(inner, D) * (0.02 / math.sqrt(2 * case["layers"])),
        "dt_bias": dt + torch.log(-torch.expm1(-dt)),
        "a_log": torch.log(1 + 15 * uniform(H)),
        "d": 1 + 0.1 * normal(H), "b_bias": 0.1 * normal(H, N), "c_bias": 0.1 * normal(H, N),
        "bc_norm.weight": 1 + 0.1 * normal(N),
    }
    if case["conv"]:
        p["conv.weight"] = (uniform(4, inner + 2 * H * N) * 2 - 1) * math.sqrt(3.0 / 4)
        p["conv.bias"] = 0.1 * normal(inner + 2 * H * N)
    return {pre + k: v for k, v in p.items()}


def _lm_params(case, g):
    D = case["d_model"]
    normal = lambda *s: torch.randn(s, device=DEV, generator=g)
    p = {"embed.weight": normal(VOCAB, D) * 0.02, "head.weight": normal(D, VOCAB) * 0.02,
         "norm_f.weight": 1 + 0.1 * normal(D)}
    for i in range(case["layers"]):
        p["stack.layers.%d.norm.weight" % i] = 1 + 0.1 * normal(D)
        p.update(_mixer_params(case, g, "stack.layers.%d.mixer." % i))
    return p


def _cache_values(case, g):
    """The cache in the middle of a generation, one dict a layer.  The angles
    stay clear of +-pi, where the last bit of a projection would decide which
    end of the circle a step's wrapped angle comes out at."""
    B, H, P, N = case["batch"], case["heads"], case["head_dim"], case["d_state"]
    normal = lambda *s: torch.randn(s, device=DEV, generator=g)
    out = []
    for _ in range(case["layers"]):
        v = {"h": normal(B, H, P, N) * 0.1,
             "angle": (torch.rand(B, H, N // 2, device=DEV, generator=g) * 2 - 1) * 2.0}
        if case["factored"]:
            v["x_prev"] = normal(B, H, P, 1).bfloat16()
            v["b_prev"] = normal(B, H, N, 1).bfloat16()
        else:
            v["last_u"] = normal(B, H, P, N) * 0.1
        if case["conv"]:
            v["conv"] = normal(B, 3, H * P + 2 * H * N).bfloat16()
        out.append(v)
    return out


def _fill_cache(cache, values):
    for c, v in zip(cache, values):
        for k, t in v.items():
            (c.conv if k == "conv" else getattr(c.ssm, k)).copy_(t)


def _cache_tensors(cache):
    names = ("h", "last_u", "x_prev", "b_prev", "angle")
    return [dict({k: getattr(c.ssm, k) for k in names if hasattr(c.ssm, k)},
                 **({} if c.conv is None else {"conv": c.conv})) for c in cache]


def _set_params(module, params):
    for name, p in module.named_parameters():
        p.set(params[name].reshape(p.shape))


def prepare(case, seed):
    from mamba3 import StateCache
    from mamba3.mixer import Mamba3Mixer
    from mamba3.lm import Mamba3Lm, Mamba3LmConfig
    kind = case["kind"]
    if kind in ("scan", "train"):
        v = _scan_inputs(case, seed)
        if kind == "train":
            v["leaves"] = [k for k in ("x", "b", "c", "dt", "a_log", "lam", "theta", "skip", "h",
                                       "last_u", "angle") if v.get(k) is not None]
            for k in v["leaves"]:
                v[k].requires_grad_()
        return dict(case=case, v=v)
    if kind == "step":
        tokens, values = _step_inputs(case, seed)
        cache = StateCache(case["layers"], case["batch"], case["heads"], case["head_dim"],
                           case["d_state"], True, DEV, factored=case["factored"],
                           rank=case["rank"], dtype=torch.float32)
        for k, t in values.items():
            getattr(cache, k).copy_(t)
        order = ("x", "b", "c", "dt", "lam", "a_log", "theta", "skip")
        return dict(case=case, cache=cache, tokens=[tuple(t[k] for k in order) for t in tokens])
    g = _gen(seed)
    if kind in ("mixer", "mixer_step"):
        mixer = Mamba3Mixer(_ssm_config(case), device=DEV, gen=_gen(0), int8_weights=True)
        _set_params(mixer, _mixer_params(case, g))
        x = torch.randn((case["batch"], case["seq"], case["d_model"]), device=DEV,
                        generator=g).bfloat16()
        s = dict(case=case, mixer=mixer, x=x)
        if kind == "mixer_step":
            s["cache"] = mixer.empty_cache(case["batch"], DEV, factored=case["factored"])
            _fill_cache([s["cache"]], _cache_values(case, g))
        return s
    lm = Mamba3Lm(Mamba3LmConfig(vocab_size=VOCAB, d_model=case["d_model"],
                                 n_layers=case["layers"], ssm=_ssm_config(case),
                                 int8_weights=True), DEV)
    _set_params(lm, _lm_params(case, g))
    ids = torch.randint(0, VOCAB, (case["batch"], case["seq"]), device=DEV, generator=g)
    s = dict(case=case, lm=lm, ids=ids)
    if kind == "lm_decode":
        s["cache"] = lm.empty_cache(case["batch"], DEV, factored=case["factored"])
        _fill_cache(s["cache"], _cache_values(case, g))
        s["graph"] = lm.capture_decode(s["cache"], case["batch"])
    return s


# ------------------------------------------------------------------ one pass
def _request(v):
    from mamba3.ssm import ScanInputs, SsmState
    si = ScanInputs(v["x"], v["b"], v["c"], v["dt"], v["a_log"], v["lam"])
    if v["theta"] is not None:
        si = si.with_theta(v["theta"])
    if v["skip"] is not None:
        si = si.with_skip(v["skip"])
    if "h" in v:
        si = si.with_state(SsmState(v["h"], v["last_u"], v["angle"]))
    return si


def run(state):
    from mamba3.ssm import mamba3_scan
    kind = state["case"]["kind"]
    if kind == "scan":
        out = mamba3_scan(_request(state["v"]))
        return {"y": out.y, "h": out.state.h, "last_u": out.state.last_u,
                "angle": out.state.angle}
    if kind == "train":
        v = state["v"]
        out = mamba3_scan(_request(v).with_state_output(False))
        grads = torch.autograd.grad(out.y, [v[k] for k in v["leaves"]], v["dy"])
        return dict({"d_" + k: t for k, t in zip(v["leaves"], grads)}, y=out.y.detach())
    if kind == "step":
        cache = state["cache"]
        ys = [cache.step_layer(i, *t) for i, t in enumerate(state["tokens"])]
        return {"y": ys, "h": cache.h, "last_u": cache.last_u, "x_prev": cache.x_prev,
                "b_prev": cache.b_prev, "angle": cache.angle}
    if kind == "mixer":
        return state["mixer"].apply(state["x"])
    if kind == "mixer_step":
        y = state["mixer"].step_(state["x"], state["cache"])
        return {"y": y, "cache": _cache_tensors([state["cache"]])}
    if kind == "lm_prefill":
        return state["lm"].forward(state["ids"])
    logits = state["graph"].step(state["ids"])
    return {"logits": logits, "cache": _cache_tensors(state["cache"])}


# ------------------------------------------------------------------ work
def work(case):
    """Bytes: each input read once, each output written once.  FLOPs: the
    products of the chunked form at 64-token chunks (training: with the three
    times as many of its backward), and the projections."""
    B, H, P, N = case["batch"], case["heads"], case["head_dim"], case["d_state"]
    T, R, kind = case.get("seq", 1), case.get("rank", 1), case["kind"]
    tok = B * T * H
    scan = tok * (2 * min(64, T) * R * R * (N + P) + 4 * R * P * N)
    if kind in ("scan", "train"):
        s = 2 if case["dtype"] == "bf16" else 4
        th = N // 2 if case["theta"] else 0
        ins = tok * ((P * R + 2 * N * R + th) * s + 8)
        st = B * H * (2 * P * N + th) * 4
        ys = tok * P * R * s
        if kind == "scan":
            return {"bytes": ins + ys + st * (2 if case["carried"] else 1), "flops": scan}
        carried = st * 2 if case["carried"] else 0
        # y written; dy read, every input's gradient written
        return {"bytes": 2 * ins + 2 * ys + carried, "flops": 3 * scan}
    cache = B * H * (2 * P * N * (4 if case["factored"] else 8) + N // 2 * 8)
    if kind == "step":
        if case["factored"]:
            cache += B * H * (P + N) * R * 8
        io = B * H * (2 * P * R + 2 * N * R + N // 2 + 2) * 4
        return {"bytes": case["layers"] * (cache + io),
                "flops": case["layers"] * 6 * B * H * R * P * N}
    D, L = case["d_model"], case["layers"]
    width = 2 * H * P + 2 * H * N + 2 * H + H * (N // 2)
    weights = D * width + H * P * D + 4 * (width + D)      # int8 codes and their scales
    proj = 2 * B * T * D * (width + H * P)
    if kind == "mixer":
        return {"bytes": weights + 4 * B * T * D, "flops": proj + scan}
    if case["conv"] and kind.endswith("step") or kind == "lm_decode" and case["conv"]:
        cache += 2 * B * 3 * (H * P + 2 * H * N) * 2
    step = 6 * B * H * P * N
    if kind == "mixer_step":
        return {"bytes": weights + cache + 4 * B * D, "flops": proj + step}
    head = 2 * D * VOCAB + B * T * (VOCAB * 2 + 8 + 2 * D)
    each = scan if kind == "lm_prefill" else step
    return {"bytes": L * (weights + (cache if kind == "lm_decode" else 0)) + head,
            "flops": L * (proj + each) + 2 * B * T * D * VOCAB}


def tolerance(case):
    """About four times the error against `exact` (relative 2-norms): f32 scans
    5e-8 to 2.6e-6 (the state's long sums; an angle summed over thousands of
    tokens up to 5e-6), their gradients up to 1.2e-6, f32 steps up to 7e-8 (a sine
    of another last bit 2e-7); bf16 scans 3.4e-3 (y and the carried states are
    rounded to bf16), their gradients 1.7e-3 (one rounding of the result); the
    mixer 5e-3 (a rounding of each intermediate row); four layers with logits
    1e-2, where a change of rounding in one travels through the others."""
    kind = case["kind"]
    if kind in ("scan", "train"):
        return {"rel": 1.3e-2 if case["dtype"] == "bf16" else 1e-5}
    if kind == "step":
        return {"rel": 1e-6}
    return {"rel": 2e-2 if kind.startswith("mixer") else 3e-2}


# ------------------------------------------------------------------ 64 bits
def _rotate(v, phi):
    """Half-split rotation by -phi: v [..., N, R], phi [..., N/2]."""
    c, s = torch.cos(phi).unsqueeze(-1), torch.sin(phi).unsqueeze(-1)
    v1, v2 = v.chunk(2, dim=-2)
    return torch.cat([v1 * c + v2 * s, v2 * c - v1 * s], dim=-2)


def _wrap(phi):
    return phi - 2 * math.pi * torch.round(phi / (2 * math.pi))


def _scan64(v, chunk=64):
    """The scan by chunks of its recurrence h_t = e_t h_{t-1} + (1 - lam_t) dt_t
    e_t u_{t-1} + lam_t dt_t u_t, e_t = exp(-exp(a_log) dt_t), u_t = sum_r x_t,r
    B~_t,r^T, y_t = h_t C~_t + D x_t, with B and C rotated by minus the running
    angle.  Returns y, h, last_u, angle."""
    x, b, c, dt, lam = v["x"], v["b"], v["c"], v["dt"], v["lam"]
    B, T, H, P, R = x.shape
    N = b.shape[3]
    la = -torch.exp(v["a_log"]) * dt
    phi = None
    if v.get("theta") is not None:
        phi = torch.cumsum(dt.unsqueeze(-1) * v["theta"], 1)
        if v.get("angle") is not None:
            phi = phi + v["angle"].unsqueeze(1)
        b, c = _rotate(b, phi), _rotate(c, phi)
    nxt = torch.cat([((1 - lam) * dt)[:, 1:], torch.zeros_like(dt[:, :1])], 1)
    g = lam * dt
    S = torch.zeros(B * H, P, N, dtype=x.dtype, device=x.device)
    if v.get("h") is not None:
        S = (v["h"] + ((1 - lam) * dt)[:, 0, :, None, None] * v["last_u"]).reshape(B * H, P, N)
    heads = lambda t: t.transpose(1, 2).reshape((B * H, t.shape[1]) + tuple(t.shape[3:]))
    ys = []
    for t0 in range(0, T, chunk):
        sl = slice(t0, min(T, t0 + chunk))
        q = sl.stop - sl.start
        xs, bs, cs = (heads(t[:, sl]).transpose(2, 3).reshape(B * H, q * R, -1) for t in (x, b, c))
        ac = torch.cumsum(heads(la[:, sl]), 1)
        gs, fs = heads(g[:, sl]), heads(nxt[:, sl])
        row = torch.arange(q, device=x.device)
        low = (row[:, None] > row[None, :]).to(x.dtype)
        eye = torch.eye(q, dtype=x.dtype, device=x.device)
        diff = ac[:, :, None] - ac[:, None, :]
        k = torch.exp(diff * (low + eye)) * (low * (gs + fs)[:, None, :] + eye * gs[:, None, :])
        k = k.repeat_interleave(R, 1).repeat_interleave(R, 2)
        band = torch.bmm(cs, bs.transpose(1, 2).contiguous()) * k
        ea = torch.exp(ac).repeat_interleave(R, 1).unsqueeze(-1)
        y = torch.bmm(band, xs) + ea * torch.bmm(cs, S.transpose(1, 2).contiguous())
        ys.append(y.reshape(B, H, q, R, P).permute(0, 2, 1, 4, 3))
        w = (torch.exp(ac[:, -1:] - ac) * (gs + fs)).repeat_interleave(R, 1).unsqueeze(-1)
        S = torch.exp(ac[:, -1])[:, None, None] * S + torch.bmm(
            (xs * w).transpose(1, 2).contiguous(), bs)
    y = torch.cat(ys, 1)
    if v.get("skip") is not None:
        y = y + v["skip"][:, None, None] * x
    last = torch.matmul(x[:, -1], b[:, -1].transpose(-1, -2).contiguous())
    return y, S.reshape(B, H, P, N), last, None if phi is None else _wrap(phi[:, -1])


def _double(v):
    return {k: t.detach().double() for k, t in v.items() if isinstance(t, torch.Tensor)}


def _step64(x, b, c, dt, lam, a_log, theta, skip, st):
    """One token [B, H, ...]; st: h, angle and last_u (or x_prev, b_prev) in 64
    bits.  Returns y and the new h, last_u, angle."""
    last_u = st.get("last_u")
    if last_u is None:
        last_u = torch.matmul(st["x_prev"], _rotate(st["b_prev"], st["angle"])
                              .transpose(-1, -2).contiguous())
    phi = st["angle"] + dt.unsqueeze(-1) * theta
    b, c = _rotate(b, phi), _rotate(c, phi)
    e = torch.exp(-torch.exp(a_log) * dt)
    u = torch.matmul(x, b.transpose(-1, -2).contiguous())
    ex = lambda t: t[..., None, None]
    h = ex(e) * st["h"] + ex((1 - lam) * dt * e) * last_u + ex(lam * dt) * u
    y = torch.matmul(h, c) + skip[:, None, None] * x
    return y, h, u, _wrap(phi)


def _codes(w):
    """The int8 grid of a weight [in, out], per output channel."""
    s = w.abs().amax(0).clamp_min(1e-12) / 127.0
    return torch.clamp(torch.round(w / s), -127, 127).double() * s.double()


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()


def _mixer64(case, p, x, cache=None):
    """The mixer on x [B, T, D]; with a cache (its values in 64 bits) one step.
    Returns the output and the new cache."""
    silu = torch.nn.functional.silu
    B, T = x.shape[:2]
    H, P, N = case["heads"], case["head_dim"], case["d_state"]
    inner = H * P
    row = x @ _codes(p["in_proj.weight"])
    z, xbc, dt, lam, th = row.split([inner, inner + 2 * H * N, H, H, H * (N // 2)], -1)
    new = {}
    if case["conv"]:
        hist = torch.zeros(B, 3, xbc.shape[-1], dtype=x.dtype, device=x.device) \
            if cache is None else cache["conv"]
        win = torch.cat([hist, xbc], 1)
        w = p["conv.weight"].double()
        new["conv"] = win[:, T:]
        xbc = sum(w[j] * win[:, j:j + T] for j in range(4)) + p["conv.bias"].double()
    xi, b, c = silu(xbc).split([inner, H * N, H * N], -1)
    xi = xi.reshape(B, T, H, P, 1)
    bc = lambda t, bias: _norm(t.reshape(B, T, H, N) + bias.double(),
                               p["bc_norm.weight"]).unsqueeze(-1)
    b, c = bc(b, p["b_bias"]), bc(c, p["c_bias"])
    dt = torch.nn.functional.softplus(dt + p["dt_bias"].double(), threshold=200)
    lam, th = torch.sigmoid(lam), th.reshape(B, T, H, N // 2)
    a_log, skip = p["a_log"].double(), p["d"].double()
    if cache is None:
        y = _scan64(dict(x=xi, b=b, c=c, dt=dt, lam=lam, a_log=a_log, theta=th, skip=skip))[0]
    else:
        y, h, u, ang = _step64(xi[:, 0], b[:, 0], c[:, 0], dt[:, 0], lam[:, 0], a_log, th[:, 0],
                               skip, cache)
        new.update(h=h, angle=ang)
        new.update(dict(x_prev=xi[:, 0], b_prev=b[:, 0]) if case["factored"]
                   else dict(last_u=u))
    y = y.reshape(B, T, inner) * silu(z)
    return y @ _codes(p["out_proj.weight"]), new


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        y, h, u, ang = _scan64(_double(_scan_inputs(case, seed)))
        return {"y": y, "h": h, "last_u": u, "angle": ang}
    if kind == "train":
        v = _double(_scan_inputs(case, seed))
        leaves = [k for k in v if k != "dy"]
        for k in leaves:
            v[k].requires_grad_()
        y = _scan64(v)[0]
        grads = torch.autograd.grad(y, [v[k] for k in leaves], v["dy"])
        return dict({"d_" + k: t for k, t in zip(leaves, grads)}, y=y.detach())
    if kind == "step":
        tokens, st = _step_inputs(case, seed)
        ys, hs, us, an = [], [], [], []
        for i, t in enumerate(tokens):
            t = _double(t)
            y, h, u, a = _step64(t["x"], t["b"], t["c"], t["dt"], t["lam"], t["a_log"],
                                 t["theta"], t["skip"], {k: s[i].double() for k, s in st.items()})
            ys.append(y), hs.append(h), us.append(u), an.append(a)
        out = {"y": ys, "h": torch.stack(hs), "angle": torch.stack(an), "last_u": None,
               "x_prev": None, "b_prev": None}
        if not case["factored"]:
            out["last_u"] = torch.stack(us)
        return out
    g = _gen(seed)
    if kind in ("mixer", "mixer_step"):
        p = _mixer_params(case, g)
        x = torch.randn((case["batch"], case["seq"], case["d_model"]), device=DEV,
                        generator=g).bfloat16().double()
        if kind == "mixer":
            return _mixer64(case, p, x)[0]
        y, new = _mixer64(case, p, x, _double(_cache_values(case, g)[0]))
        return {"y": y, "cache": [new]}
    p = _lm_params(case, g)
    ids = torch.randint(0, VOCAB, (case["batch"], case["seq"]), device=DEV, generator=g)
    cache = _cache_values(case, g) if kind == "lm_decode" else None
    x = p["embed.weight"].bfloat16().double()[ids]
    news = []
    for i in range(case["layers"]):
        pre = "stack.layers.%d." % i
        lp = {k[len(pre) + 6:]: t for k, t in p.items() if k.startswith(pre + "mixer.")}
        y, new = _mixer64(case, lp, _norm(x, p[pre + "norm.weight"]),
                          None if cache is None else _double(cache[i]))
        x = x + y
        news.append(new)
    logits = _norm(x, p["norm_f.weight"]) @ p["head.weight"].bfloat16().double()
    return logits if kind == "lm_prefill" else {"logits": logits, "cache": news}
