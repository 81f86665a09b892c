// Backward of the chunked SSD scan (mamba3_scan, src/ssm/scan.rs:458-638) for
// gfx950: the gradient the reference obtains by autodiff through the composed
// scan, whose hand-written adjoints are ssd_band_backward
// (src/tensor/ops/fused.rs:2080-2138), exp_decay_backward (2326-2382) and
// trapezoid_weights_backward (2513-2549).  Shapes as the chunk-parallel
// forward: head_dim 64, d_state 64/128, rank 1/2/4; f32 or bf16 storage,
// f32 arithmetic (MFMA f32 16x16x4 over f32 operands in LDS).
//
// Chunks of 32 rows (token, rank).  In chunk k's own rotating frame, with alpha the in-chunk inclusive cumsum of a = dt A, K_ts = W_ts e^{alpha_t -
// alpha_s} (W = g on the token diagonal, w below it), CB = C~ B~^T, M = CB o K,
// wbar_s = e^{alpha_E - alpha_s} w_s, S_k the state entering the chunk and
// Gh_k = dL/d(e_k S_k + U_k) = R(-Phi_k) G_{k+1}:
//
//   dX       = M^T dY + D dY + diag(wbar) B~ Gh^T
//   dC~      = (dY X^T o K) B~ + diag(e^alpha) dY S
//   dB~      = (dY X^T o K)^T C~ + diag(wbar) X Gh
//   G_k      = e_k Gh_k + (diag(e^alpha) dY)^T C~            (reverse state pass)
//   dalpha_t = sum_{s<t} L_ts - sum_{t'>t} L_t't + e^{alpha_t} dy_t . (S C~_t)
//              - wbar_t x_t . (Gh B~_t)   (+ the alpha_E terms on the last row),
//              L = dM o M;  da = in-chunk reverse cumsum of dalpha
//   dphi_t   = sum_pairs dB~1 B~2 - dB~2 B~1 + dC~1 C~2 - dC~2 C~1, invariant
//              under the frame rotation, so the global angle gradient is its
//              reverse cumsum over the whole sequence.
//
// Launches: bwd_passes_kernel (the forward recurrence giving S_k, each
// chunk's U_k, the forward's chunk state, formed in place with f32 operands;
// and the reverse one giving G and Gh per chunk, with each chunk's V_k, its
// direct share of G, and dh0 / dlast_u0; side by side), bwd_chunk_kernel (dx, db, dc and
// the per-token da, dg, dw and angle sums), bwd_angle_kernel (the angle sums
// of later chunks), bwd_token_kernel (dtheta, ddt, dlambda: trapezoid_weights
// backward, the decay and angle chains) and bwd_head_kernel (da_log, dD).
#include <algorithm>

#include "scan_common.hpp"

namespace m3 {

namespace {

constexpr int kP = 64;
constexpr int kRows = 32;    // (token, rank) rows of a chunk
constexpr int kWaves = 8;    // of the chunk kernel
constexpr int kBT = 64 * kWaves;

struct BwdArgs {
    const void *dy;           // [B,T,H,P,R]
    const float *dh_out;      // [B,H,P,N] or null
    const float *dangle_out;  // [B,H,N/2] or null
    const float *dlast_u_out; // [B,H,P,N] or null
    void *dx, *db, *dc;       // storage type
    float *ddt, *dlambda;     // [B,T,H]
    float *da_log;            // [H]
    void *dtheta;             // [B,T,H,N/2] or null
    float *dd_skip;           // [H] or null
    float *dh0, *dlast_u0;    // [B,H,P,N] or null
    float *dangle0;           // [B,H,N/2] or null
    bool add_sums;            // da_log and dd_skip are added to
};

// Backward workspace, 256-byte aligned sections.  Per (batch, head, chunk):
// S_k and Gh_k as f32 [p-tile][n-tile][lane][4] MFMA D-layout records of the
// [P][N] state and the chunk decay e_k, for a window of `wn` chunks of every
// sequence (all of them where the workspace holds that): the passes and the
// chunk kernel run once a window, each of whose passes walks the whole sequence
// and writes its own chunks' records.  pd and pa add up over the windows.
// With an upstream gradient of the outgoing last_u: the angle seed (that
// gradient's angle term plus dL/dangle) and the last token's dx and db terms.
struct BwdLayout {
    size_t s, gh, eda, cin, ctot, da, dg, dw, pd, pa, pfirst;
    size_t seed, lux, lub, total;
};

size_t balign(size_t v) { return (v + 255) & ~size_t(255); }

BwdLayout bwd_layout(size_t bh, size_t nck, size_t wn, size_t seq, size_t n, size_t r) {
    const size_t bhw = bh * wn, rec = bhw * kP * n * 4, pairs = bh * nck * (n / 2) * 4;
    BwdLayout l;
    size_t o = 0;
    l.s = o;      o = balign(o + rec);
    l.gh = o;     o = balign(o + rec);
    l.eda = o;    o = balign(o + bhw * 4);
    l.cin = o;    o = balign(o + bh * seq * (n / 2) * 4);
    l.ctot = o;   o = balign(o + pairs);
    l.da = o;     o = balign(o + bh * seq * 4);
    l.dg = o;     o = balign(o + bh * seq * 4);
    l.dw = o;     o = balign(o + bh * seq * 4);
    l.pd = o;     o = balign(o + bhw * 4);
    l.pa = o;     o = balign(o + bhw * 4);
    l.pfirst = o; o = balign(o + bh * (n / 32) * 4);
    l.seed = o;   o = balign(o + bh * (n / 2) * 4);
    l.lux = o;    o = balign(o + bh * kP * r * 4);
    l.lub = o;    o = balign(o + bh * n * r * 4);
    l.total = o;
    return l;
}

struct BwdWs {
    float *s, *gh, *eda;
    float *cin, *ctot, *da, *dg, *dw, *pd, *pa, *pfirst;
    float *seed, *lux, *lub;
    int k0, wn;   // the window: chunks k0 .. k0 + wn - 1 of each sequence
};

// element access in the storage type
template <typename T> __device__ __forceinline__ float ldv(const void *p, size_t i);
template <> __device__ __forceinline__ float ldv<float>(const void *p, size_t i) {
    return static_cast<const float *>(p)[i];
}
template <> __device__ __forceinline__ float ldv<bf16_t>(const void *p, size_t i) {
    return to_f32(static_cast<const bf16_t *>(p)[i]);
}
template <typename T> __device__ __forceinline__ void stv(void *p, size_t i, float v);
template <> __device__ __forceinline__ void stv<float>(void *p, size_t i, float v) {
    static_cast<float *>(p)[i] = v;
}
template <> __device__ __forceinline__ void stv<bf16_t>(void *p, size_t i, float v) {
    static_cast<bf16_t *>(p)[i] = from_f32<bf16_t>(v);
}

// Four elements i, i + R, i + 2R, i + 3R in the storage type: one 16-byte
// (f32) or 8-byte (bf16) store when they are adjacent (rank 1; i is then a
// multiple of 4 in a 16-byte aligned buffer), else four scalar stores.
template <typename T, int R>
__device__ __forceinline__ void st4(void *p, size_t i, f32x4 v) {
    if constexpr (R == 1) {
        if constexpr (sizeof(T) == 4) {
            *reinterpret_cast<f32x4 *>(static_cast<float *>(p) + i) = v;
        } else {
            bf16x4 h;
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = to_bf16(v[r]);
            *reinterpret_cast<bf16x4 *>(static_cast<bf16_t *>(p) + i) = h;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) stv<T>(p, i + r * R, v[r]);
    }
}

__device__ __forceinline__ float clamp_exp(float d) {
    return expf(fminf(fmaxf(d, -60.0f), 0.0f));
}

// dt A on a 2^-14 grid and what is left of it (with the product's own
// rounding): prefix sums of the grid part are exact in f32 up to 2^10, and
// those of the rest some 2^-40 off, so the difference of two prefixes is as
// exact as the step between them.  One f32 prefix of a long, fast-decaying
// chunk (about -50 at its end) holds 4e-6, which came out whole in every decay
// factor of its last rows and in da_log.
// A decay past -1e30 (infinite ones too) is taken there, where a prefix of 32
// and its grid still have a finite difference of zero with itself.
__device__ __forceinline__ void split_decay(float dt, float A, float &hi, float &lo) {
    const float v0 = dt * A, v = fmaxf(v0, -1e30f);
    hi = rintf(v * 16384.0f) * (1.0f / 16384.0f);
    lo = (v - hi) + (v == v0 ? __builtin_fmaf(dt, A, -v) : 0.0f);
}

// sin and cos of an angle, to about an ulp: the argument less the nearest
// multiple of pi / 2 by Cody and Waite's method (three parts of pi / 2 and
// fused multiply-adds, good while the multiple is an exact f32 integer and the
// last part's error stays below the result's: |x| < 2^13 here, past which the
// library's sincosf takes over), then the Taylor polynomials to r^9 and r^10
// on |r| <= pi / 4 and the quadrant's swap and signs: over every f32 of its range
// within 7.2e-8 of f64 and 1.7e-8 in the mean square (sincosf 7.2e-8 and 1.8e-8, an
// exact result rounded 3.0e-8).  34 instructions where sincosf compiles to 147,
// both its paths counted, and the backward forms three per (token, pair): a
// forward and backward of 2 x 4096 tokens, 8 heads, d_state 64, bf16 storage,
// 318 -> 305 us, of 1 x 1154, 8 heads, 128, rank 4, f32, 434 -> 418; no change
// where the chip is full (8 x 2048, 12 heads).
__device__ __forceinline__ void sincos_turn(float x, float &sn, float &cs) {
    const float k = rintf(x * 0.63661977236758134f);                 // 2 / pi
    float r = __builtin_fmaf(k, -1.5707963267948966f, x);            // pi / 2 rounded to f32,
    r = __builtin_fmaf(k, 4.3711388286737929e-08f, r);               // less what that is over,
    r = __builtin_fmaf(k, 1.7151245100058819e-15f, r);               // and the rest
    const float r2 = r * r;
    float p = __builtin_fmaf(r2, 2.7557319223985893e-06f, -1.9841269841269841e-04f);
    p = __builtin_fmaf(p, r2, 8.3333333333333333e-03f);
    p = __builtin_fmaf(p, r2, -1.6666666666666667e-01f);
    const float s = __builtin_fmaf(p * r2, r, r);
    float q = __builtin_fmaf(r2, -2.7557319223985888e-07f, 2.4801587301587302e-05f);
    q = __builtin_fmaf(q, r2, -1.3888888888888889e-03f);
    q = __builtin_fmaf(q, r2, 4.1666666666666667e-02f);
    q = __builtin_fmaf(q, r2, -0.5f);
    const float c = __builtin_fmaf(q, r2, 1.0f);
    const int n = static_cast<int>(k);
    const float a = (n & 1) ? c : s, b = (n & 1) ? s : c;
    sn = __uint_as_float(__float_as_uint(a) ^ (static_cast<uint32_t>(n & 2) << 30));
    cs = __uint_as_float(__float_as_uint(b) ^ (static_cast<uint32_t>((n + 1) & 2) << 30));
    if (__builtin_expect(!(fabsf(x) < 8192.0f), 0)) sincosf(x, &sn, &cs);
}

// Four consecutive elements of a row as they are loaded: 8 bytes of bf16
// storage, 16 of f32.  An address off the 4-byte grid (a bf16 dy the caller
// placed there) is read element by element.
template <typename T> struct Raw4 { u32x2 q; };
template <> struct Raw4<float> { u32x4 q; };
__device__ __forceinline__ void ld4(Raw4<bf16_t> &d, rsrc_t r, uint32_t off, bool aligned = true) {
    if (aligned) {
        d.q = bld8(r, off);
    } else {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            h[i] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(r, off + 2 * i, 0, 0));
        d.q = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
}
__device__ __forceinline__ void ld4(Raw4<float> &d, rsrc_t r, uint32_t off, bool = true) { d.q = bld16(r, off); }
__device__ __forceinline__ void un4(const Raw4<bf16_t> &d, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        v[2 * i] = __uint_as_float(d.q[i] << 16);
        v[2 * i + 1] = __uint_as_float(d.q[i] & 0xFFFF0000u);
    }
}
__device__ __forceinline__ void un4(const Raw4<float> &d, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(d.q[i]);
}
// PN consecutive theta values (2 or 4)
template <typename T, int PN>
__device__ __forceinline__ void ldth(rsrc_t r, uint32_t off, uint32_t (&q)[PN]) {
    if constexpr (sizeof(T) == 4) {
        if constexpr (PN == 4) {
            const u32x4 v = bld16(r, off);
            q[0] = v[0]; q[1] = v[1]; q[2] = v[2]; q[3] = v[3];
        } else {
            const u32x2 v = bld8(r, off);
            q[0] = v[0]; q[1] = v[1];
        }
    } else if constexpr (PN == 4) {
        const u32x2 v = bld8(r, off);
        q[0] = v[0]; q[1] = v[1];
    } else {
        q[0] = bld4(r, off);
    }
}
template <typename T, int PN>
__device__ __forceinline__ void unth(const uint32_t (&q)[PN], float (&v)[PN]) {
#pragma unroll
    for (int i = 0; i < PN; ++i)
        v[i] = sizeof(T) == 4 ? __uint_as_float(q[i])
                              : __uint_as_float((i & 1) ? (q[i >> 1] & 0xFFFF0000u) : (q[i >> 1] << 16));
}

// Elements e .. e + 3 (column e / R, rank e % R) of token t into a row-major
// [row][pitch] tile of (token, rank) rows.
template <int R>
__device__ __forceinline__ void put4(float *tile, int pitch, int t, int e, const float (&v)[4]) {
    if constexpr (R == 1) {
        *reinterpret_cast<f32x4 *>(tile + t * pitch + e) = f32x4{v[0], v[1], v[2], v[3]};
    } else if constexpr (R == 2) {
        *reinterpret_cast<f32x2 *>(tile + (2 * t) * pitch + e / 2) = f32x2{v[0], v[2]};
        *reinterpret_cast<f32x2 *>(tile + (2 * t + 1) * pitch + e / 2) = f32x2{v[1], v[3]};
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) tile[(4 * t + r) * pitch + e / 4] = v[r];
    }
}

// Inclusive scans over 32-lane segments of PN values at once.
template <int PN>
__device__ __forceinline__ void scan32(float (&v)[PN]) {
    if constexpr (PN == 4) {
        seg_scan4<32>(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int i = 0; i < PN; ++i) v[i] = seg_scan<32>(v[i]);
    }
}
// The wave's sum, in every lane (DPP; a shuffle tree is six LDS round trips).
__device__ __forceinline__ float wave_sum(float v) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(seg_scan<64>(v)), 63));
}

__device__ __forceinline__ float block_sum(float v, float *red) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.0f;
    for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) s += red[w];
    return s;
}

// ---------------------------------------------------------------- state passes
// The recompute's sequential parts, each with its chunk term formed in place:
//   forward: S_0 = R(angle0)(h0 + (1 - lambda_0) dt_0 last_u0) (scan.rs:521-535),
//     S_{k+1} = R(Phi_k)(e_k S_k + U_k), S_k written for every chunk
//     (scan.rs:244-251 in chunk frames), with
//     U_k^T[n][p] = sum_rho wbar B~[rho][n] X[rho][p], the chunk's contribution
//     to the state (the forward's chunk state, scan.rs:207-251), f32 operands;
//   reverse: G_C = R(phi_end) dh_out (or 0); for k = C-1 .. 0: Gh_k =
//     R(-Phi_k) G_{k+1}, G_k = e_k Gh_k + V_k, with V_k^T[n][p] =
//     sum_rho C~[rho][n] e^{alpha} dY[rho][p], the chunk's direct share of
//     dL/dS_k (the carry-in product y += e^alpha C~ S, scan.rs:253-263); then
//     dh0, dlast_u0 and the gradient of (1 - lambda_0) dt_0.
// One workgroup per (batch, head, 16 rotation pairs) and direction; the
// state's 32 columns of those pairs, for all 64 p, stay in registers in the
// MFMA D layout (lane (c, g) of wave pt: column n = 16 i1 + c and its partner,
// p = 16 pt + 4 g + r), which is also how the chunk kernel's operands read the
// records.  Per chunk the workgroup stages the token scalars and its pairs'
// in-chunk angles (the scans of the chunk kernel, so every value is the same),
// rotates its 32 columns of B (or C) into LDS scaled by wbar (or not), stages
// X (or e^alpha dY) as rows, and forms U (or V) by f32 MFMA.  The raw inputs
// are loaded ahead into registers, four elements a load; no per-chunk record
// but S_k (Gh_k) leaves the workgroup.
//
// The recurrence is serial over the chunks, so with few sequences the time is
// the chain of one step (barriers, scans, sine, products): a step is two
// chunks, whose chains run side by side between the same two barriers.  A
// forward and backward against one chunk a step: 2 x 4096 tokens, 8 heads,
// d_state 64, bf16 storage, 305 -> 261 us; 1 x 1154, 8 heads, 128, rank 4, f32,
// 418 -> 361; 2 x 1777, 12 heads, 128, f32, 243 -> 229.  With the chip full it
// is bandwidth and issue that bound them: batch 8 x 2048, 12 heads, d_state 128,
// 205 us either way, for 500 MB (100 us at the rate of a large copy).
template <int R>
struct PassSmem {
    static constexpr int QT = kRows / R, LDR = kRows + 4, LX = kP + 4, AP = 17;
    // per chunk of the step
    float As[2][32 * LDR];      // rotated columns: [column][rho], lo pairs then hi
    float Xs[2][kRows * LX];    // X or e^alpha dY: [rho][p]
    // per step parity and chunk: cos / sin of the in-chunk angle [token][pair],
    // the decay prefix, the token and per-token scales
    float acs[2][2][QT * AP], asn[2][2][QT * AP];
    float acum[2][2][QT], aclo[2][2][QT], ww[2][2][QT], scal[2][2][QT];
    float phi[2][16];           // the sequence's angle total per pair (reverse pass)
    float red[16];
};

template <typename T, int N, int R, bool FWD>
__device__ void state_pass(const ScanLaunch &a, const BwdArgs &g, const BwdWs &w, int nck,
                           size_t blk, PassSmem<R> &sm) {
    using S = PassSmem<R>;
    constexpr int NTN = N / 16, HT = NTN / 2, NH = N / 2, QT = S::QT, LDR = S::LDR, LX = S::LX, AP = S::AP;
    constexpr int PN = 4;                       // pairs a half-wave scans
    constexpr int JX = 2;                       // four-element items of X (dY) per thread and chunk
    const int tid = threadIdx.x, lane = tid & 63;
    const int pt = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, gq = lane >> 4;
    const int i1 = static_cast<int>(blk % HT);
    const size_t bh = blk / HT;
    const size_t H = a.heads, L = a.seq;
    const size_t bb = bh / H, hh = bh % H;
    const bool rot = a.theta != nullptr;
    const float A = 0.0f - expf(a.a_log[hh]);
    const int p0 = 16 * pt + 4 * gq, nlo = 16 * i1 + c;
    const size_t sbase = bh * kP * N + static_cast<size_t>(p0) * N + nlo;   // state (p0, nlo)
    const int tl = lane & 31, hl = lane >> 5;   // the scans: lane -> token tl of the step's chunk hl
    const int ip = PN * pt;                     // and pairs ip ..
    auto rot4 = [](f32x4 &lo, f32x4 &hi, float cs, float sn) {
        const f32x4 l = lo;
        lo = l * cs - hi * sn;
        hi = l * sn + hi * cs;
    };
    auto ld_state = [&](const float *p, f32x4 &lo, f32x4 &hi) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            lo[r] = p[sbase + r * N];
            hi[r] = p[sbase + r * N + NH];
        }
    };
    auto st_state = [&](float *p, f32x4 lo, f32x4 hi) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[sbase + r * N] = lo[r];
            p[sbase + r * N + NH] = hi[r];
        }
    };

    // Steps of two chunks: half the barriers, and the chains of one chunk
    // (scan, sine, products) beside the other's.  A second chunk past the
    // sequence's end is all zeros: decay one, no angle, nothing added.
    const int ns = (nck + 1) / 2;
    struct In {
        float dt, lam, dtn, lamn, dtl;
        uint32_t th[PN];
        Raw4<T> b1, b2, x[2 * JX];
    };
    // Step s's raw inputs, by buffer loads over this sequence's tokens: a
    // token at or past the sequence end reads as zero.  A thread's items sit
    // at fixed byte offsets from its step-0 offsets.
    constexpr uint32_t SZ = sizeof(T);
    const scan::SeqBufs rs = scan::seq_bufs<T, N, kP, R>(a, bb, hh);
    const rsrc_t rbc = FWD ? rs.b : rs.c;
    const rsrc_t rxy = FWD ? rs.x
                           : make_rsrc(static_cast<const char *>(g.dy) + (bb * L * H + hh) * kP * R * SZ,
                                       static_cast<uint32_t>((L * H - hh) * kP * R * SZ));
    const bool xal = FWD || (reinterpret_cast<uintptr_t>(g.dy) & 3u) == 0;
    const int tk = hl * QT + (tl < QT ? tl : 0);                 // this lane's token of the step
    const uint32_t o_s = tk * rs.tok_s;
    const uint32_t o_th = tk * rs.tok_th + (16 * i1 + ip) * SZ;
    // B (C) items: 128 a chunk, one a thread; X (dY): 512 a chunk
    const int tb = tid / (4 * R) % QT, sb_ = tid >> 7, eb = (tid % (4 * R)) * 4;
    const uint32_t o_bc = (sb_ * QT + tb) * rs.tok_bc + (16 * i1 * R + eb) * SZ;
    const int tx = tid / (16 * R), ex = (tid % (16 * R)) * 4;    // item tid + 256 j: token tx + j XJ
    constexpr int XJ = 256 / (16 * R);
    const uint32_t o_xy = tx * rs.tok_x + ex * SZ;
    auto load = [&](int st, In &d) {
        const int ss = st < 0 ? 0 : (st < ns ? st : ns - 1);   // outside: re-read, unused
        const uint32_t t0 = static_cast<uint32_t>(ss) * (2 * QT);
        d.dtl = bldf(rs.s0, o_s + t0 * rs.tok_s);
        if (pt == 0) {
            d.lam = bldf(rs.s1, o_s + t0 * rs.tok_s);
            d.dtn = bldf(rs.s0, o_s + (t0 + 1) * rs.tok_s);
            d.lamn = bldf(rs.s1, o_s + (t0 + 1) * rs.tok_s);
        }
        if (rot) ldth<T, PN>(rs.th, o_th + t0 * rs.tok_th, d.th);
        ld4(d.b1, rbc, o_bc + t0 * rs.tok_bc);
        ld4(d.b2, rbc, o_bc + t0 * rs.tok_bc + NH * R * SZ);
#pragma unroll
        for (int j = 0; j < 2 * JX; ++j) ld4(d.x[j], rxy, o_xy + (t0 + j * XJ) * rs.tok_x, xal);
    };
    // The step's work in four pieces, software-pipelined over two sets of the
    // per-step tables (sb = step parity): the scalars and decay prefixes (p1)
    // and the angles (p2) of the next step run in the same two barrier phases
    // as the staging (p3) and the products (p4) of this one.
    //   phase X: p3(s), p1(s + 1);  barrier;  phase Y: p4(s), p2(s + 1);  barrier
    // token scalars, the decay prefix (fused.rs:2494-2498)
    auto p1 = [&](const In &d, int sb) {
        if (pt == 0) {
            const float dt = tl < QT ? d.dtl : 0.0f;
            float hi, lo;
            split_decay(dt, A, hi, lo);
            hi = seg_scan<32>(hi);
            lo = seg_scan<32>(lo);
            if (tl < QT) {
                sm.ww[sb][hl][tl] = d.lam * dt + (1.0f - d.lamn) * d.dtn;
                sm.acum[sb][hl][tl] = hi;
                sm.aclo[sb][hl][tl] = lo;
            }
        }
    };
    // the in-chunk angle of this workgroup's pairs and its cos / sin; per
    // token wbar (B~'s scale) or e^alpha (dY's)
    auto p2 = [&](const In &d, int sb) {
        if (rot) {
            float v[PN];
            unth<T, PN>(d.th, v);
#pragma unroll
            for (int j = 0; j < PN; ++j) v[j] = tl < QT ? d.dtl * v[j] : 0.0f;
            scan32<PN>(v);
            if (tl < QT) {
#pragma unroll
                for (int j = 0; j < PN; ++j) {
                    float sv, cv;
                    sincos_turn(v[j], sv, cv);
                    sm.acs[sb][hl][tl * AP + ip + j] = cv;
                    sm.asn[sb][hl][tl * AP + ip + j] = sv;
                }
            }
        }
        if (pt == 0 && tl < QT) {
            const float hi = sm.acum[sb][hl][tl], lo = sm.aclo[sb][hl][tl];
            sm.scal[sb][hl][tl] = FWD ? clamp_exp((sm.acum[sb][hl][QT - 1] - hi) + (sm.aclo[sb][hl][QT - 1] - lo)) *
                                            sm.ww[sb][hl][tl]
                                      : clamp_exp(hi + lo);
        }
    };
    // rotation by the negative in-chunk angle (fused.rs:610-617) into LDS;
    // the chunks' decays
    auto p3 = [&](const In &d, int sb, float (&e)[2]) {
        {
            float b1[4], b2[4];
            un4(d.b1, b1);
            un4(d.b2, b2);
            const float sc = FWD ? sm.scal[sb][sb_][tb] : 1.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = (eb + j) / R, rho = tb * R + (eb + j) % R;
                float sn = 0.0f, cs = 1.0f;
                if (rot) {
                    cs = sm.acs[sb][sb_][tb * AP + q];
                    sn = sm.asn[sb][sb_][tb * AP + q];
                }
                sm.As[sb_][q * LDR + rho] = (b1[j] * cs + b2[j] * sn) * sc;
                sm.As[sb_][(16 + q) * LDR + rho] = (-b1[j] * sn + b2[j] * cs) * sc;
            }
        }
#pragma unroll
        for (int j = 0; j < 2 * JX; ++j) {
            const int u = j / JX, t = tx + (j % JX) * XJ;
            float v[4];
            un4(d.x[j], v);
            if constexpr (!FWD) {
                const float sc = sm.scal[sb][u][t];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] *= sc;
            }
            put4<R>(sm.Xs[u], LX, t, ex, v);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) e[u] = clamp_exp(sm.acum[sb][u][QT - 1] + sm.aclo[sb][u][QT - 1]);
    };
    // U (V) of the two chunks at this lane's (p, n): A(m = p, k = rho), B(k =
    // rho, col = n), with k slot 4 g + r of a block of 16 the rho of MFMA r's
    // lane group g; the rotations by the chunks' angle totals, the in-chunk
    // angles of their last rows
    auto p4 = [&](int sb, f32x4 (&alo)[2], f32x4 (&ahi)[2], float (&pc)[2], float (&ps)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) alo[u] = ahi[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < kRows / 16; ++kb) {
            f32x4 bl[2], bhv[2];
            float av[2][4];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bl[u] = *reinterpret_cast<const f32x4 *>(sm.As[u] + c * LDR + 16 * kb + 4 * gq);
                bhv[u] = *reinterpret_cast<const f32x4 *>(sm.As[u] + (16 + c) * LDR + 16 * kb + 4 * gq);
#pragma unroll
                for (int r = 0; r < 4; ++r) av[u][r] = sm.Xs[u][(16 * kb + 4 * gq + r) * LX + 16 * pt + c];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    alo[u] = mfma_f32(av[u][r], bl[u][r], alo[u]);
                    ahi[u] = mfma_f32(av[u][r], bhv[u][r], ahi[u]);
                }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            pc[u] = rot ? sm.acs[sb][u][(QT - 1) * AP + c] : 1.0f;
            ps[u] = rot ? sm.asn[sb][u][(QT - 1) * AP + c] : 0.0f;
        }
    };
    const uint32_t nw = static_cast<uint32_t>(min(w.wn, nck - w.k0));   // chunks in the window
    auto put_record = [&](float *base, int k, f32x4 lo, f32x4 hi) {
        const uint32_t kw = static_cast<uint32_t>(k - w.k0);
        if (kw >= nw) return;
        float *o = base + (bh * w.wn + kw) * kP * N + ((pt * NTN + i1) * 64 + lane) * 4;
        *reinterpret_cast<f32x4 *>(o) = lo;
        *reinterpret_cast<f32x4 *>(o + HT * 256) = hi;
    };

    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    In d[2];
    if constexpr (FWD) {
        if (a.h0 != nullptr) {
            ld_state(a.h0, lo, hi);
            if (a.last_u0 != nullptr) {
                const size_t i0 = (bb * L) * H + hh;
                const float first = (1.0f - a.lambda[i0]) * a.dt[i0];
                f32x4 ul, uh;
                ld_state(a.last_u0, ul, uh);
                lo += ul * first;
                hi += uh * first;
            }
        }
        if (rot && a.angle0 != nullptr) {
            float sn, cs;
            sincosf(a.angle0[bh * NH + nlo], &sn, &cs);
            rot4(lo, hi, cs, sn);
        }
        load(0, d[0]);
        load(1, d[1]);
        p1(d[0], 0);
        __syncthreads();
        p2(d[0], 0);
        __syncthreads();
        for (int k = 0; k < ns; k += 2) {
#pragma unroll
            for (int sb = 0; sb < 2; ++sb) {
                const int st = k + sb;
                if (st < ns) {
                    float e[2], pc[2], ps[2];
                    p3(d[sb], sb, e);
                    p1(d[sb ^ 1], sb ^ 1);
                    load(st + 2, d[sb]);
                    __syncthreads();
                    f32x4 ulo[2], uhi[2];
                    p4(sb, ulo, uhi, pc, ps);
                    p2(d[sb ^ 1], sb ^ 1);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        put_record(w.s, 2 * st + u, lo, hi);
                        lo = lo * e[u] + ulo[u];
                        hi = hi * e[u] + uhi[u];
                        if (rot && 2 * st + u < nck) rot4(lo, hi, pc[u], ps[u]);   // R(Phi_k)
                        const uint32_t kw = static_cast<uint32_t>(2 * st + u - w.k0);
                        if (i1 == 0 && tid == 0 && kw < nw) w.eda[bh * w.wn + kw] = e[u];
                    }
                    __syncthreads();
                }
            }
        }
    } else {
        if (g.dh_out != nullptr) {
            ld_state(g.dh_out, lo, hi);
            if (rot) {
                // phi_end = angle0 + sum_k Phi_k: the final frame, S_C = R(phi_end) h_out.
                // Each Phi_k is the in-chunk scan's last value; a half-wave sums
                // every second chunk.
                constexpr int DT = 4;
                float ph[PN], dq[DT];
                uint32_t tq[DT][PN];
#pragma unroll
                for (int j = 0; j < PN; ++j) ph[j] = 0.0f;
                auto tload = [&](int st, float &dv, uint32_t (&tv)[PN]) {
                    const uint32_t t0 = static_cast<uint32_t>(st < ns ? st : ns - 1) * (2 * QT);
                    dv = bldf(rs.s0, o_s + t0 * rs.tok_s);
                    ldth<T, PN>(rs.th, o_th + t0 * rs.tok_th, tv);
                };
#pragma unroll
                for (int q = 0; q < DT; ++q) tload(q, dq[q], tq[q]);
                for (int k = 0; k < ns; k += DT) {
#pragma unroll
                    for (int q = 0; q < DT; ++q) {
                        if (k + q < ns) {
                            float v[PN];
                            unth<T, PN>(tq[q], v);
#pragma unroll
                            for (int j = 0; j < PN; ++j) v[j] = tl < QT ? dq[q] * v[j] : 0.0f;
                            scan32<PN>(v);
#pragma unroll
                            for (int j = 0; j < PN; ++j) ph[j] += v[j];
                        }
                        tload(k + DT + q, dq[q], tq[q]);
                    }
                }
                if (tl == QT - 1) {
#pragma unroll
                    for (int j = 0; j < PN; ++j) sm.phi[hl][ip + j] = ph[j];
                }
                __syncthreads();
                const float pe = (a.angle0 != nullptr ? a.angle0[bh * NH + nlo] : 0.0f) + sm.phi[0][c] + sm.phi[1][c];
                float sn, cs;
                sincosf(pe, &sn, &cs);
                rot4(lo, hi, cs, sn);
            }
        }
        const int top = (ns - 1) | 1;   // the odd step of the last two; past the end if ns is odd
        load(top < ns ? top : top - 2, d[1]);
        load(top - 1, d[0]);
        if (top < ns) p1(d[1], 1); else p1(d[0], 0);
        __syncthreads();
        if (top < ns) p2(d[1], 1); else p2(d[0], 0);
        __syncthreads();
        for (int k = top; k >= 0; k -= 2) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int sb = 1 - q, st = k - q;
                if (st < ns) {
                    float e[2], pc[2], ps[2];
                    p3(d[sb], sb, e);
                    p1(d[sb ^ 1], sb ^ 1);
                    load(st - 2, d[sb]);
                    __syncthreads();
                    f32x4 vlo[2], vhi[2];
                    p4(sb, vlo, vhi, pc, ps);
                    p2(d[sb ^ 1], sb ^ 1);
#pragma unroll
                    for (int u = 1; u >= 0; --u) {
                        if (rot && 2 * st + u < nck) rot4(lo, hi, pc[u], -ps[u]);   // R(-Phi_k)
                        put_record(w.gh, 2 * st + u, lo, hi);
                        lo = lo * e[u] + vlo[u];
                        hi = hi * e[u] + vhi[u];
                    }
                    __syncthreads();
                }
            }
        }
        // into the global frame: dZ0 = R(-angle0) G_0
        if (rot && a.angle0 != nullptr) {
            float sn, cs;
            sincosf(a.angle0[bh * NH + nlo], &sn, &cs);
            rot4(lo, hi, cs, -sn);
        }
        float dfirst = 0.0f;
        if (a.h0 != nullptr && w.k0 + w.wn >= nck) {   // (the last window: every read of dh is done)
            if (g.dh0 != nullptr) st_state(g.dh0, lo, hi);
            if (a.last_u0 != nullptr) {
                const size_t i0 = (bb * L) * H + hh;
                const float first = (1.0f - a.lambda[i0]) * a.dt[i0];
                f32x4 ul, uh;
                ld_state(a.last_u0, ul, uh);
                for (int r = 0; r < 4; ++r) dfirst += lo[r] * ul[r] + hi[r] * uh[r];
                if (g.dlast_u0 != nullptr) st_state(g.dlast_u0, lo * first, hi * first);
            }
        }
        dfirst = block_sum(dfirst, sm.red);
        if (tid == 0) w.pfirst[blk] = dfirst;   // of the last window in the end
    }
}

// Both sequential passes in one launch (they are independent): workgroups
// [0, nb) run the forward recurrence, [nb, 2 nb) the reverse one.
template <typename T, int N, int R>
__global__ void __launch_bounds__(256) bwd_passes_kernel(ScanLaunch a, BwdArgs g, BwdWs w, int nck) {
    __shared__ __attribute__((aligned(16))) PassSmem<R> sm;
    const size_t nb = a.batch * a.heads * (N / 32);
    if (blockIdx.x < nb)
        state_pass<T, N, R, true>(a, g, w, nck, blockIdx.x, sm);
    else
        state_pass<T, N, R, false>(a, g, w, nck, blockIdx.x - nb, sm);
}

// ---------------------------------------------------------------- chunk gradients
// One workgroup of eight waves per chunk, two to a CU (80 KB of LDS and 128
// VGPRs each): a chunk is a chain of six barriers, so one workgroup leaves
// every unit idle most of the time, and the other fills in.  Measured at batch 8
// x 2048, 12 heads, d_state 128, bf16 storage: sixteen waves with everything in
// 158 KB of LDS, one to a CU, operands read by words, 445 us (MFMA busy 23 % of
// the time, LDS 44 %); this form 297 us, against some 140 us for its 700 MB at
// the rate of a large copy and 106 us of f32 MFMA.  What keeps it in 80 KB: the state S entering the chunk and Gh never go through LDS.  Their
// records' lane layout (column n = 16 i + c, p = 16 pt + 4 g + r) is the MFMA
// operand of the dC~ and dB~ products as it stands (k = p, 16 bytes a lane);
// the Gh B~^T product reads Gh's record by words.  Operand rows in LDS are read
// 16 bytes a lane, k slot 4 g + r of a block of 16 being lane group g's of MFMA
// r, and read transposed in the same order, whose four lane groups then sit 4
// rows apart, on banks of their own.
template <int N, int R>
struct Smem {
    static constexpr int QT = kRows / R, NH = N / 2, NTN = N / 16, PT = NTN / 2;
    static constexpr int LB = N + 12;       // B~, C~ rows
    static constexpr int LX = kP + 4;       // X, dY rows
    static constexpr int LM = kRows + 4;    // M, dCB rows
    static constexpr int AP = NH + 1;
    float Bs[kRows * LB], Cs[kRows * LB];
    float Xs[kRows * LX], Ys[kRows * LX];   // Xs: the band's column sums once X has been used
    float Ms[kRows * LM], Ds[kRows * LM];
    // per token and pair: cos and sin of the in-chunk angle; once every reader
    // holds its values, the two halves of the angle sums
    float acs[QT * AP], asn[QT * AP];
    float acum[QT], aclo[QT], gw[QT], ww[QT], eac[QT], ebar[QT], wbar[QT];
    float rin[kRows], dgr[kRows];
    float rcr[PT][kRows], qv[PT][kRows];    // per pair tile: rows' S and Gh sums
    float red[3][kWaves];
};

template <typename T, int N, int R>
__global__ void __launch_bounds__(kBT, 4) bwd_chunk_kernel(ScanLaunch a, BwdArgs g, BwdWs w, int nck) {
    using S = Smem<N, R>;
    constexpr int QT = S::QT, NH = S::NH, NTN = S::NTN, PT = S::PT;
    constexpr int LB = S::LB, LX = S::LX, LM = S::LM, AP = S::AP;
    constexpr uint32_t SZ = sizeof(T);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    S &sm = *reinterpret_cast<S *>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, gq = lane >> 4;
    const size_t bhw = blockIdx.x;   // the record
    const int ck = w.k0 + static_cast<int>(bhw % w.wn);
    const size_t bh = bhw / w.wn;
    if (ck >= nck) return;           // the last window's end
    const size_t H = a.heads, L = a.seq;
    const size_t bb = bh / H, hh = bh % H;
    const bool rot = a.theta != nullptr;
    const float D = a.d_skip ? a.d_skip[hh] : 0.0f;
    const float A = 0.0f - expf(a.a_log[hh]);
    const uint32_t t0 = static_cast<uint32_t>(ck) * QT;

    // ---- loads, all in flight together: tokens past the end read as zeros
    const scan::SeqBufs rs = scan::seq_bufs<T, N, kP, R>(a, bb, hh);
    const rsrc_t rdy = make_rsrc(static_cast<const char *>(g.dy) + (bb * L * H + hh) * kP * R * SZ,
                                 static_cast<uint32_t>((L * H - hh) * kP * R * SZ));
    const bool yal = (reinterpret_cast<uintptr_t>(g.dy) & 3u) == 0;
    // the angle scans: lane -> token tl, pairs i0 ..
    constexpr int PN = NH / 16;
    const int tl = lane & 31, hl = lane >> 5;
    const int i0 = (NH / kWaves) * wave + PN * hl;
    float dtl = 0.0f;
    uint32_t thq[PN];
    if (rot) {
        const uint32_t t = t0 + (tl < QT ? tl : 0);
        dtl = bldf(rs.s0, t * rs.tok_s);
        ldth<T, PN>(rs.th, t * rs.tok_th + i0 * SZ, thq);
    }
    float dt = 0.0f, lam = 0.0f, dtn = 0.0f, lamn = 0.0f;
    if (tid < QT) {
        dt = bldf(rs.s0, (t0 + tid) * rs.tok_s);
        lam = bldf(rs.s1, (t0 + tid) * rs.tok_s);
        dtn = bldf(rs.s0, (t0 + tid + 1) * rs.tok_s);
        lamn = bldf(rs.s1, (t0 + tid + 1) * rs.tok_s);
    }
    // four elements of each half row of B and C, of a row of X and dY
    constexpr int IB = NH * R / 4, IX = kP * R / 4;   // items per token
    static_assert(QT * IX == kBT && QT * IB <= kBT, "one item a thread");
    const bool has_b = tid < QT * IB;
    const int tb = tid / IB, eb = (tid % IB) * 4, tx = tid / IX, ex = (tid % IX) * 4;
    Raw4<T> b1, b2, c1, c2, xq, yq;
    ld4(xq, rs.x, (t0 + tx) * rs.tok_x + ex * SZ);
    ld4(yq, rdy, (t0 + tx) * rs.tok_x + ex * SZ, yal);
    if (has_b) {
        const uint32_t o = (t0 + tb) * rs.tok_bc + eb * SZ;
        ld4(b1, rs.b, o);
        ld4(b2, rs.b, o + NH * R * SZ);
        ld4(c1, rs.c, o);
        ld4(c2, rs.c, o + NH * R * SZ);
    }
    // The wave's dC~ (waves 0-3) or dB~ job: pair tile ji, JR row tiles from rt0
    // on; S or Gh of its columns
    constexpr int JR = PT == 4 ? 2 : 1;
    static_assert(2 * PT * (2 / JR) == kWaves, "one job a wave");
    const bool isb = wave >= kWaves / 2;
    const int ji = wave % PT, rt0 = PT == 4 ? 0 : (wave / PT) & 1;
    const size_t rec = bhw * kP * N;
    const float eda = w.eda[bhw];
    f32x4 fl[4], fh[4];
    {
        const f32x4 *r4 = reinterpret_cast<const f32x4 *>((isb ? w.gh : w.s) + rec) + lane;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fl[q] = r4[(q * NTN + ji) * 64];
            fh[q] = r4[(q * NTN + ji + PT) * 64];
        }
    }

    // ---- per-token scalars, the decay prefix, the in-chunk angles (inclusive
    // cumsums of dt theta) and their cos / sin; X and dY
    if (tid < QT) {
        sm.gw[tid] = lam * dt;                          // fused.rs:2494
        sm.ww[tid] = lam * dt + (1.0f - lamn) * dtn;    // fused.rs:2496-2498
    }
    if (wave == 0) {
        float hi, lo;
        split_decay(dt, A, hi, lo);
        hi = seg_scan<32>(hi);
        lo = seg_scan<32>(lo);
        if (lane < QT) {
            sm.acum[lane] = hi;
            sm.aclo[lane] = lo;
        }
    }
    if (rot) {
        float v[PN];
        unth<T, PN>(thq, v);
#pragma unroll
        for (int j = 0; j < PN; ++j) v[j] = tl < QT ? dtl * v[j] : 0.0f;
        scan32<PN>(v);
        if (tl < QT) {
#pragma unroll
            for (int j = 0; j < PN; ++j) {
                float sv, cv;
                sincos_turn(v[j], sv, cv);
                sm.acs[tl * AP + i0 + j] = cv;
                sm.asn[tl * AP + i0 + j] = sv;
            }
        }
    }
    float dsum = 0.0f, gsum = 0.0f, asum = 0.0f;
    {
        float xv[4], yv[4];
        un4(xq, xv);
        un4(yq, yv);
#pragma unroll
        for (int j = 0; j < 4; ++j) dsum = __builtin_fmaf(xv[j], yv[j], dsum);
        put4<R>(sm.Xs, LX, tx, ex, xv);
        put4<R>(sm.Ys, LX, tx, ex, yv);
    }
    __syncthreads();
    if (tid < QT) {
        const float hi = sm.acum[tid], lo = sm.aclo[tid];
        sm.eac[tid] = clamp_exp(hi + lo);
        sm.ebar[tid] = clamp_exp((sm.acum[QT - 1] - hi) + (sm.aclo[QT - 1] - lo));
        sm.wbar[tid] = sm.ebar[tid] * sm.ww[tid];
    }
    // rotation by the negative in-chunk angle (fused.rs:610-617) into LDS
    if (has_b) {
        float u1[4], u2[4], v1[4], v2[4], cs[4], sn[4];
        un4(b1, u1);
        un4(b2, u2);
        un4(c1, v1);
        un4(c2, v2);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cs[j] = rot ? sm.acs[tb * AP + (eb + j) / R] : 1.0f;
            sn[j] = rot ? sm.asn[tb * AP + (eb + j) / R] : 0.0f;
        }
        float lo[4], hi[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo[j] = u1[j] * cs[j] + u2[j] * sn[j];
            hi[j] = -u1[j] * sn[j] + u2[j] * cs[j];
        }
        put4<R>(sm.Bs, LB, tb, eb, lo);
        put4<R>(sm.Bs + NH, LB, tb, eb, hi);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo[j] = v1[j] * cs[j] + v2[j] * sn[j];
            hi[j] = -v1[j] * sn[j] + v2[j] * cs[j];
        }
        put4<R>(sm.Cs, LB, tb, eb, lo);
        put4<R>(sm.Cs + NH, LB, tb, eb, hi);
    }
    __syncthreads();

    // Three phases.  Phase 1 is everything that does not need the band: the
    // band products themselves, the Gh B~^T half of dX, the S dY / Gh X half of
    // each dC~ / dB~ job with its row sums, and the jobs' sines.  Phase 2 is
    // the band, elementwise.  Phase 3 finishes dX and the jobs with M and dCB.

    // ---- phase 1a: dX^T[p][s] = sum_n Gh[p][n] B~[s][n] (x wbar_s, + phase 3),
    // one 16 x 16 tile a wave: A(p = c, k): word c & 3 of the record's lane of
    // (n, p >> 2), the four lane groups at n = 16 i + 4 j + g
    const int xpt = wave & 3, xst = wave >> 2;
    f32x4 xacc = {0.f, 0.f, 0.f, 0.f};
    {
        const float *gr = w.gh + rec + (xpt * NTN * 64 + gq + 16 * (c >> 2)) * 4 + (c & 3);
        const float *br = sm.Bs + (16 * xst + c) * LB + gq;
        constexpr int HB = NTN / 2;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float av[HB][4];
#pragma unroll
            for (int i = 0; i < HB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) av[i][j] = gr[((half * HB + i) * 64 + 4 * j) * 4];
#pragma unroll
            for (int i = 0; i < HB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    xacc = mfma_f32(av[i][j], br[16 * (half * HB + i) + 4 * j], xacc);
        }
    }
    // ---- phase 1b: dC~ and dB~ as [n][row] tiles
    f32x4 lo[JR], hi[JR];
    float cs[JR][4], sn[JR][4];
    const int n0 = 16 * ji + 4 * gq;
    // the job's own rotated operand (C~ for dC~, B~ for dB~) at its elements
    const float *own = isb ? sm.Bs : sm.Cs;
    {
        const float *xr = isb ? sm.Xs : sm.Ys;
#pragma unroll
        for (int jr = 0; jr < JR; ++jr) {
            lo[jr] = f32x4{0.f, 0.f, 0.f, 0.f};
            hi[jr] = lo[jr];
        }
        // dC~^T[n][t] = e^{alpha_t} sum_p S[p][n] dY[t][p], dB~^T[n][s] = wbar_s
        // sum_p Gh[p][n] X[s][p] (+ phase 3)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int jr = 0; jr < JR; ++jr) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(xr + (16 * (rt0 + jr) + c) * LX + 16 * q + 4 * gq);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    lo[jr] = mfma_f32(fl[q][r], v[r], lo[jr]);
                    hi[jr] = mfma_f32(fh[q][r], v[r], hi[jr]);
                }
            }
        if (!isb && rt0 == 0) {
            // <Gh, S> over the job's columns
            const f32x4 *r4 = reinterpret_cast<const f32x4 *>(w.gh + rec) + lane;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 ga = r4[(q * NTN + ji) * 64], gb = r4[(q * NTN + ji + PT) * 64];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    gsum = __builtin_fmaf(ga[r], fl[q][r], gsum);
                    gsum = __builtin_fmaf(gb[r], fh[q][r], gsum);
                }
            }
        }
#pragma unroll
        for (int jr = 0; jr < JR; ++jr) {
            const int row = 16 * (rt0 + jr) + c, tr = row / R;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                cs[jr][r] = rot ? sm.acs[tr * AP + n0 + r] : 1.0f;
                sn[jr][r] = rot ? sm.asn[tr * AP + n0 + r] : 0.0f;
            }
            if (!isb) {
                const float ea = sm.eac[tr];
                lo[jr] = lo[jr] * ea;
                hi[jr] = hi[jr] * ea;
            }
            // row . (S or Gh part): the e^alpha dy.(S C~) and x.(Gh B~) terms
            const f32x4 o1 = *reinterpret_cast<const f32x4 *>(own + row * LB + n0);
            const f32x4 o2 = *reinterpret_cast<const f32x4 *>(own + row * LB + n0 + NH);
            float q = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) q += lo[jr][r] * o1[r] + hi[jr][r] * o2[r];
            q += __shfl_xor(q, 16, 64);
            q += __shfl_xor(q, 32, 64);
            if (gq == 0) (isb ? sm.qv : sm.rcr)[ji][row] = q;
            if (isb) {
                const float wb = sm.wbar[tr];
                lo[jr] = lo[jr] * wb;
                hi[jr] = hi[jr] * wb;
            }
        }
    }
    // ---- phase 1c: band products, raw: CB[t][s] = sum_n C~[t][n] B~[s][n]
    // into Ms and dM[t][s] = sum_p dY[t][p] X[s][p] into Ds, for the three
    // tiles on and below the diagonal (the tile above lies above the token
    // diagonal)
    if (wave < 6) {
        const int q = wave % 3, tj = q > 0, si = q > 1;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float *dst;
        if (wave < 3) {
#pragma unroll
            for (int kb = 0; kb < N / 16; ++kb)
                acc = scan::mma_kb(sm.Cs + (16 * tj + c) * LB + 16 * kb, sm.Bs + (16 * si + c) * LB + 16 * kb, acc, gq);
            dst = sm.Ms;
        } else {
#pragma unroll
            for (int kb = 0; kb < kP / 16; ++kb)
                acc = scan::mma_kb(sm.Ys + (16 * tj + c) * LX + 16 * kb, sm.Xs + (16 * si + c) * LX + 16 * kb, acc, gq);
            dst = sm.Ds;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(16 * tj + 4 * gq + r) * LM + 16 * si + c] = acc[r];
    }
    __syncthreads();

    // ---- phase 2: the band, elementwise (two (t, s) a thread, s fastest): K =
    // W e^{alpha_t - alpha_s}, M = CB o K, dCB = dM o K; the diagonal's dg
    // sums, and off it L = dM o M (row sums, column sums), the dw sums and the
    // sum of L (alpha_t - alpha_s).  Sums are stored, not added atomically, and
    // added in a fixed order: the gradients repeat bit for bit.
    float *const cpl = sm.Xs, *const cpw = sm.Xs + 2 * kWaves * kRows;   // [16][32] column sums
    {
        float cl = 0.0f, cw = 0.0f;
#pragma unroll
        for (int it = 0; it < kRows * kRows / kBT; ++it) {
            const int e = tid + it * kBT, t = e / kRows, s = e % kRows;
            const int tt = t / R, ts = s / R;
            float m = 0.0f, d = 0.0f, lm = 0.0f, dgd = 0.0f;
            if (tt >= ts) {
                const float cb = sm.Ms[t * LM + s], dm = sm.Ds[t * LM + s];
                const float step = (sm.acum[tt] - sm.acum[ts]) + (sm.aclo[tt] - sm.aclo[ts]);
                const float E = clamp_exp(step);
                const float K = (tt == ts ? sm.gw[ts] : sm.ww[ts]) * E;
                m = cb * K;
                d = dm * K;
                if (tt == ts) {
                    dgd = dm * cb;
                } else {
                    lm = dm * m;
                    cw += dm * cb * E;
                    asum = __builtin_fmaf(lm, step, asum);
                }
            }
            sm.Ms[t * LM + s] = m;
            sm.Ds[t * LM + s] = d;
            cl += lm;
            // row sums: a row is 32 consecutive lanes of a wave
            const float row = seg_scan<32>(lm);
            if ((lane & 31) == 31) sm.rin[t] = row;
            if constexpr (R >= 2) dgd += __shfl_xor(dgd, 1, 64);
            if constexpr (R >= 4) dgd += __shfl_xor(dgd, 2, 64);
            if (tt == ts && s % R == 0) sm.dgr[t] = dgd;
        }
        cpl[(2 * wave + hl) * kRows + tl] = cl;
        cpw[(2 * wave + hl) * kRows + tl] = cw;
    }
    __syncthreads();

    // ---- phase 3a: dX^T[p][s] += sum_t dY[t][p] M[t][s] + D dY[s][p]
    {
        const int s = 16 * xst + c, ts = s / R, rr = s % R;
        f32x4 acc = xacc * sm.wbar[ts];
#pragma unroll
        for (int kb = 0; kb < kRows / 16; ++kb) {
            float av[4], bv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = 16 * kb + 4 * gq + r;
                av[r] = sm.Ys[t * LX + 16 * xpt + c];
                bv[r] = sm.Ms[t * LM + s];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) acc = mfma_f32(av[r], bv[r], acc);
        }
        const size_t tg = t0 + ts;
        if (tg < L) {
            const size_t base = ((bb * L + tg) * H + hh) * kP * R;
            const int p0 = 16 * xpt + 4 * gq;
            const f32x4 yv = *reinterpret_cast<const f32x4 *>(sm.Ys + s * LX + p0);
            acc += yv * D;
            st4<T, R>(g.dx, base + p0 * R + rr, acc);
        }
    }
    // ---- phase 3b: the band halves of dC~ and dB~
    //   dC~^T[n][t] += sum_s B~[s][n] dCB[t][s],  dB~^T[n][s] += sum_t C~[t][n] dCB[t][s]
    // then the angle sums (every cos / sin was read in phase 1: asn receives
    // the dB~ half, acs the dC~ half, one lane per (token, pair)) and the
    // rotation back, d = R(psi) d~ (the transpose of fused.rs:610-617)
    {
        const float *ar = isb ? sm.Cs : sm.Bs;
#pragma unroll
        for (int kb = 0; kb < kRows / 16; ++kb) {
            float al[4], ah[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float *x = ar + (16 * kb + 4 * gq + r) * LB + 16 * ji + c;
                al[r] = x[0];
                ah[r] = x[NH];
            }
#pragma unroll
            for (int jr = 0; jr < JR; ++jr) {
                const int rt = 16 * (rt0 + jr) + c;
                f32x4 bv;
                if (isb) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) bv[r] = sm.Ds[(16 * kb + 4 * gq + r) * LM + rt];
                } else {
                    bv = *reinterpret_cast<const f32x4 *>(sm.Ds + rt * LM + 16 * kb + 4 * gq);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    lo[jr] = mfma_f32(al[r], bv[r], lo[jr]);
                    hi[jr] = mfma_f32(ah[r], bv[r], hi[jr]);
                }
            }
        }
#pragma unroll
        for (int jr = 0; jr < JR; ++jr) {
            const int row = 16 * (rt0 + jr) + c, tr = row / R, rr = row % R;
            if (rot) {
                float *half = isb ? sm.asn : sm.acs;
                const f32x4 o1 = *reinterpret_cast<const f32x4 *>(own + row * LB + n0);
                const f32x4 o2 = *reinterpret_cast<const f32x4 *>(own + row * LB + n0 + NH);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float cr = lo[jr][r] * o2[r] - hi[jr][r] * o1[r];
                    // the R rows of a token sit in adjacent lanes
                    if constexpr (R >= 2) cr += __shfl_xor(cr, 1, 64);
                    if constexpr (R >= 4) cr += __shfl_xor(cr, 2, 64);
                    if (rr == 0) half[tr * AP + n0 + r] = cr;
                }
            }
            f32x4 v1, v2;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v1[r] = lo[jr][r] * cs[jr][r] - hi[jr][r] * sn[jr][r];
                v2[r] = lo[jr][r] * sn[jr][r] + hi[jr][r] * cs[jr][r];
            }
            const size_t tg = t0 + tr;
            if (tg < L) {
                void *dst = isb ? g.db : g.dc;
                const size_t base = ((bb * L + tg) * H + hh) * N * R;
                st4<T, R>(dst, base + n0 * R + rr, v1);
                st4<T, R>(dst, base + (n0 + NH) * R + rr, v2);
            }
        }
    }
    // ---- <Gh, S>, the skip's sum dY . X and the band's share of da_log
    gsum = wave_sum(gsum);
    dsum = wave_sum(dsum);
    asum = wave_sum(asum);
    if (lane == 0) {
        sm.red[0][wave] = gsum;
        sm.red[1][wave] = dsum;
        sm.red[2][wave] = asum;
    }
    __syncthreads();

    // ---- in-chunk reverse cumsums of the angle sums, over lanes in reverse
    // token order (lane tl holds token QT - 1 - tl), four (two) pairs at once
    if (rot) {
        const int t = QT - 1 - tl;
        float v[PN];
#pragma unroll
        for (int j = 0; j < PN; ++j)
            v[j] = tl < QT ? sm.acs[t * AP + i0 + j] + sm.asn[t * AP + i0 + j] : 0.0f;
        scan32<PN>(v);
        const size_t tg = t0 + t;
        if (tl < QT && tg < L) {
            float *dst = w.cin + (bh * L + tg) * NH + i0;
            if constexpr (PN == 4)
                *reinterpret_cast<f32x4 *>(dst) = f32x4{v[0], v[1], v[2], v[3]};
            else
                *reinterpret_cast<f32x2 *>(dst) = f32x2{v[0], v[1]};
        }
        if (tl == QT - 1) {
#pragma unroll
            for (int j = 0; j < PN; ++j) w.ctot[(bh * nck + ck) * NH + i0 + j] = v[j];
        }
    }
    // ---- per-token scalars (lane = row, then the row's token at lane t R)
    if (wave == 0) {
        float gs = 0.0f, ds = 0.0f, pa = 0.0f;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) {
            gs += sm.red[0][q];
            ds += sm.red[1][q];
            pa += sm.red[2][q];
        }
        // lanes 0-31 the column sums of L, lanes 32-63 those of dw
        const float *cp = hl ? cpw : cpl;
        float col = 0.0f;
#pragma unroll
        for (int q = 0; q < 2 * kWaves; ++q) col += cp[q * kRows + tl];
        const float dwi = __shfl(col, tl + 32, 64);
        float rc = 0.0f, qv = 0.0f;
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            rc += sm.rcr[q][tl];
            qv += sm.qv[q][tl];
        }
        const int t = tl / R;   // both halves of the wave form the rows; the first keeps them
        const float wb = sm.wbar[t];
        // da_log's share (a = -e^{a_log} dt, so da_log = sum of a da): every
        // term weighs the decay it crossed, alpha_t for the carry-in, alpha_E -
        // alpha_s for the state, alpha_E for what passes through.  The sum of
        // dt da, whose cumsums cancel most of each row and column sum, was off
        // by up to 1.3e-5.
        const float alt = sm.acum[t] + sm.aclo[t];
        const float ale = sm.acum[QT - 1] + sm.aclo[QT - 1];
        const float toe = (sm.acum[QT - 1] - sm.acum[t]) + (sm.aclo[QT - 1] - sm.aclo[t]);
        const float egs = eda * gs;
        pa += wave_sum(hl ? 0.0f : rc * alt + qv * wb * toe) + egs * ale;
        const float et = wave_sum(hl ? 0.0f : qv * wb);
        float d = sm.rin[tl] - col + rc - qv * wb;
        float dw = dwi + qv * sm.ebar[t], dg = sm.dgr[tl];
        if constexpr (R >= 2) {
            d += __shfl_xor(d, 1, 64);
            dw += __shfl_xor(dw, 1, 64);
            dg += __shfl_xor(dg, 1, 64);
        }
        if constexpr (R >= 4) {
            d += __shfl_xor(d, 2, 64);
            dw += __shfl_xor(dw, 2, 64);
            dg += __shfl_xor(dg, 2, 64);
        }
        // the alpha_E terms of the last token; da its reverse cumsum
        if (t == QT - 1) d += et + egs;
        const int rt = QT - 1 - tl;
        float da = __shfl(d, (rt < 0 ? 0 : rt) * R, 64);
        da = seg_scan<32>(tl < QT ? da : 0.0f);
        if (lane == 0) {
            if (w.k0 > 0) {
                ds += w.pd[bhw];
                pa += w.pa[bhw];
            }
            w.pd[bhw] = ds;
            w.pa[bhw] = pa;
        }
        if (lane < QT && t0 + rt < L) w.da[bh * L + t0 + rt] = da;
        if (lane < kRows && tl % R == 0 && t0 + t < L) {
            w.dg[bh * L + t0 + t] = dg;
            w.dw[bh * L + t0 + t] = dw;
        }
    }
}

// ---------------------------------------------------------------- angle sums of later chunks
template <int N>
__global__ void bwd_angle_kernel(ScanLaunch a, BwdArgs g, BwdWs w, int nck) {
    constexpr int NH = N / 2, D = 8;
    const size_t bh = blockIdx.x;
    const int i = threadIdx.x;
    if (i >= NH) return;
    float run = g.dangle_out ? g.dangle_out[bh * NH + i] : 0.0f;
    // eight chunk totals in flight ahead of the running sum, which takes their place
    for (int k0 = nck - 1; k0 >= 0; k0 -= D) {
        float v[D];
#pragma unroll
        for (int j = 0; j < D; ++j) v[j] = k0 - j >= 0 ? w.ctot[(bh * nck + k0 - j) * NH + i] : 0.0f;
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (k0 - j < 0) break;
            w.ctot[(bh * nck + k0 - j) * NH + i] = run;
            run += v[j];
        }
    }
    if (g.dangle0 != nullptr) g.dangle0[bh * NH + i] = run;
}

// ---------------------------------------------------------------- per token
// dtheta_t = dt_t dphi_t, ddt_t = theta_t . dphi_t + A da_t
//   + lambda_t (dg_t + dw_t) + (1 - lambda_t) dw_{t-1},
// dlambda_t = dt_t (dg_t + dw_t) - dt_t dw_{t-1}    (trapezoid_weights_backward,
// fused.rs:2513-2549), plus the carried-in boundary term at t = 0.
// One workgroup per chunk, one wave per token, lane = rotation pair.
template <typename T, int N, int R>
__global__ void __launch_bounds__(256) bwd_token_kernel(ScanLaunch a, BwdArgs g, BwdWs w, int nck) {
    constexpr int NH = N / 2, QT = kRows / R;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t bhk = blockIdx.x;
    const int ck = static_cast<int>(bhk % nck);
    const size_t bh = bhk / nck;
    const size_t H = a.heads, L = a.seq;
    const size_t bb = bh / H, hh = bh % H;
    const float A = 0.0f - expf(a.a_log[hh]);
    const bool rot = a.theta != nullptr;
    constexpr int TW = (QT + 3) / 4;   // tokens per wave: wave + 4 j
    static_assert(TW <= 64, "tokens per wave");
    // the per-token scalars of the second part (lane j = token wave + 4 j)
    // go out first: they depend on nothing below
    const int tk = wave + 4 * lane;
    const size_t tkg = static_cast<size_t>(ck) * QT + tk;
    const bool tk_live = lane < TW && tk < QT && tkg < L;
    const size_t tkc = tk_live ? tkg : 0;
    const size_t tkx = (bb * L + tkc) * H + hh;
    const float dt = a.dt[tkx], lam = a.lambda[tkx];
    const float da = w.da[bh * L + tkc];
    const float dgw = w.dg[bh * L + tkc] + w.dw[bh * L + tkc];
    const float dwv = w.dw[bh * L + (tkc > 0 ? tkc - 1 : 0)];
    // per pair (lane = pair): dtheta and the angle part of ddt, with every
    // load issued first (unconditional at clamped indices)
    float cin[TW], th[TW];
    const int pl = lane < NH ? lane : 0;
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        const int t = wave + 4 * j;
        const size_t tg = static_cast<size_t>(ck) * QT + t;
        const bool live = t < QT && tg < L && lane < NH;
        const size_t tc = live ? tg : 0;
        const size_t ix = (bb * L + tc) * H + hh;
        float u = 0.0f, v = 0.0f;
        if (rot) {
            u = w.cin[(bh * L + tc) * NH + pl];
            v = ldv<T>(a.theta, ix * NH + pl);
        }
        cin[j] = live ? u : 0.0f;
        th[j] = live ? v : 0.0f;
    }
    const float off = rot ? w.ctot[bhk * NH + pl] : 0.0f;   // the later chunks' sum
    float mine = 0.0f;   // lane j keeps token wave + 4 j's angle part
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        const int t = wave + 4 * j;
        const size_t tg = static_cast<size_t>(ck) * QT + t;
        float part = 0.0f;
        if (rot && t < QT && tg < L && lane < NH) {
            const size_t ix = (bb * L + tg) * H + hh;
            const float dphi = cin[j] + off;
            if (g.dtheta != nullptr) stv<T>(g.dtheta, ix * NH + lane, a.dt[ix] * dphi);
            part = th[j] * dphi;
        }
        part = group_sum(part, 64);
        if (lane == j) mine = part;
    }
    // per token (lane j = token wave + 4 j): trapezoid and decay chains
    const float dwp = tkc > 0 ? dwv : 0.0f;
    float ddt = mine + A * da + lam * dgw + (1.0f - lam) * dwp;
    float dlam = dt * dgw - dt * dwp;
    if (tk_live && tkg == 0 && a.h0 != nullptr && a.last_u0 != nullptr) {
        float dfirst = 0.0f;
        for (int q = 0; q < N / 32; ++q) dfirst += w.pfirst[bh * (N / 32) + q];
        ddt += (1.0f - lam) * dfirst;
        dlam -= dt * dfirst;
    }
    if (tk_live) {
        g.ddt[tkx] = ddt;
        g.dlambda[tkx] = dlam;
    }
}

// ---------------------------------------------------------------- per head
__global__ void __launch_bounds__(256) bwd_head_kernel(ScanLaunch a, BwdArgs g, BwdWs w) {
    __shared__ float red[16];
    const size_t hh = blockIdx.x;
    const size_t H = a.heads;
    float sa = 0.0f, sd = 0.0f;
    const size_t n = a.batch * static_cast<size_t>(w.wn);
    for (size_t j = threadIdx.x; j < n; j += blockDim.x) {
        const size_t bb = j / w.wn, k = j % w.wn;
        const size_t bhw = (bb * H + hh) * w.wn + k;
        sa += w.pa[bhw];
        sd += w.pd[bhw];
    }
    sa = block_sum(sa, red);
    sd = block_sum(sd, red + 8);
    if (threadIdx.x == 0) {
        g.da_log[hh] = g.add_sums ? g.da_log[hh] + sa : sa;
        if (g.dd_skip != nullptr) g.dd_skip[hh] = g.add_sums ? g.dd_skip[hh] + sd : sd;
    }
}

// ---------------------------------------------------------------- outgoing last_u
// last_u = sum_r x_{L-1,r} (R(-phi_{L-1}) B_{L-1,r})^T (scan.rs:599-618), so an
// upstream gradient G of it adds, at the last token,
//   dx[p][r]  += sum_n G[p][n] B~[n][r]
//   dB~[n][r]  = sum_p G[p][n] x[p][r],   dB = R(+phi) dB~
//   dphi_i    += sum_r dB~_1 B~_2 - dB~_2 B~_1   (d B~_1/dphi = B~_2, d B~_2/dphi = -B~_1)
// The angle term joins dL/dangle as the seed of the angle gradient's reverse
// cumsum (bwd_angle_kernel); the dx and db terms wait in the workspace for
// bwd_last_add_kernel.  One workgroup per (batch, head).
template <typename T, int N, int R>
__global__ void __launch_bounds__(256) bwd_last_u_kernel(ScanLaunch a, BwdArgs g, BwdWs w) {
    constexpr int NH = N / 2, P = kP;
    __shared__ float sphi[4][NH];
    __shared__ float sx[P * R];
    __shared__ float sb[N * R];      // B~ of the last token
    __shared__ float sdb[N * R];     // dB~
    const int tid = threadIdx.x;
    const size_t bh = blockIdx.x;
    const size_t H = a.heads, L = a.seq;
    const size_t bb = bh / H, hh = bh % H;
    const bool rot = a.theta != nullptr;
    const size_t tl = (bb * L + (L - 1)) * H + hh;   // (b, L-1, h)
    // phi_{L-1} = angle0 + sum_t dt_t theta_t, four token stripes per pair
    if (rot) {
        const int i = tid % NH, q = tid / NH;        // NH <= 64: q < 4 covers 256 threads
        float acc = 0.0f;
        if (i < NH && q < 4) {
            for (size_t t = q; t < L; t += 4) {
                const size_t row = (bb * L + t) * H + hh;
                acc += a.dt[row] * ldv<T>(a.theta, row * NH + i);
            }
            sphi[q][i] = acc;
        }
    }
    for (int e = tid; e < P * R; e += 256) sx[e] = ldv<T>(a.x, tl * P * R + e);
    __syncthreads();
    for (int i = tid; i < NH; i += 256) {
        float phi = 0.0f, cs = 1.0f, sn = 0.0f;
        if (rot) {
            phi = sphi[0][i] + sphi[1][i] + sphi[2][i] + sphi[3][i];
            if (a.angle0 != nullptr) phi += a.angle0[bh * NH + i];
            sincosf(wrap_angle(phi), &sn, &cs);
        }
        sphi[0][i] = cs;
        sphi[1][i] = sn;
        for (int r = 0; r < R; ++r) {
            const float b1 = ldv<T>(a.b, (tl * N + i) * R + r);
            const float b2 = ldv<T>(a.b, (tl * N + i + NH) * R + r);
            sb[i * R + r] = b1 * cs + b2 * sn;              // fused.rs:610-617
            sb[(i + NH) * R + r] = -b1 * sn + b2 * cs;
        }
    }
    __syncthreads();
    const float *G = g.dlast_u_out + bh * P * N;
    // dB~[n][r] = sum_p G[p][n] x[p][r]
    for (int e = tid; e < N * R; e += 256) {
        const int n = e / R, r = e % R;
        float acc = 0.0f;
        for (int p = 0; p < P; ++p) acc += G[p * N + n] * sx[p * R + r];
        sdb[e] = acc;
    }
    // dx[p][r] = sum_n G[p][n] B~[n][r]
    for (int e = tid; e < P * R; e += 256) {
        const int p = e / R, r = e % R;
        float acc = 0.0f;
        for (int n = 0; n < N; ++n) acc += G[p * N + n] * sb[n * R + r];
        w.lux[bh * P * R + e] = acc;
    }
    __syncthreads();
    for (int i = tid; i < NH; i += 256) {
        const float cs = sphi[0][i], sn = sphi[1][i];
        float dphi = 0.0f;
        for (int r = 0; r < R; ++r) {
            const float d1 = sdb[i * R + r], d2 = sdb[(i + NH) * R + r];
            dphi += d1 * sb[(i + NH) * R + r] - d2 * sb[i * R + r];
            w.lub[(bh * N + i) * R + r] = d1 * cs - d2 * sn;          // R(+phi) dB~
            w.lub[(bh * N + i + NH) * R + r] = d1 * sn + d2 * cs;
        }
        if (rot) w.seed[bh * NH + i] = (g.dangle_out ? g.dangle_out[bh * NH + i] : 0.0f) + dphi;
    }
}

// The last token's dx and db terms of the outgoing last_u, added to the
// gradients the main passes wrote (in their storage type).
template <typename T, int N, int R>
__global__ void __launch_bounds__(256) bwd_last_add_kernel(ScanLaunch a, BwdArgs g, BwdWs w) {
    constexpr int P = kP;
    const size_t bh = blockIdx.x;
    const size_t H = a.heads, L = a.seq;
    const size_t bb = bh / H, hh = bh % H;
    const size_t tl = (bb * L + (L - 1)) * H + hh;
    for (int e = threadIdx.x; e < P * R; e += 256)
        stv<T>(g.dx, tl * P * R + e, ldv<T>(g.dx, tl * P * R + e) + w.lux[bh * P * R + e]);
    for (int e = threadIdx.x; e < N * R; e += 256)
        stv<T>(g.db, tl * N * R + e, ldv<T>(g.db, tl * N * R + e) + w.lub[bh * N * R + e]);
}

template <typename K>
hipError_t set_lds(K kern, size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
}

hipError_t launched(int &launches) {
    ++launches;
    return hipGetLastError();
}

template <typename T, int N, int R>
hipError_t launch_bwd(const ScanLaunch &a, const BwdArgs &g, char *base, size_t bytes, hipStream_t s,
                      int &launches) {
    constexpr int QT = kRows / R;
    const int nck = static_cast<int>((a.seq + QT - 1) / QT);
    const size_t bh = a.batch * a.heads, bhk = bh * nck;
    BwdLayout l = bwd_layout(bh, nck, nck, a.seq, N, R);
    int wn = nck;
    if (l.total > bytes) {   // two windows (scan_backward_workspace_least)
        wn = (nck + 1) / 2;
        l = bwd_layout(bh, nck, wn, a.seq, N, R);
    }
    BwdWs w;
    auto f = [base](size_t off) { return reinterpret_cast<float *>(base + off); };
    w.s = f(l.s);
    w.gh = f(l.gh);
    w.eda = f(l.eda);
    w.cin = f(l.cin);
    w.ctot = f(l.ctot);
    w.da = f(l.da);
    w.dg = f(l.dg);
    w.dw = f(l.dw);
    w.pd = f(l.pd);
    w.pa = f(l.pa);
    w.pfirst = f(l.pfirst);
    w.seed = f(l.seed);
    w.lux = f(l.lux);
    w.lub = f(l.lub);
    w.k0 = 0;
    w.wn = wn;

    static_assert(sizeof(Smem<N, R>) <= 80 * 1024, "two chunk workgroups a CU");
    const size_t lds = sizeof(Smem<N, R>);
    static const hipError_t a2 = set_lds(bwd_chunk_kernel<T, N, R>, lds);
    if (a2 != hipSuccess) return a2;
    hipError_t e;
    BwdArgs gm = g;
    if (g.dlast_u_out != nullptr) {
        // the outgoing last_u's terms; its angle term seeds the angle passes
        hipLaunchKernelGGL((bwd_last_u_kernel<T, N, R>), dim3(bh), dim3(256), 0, s, a, g, w);
        if ((e = launched(launches)) != hipSuccess) return e;
        if (a.theta != nullptr) gm.dangle_out = w.seed;
    }
    const BwdArgs &g2 = gm;
    for (w.k0 = 0; w.k0 < nck; w.k0 += wn) {
        hipLaunchKernelGGL((bwd_passes_kernel<T, N, R>), dim3(2 * bh * (N / 32)), dim3(256), 0, s, a, g2, w,
                           nck);
        if ((e = launched(launches)) != hipSuccess) return e;
        hipLaunchKernelGGL((bwd_chunk_kernel<T, N, R>), dim3(bh * wn), dim3(kBT), lds, s, a, g2, w, nck);
        if ((e = launched(launches)) != hipSuccess) return e;
    }
    if (a.theta != nullptr) {
        hipLaunchKernelGGL((bwd_angle_kernel<N>), dim3(bh), dim3(64), 0, s, a, g2, w, nck);
        if ((e = launched(launches)) != hipSuccess) return e;
    }
    hipLaunchKernelGGL((bwd_token_kernel<T, N, R>), dim3(bhk), dim3(256), 0, s, a, g2, w, nck);
    if ((e = launched(launches)) != hipSuccess) return e;
    hipLaunchKernelGGL(bwd_head_kernel, dim3(a.heads), dim3(256), 0, s, a, g2, w);
    if ((e = launched(launches)) != hipSuccess) return e;
    if (g.dlast_u_out != nullptr) {
        hipLaunchKernelGGL((bwd_last_add_kernel<T, N, R>), dim3(bh), dim3(256), 0, s, a, g, w);
        if ((e = launched(launches)) != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename T>
hipError_t launch_bwd_t(const ScanLaunch &a, const BwdArgs &g, char *ws, size_t bytes, hipStream_t s,
                        int &launches) {
    const size_t n = a.d_state, r = a.rank;
    if (n == 128) {
        if (r == 1) return launch_bwd<T, 128, 1>(a, g, ws, bytes, s, launches);
        if (r == 2) return launch_bwd<T, 128, 2>(a, g, ws, bytes, s, launches);
        if (r == 4) return launch_bwd<T, 128, 4>(a, g, ws, bytes, s, launches);
    } else if (n == 64) {
        if (r == 1) return launch_bwd<T, 64, 1>(a, g, ws, bytes, s, launches);
        if (r == 2) return launch_bwd<T, 64, 2>(a, g, ws, bytes, s, launches);
        if (r == 4) return launch_bwd<T, 64, 4>(a, g, ws, bytes, s, launches);
    }
    return hipErrorNotSupported;
}

}  // namespace

bool scan_backward_supported(const ScanLaunch &a) {
    return a.mode_raw && a.seq > 0 && scan_fast_supported(a);
}

size_t scan_backward_workspace(const ScanLaunch &a) {
    if (!scan_backward_supported(a)) return 0;
    const size_t qt = kRows / a.rank;
    const size_t nck = (a.seq + qt - 1) / qt;
    return bwd_layout(a.batch * a.heads, nck, nck, a.seq, a.d_state, a.rank).total;
}

// bf16 storage at d_state 64 took 64-row chunks once, and half the records;
// their workspace still runs, in two windows.  Batch 12 x 1024, 24 heads, us:
// 64-row chunks 790 in 194 MB, 32-row ones 479 in 345 MB, in two windows 592 in
// 194; 2 x 512, 4 heads 73.5, 42.8 and 73.5.
size_t scan_backward_workspace_least(const ScanLaunch &a) {
    if (!scan_backward_supported(a)) return 0;
    const size_t qt = kRows / a.rank;
    const size_t nck = (a.seq + qt - 1) / qt, wn = a.bf16 && a.d_state == 64 ? (nck + 1) / 2 : nck;
    return bwd_layout(a.batch * a.heads, nck, wn, a.seq, a.d_state, a.rank).total;
}

hipError_t launch_scan_backward(const ScanLaunch &a, const ScanGrads &gr, void *workspace, size_t bytes,
                                hipStream_t stream, int &launches) {
    if (!scan_backward_supported(a) || bytes < scan_backward_workspace_least(a)) return hipErrorNotSupported;
    BwdArgs g;
    g.dy = gr.dy;
    g.dh_out = gr.dh_out;
    g.dangle_out = gr.dangle_out;
    g.dlast_u_out = gr.dlast_u_out;
    g.dx = gr.dx;
    g.db = gr.db;
    g.dc = gr.dc;
    g.ddt = gr.ddt;
    g.dlambda = gr.dlambda;
    g.da_log = gr.da_log;
    g.dtheta = gr.dtheta;
    g.dd_skip = gr.dd_skip;
    g.dh0 = gr.dh0;
    g.dlast_u0 = gr.dlast_u0;
    g.dangle0 = gr.dangle0;
    g.add_sums = gr.add_sums != 0;
    char *ws = static_cast<char *>(workspace);
    if (a.bf16) return launch_bwd_t<bf16_t>(a, g, ws, bytes, stream, launches);
    return launch_bwd_t<float>(a, g, ws, bytes, stream, launches);
}

}  // namespace m3
