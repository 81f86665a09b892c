// Linear::apply for a handful of rows (a decode step of one or a few
// sequences) on gfx950:
//   y[m, n] = (x[m, :] . w^T[n, :]) * scale[n] + res[m, n]
// bf16 x [M, K] and w^T [N, K], f32 accumulation, the per-column scale and the
// residual in the epilogue, bf16 y (nn/linear.rs:155-185).
//
// The product is a stream over the weights, each read once; what bounds a
// call of a few MB is how soon enough of it is in flight.  A workgroup owns 16
// NT columns of y and its WK waves split K: wave q takes the 64-k blocks q, q +
// WK, ..., each lane loading its weights and x straight into the registers the
// MFMA reads them from (row c, k = 16 g .. 16 g + 15 of the block: two 16-byte
// loads a tile, whole 128-byte lines a row; no LDS, no barrier on the way),
// two groups of U blocks in flight.  bf16 MFMA 16x16x32 forms y^T = W^T X^T,
// so one to sixteen rows cost the same; rows and columns past the end read as
// zeros.  The waves' partial sums meet in LDS, in wave order.
//
// Measured on MI355X (us per call, captured, weights from HBM, against the
// product's route before: hipBLASLt from 4096 columns on, skinny_gemm.hip
// below), K x N at 1 / 16 rows: 1536 x 10800 11.6 -> 8.4 / 13.5 -> 11.6 (33 MB,
// 4.0 TB/s); 1536 x 1536 7.1 -> 4.2 / 7.3 -> 5.3; 1536 x 32000 24.9 -> 18.4
// (5.3 TB/s) / 25.9 -> 22.1; 768 x 5400 6.1 -> 4.6 / 6.1 -> 5.3.  One row of 8 or
// 16 waves splitting K, or two column tiles a wave, were slower there (9.1,
// 10.3 and 10.0 at 1536 x 10800).
#include "m3_internal.hpp"
#include "scan_common.hpp"

namespace m3 {

namespace {

using namespace scan;

// NORM: x is RMS-normalised on the way (nn/norm.rs:95-105), x rsqrt(mean x^2 +
// eps) gain.  The operand is bf16(x gain); the row's factor, known only when
// all of K has been read, multiplies the sums in f32: as many roundings as the
// norm's own bf16 output has.  The waves form the operand's rows in LDS while
// the first weights are on their way.  Measured (us, a norm and a product
// against this, K x N at 1 / 4 rows): 1536 x 10800 11.2 -> 9.8 / 12.0 -> 10.7,
// 1536 x 32000 21.1 -> 20.3 / 22.4 -> 21.9, 768 x 5400 6.7 -> 5.0 / 7.1 -> 6.0.
// Past four rows forming them in every workgroup costs what the norm's launch
// does (8 rows 7.0 -> 7.5 at 768 x 5400).  Scaling the lanes' own x registers
// instead, sixteen lanes a row for one live row, took 15.2 us a call over a
// decode step's projections against 12.2.
constexpr uint32_t kNormRows = 4;
template <int MT, int NT, int WK, int U, bool NORM>
__global__ void __launch_bounds__(64 * WK)
few_rows_kernel(uint32_t M, uint32_t K, uint32_t N, const void *x, const float *gain, float eps,
                const void *w, const float *scale, const void *res, void *y) {
    static_assert(!NORM || MT == 1, "the normed rows are one tile's");
    extern __shared__ __attribute__((aligned(16))) unsigned char xs[];   // NORM: [M][2 K + 16]
    __shared__ __attribute__((aligned(16))) f32x4 part[WK][NT * MT][64];
    __shared__ float squares[NORM ? WK : 1][kNormRows];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const uint32_t n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * (16 * MT);
    const rsrc_t rx = make_rsrc(x, M * K * 2u), rw = make_rsrc(w, N * K * 2u);
    const int nb = static_cast<int>(K / 64);
    const uint32_t pitch = 2 * K + 16;   // of a row in LDS
    uint32_t ow[NT], ox[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) ow[i] = ((n0 + 16 * i + c) * K + 16 * g) * 2u;
#pragma unroll
    for (int j = 0; j < MT; ++j)
        ox[j] = NORM ? min(static_cast<uint32_t>(c), M - 1) * pitch + 32 * g
                     : ((m0 + 16 * j + c) * K + 16 * g) * 2u;

    struct Group {
        u32x4 w[U][NT][2], x[U][NORM ? 1 : MT][2];
    };
    auto load = [&](int b, Group &d) {   // blocks b, b + WK, ... of this wave
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kb = b + u * WK;
            if (kb >= nb) break;
            const uint32_t o = static_cast<uint32_t>(kb) * 128u;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                d.w[u][i][0] = bld16(rw, ow[i] + o);
                d.w[u][i][1] = bld16(rw, ow[i] + o + 16);
            }
            if constexpr (!NORM)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    d.x[u][j][0] = bld16(rx, ox[j] + o);
                    d.x[u][j][1] = bld16(rx, ox[j] + o + 16);
                }
        }
    };
    f32x4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](int b, const Group &d) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kb = b + u * WK;
            if (kb >= nb) break;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    u32x4 xv;
                    if constexpr (NORM)
                        xv = *reinterpret_cast<const u32x4 *>(xs + ox[j] + kb * 128 + 16 * h);
                    else
                        xv = d.x[u][j][h];
#pragma unroll
                    for (int i = 0; i < NT; ++i)
                        acc[i][j] = mfma_bf16(__builtin_bit_cast(bf16x8, d.w[u][i][h]),
                                              __builtin_bit_cast(bf16x8, xv), acc[i][j]);
                }
        }
    };
    Group d0, d1;
    float sq[kNormRows] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (NORM) {
        // eight k of every row a thread; the rows and the gain are asked for
        // before the weights, which arrive in order behind them
        constexpr uint32_t STEP = 64 * WK * 8;
        u32x4 v[kNormRows];
        f32x4 gn[2];
        auto load_rows = [&](uint32_t i) {   // rows past M read as zeros
            gn[0] = gn[1] = f32x4{1.f, 1.f, 1.f, 1.f};
            if (gain != nullptr && i < K) {
                gn[0] = *reinterpret_cast<const f32x4 *>(gain + i);
                gn[1] = *reinterpret_cast<const f32x4 *>(gain + i + 4);
            }
#pragma unroll
            for (uint32_t r = 0; r < kNormRows; ++r) v[r] = bld16(rx, (r * K + i) * 2u);
        };
        auto form_rows = [&](uint32_t i) {
#pragma unroll
            for (uint32_t r = 0; r < kNormRows; ++r) {
                if (r >= M || i >= K) continue;
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = __uint_as_float(v[r][e] << 16);
                    const float hi = __uint_as_float(v[r][e] & 0xFFFF0000u);
                    sq[r] = __builtin_fmaf(lo, lo, sq[r]);
                    sq[r] = __builtin_fmaf(hi, hi, sq[r]);
                    o[e] = pack_bf16x2(lo * gn[e >> 1][2 * (e & 1)], hi * gn[e >> 1][2 * (e & 1) + 1]);
                }
                *reinterpret_cast<u32x4 *>(xs + r * pitch + i * 2) = o;
            }
        };
        uint32_t i = tid * 8;
        load_rows(i);
        load(wave, d0);
        form_rows(i);
        for (i += STEP; i < K; i += STEP) {
            load_rows(i);
            form_rows(i);
        }
        __syncthreads();
    } else {
        load(wave, d0);
    }
#pragma unroll 1
    for (int b = wave; b < nb; b += 2 * U * WK) {
        load(b + U * WK, d1);
        mul(b, d0);
        load(b + 2 * U * WK, d0);
        mul(b + U * WK, d1);
    }

    // ---- the waves' sums, then lane (c, g) of tile (i, j) holds y[m][n .. n + 3]
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    if constexpr (NORM) {
#pragma unroll
        for (int r = 0; r < static_cast<int>(kNormRows); ++r) {
            const float ss = group_sum(sq[r], 64);
            if (lane == 0) squares[wave][r] = ss;
        }
    }
    __syncthreads();
    float norm = 1.0f;
    if constexpr (NORM) {
        const int row = min(c, static_cast<int>(kNormRows) - 1);
        float ss = squares[0][row];
#pragma unroll
        for (int q = 1; q < WK; ++q) ss += squares[q][row];
        norm = 1.0f / sqrtf(ss / static_cast<float>(K) + eps);
    }
    for (int t = wave; t < NT * MT; t += WK) {
        f32x4 v = part[0][t][lane];
#pragma unroll
        for (int q = 1; q < WK; ++q) v += part[q][t][lane];
        if constexpr (NORM) v = v * norm;
        const uint32_t n = n0 + 16 * (t / MT) + 4 * g, m = m0 + 16 * (t % MT) + c;
        if (n >= N || m >= M) continue;
        if (scale) v = v * *reinterpret_cast<const f32x4 *>(scale + n);
        const size_t o = static_cast<size_t>(m) * N + n;
        if (res) {
            const u32x2 rv = *reinterpret_cast<const u32x2 *>(static_cast<const uint16_t *>(res) + o);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] += __uint_as_float((r & 1) ? (rv[r >> 1] & 0xFFFF0000u) : (rv[r >> 1] << 16));
        }
        *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(y) + o) =
            u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
}

template <int MT, int NT, int WK, int U, bool NORM = false>
void launch_cfg(uint32_t M, uint32_t K, uint32_t N, const void *x, const void *w, const float *scale,
                const void *res, void *y, hipStream_t s, const float *gain = nullptr, float eps = 0.0f) {
    const dim3 grid((N + 16 * NT - 1) / (16 * NT), (M + 16 * MT - 1) / (16 * MT));
    hipLaunchKernelGGL((few_rows_kernel<MT, NT, WK, U, NORM>), grid, dim3(64 * WK),
                       NORM ? M * (2 * K + 16) : 0, s, M, K, N, x, gain, eps, w, scale, res, y);
}

// The x a call reads from L2, every row once per workgroup of 32 columns.
size_t x_reads(size_t m, size_t k, size_t n) { return (n + 31) / 32 * m * k * 2; }

}  // namespace

// What the kernel takes.
static bool fits(size_t m, size_t k, size_t n, const void *x, const void *w, bool w_transposed,
                 const float *scale, const void *res, const void *y) {
    auto al = [](const void *p, uintptr_t b) { return reinterpret_cast<uintptr_t>(p) % b == 0; };
    if (!w_transposed || m < 1 || k < 64 || k % 64 != 0 || n < 16 || n % 4 != 0) return false;
    if (k * n * 2 >= (size_t(1) << 31) || !al(x, 16) || !al(w, 16) || !al(scale, 16) || !al(res, 8) ||
        !al(y, 8))
        return false;
    return true;
}

// Where the lines lie (us per call, hipBLASLt's plan of its own probe / this
// kernel; K x N).  Under 4096 columns, against skinny_gemm.hip, it is the faster
// one to 32 rows at every size: 16384 x 1024 54 / 20 (1 row), 1536 x 1536 7.3 / 6.5 (32),
// 3072 x 768 12.1 / 10.5 (32), 4096 x 4088 16.4 / 13.7 (32); at 48 rows 8.6 against 7.7
// the other way round: x's re-reads by every column tile take over.  From 4096 columns
// on hipBLASLt splits a long K where the columns leave CUs idle, and has tiles
// of 32 and 64 rows:
// - to 4 rows: 2048 x 4096 6.4 / 6.0, 2816 x 6144 10.7 / 10.2, 4096 x 12288 24.0 / 20.8; but
//   3072 x 6144 9.4 / 10.3, 4096 x 4608 9.9 / 12.8, 8192 x 8192 27.8 / 29.1; 64 x 65536, one
//   block of K for four waves, 5.5 / 6.3.
// - to 16: 1536 x 4608 and up to 1536 x 16384 11.1 / 10.7 (16 rows), any K to 4096 x 32000
//   56.1 / 55.0; but 2048 x 12288 12.3 / 14.0, 3072 x 10240 13.4 / 18.6, 8192 x 4608 19.8 /
//   24.8; at 4096 columns, half the CUs, 1024 6.4 / 5.4, 1536 5.9 / 6.3, 3072 7.7 / 10.6.
// - to 32: 2048 x 4608 11.7 / 9.8 (28), 1024 x 12288 10.4 / 9.5 (24), 512 x 32000 11.3 / 10.7
//   (20); but at exactly 32 2048 x 4608 9.1 / 10.2, 1536 x 4608 7.6 / 8.0; 1536 x 10800 11.7 /
//   12.8 (20), 3072 x 4608 11.2 / 12.2 (20), 256 x 32000 6.9 / 7.9 (28).
// - to 64, while each of its workgroups has a CU (8192 columns): 768 x 5400 10.0 / 6.7
//   (48) and 7.6 / 7.2 (64), 512 x 8192 8.1 / 6.0 (64); but 1024 x 4608 8.4 / 8.6 (64), 256 x
//   16384 6.6 / 7.9, 256 x 32000 7.4 / 11.9 (33).
bool few_rows_supported(size_t m, size_t k, size_t n, const void *x, const void *w, bool w_transposed,
                        const float *scale, const void *res, const void *y) {
    if (!fits(m, k, n, x, w, w_transposed, scale, res, y)) return false;
    if (n < 4096) return m <= 32;
    if (m <= 4) return (k <= 2816 || (n > 8192 && k <= 4096)) && (k >= 128 || n <= 32768);
    if (m <= 16) return k <= (n > 16384 ? 4096 : n >= 4608 ? 1536 : 1024);
    if (x_reads(m, k, n) > (size_t(20) << 20)) return false;
    if (m <= 32)
        return k <= (n >= 4608 && n <= 8192 && m < 32 ? 2048 : 1024) && (n <= 16384 || k >= 512);
    return m <= 64 && n <= 8192 && m * k <= 57344;
}

hipError_t launch_few_rows(size_t m, size_t k, size_t n, const void *x, const void *w,
                           const float *scale, const void *res, void *y, hipStream_t s) {
    const uint32_t M = static_cast<uint32_t>(m), K = static_cast<uint32_t>(k),
                   N = static_cast<uint32_t>(n);
    // two column tiles a wave halve x's re-reads of wide products (16 rows at
    // 1536 x 10800 11.6 against 12.5, at 1536 x 32000 22.1 against 27.5); up
    // to four rows there is next to nothing to re-read (10.0 against 8.4)
    if (m <= 16 && (m <= 4 || n < 4096))
        launch_cfg<1, 1, 4, 3>(M, K, N, x, w, scale, res, y, s);
    else if (m <= 16)
        launch_cfg<1, 2, 4, 2>(M, K, N, x, w, scale, res, y, s);
    else if (m <= 32 && n < 4096)
        launch_cfg<2, 1, 4, 2>(M, K, N, x, w, scale, res, y, s);
    else if (m <= 32)
        launch_cfg<2, 2, 4, 2>(M, K, N, x, w, scale, res, y, s);
    else
        launch_cfg<4, 2, 8, 1>(M, K, N, x, w, scale, res, y, s);
    return hipGetLastError();
}

bool norm_few_rows_supported(size_t m, size_t k, size_t n, const void *x, const float *gain,
                             const void *w, const float *scale, const void *res, const void *y) {
    // (the rows' copies in LDS, beside the partial sums).  With the norm's launch
    // and row in it this is the faster form at any K and N: 4096 x 4608 18.5 / 12.8 us
    // (1 row), 4096 x 12288 33.9 / 22.7 (4), 64 x 32000 6.5 / 5.9.
    return m <= kNormRows && m * (2 * k + 16) <= (size_t(50) << 10) &&
           reinterpret_cast<uintptr_t>(gain) % 16 == 0 &&
           fits(m, k, n, x, w, true, scale, res, y);
}

hipError_t launch_norm_few_rows(size_t m, size_t k, size_t n, const void *x, const float *gain, float eps,
                                const void *w, const float *scale, const void *res, void *y,
                                hipStream_t s) {
    const uint32_t M = static_cast<uint32_t>(m), K = static_cast<uint32_t>(k),
                   N = static_cast<uint32_t>(n);
    launch_cfg<1, 1, 4, 3, true>(M, K, N, x, w, scale, res, y, s, gain, eps);
    return hipGetLastError();
}

}  // namespace m3
