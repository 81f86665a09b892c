// The scan and its backward for the heads of small models (head_dim up to 32,
// d_state up to 64, rank 1, 2 or 4), on the chunk-parallel kernels of the
// 64 x 64 head: the inputs are copied into zero-padded rows, the kernels run
// on those, and the outputs' live parts are copied back.  Zero columns of x
// and zero state pairs of B, C and theta add exact zeros to every sum, so the
// results are those kernels' own.
//
// The kernels these shapes took before walk each sequence with one workgroup:
// the forward in 32- or 64-row chunks, the backward token by token.  What
// bounds them is that serial chain, not work: at batch 4 x 512, 4 heads of 16,
// d_state 16, f32, 16 of the 256 CUs are busy for 233 us (forward) and
// 5613 us (backward).  Padded, the 16 sequences are cut in chunks that run side by
// side: 33 and 59 us, for the most part launches and their gaps.
#include <algorithm>

#include "m3_device.hpp"
#include "m3_internal.hpp"

namespace m3 {

namespace {

constexpr size_t kPadP = 64, kPadN = 64;
constexpr int kPadThreads = 256;

// How an array's elements move: as they are, or bf16 in the caller's array and
// f32 in the padded one.
enum PadKind : uint32_t { kPad16, kPad32, kPadWiden };

// One array of rows: a source row of `lo` + `hi` elements stands at the front
// of each half of a padded row of 2 `half` elements (hi = 0: at the front of
// the row, lo <= 2 half).  Rows come in groups of `live` source rows padded to
// 1 << group_log rows (1 and 0 for token rows).
struct PadArray {
    const void *src;      // the caller's (written by the unpad)
    void *dst;            // the padded copy
    uint32_t groups;      // row groups
    uint32_t lo, hi;      // source elements in each half
    uint32_t half;        // elements of a padded half row
    uint32_t quad_log;    // log2 of a padded row's four-element pieces
    uint32_t live, group_log;
    uint32_t kind;
};
constexpr int kPadArrays = 12;
struct PadTable {
    PadArray a[kPadArrays];
};

template <typename S, typename D>
__device__ __forceinline__ void pad_rows(const PadArray &A) {
    const S *src = static_cast<const S *>(A.src);
    D *dst = static_cast<D *>(A.dst);
    const uint32_t items = A.groups << (A.group_log + A.quad_log);
    for (uint32_t it = blockIdx.x * kPadThreads + threadIdx.x; it < items;
         it += gridDim.x * kPadThreads) {
        const uint32_t row = it >> A.quad_log;
        const uint32_t e = (it & ((1u << A.quad_log) - 1)) * 4;
        const uint32_t g = row >> A.group_log, p = row & ((1u << A.group_log) - 1);
        const bool second = A.hi != 0 && e >= A.half;
        const uint32_t j = second ? e - A.half : e;
        const uint32_t n = p < A.live ? (second ? A.hi : A.lo) : 0;
        const size_t s = (static_cast<size_t>(g) * A.live + p) * (A.lo + A.hi) + (second ? A.lo : 0) + j;
        typedef D D4 __attribute__((ext_vector_type(4)));
        D4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = D(0);
            if (j + q < n) {
                if constexpr (sizeof(S) == sizeof(D))
                    v[q] = src[s + q];
                else   // bf16 bits to f32
                    v[q] = __uint_as_float(static_cast<uint32_t>(src[s + q]) << 16);
            }
        }
        *reinterpret_cast<D4 *>(dst + static_cast<size_t>(it) * 4) = v;
    }
}

// src -> dst zero-padded, one array per blockIdx.y; bound by the writes.
__global__ void __launch_bounds__(kPadThreads) pad_kernel(PadTable t) {
    const PadArray &A = t.a[blockIdx.y];
    if (A.kind == kPad32)
        pad_rows<float, float>(A);
    else if (A.kind == kPad16)
        pad_rows<uint16_t, uint16_t>(A);
    else
        pad_rows<uint16_t, float>(A);
}

template <typename S, typename D>
__device__ __forceinline__ void unpad_rows(const PadArray &A) {
    const D *src = static_cast<const D *>(A.dst);
    S *dst = static_cast<S *>(const_cast<void *>(A.src));
    const uint32_t len = A.lo + A.hi, items = A.groups * A.live * len;
    for (uint32_t it = blockIdx.x * kPadThreads + threadIdx.x; it < items;
         it += gridDim.x * kPadThreads) {
        const uint32_t row = it / len, e = it - row * len;
        const uint32_t g = A.live == 1 ? row : row / A.live;
        const uint32_t p = row - g * A.live;
        const size_t o = ((static_cast<size_t>(g) << A.group_log) + p) * (4u << A.quad_log) +
                         (e < A.lo ? e : A.half + e - A.lo);
        if constexpr (sizeof(S) == sizeof(D))
            dst[it] = src[o];
        else
            dst[it] = from_f32<bf16_t>(src[o]);
    }
}

// The live parts of the padded outputs (dst) back into the caller's (src).
__global__ void __launch_bounds__(kPadThreads) unpad_kernel(PadTable t) {
    const PadArray &A = t.a[blockIdx.y];
    if (A.kind == kPad32)
        unpad_rows<float, float>(A);
    else if (A.kind == kPad16)
        unpad_rows<uint16_t, uint16_t>(A);
    else
        unpad_rows<bf16_t, float>(A);
}

// The table's arrays and the largest one's items (four-element pieces to pad,
// elements to unpad).
struct Pads {
    PadTable t{};
    int n = 0;
    size_t items = 0;
    void add(const PadArray &p) {
        t.a[n++] = p;
        items = std::max(items, static_cast<size_t>(p.groups) << (p.group_log + p.quad_log));
    }
    dim3 grid() const {
        const size_t b = (items + kPadThreads - 1) / kPadThreads;
        return dim3(static_cast<unsigned>(b < 2048 ? b : 2048), static_cast<unsigned>(n));
    }
};

size_t up256(size_t v) { return (v + 255) & ~size_t(255); }

// Sections of the padded copies in the workspace; the kernels' own workspace
// follows.  Sized for every optional array, present or not.
struct PadLayout {
    size_t x, b, c, theta, y, h, lu, ang, dh, dlu, dang;         // inputs
    size_t dx, db, dc, dtheta, dh0, dlu0, dang0, hout, luout, angout;
    size_t total;
};
PadLayout pad_layout(const ScanLaunch &a, bool backward) {
    const size_t es = backward && a.bf16 ? 2 : 4, rows = a.batch * a.seq * a.heads, bh = a.batch * a.heads;
    const size_t xr = up256(rows * kPadP * a.rank * es), br = up256(rows * kPadN * a.rank * es);
    const size_t tr = up256(rows * (kPadN / 2) * es), st = up256(bh * kPadP * kPadN * 4);
    const size_t an = up256(bh * (kPadN / 2) * 4);
    PadLayout l{};
    size_t o = 0;
    auto take = [&o](size_t v) { const size_t at = o; o += v; return at; };
    l.x = take(xr);
    l.b = take(br);
    l.c = take(br);
    l.theta = take(tr);
    l.y = take(xr);            // y, or the backward's dy
    l.h = take(st);
    l.lu = take(st);
    l.ang = take(an);
    if (backward) {
        l.dh = take(st);
        l.dlu = take(st);
        l.dang = take(an);
        l.dx = take(xr);
        l.db = take(br);
        l.dc = take(br);
        l.dtheta = take(tr);
        l.dh0 = take(st);
        l.dlu0 = take(st);
        l.dang0 = take(an);
    } else {
        l.hout = take(st);
        l.luout = take(st);
        l.angout = take(an);
    }
    l.total = o;
    return l;
}

uint32_t log2u(size_t v) {
    uint32_t k = 0;
    while ((size_t(1) << k) < v) ++k;
    return k;
}

// The arrays of a launch in the padded layout.
struct PadShapes {
    PadArray x, bc, theta, state, angle;
    PadShapes(const ScanLaunch &a, bool backward) {
        const uint32_t rows = static_cast<uint32_t>(a.batch * a.seq * a.heads);
        const uint32_t bh = static_cast<uint32_t>(a.batch * a.heads);
        const uint32_t P = static_cast<uint32_t>(a.head_dim), N = static_cast<uint32_t>(a.d_state);
        const uint32_t R = static_cast<uint32_t>(a.rank);
        // rotation pairs keep their places in the two halves; an odd d_state
        // (real dynamics, no pairs) fills them in order
        const uint32_t lo = N / 2 > 0 ? N / 2 : N, hi = N - lo;
        const uint32_t q = log2u(kPadP * R / 4);
        const PadKind t = !a.bf16 ? kPad32 : backward ? kPad16 : kPadWiden;
        x = PadArray{nullptr, nullptr, rows, P * R, 0, static_cast<uint32_t>(kPadP) * R / 2, q, 1, 0, t};
        bc = PadArray{nullptr, nullptr, rows, lo * R, hi * R, static_cast<uint32_t>(kPadN) * R / 2, q, 1, 0, t};
        theta = PadArray{nullptr, nullptr, rows, N / 2, 0, static_cast<uint32_t>(kPadN) / 4, log2u(kPadN / 8), 1, 0, t};
        state = PadArray{nullptr, nullptr, bh, lo, hi, static_cast<uint32_t>(kPadN) / 2, log2u(kPadN / 4), P, log2u(kPadP), kPad32};
        angle = PadArray{nullptr, nullptr, bh, N / 2, 0, static_cast<uint32_t>(kPadN) / 4, log2u(kPadN / 8), 1, 0, kPad32};
    }
};

PadArray with(PadArray p, const void *src, void *dst) {
    p.src = src;
    p.dst = dst;
    return p;
}

// The launch on the padded copies under `base` (inputs only; states where the
// caller has them).
ScanLaunch padded(const ScanLaunch &a, const PadLayout &l, char *base, const PadShapes &s, Pads &in) {
    ScanLaunch p = a;
    p.head_dim = kPadP;
    p.d_state = kPadN;
    p.bf16 = s.x.kind == kPad16;
    auto put = [&](const PadArray &shape, const void *src, size_t off) -> void * {
        if (src == nullptr) return nullptr;
        in.add(with(shape, src, base + off));
        return base + off;
    };
    p.x = put(s.x, a.x, l.x);
    p.b = put(s.bc, a.b, l.b);
    p.c = put(s.bc, a.c, l.c);
    p.theta = put(s.theta, a.theta, l.theta);
    p.h0 = static_cast<const float *>(put(s.state, a.h0, l.h));
    p.last_u0 = static_cast<const float *>(put(s.state, a.last_u0, l.lu));
    p.angle0 = static_cast<const float *>(put(s.angle, a.angle0, l.ang));
    return p;
}

// The launch's shape on the padded head, with aligned pointers (sizing).  The
// forward widens bf16 storage: the bf16 chunk kernels round the states between
// chunks to bf16, which the kernel these shapes took before does not.
ScanLaunch padded_shape(const ScanLaunch &a, bool backward) {
    alignas(16) static float dummy[4] = {0, 0, 0, 0};
    ScanLaunch p = a;
    p.head_dim = kPadP;
    p.d_state = kPadN;
    p.bf16 = backward ? a.bf16 : 0;
    p.x = p.b = p.c = p.y = dummy;
    p.theta = a.theta ? dummy : nullptr;
    p.h0 = p.last_u0 = p.angle0 = p.init_state = nullptr;
    p.h_out = p.last_u_out = p.angle_out = nullptr;
    return p;
}

bool pad_shape(const ScanLaunch &a, bool backward) {
    return a.mode_raw && a.seq > 0 && a.theta_stride == 0 && a.head_dim >= 1 && a.head_dim <= 32 &&
           a.d_state >= 1 && a.d_state <= kPadN && (a.rank == 1 || a.rank == 2 || a.rank == 4) &&
           a.batch * a.seq * a.heads * kPadP * a.rank < (size_t(1) << 31) &&
           a.batch * a.heads * kPadP * kPadN < (size_t(1) << 31) &&
           scan_fast_supported(padded_shape(a, backward));
}

hipError_t launch_pads(const Pads &p, bool out, hipStream_t s) {
    if (p.n == 0) return hipSuccess;
    if (out)
        hipLaunchKernelGGL(unpad_kernel, p.grid(), dim3(kPadThreads), 0, s, p.t);
    else
        hipLaunchKernelGGL(pad_kernel, p.grid(), dim3(kPadThreads), 0, s, p.t);
    return hipGetLastError();
}

}  // namespace

// Measured on MI355X (f32, head_dim and d_state 16, us per call, one workgroup
// per sequence against padded): 8 sequences of 128 tokens 65 against 24; 16 of
// 512 233 against 33; 64 of 400 (heads of 32) 153 against 50; 512 of 512 340
// against 211; 1024 of 512 344 against 403, for a thousand sequences fill the
// chip as they are.  The line at 128 rows is where the two met (8 of 64 / 96
// 38 / 51 against 38 / 53) before the padded windows were cut into as many
// segments as they are now; 4 of 33 at rank 4 were 54 against 56, 4096 of 64 160
// against 268.
bool scan_pad_wanted(const ScanLaunch &a) {
    return a.seq * a.rank >= 128 && a.batch * a.heads <= 512 && pad_shape(a, false);
}

size_t scan_pad_workspace(const ScanLaunch &a) {
    if (!scan_pad_wanted(a)) return 0;
    return pad_layout(a, false).total + scan_chunked_workspace(padded_shape(a, false));
}

hipError_t launch_scan_pad(const ScanLaunch &a, void *workspace, hipStream_t stream, int &launches) {
    const PadLayout l = pad_layout(a, false);
    const PadShapes s(a, false);
    char *base = static_cast<char *>(workspace);
    Pads in, out;
    ScanLaunch p = padded(a, l, base, s, in);
    auto get = [&](const PadArray &shape, void *dst, size_t off) -> void * {
        if (dst == nullptr) return nullptr;
        out.add(with(shape, dst, base + off));
        return base + off;
    };
    p.y = get(s.x, a.y, l.y);
    p.h_out = static_cast<float *>(get(s.state, a.h_out, l.hout));
    p.last_u_out = static_cast<float *>(get(s.state, a.last_u_out, l.luout));
    p.angle_out = static_cast<float *>(get(s.angle, a.angle_out, l.angout));
    hipError_t e = launch_pads(in, false, stream);
    if (e != hipSuccess) return e;
    if (scan_chunked_workspace(p) > 0) {
        e = launch_scan_chunked(p, base + l.total, stream, launches);
    } else {
        e = launch_scan(p, stream);
        ++launches;
    }
    if (e != hipSuccess) return e;
    launches += 2;
    return launch_pads(out, true, stream);
}

// The token walk against padded (f32, head_dim and d_state 16, us per call): 2
// sequences of 8 / 64 tokens 98 / 701 against 32 / 33; 16 of 512 5613 against 59;
// 1024 of 512 8507 against 1160; 8192 of 32 4471 against 815; 2 of 1 token 20 by
// the walk.  The line at 8 tokens was drawn with the chunk kernels at 50 us, which
// met the walk at 4 (52).  Heads over 32, states over 64 and other ranks keep the
// walk's two launches.
bool scan_backward_pad_wanted(const ScanLaunch &a) { return a.seq >= 8 && pad_shape(a, true); }

size_t scan_backward_pad_workspace(const ScanLaunch &a) {
    if (!scan_backward_pad_wanted(a)) return 0;
    return pad_layout(a, true).total + scan_backward_workspace(padded_shape(a, true));
}

hipError_t launch_scan_backward_pad(const ScanLaunch &a, const ScanGrads &g, void *workspace,
                                    hipStream_t stream) {
    const PadLayout l = pad_layout(a, true);
    const PadShapes s(a, true);
    char *base = static_cast<char *>(workspace);
    Pads in, out;
    const ScanLaunch p = padded(a, l, base, s, in);
    ScanGrads q = g;
    auto put = [&](const PadArray &shape, const void *src, size_t off) -> void * {
        if (src == nullptr) return nullptr;
        in.add(with(shape, src, base + off));
        return base + off;
    };
    auto get = [&](const PadArray &shape, void *dst, size_t off) -> void * {
        if (dst == nullptr) return nullptr;
        out.add(with(shape, dst, base + off));
        return base + off;
    };
    q.dy = put(s.x, g.dy, l.y);
    q.dh_out = static_cast<const float *>(put(s.state, g.dh_out, l.dh));
    q.dlast_u_out = static_cast<const float *>(put(s.state, g.dlast_u_out, l.dlu));
    q.dangle_out = static_cast<const float *>(put(s.angle, g.dangle_out, l.dang));
    q.dx = get(s.x, g.dx, l.dx);
    q.db = get(s.bc, g.db, l.db);
    q.dc = get(s.bc, g.dc, l.dc);
    q.dtheta = get(s.theta, g.dtheta, l.dtheta);
    q.dh0 = static_cast<float *>(get(s.state, g.dh0, l.dh0));
    q.dlast_u0 = static_cast<float *>(get(s.state, g.dlast_u0, l.dlu0));
    q.dangle0 = static_cast<float *>(get(s.angle, g.dangle0, l.dang0));
    hipError_t e = launch_pads(in, false, stream);
    if (e != hipSuccess) return e;
    e = launch_scan_backward(p, q, base + l.total, stream);
    if (e != hipSuccess) return e;
    return launch_pads(out, true, stream);
}

}  // namespace m3
