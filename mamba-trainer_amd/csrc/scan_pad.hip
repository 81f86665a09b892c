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
// side: 32 and 57 us, for the most part launches and their gaps.
#include <algorithm>

#include "m3_device.hpp"
#include "m3_internal.hpp"

namespace m3 {

namespace {

constexpr size_t kPadP = 64, kPadN = 64;
constexpr int kPadThreads = 256;

// How an array's elements move: as they are, or bf16 in the caller's array and
// f32 in the padded one; kMove32: one f32 a row, unpadded.
enum PadKind : uint32_t { kPad16, kPad32, kPadWiden, kMove32 };

// One array of rows: a source row of `lo` + `hi` elements stands at the front
// of each half of a padded row of 2 `half` elements (hi = 0: at the front of
// the row, lo <= 2 half).  Rows come in groups of `live` source rows padded to
// 1 << group_log rows (1 and 0 for token rows).  The caller's groups are those
// of `nh` heads out of `heads`: group g of the copy is (g / nh) heads + g % nh
// from `src` on.
struct PadArray {
    const void *src;      // the caller's (written by the unpad)
    void *dst;            // the padded copy
    uint32_t groups;      // row groups
    uint32_t lo, hi;      // source elements in each half
    uint32_t half;        // elements of a padded half row
    uint32_t quad_log;    // log2 of a padded row's four-element pieces
    uint32_t live, group_log;
    uint32_t kind;
    uint32_t nh, heads;
};
constexpr int kPadArrays = 13;   // the backward's inputs: x, b, c, theta, dt, lambda, dy, six of states
struct PadTable {
    PadArray a[kPadArrays];
};

__device__ __forceinline__ uint32_t src_group(const PadArray &A, uint32_t g) {
    return A.nh == A.heads ? g : g / A.nh * A.heads + g % A.nh;
}

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
        const size_t s = (static_cast<size_t>(src_group(A, g)) * A.live + p) * (A.lo + A.hi) +
                         (second ? A.lo : 0) + j;
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

// One f32 a row, to the copy or back.
template <bool OUT>
__device__ __forceinline__ void move_rows(const PadArray &A) {
    float *src = static_cast<float *>(const_cast<void *>(A.src)), *dst = static_cast<float *>(A.dst);
    for (uint32_t g = blockIdx.x * kPadThreads + threadIdx.x; g < A.groups; g += gridDim.x * kPadThreads) {
        if constexpr (OUT)
            src[src_group(A, g)] = dst[g];
        else
            dst[g] = src[src_group(A, g)];
    }
}

// src -> dst zero-padded, one array per blockIdx.y; bound by the writes.
__global__ void __launch_bounds__(kPadThreads) pad_kernel(PadTable t) {
    const PadArray &A = t.a[blockIdx.y];
    if (A.kind == kPad32)
        pad_rows<float, float>(A);
    else if (A.kind == kPad16)
        pad_rows<uint16_t, uint16_t>(A);
    else if (A.kind == kPadWiden)
        pad_rows<uint16_t, float>(A);
    else
        move_rows<false>(A);
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
        const size_t d = (static_cast<size_t>(src_group(A, g)) * A.live + p) * len + e;
        if constexpr (sizeof(S) == sizeof(D))
            dst[d] = src[o];
        else
            dst[d] = from_f32<bf16_t>(src[o]);
    }
}

// The live parts of the padded outputs (dst) back into the caller's (src).
__global__ void __launch_bounds__(kPadThreads) unpad_kernel(PadTable t) {
    const PadArray &A = t.a[blockIdx.y];
    if (A.kind == kPad32)
        unpad_rows<float, float>(A);
    else if (A.kind == kPad16)
        unpad_rows<uint16_t, uint16_t>(A);
    else if (A.kind == kPadWiden)
        unpad_rows<bf16_t, float>(A);
    else
        move_rows<true>(A);
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

// A call's sequences are copied and run in parts, of whole batch entries or of
// some heads of one, whose copies and kernels' workspace fit the room there is:
// the padded rows are up to 16 times the caller's and the backward's records 64 x
// 64 a chunk, 3.4 KB of both a token of a head of 16, so all of a long batch at
// once would take gigabytes.  A forward sequence whose own copies do not fit the
// static scratch runs in windows of its tokens, the state of one entering the
// next.
struct PadPart {
    size_t b0, nb, h0, nh, t0, nt;
};

// The part as a call of its own, but for the pointers into the arrays.
ScanLaunch part_of(const ScanLaunch &a, const PadPart &q) {
    ScanLaunch p = a;
    p.batch = q.nb;
    p.heads = q.nh;
    p.seq = q.nt;
    p.a_log = a.a_log ? a.a_log + q.h0 : nullptr;
    p.d_skip = a.d_skip ? a.d_skip + q.h0 : nullptr;
    return p;
}

// Sections of a part's padded copies in the workspace; the kernels' own
// workspace follows.  Sized for every optional array, present or not; dt,
// lambda and their gradients are copied for some heads of a batch entry only.
struct PadLayout {
    size_t x, b, c, theta, y, h, lu, ang, dh, dlu, dang;         // inputs
    size_t dx, db, dc, dtheta, dh0, dlu0, dang0, hout, luout, angout;
    size_t dt, lam, ddt, dlam;
    size_t total;
};
PadLayout pad_layout(const ScanLaunch &a, const PadPart &q, bool backward) {
    const size_t es = backward && a.bf16 ? 2 : 4, rows = q.nb * q.nt * q.nh, bh = q.nb * q.nh;
    const size_t xr = up256(rows * kPadP * a.rank * es), br = up256(rows * kPadN * a.rank * es);
    const size_t tr = up256(rows * (kPadN / 2) * es), st = up256(bh * kPadP * kPadN * 4);
    const size_t an = up256(bh * (kPadN / 2) * 4), sc = q.nh < a.heads ? up256(rows * 4) : 0;
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
    l.dt = take(sc);
    l.lam = take(sc);
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
        l.ddt = take(sc);
        l.dlam = take(sc);
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

// The arrays of a part in the padded layout; `first`: the byte of the caller's
// array that the part begins at.
struct PadShape {
    PadArray a;
    size_t first;
};
struct PadShapes {
    PadShape x, bc, theta, state, angle, scalar;
    PadShapes(const ScanLaunch &a, const PadPart &part, bool backward) {
        const uint32_t rows = static_cast<uint32_t>(part.nb * part.nt * part.nh);
        const uint32_t bh = static_cast<uint32_t>(part.nb * part.nh);
        const uint32_t nh = static_cast<uint32_t>(part.nh), H = static_cast<uint32_t>(a.heads);
        const uint32_t P = static_cast<uint32_t>(a.head_dim), N = static_cast<uint32_t>(a.d_state);
        const uint32_t R = static_cast<uint32_t>(a.rank);
        // rotation pairs keep their places in the two halves; an odd d_state
        // (real dynamics, no pairs) fills them in order
        const uint32_t lo = N / 2 > 0 ? N / 2 : N, hi = N - lo;
        const uint32_t q = log2u(kPadP * R / 4);
        const PadKind t = !a.bf16 ? kPad32 : backward ? kPad16 : kPadWiden;
        const size_t row0 = (part.b0 * a.seq + part.t0) * a.heads + part.h0, seq0 = part.b0 * a.heads + part.h0;
        const size_t es = a.bf16 ? 2 : 4;
        x = {{nullptr, nullptr, rows, P * R, 0, static_cast<uint32_t>(kPadP) * R / 2, q, 1, 0, t, nh, H},
             row0 * P * R * es};
        bc = {{nullptr, nullptr, rows, lo * R, hi * R, static_cast<uint32_t>(kPadN) * R / 2, q, 1, 0, t, nh, H},
              row0 * N * R * es};
        theta = {{nullptr, nullptr, rows, N / 2, 0, static_cast<uint32_t>(kPadN) / 4, log2u(kPadN / 8), 1, 0, t, nh, H},
                 row0 * (N / 2) * es};
        state = {{nullptr, nullptr, bh, lo, hi, static_cast<uint32_t>(kPadN) / 2, log2u(kPadN / 4), P,
                  log2u(kPadP), kPad32, nh, H},
                 seq0 * P * N * 4};
        angle = {{nullptr, nullptr, bh, N / 2, 0, static_cast<uint32_t>(kPadN) / 4, log2u(kPadN / 8), 1, 0, kPad32,
                  nh, H},
                 seq0 * (N / 2) * 4};
        scalar = {{nullptr, nullptr, rows, 1, 0, 0, 0, 1, 0, kMove32, nh, H}, row0 * 4};
    }
};

// A part's arrays as the kernels take them: those copied into `in` before them
// and out of `out` after them.
struct PadCopies {
    char *base;
    bool some_heads;
    Pads in, out;
    const void *put(const PadShape &s, const void *src, size_t off) {
        return add(in, s, const_cast<void *>(src), off);
    }
    void *get(const PadShape &s, void *dst, size_t off) { return add(out, s, dst, off); }
    // one value a row: in place where the part's rows are the caller's
    const float *put_row(const PadShape &s, const float *src, size_t off) {
        return some_heads ? static_cast<const float *>(put(s, src, off)) : src + s.first / 4;
    }
    float *get_row(const PadShape &s, float *dst, size_t off) {
        return some_heads ? static_cast<float *>(get(s, dst, off)) : dst + s.first / 4;
    }

private:
    void *add(Pads &to, const PadShape &s, void *ptr, size_t off) {
        if (ptr == nullptr) return nullptr;
        PadArray p = s.a;
        p.src = static_cast<char *>(ptr) + s.first;
        p.dst = base + off;
        to.add(p);
        return base + off;
    }
};

// The launch on a part's padded copies (inputs only; states where the caller
// has them).
ScanLaunch padded(const ScanLaunch &a, const PadPart &part, const PadLayout &l, const PadShapes &s,
                  PadCopies &c) {
    ScanLaunch p = part_of(a, part);
    p.head_dim = kPadP;
    p.d_state = kPadN;
    p.bf16 = s.x.a.kind == kPad16;
    p.x = c.put(s.x, a.x, l.x);
    p.b = c.put(s.bc, a.b, l.b);
    p.c = c.put(s.bc, a.c, l.c);
    p.theta = c.put(s.theta, a.theta, l.theta);
    p.dt = c.put_row(s.scalar, a.dt, l.dt);
    p.lambda = c.put_row(s.scalar, a.lambda, l.lam);
    if (part.t0 == 0) {   // a later window's state is where the one before left it
        p.h0 = static_cast<const float *>(c.put(s.state, a.h0, l.h));
        p.last_u0 = static_cast<const float *>(c.put(s.state, a.last_u0, l.lu));
        p.angle0 = static_cast<const float *>(c.put(s.angle, a.angle0, l.ang));
    }
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

size_t part_bytes(const ScanLaunch &a, const PadPart &q, bool backward) {
    ScanLaunch p = padded_shape(part_of(a, q), backward);
    size_t kernels = backward ? scan_backward_workspace(p) : scan_chunked_workspace(p);
    if (a.seq % q.nt != 0) {   // the last window may be cut into more segments than a longer one
        p.seq = a.seq % q.nt;
        kernels = std::max(kernels, scan_chunked_workspace(p));
    }
    return pad_layout(a, q, backward).total + kernels;
}

// The largest of n counts from 1 on that fits; 0 if none does.
template <typename F>
size_t largest(size_t n, F fits) {
    size_t lo = 0, hi = n;
    while (lo < hi) {
        const size_t mid = lo + (hi - lo + 1) / 2;
        if (fits(mid))
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// The first (and largest) part within `room` bytes: the whole call, else as
// many batch entries as fit, shared out evenly, else as many heads of one; one
// sequence at the least for the backward (heads of 64 ask for as much; one of
// 170,000 tokens, rank 1 in f32, 5.8 ms in 522 MiB, where the token walk takes 11 us a
// token), nb = 0 for the forward where that does not fit.  Parts of 64 / 256 / 512 / 1024 MiB, us
// a call, heads of 16, f32: backward, 512 sequences of 512 tokens 1022 / 611 /
// 608 / 591, 256 of 2048 3642 / 1387 / 1241 / 1157 (1137 at once, in 1.7 GB), 8 of
// 16384 4410 / 1279 / 793 / 795; forward, 256 of 2048 889 / 503 / 480 / 428.  The
// kernels these shapes took before need 8 ms and 40 ms for the first two.
// A sequence past the static scratch is cut into windows by that, whatever the
// room, so that both of the forward's callers cut alike: 2 of 31000 tokens 421 us in
// windows, 156 at once in 93 MB, 15816 by one workgroup each; 8 of them 1692, 253 and
// 18702.
PadPart pad_part(const ScanLaunch &a, bool backward, size_t room) {
    auto fits = [&](size_t nb, size_t nh) {
        return part_bytes(a, PadPart{0, nb, 0, nh, 0, a.seq}, backward) <= room;
    };
    // the most of n that fit, or fewer in as many parts of one size
    auto share = [](size_t n, auto ok) {
        const size_t most = largest(n, ok);
        if (most == 0) return most;
        const size_t parts = (n + most - 1) / most, even = (n + parts - 1) / parts;
        return ok(even) ? even : most;
    };
    if (!backward && part_bytes(a, PadPart{0, 1, 0, 1, 0, a.seq}, false) > kNoAllocScratchBytes) {
        const size_t tiles = share((a.seq + 63) / 64, [&](size_t v) {
            return part_bytes(a, PadPart{0, 1, 0, 1, 0, 64 * v}, false) <= kNoAllocScratchBytes;
        });
        return tiles > 0 ? PadPart{0, 1, 0, 1, 0, 64 * tiles} : PadPart{};
    }
    if (fits(a.batch, a.heads)) return PadPart{0, a.batch, 0, a.heads, 0, a.seq};
    const size_t nb = share(a.batch, [&](size_t v) { return fits(v, a.heads); });
    if (nb > 0) return PadPart{0, nb, 0, a.heads, 0, a.seq};
    const size_t nh = share(a.heads, [&](size_t v) { return fits(1, v); });
    if (nh > 0) return PadPart{0, 1, 0, nh, 0, a.seq};
    return backward ? PadPart{0, 1, 0, 1, 0, a.seq} : PadPart{};
}

// f(part) for every part of the call, whose first is q; a sequence's windows in
// order.
template <typename F>
hipError_t each_part(const ScanLaunch &a, PadPart q, F f) {
    const size_t nb = q.nb, nh = q.nh, nt = q.nt;
    if (nb == 0) return hipErrorNotSupported;
    for (q.b0 = 0; q.b0 < a.batch; q.b0 += nb) {
        q.nb = std::min(nb, a.batch - q.b0);
        for (q.h0 = 0; q.h0 < a.heads; q.h0 += nh) {
            q.nh = std::min(nh, a.heads - q.h0);
            for (q.t0 = 0; q.t0 < a.seq; q.t0 += nt) {
                q.nt = std::min(nt, a.seq - q.t0);
                const hipError_t e = f(q);
                if (e != hipSuccess) return e;
            }
        }
    }
    return hipSuccess;
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

// Measured on MI355X (f32, us per call, one workgroup per sequence / padded):
// - head_dim and d_state 16, 8 sequences of 33 tokens 28.8 / 24.5, 64 34.3 / 24.4, 96
//   47.9 / 26.1, 128 61.7 / 25.7; 16 of 512 227 / 32; rank 4, 8 of 8 tokens 16.8 / 24.9, 16
//   26.1 / 25.7, 24 35.7 / 26.7, 32 44.9 / 26.1;
// - heads of 32, d_state 32: 8 of 33 25.2 / 25.5, 64 28.8 / 25.6, 96 39.7 / 26.5, 128 50.5 /
//   26.2; 64 of 400 148 / 48; d_state 64, 8 of 33 32.9 / 26.5, 64 37.8 / 25.8;
// - many sequences of 512 tokens, heads of 16: 256 314 / 98, 512 322 / 206, 640 326 /
//   427, 768 326 / 329, 1024 326 / 469; of 128 tokens 512 88 / 55, 1024 95 / 92.
// The line at 512 sequences lies where a thousand fill the chip as they are.  The
// line at 128 rows is older than the segments of less than 64 tokens, which moved
// the meeting point to some 33 rows (rank 4: 64): windows between are left on the
// slower kernel.  Heads of 33 to 63, and head_dim 64 at d_state below 64, were not
// measured.
bool scan_pad_wanted(const ScanLaunch &a) {
    return a.seq * a.rank >= 128 && a.batch * a.heads <= 512 && pad_shape(a, false);
}

// The call with its cut decided, by the part that kPadBytes hold: the same
// results through any room, and m3_scan_no_alloc's those of m3_scan.
static ScanLaunch planned(const ScanLaunch &a) {
    const PadPart q = pad_part(a, false, kPadBytes);
    ScanLaunch p = a;
    p.plan_seqs = q.nb * q.nh;
    return p;
}

size_t scan_pad_workspace(const ScanLaunch &a, size_t room) {
    if (!scan_pad_wanted(a)) return 0;
    const ScanLaunch p = planned(a);
    return part_bytes(p, pad_part(p, false, room), false);
}

hipError_t launch_scan_pad(const ScanLaunch &call, void *workspace, size_t room, hipStream_t stream,
                           int &launches) {
    const ScanLaunch a = planned(call);
    const PadPart first = pad_part(a, false, room);
    return each_part(a, first, [&](const PadPart &q) {
        PadPart longest = q;   // windows share the layout of the longest
        longest.nt = first.nt;
        const PadLayout l = pad_layout(a, longest, false);
        const PadShapes s(a, q, false);
        PadCopies c{static_cast<char *>(workspace), q.nh < a.heads, {}, {}};
        ScanLaunch p = padded(a, q, l, s, c);
        p.y = c.get(s.x, a.y, l.y);
        // the state entering and leaving a window change places with each
        const bool odd = q.t0 / first.nt % 2 != 0;
        auto at = [&](size_t off) { return reinterpret_cast<float *>(c.base + off); };
        const size_t hi = odd ? l.hout : l.h, ui = odd ? l.luout : l.lu, ai = odd ? l.angout : l.ang;
        const size_t ho = odd ? l.h : l.hout, uo = odd ? l.lu : l.luout, ao = odd ? l.ang : l.angout;
        if (q.t0 > 0) {
            p.h0 = at(hi);
            p.last_u0 = at(ui);
            p.angle0 = a.theta ? at(ai) : nullptr;
        }
        if (q.t0 + q.nt < a.seq) {
            p.h_out = at(ho);
            p.last_u_out = at(uo);
            p.angle_out = a.theta ? at(ao) : nullptr;
        } else {
            p.h_out = static_cast<float *>(c.get(s.state, a.h_out, ho));
            p.last_u_out = static_cast<float *>(c.get(s.state, a.last_u_out, uo));
            p.angle_out = static_cast<float *>(c.get(s.angle, a.angle_out, ao));
        }
        const size_t kernels = scan_chunked_workspace(p);
        if (l.total + kernels > room) return hipErrorInvalidValue;
        hipError_t e = launch_pads(c.in, false, stream);
        if (e != hipSuccess) return e;
        if (kernels > 0) {
            e = launch_scan_chunked(p, c.base + l.total, stream, launches);
        } else {
            e = launch_scan(p, stream);
            ++launches;
        }
        if (e != hipSuccess) return e;
        launches += 2;
        return launch_pads(c.out, true, stream);
    });
}

// The token walk / padded (f32, head_dim and d_state 16, us per call): 2 sequences
// of 8 tokens 94 / 34, of 64 701 / 38; 16 of 512 5637 / 57; 1024 of 512 8445 / 1219 (in
// parts, 447 MB; at once 1155 in 1.8 GB), 8192 of 32 5248 / 802; 2 of 1 token 20 by the
// walk.  The line at 8 tokens was drawn with the chunk kernels at 50 us, which
// met the walk at 4 (52).  Heads over 32, states over 64 and other ranks keep the
// walk's two launches; its line against them was not measured.
bool scan_backward_pad_wanted(const ScanLaunch &a) { return a.seq >= 8 && pad_shape(a, true); }

size_t scan_backward_pad_workspace(const ScanLaunch &a) {
    if (!scan_backward_pad_wanted(a)) return 0;
    const PadPart q = pad_part(a, true, kPadBytes);
    return q.nb > 0 ? part_bytes(a, q, true) : 0;
}

hipError_t launch_scan_backward_pad(const ScanLaunch &a, const ScanGrads &g, void *workspace,
                                    hipStream_t stream, int &launches) {
    return each_part(a, pad_part(a, true, kPadBytes), [&](const PadPart &part) {
        const PadLayout l = pad_layout(a, part, true);
        const PadShapes s(a, part, true);
        PadCopies c{static_cast<char *>(workspace), part.nh < a.heads, {}, {}};
        const ScanLaunch p = padded(a, part, l, s, c);
        ScanGrads q = g;
        q.dy = c.put(s.x, g.dy, l.y);
        q.dh_out = static_cast<const float *>(c.put(s.state, g.dh_out, l.dh));
        q.dlast_u_out = static_cast<const float *>(c.put(s.state, g.dlast_u_out, l.dlu));
        q.dangle_out = static_cast<const float *>(c.put(s.angle, g.dangle_out, l.dang));
        q.dx = c.get(s.x, g.dx, l.dx);
        q.db = c.get(s.bc, g.db, l.db);
        q.dc = c.get(s.bc, g.dc, l.dc);
        q.ddt = c.get_row(s.scalar, g.ddt, l.ddt);
        q.dlambda = c.get_row(s.scalar, g.dlambda, l.dlam);
        q.dtheta = c.get(s.theta, g.dtheta, l.dtheta);
        q.dh0 = static_cast<float *>(c.get(s.state, g.dh0, l.dh0));
        q.dlast_u0 = static_cast<float *>(c.get(s.state, g.dlast_u0, l.dlu0));
        q.dangle0 = static_cast<float *>(c.get(s.angle, g.dangle0, l.dang0));
        // the sums over the batch, part after part
        q.da_log = g.da_log + part.h0;
        q.dd_skip = g.dd_skip ? g.dd_skip + part.h0 : nullptr;
        q.add_sums = part.b0 > 0;
        hipError_t e = launch_pads(c.in, false, stream);
        if (e != hipSuccess) return e;
        e = launch_scan_backward(p, q, c.base + l.total, scan_backward_workspace(p), stream, launches);
        if (e != hipSuccess) return e;
        launches += 2;
        return launch_pads(c.out, true, stream);
    });
}

}  // namespace m3
