// Separable wavelet transforms for gfx950: CDF 9/7 (fp32) and reversible CDF 5/3 (int16).
//
// Math: src/cudaCompress/util/DWTFloatKernels.cui:14-81 (9/7 analysis), :433-503 (synthesis),
// src/cudaCompress/util/DWTFloatFilters.cuh:42-49 (coefficients), src/cudaCompress/util/
// DWTIntKernels.cui:15-100, :597-687 (5/3 lifting), src/cudaCompress/util/DWTCommon.cuh:54-142
// (extensions, div2/div4).  Pass order and buffer use follow src/cudaCompress/util/DWTFloat.cu:
// 85-463 and DWTInt.cu:79-317 so callers that alias source, buffers and destination the way the
// reference's callers do (src/examples/CompressVolume.cpp:341-347, :503-507) get the same result.
//
// Layout of the work: the x and y axes in one pass, streaming along y (fwd_xy, inv_yx), then z
// (fwd_cols, inv_cols), streaming along z; every element is read and written once a pass, the filter
// windows stay in registers and neighbours along x are fetched from the next lanes, so there is no LDS
// and no barrier.  Where a caller's buffers do not allow the fused pass (it reads rows that another
// workgroup may have replaced already), or an axis is shorter than 8, x and y run one after the other
// (fwd_x, inv_x and the column passes).  9/7 sums are explicit fmaf chains in filter order (no
// reassociation), which is what the reference's `sum += c*v` loop compiles to, so every route gives the
// same bits.  Memory bounds the passes: three levels of 256^3 floats move 153 MB a pass, xy 46, z 35, its
// inverse 33 and yx 44 us (3.3 to 4.6 TB/s; a copy reaches 4.8).  With LDS tiles, one pass per axis and
// rows walked by one wave the four passes' work took 290 us.
#include "../kernels.hpp"
#include "dwt_ops.hpp"

#include <type_traits>

namespace cca {
namespace {

constexpr int XP = 64;  // pairs per X-pass chunk (one per lane)

// Byte images enter the first analysis pass as value - 128 and leave the last synthesis pass
// rounded half up and clamped to [0, 255] (toFloat/fromFloat, src/cudaCompress/util/
// DWTCommon.cuh:16-34).
template <class T>
__device__ __forceinline__ T load_in(T v) { return v; }
__device__ __forceinline__ float load_in(uint8_t v) { return float(v) - 128.0f; }
template <class TOut, class T>
__device__ __forceinline__ TOut store_out(T v) {
    if constexpr (std::is_same<TOut, uint8_t>::value)
        return (uint8_t)fminf(fmaxf(v + 128.5f, 0.0f), 255.0f);
    else
        return v;
}

// mirror, ext_low and ext_high for lines of at least kLine samples, where one reflection is enough
// whatever the filter: no loop, so that loads around them can be issued together.
constexpr int kLine = 8;
__device__ __forceinline__ int mirror1(int j, int n) {
    const int a = max(j, -j);
    return min(a, 2 * (n - 1) - a);
}
__device__ __forceinline__ int ext_low1(int g, int m) {
    const int a = max(g, -g);
    return min(a, 2 * m - 1 - a);
}
__device__ __forceinline__ int ext_high1(int g, int m) {
    const int a = max(g, -g - 1);
    return min(a, 2 * m - 2 - a);
}

// ---- X pass (contiguous axis): a wave per row and chunk of XP pairs ------------------------------
// LO: only the lowpass half is written (the lowpass-only transforms).
template <class Op, int CH, class TIn = typename Op::T, bool LO = false>
__global__ __launch_bounds__(256) void fwd_x(typename Op::T* __restrict__ dst, const TIn* __restrict__ src,
                                             int n, int rows, int sy, int dRow, int dSlice, int sRow, int sSlice) {
    using T = typename Op::T;
    constexpr int W = 2 * XP + 2 * Op::H;
    __shared__ T lds[4][W + 2];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned rb = ((unsigned)rows + 3) / 4, chunk = blockIdx.x / rb;
    const int row = (int)(blockIdx.x - chunk * rb) * 4 + wave;
    const bool active = row < rows;
    const int y = active ? row % sy : 0, z = active ? row / sy : 0;
    const TIn* s = src + (long long)z * sSlice + (long long)y * sRow;
    T* d = dst + (long long)z * dSlice + (long long)y * dRow;
    const int m = n / 2;
    const int k0 = (int)chunk * XP;
    if (active) {
        for (int i = lane; i < W; i += 64) {
            int p = 2 * k0 - Op::H + i;
            if (p < n + Op::H) lds[wave][i] = load_in(s[(long long)mirror(p, n) * CH]);
        }
    }
    __syncthreads();
    const int k = k0 + lane;
    if (active && k < m) {
        T lo, hi;
        Op::pair(lds[wave], lane, lo, hi);
        d[k] = lo;
        if (!LO) d[m + k] = hi;
    }
}

template <class Op, int CH, class TOut = typename Op::T>
__global__ __launch_bounds__(256) void inv_x(TOut* __restrict__ dst, const typename Op::T* __restrict__ src,
                                             int n, int rows, int sy, int dRow, int dSlice, int sRow, int sSlice) {
    using T = typename Op::T;
    constexpr int W = 2 * (XP + 2 * Op::G);
    __shared__ T lds[4][W + 2];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned rb = ((unsigned)rows + 3) / 4, chunk = blockIdx.x / rb;
    const int row = (int)(blockIdx.x - chunk * rb) * 4 + wave;
    const bool active = row < rows;
    const int y = active ? row % sy : 0, z = active ? row / sy : 0;
    const T* s = src + (long long)z * sSlice + (long long)y * sRow;
    TOut* d = dst + (long long)z * dSlice + (long long)y * dRow;
    const int m = n / 2;
    const int k0 = (int)chunk * XP;
    if (active) {
        for (int q = lane; q < XP + 2 * Op::G; q += 64) {
            int g = k0 - Op::G + q;
            if (g < m + Op::G) {
                lds[wave][2 * q] = s[ext_low(g, m)];
                lds[wave][2 * q + 1] = s[m + ext_high(g, m)];
            }
        }
    }
    __syncthreads();
    if (!active) return;
    if constexpr (Op::G == 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int t = lane + 64 * h;
            int j = 2 * k0 + t;
            if (j < n) d[(long long)j * CH] = store_out<TOut>(Op::out(lds[wave] + t, t & 1));
        }
    } else {
        int k = k0 + lane;
        if (k < m) {
            T e, o;
            Op::pair_out(lds[wave] + 2 * lane, e, o);
            d[(long long)(2 * k) * CH] = store_out<TOut>(e);
            d[(long long)(2 * k + 1) * CH] = store_out<TOut>(o);
        }
    }
}

// ---- Y/Z pass (strided axis): a thread per column and segment of `seg` pairs --------------------
// Columns are numbered x first, then the other axis, so a wave reads and writes 64 consecutive elements
// a row (or, for narrow levels, several short rows).  The loads run kAhead pairs ahead of the filter.
constexpr int kAhead = 4;
struct Columns {
    int sx, n, seg, nseg;
    long long cols;                 // sx * size of the other axis
    long long aStride, oStride;     // source: along the axis, of the other one
    long long dA, dO;               // destination
    // the thread's column, segment and whether it has one
    __device__ bool place(int& x, int& other, int& k0, int& k1) const {
        const unsigned w = (unsigned)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
        const unsigned ct = (unsigned)((cols + 63) / 64);
        const int s = (int)(w / ct);
        const long long c = (long long)(w - s * ct) * 64 + (threadIdx.x & 63);
        other = cols < (1LL << 32) ? (int)((uint32_t)c / (uint32_t)sx) : (int)(c / sx);
        x = (int)(c - (long long)other * sx);
        k0 = s * seg;
        k1 = min(k0 + seg, n / 2);
        return s < nseg && c < cols;
    }
};

template <class Op, bool LO = false>
__global__ __launch_bounds__(256) void fwd_cols(typename Op::T* __restrict__ dst, const typename Op::T* __restrict__ src,
                                                Columns C) {
    using T = typename Op::T;
    constexpr int W = 2 * Op::H + 2;
    int x, other, k0, k1;
    if (!C.place(x, other, k0, k1)) return;
    const T* s = src + other * C.oStride + x;
    T* d = dst + other * C.dO + x;
    const int n = C.n, m = n / 2;
    T w[W];  // positions 2k - H .. 2k + H + 1
#pragma unroll
    for (int j = 0; j < W - 2; j++) w[j] = s[mirror1(2 * k0 - Op::H + j, n) * C.aStride];
    auto step = [&](int k, T a, T b) {
        w[W - 2] = a;
        w[W - 1] = b;
        T lo, hi;
        Op::pair(w, 0, lo, hi);
        d[k * C.dA] = lo;
        if (!LO) d[(m + k) * C.dA] = hi;
#pragma unroll
        for (int t = 0; t < W - 2; t++) w[t] = w[t + 2];
    };
    int k = k0;
    for (; k + kAhead <= k1; k += kAhead) {
        T v[2 * kAhead];
#pragma unroll
        for (int j = 0; j < 2 * kAhead; j++) v[j] = s[mirror1(2 * k + Op::H + j, n) * C.aStride];
#pragma unroll
        for (int u = 0; u < kAhead; u++) step(k + u, v[2 * u], v[2 * u + 1]);
    }
    for (; k < k1; k++) step(k, s[mirror1(2 * k + Op::H, n) * C.aStride], s[mirror1(2 * k + Op::H + 1, n) * C.aStride]);
}

// Source of a synthesis column pass: column() gives the thread's column; low(k) and high(k) load what
// is stored of its k-th lowpass and highpass coefficient, which low_value and high_value turn into the
// coefficient, so the loads of several steps can be under way before the first is looked at.
struct PlainFetch {
    template <class T>
    struct Column {
        const T* p;
        long long stride, high_at;
        __device__ T low(int k) const { return p[k * stride]; }
        __device__ T high(int k) const { return p[high_at + k * stride]; }
        __device__ T low_value(T v) const { return v; }
        __device__ T high_value(T v) const { return v; }
    };
    template <class T>
    __device__ Column<T> column(const T* src, int x, int other, const Columns& C) const {
        return Column<T>{src + x + other * C.oStride, C.aStride, C.n / 2 * C.aStride};
    }
};

// Outputs of one synthesis window: interleaved pairs u - G .. u + G -> outputs 2u, 2u + 1.
template <class Op, class T>
__device__ __forceinline__ void synth(const T* w, T& even, T& odd) {
    if constexpr (Op::G == 2) {
        even = Op::out(w, 0);
        odd = Op::out(w + 1, 1);
    } else {
        Op::pair_out(w, even, odd);
    }
}

template <class Op, class Fetch>
__global__ __launch_bounds__(256) void inv_cols(typename Op::T* __restrict__ dst, const typename Op::T* __restrict__ src,
                                                Columns C, Fetch fetch) {
    using T = typename Op::T;
    constexpr int W = 4 * Op::G + 2;
    int x, other, k0, k1;
    if (!C.place(x, other, k0, k1)) return;
    T* d = dst + other * C.dO + x;
    const int m = C.n / 2;
    const auto col = fetch.column(src, x, other, C);
    auto low = [&](int g) { return col.low(ext_low1(g, m)); };
    auto high = [&](int g) { return col.high(ext_high1(g, m)); };
    T w[W];  // interleaved pairs u - G .. u + G
    auto step = [&](int u, T a, T b) {
        w[W - 2] = a;
        w[W - 1] = b;
        T e, o;
        synth<Op>(w, e, o);
        d[2 * u * C.dA] = e;
        d[(2 * u + 1) * C.dA] = o;
#pragma unroll
        for (int t = 0; t < W - 2; t++) w[t] = w[t + 2];
    };
    decltype(low(0)) fl[2 * Op::G], vl[kAhead];
    decltype(high(0)) fh[2 * Op::G], vh[kAhead];
#pragma unroll
    for (int j = 0; j < 2 * Op::G; j++) {
        fl[j] = low(k0 - Op::G + j);
        fh[j] = high(k0 - Op::G + j);
    }
    int u = k0;
    auto load = [&] {
#pragma unroll
        for (int j = 0; j < kAhead; j++) {
            vl[j] = low(u + Op::G + j);
            vh[j] = high(u + Op::G + j);
        }
    };
    const bool batch = u + kAhead <= k1;
    if (batch) load();
#pragma unroll
    for (int j = 0; j < 2 * Op::G; j++) {
        w[2 * j] = col.low_value(fl[j]);
        w[2 * j + 1] = col.high_value(fh[j]);
    }
    if (batch) {
        for (;;) {
#pragma unroll
            for (int j = 0; j < kAhead; j++) step(u + j, col.low_value(vl[j]), col.high_value(vh[j]));
            u += kAhead;
            if (u + kAhead > k1) break;
            load();
        }
    }
    for (; u < k1; u++) step(u, col.low_value(low(u + Op::G)), col.high_value(high(u + Op::G)));
}

// The same for columns of at most kWhole samples whose source and destination share memory (a thread
// reads its whole column before it writes), and for those shorter than kLine.
constexpr int kWhole = 64;
template <class Op, bool LO = false>
__global__ __launch_bounds__(256) void fwd_cols_whole(typename Op::T* dst, const typename Op::T* src, Columns C) {
    using T = typename Op::T;
    int x, other, k0, k1;
    if (!C.place(x, other, k0, k1)) return;
    const T* s = src + other * C.oStride + x;
    T* d = dst + other * C.dO + x;
    const int n = C.n, m = n / 2;
    T v[kWhole + 2 * Op::H];
#pragma unroll
    for (int j = 0; j < kWhole + 2 * Op::H; j++)
        v[j] = j < n + 2 * Op::H ? s[mirror(j - Op::H, n) * C.aStride] : T(0);
#pragma unroll
    for (int k = 0; k < kWhole / 2; k++) {
        if (k < m) {
            T lo, hi;
            Op::pair(v, k, lo, hi);
            d[k * C.dA] = lo;
            if (!LO) d[(m + k) * C.dA] = hi;
        }
    }
}

template <class Op, class Fetch>
__global__ __launch_bounds__(256) void inv_cols_whole(typename Op::T* dst, const typename Op::T* src, Columns C,
                                                      Fetch fetch) {
    using T = typename Op::T;
    int x, other, k0, k1;
    if (!C.place(x, other, k0, k1)) return;
    T* d = dst + other * C.dO + x;
    const int m = C.n / 2;
    const auto col = fetch.column(src, x, other, C);
    T v[kWhole + 4 * Op::G];
#pragma unroll
    for (int j = 0; j < kWhole / 2 + 2 * Op::G; j++) {
        const int g = j - Op::G;
        const bool in = g < m + Op::G;
        v[2 * j] = in ? col.low_value(col.low(ext_low(g, m))) : T(0);
        v[2 * j + 1] = in ? col.high_value(col.high(ext_high(g, m))) : T(0);
    }
#pragma unroll
    for (int u = 0; u < kWhole / 2; u++) {
        if (u < m) {
            T e, o;
            synth<Op>(v + 2 * u, e, o);
            d[2 * u * C.dA] = e;
            d[(2 * u + 1) * C.dA] = o;
        }
    }
}

// ---- X and Y in one pass ------------------------------------------------------------------------
// A wave serves `per` x pairs of one z-slice (lane: one pair, with the HP halo pairs of the x filter on
// either side, which compute along and store nothing) and a segment of `seg` y pairs.  Going down the
// rows, a lane's own samples and its neighbours' (lane moves) give the x filter its window; the y
// windows stay in registers.  Against two passes by way of a buffer it saves a write and a read of the
// level (67 MB each at 256^3).
constexpr int kRowsAhead = 4;  // y pairs whose rows are loaded together
struct XYShape {
    int nx, ny, nz;
    int tiles, per, seg, nseg;
    long long dRow, dSlice, sRow, sSlice;
    __device__ bool place(int& k0, int& cnt, int& y0, int& y1, int& z) const {
        const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
        const int t = w % tiles, r = w / tiles;
        const int s = r % nseg;
        z = r / nseg;
        k0 = t * per;
        cnt = min(per, nx / 2 - k0);
        y0 = s * seg;
        y1 = min(y0 + seg, ny / 2);
        return z < nz;
    }
};
template <class T>
struct Two {
    T a, b;
};
// the previous (next) lane's pair
template <int Ctl>
__device__ __forceinline__ int lane_move(int v) {
    return __builtin_amdgcn_update_dpp(0, v, Ctl, 0xf, 0xf, false);
}
template <int Ctl>
__device__ __forceinline__ Two<float> lane_move(Two<float> p) {
    return Two<float>{__int_as_float(lane_move<Ctl>(__float_as_int(p.a))),
                      __int_as_float(lane_move<Ctl>(__float_as_int(p.b)))};
}
template <int Ctl>
__device__ __forceinline__ Two<int16_t> lane_move(Two<int16_t> p) {
    const uint32_t v = (uint32_t)lane_move<Ctl>((int)((uint32_t)(uint16_t)p.a | ((uint32_t)(uint16_t)p.b << 16)));
    return Two<int16_t>{(int16_t)(v & 0xFFFFu), (int16_t)(v >> 16)};
}
constexpr int kPrevLane = 0x138, kNextLane = 0x130;  // wave_shr:1, wave_shl:1
// pairs k - HP .. k + HP around each lane's, interleaved
template <int HP, class T>
__device__ __forceinline__ void x_window(Two<T> c, T* w) {
    Two<T> l = c, r = c;
    w[2 * HP] = c.a;
    w[2 * HP + 1] = c.b;
#pragma unroll
    for (int i = 1; i <= HP; i++) {
        l = lane_move<kPrevLane>(l);
        r = lane_move<kNextLane>(r);
        w[2 * (HP - i)] = l.a;
        w[2 * (HP - i) + 1] = l.b;
        w[2 * (HP + i)] = r.a;
        w[2 * (HP + i) + 1] = r.b;
    }
}
// two neighbouring elements (at least element-aligned)
template <class T>
__device__ __forceinline__ Two<T> load_two(const T* p) {
    Two<T> v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}

template <class Op, int CH, class TIn>
__global__ __launch_bounds__(256) void fwd_xy(typename Op::T* __restrict__ dst, const TIn* __restrict__ src, XYShape g) {
    using T = typename Op::T;
    constexpr int HP = Op::H / 2, W = 2 * Op::H + 2;
    int k0, cnt, y0, y1, z;
    if (!g.place(k0, cnt, y0, y1, z)) return;
    const int lane = threadIdx.x & 63, mx = g.nx / 2, my = g.ny / 2;
    const int gp = min(k0 - HP + lane, mx + HP - 1);  // this lane's x pair, past the ends: its reflection
    const int xa = mirror1(2 * gp, g.nx), xb = mirror1(2 * gp + 1, g.nx);
    const bool out = lane >= HP && lane < HP + cnt;
    const TIn* s = src + z * g.sSlice;
    auto row = [&](int p) -> Two<T> {
        const TIn* q = s + mirror1(p, g.ny) * g.sRow;
        if constexpr (CH == 1 && std::is_same<TIn, T>::value) {  // the two samples are neighbours, in either order
            const Two<T> v = load_two(q + min(xa, xb));
            return xa < xb ? v : Two<T>{v.b, v.a};
        } else {
            return Two<T>{load_in(q[(long long)xa * CH]), load_in(q[(long long)xb * CH])};
        }
    };
    T* d = dst + z * g.dSlice + gp;
    T wl[W], wh[W];  // y windows of the columns gp and mx + gp: rows 2k - H .. 2k + H + 1
    auto filter_x = [&](Two<T> v, T& lo, T& hi) {
        T w[4 * HP + 2];
        x_window<HP>(v, w);
        Op::pair(w, 0, lo, hi);
    };
    {
        Two<T> v[W - 2];
#pragma unroll
        for (int j = 0; j < W - 2; j++) v[j] = row(2 * y0 - Op::H + j);
#pragma unroll
        for (int j = 0; j < W - 2; j++) filter_x(v[j], wl[j], wh[j]);
    }
    auto step = [&](int k, Two<T> a, Two<T> b) {
        filter_x(a, wl[W - 2], wh[W - 2]);
        filter_x(b, wl[W - 1], wh[W - 1]);
        T l0, h0, l1, h1;
        Op::pair(wl, 0, l0, h0);
        Op::pair(wh, 0, l1, h1);
        if (out) {
            T* r0 = d + k * g.dRow;
            T* r1 = d + (my + k) * g.dRow;
            r0[0] = l0;
            r0[mx] = l1;
            r1[0] = h0;
            r1[mx] = h1;
        }
#pragma unroll
        for (int t = 0; t < W - 2; t++) {
            wl[t] = wl[t + 2];
            wh[t] = wh[t + 2];
        }
    };
    int k = y0;
    for (; k + kRowsAhead <= y1; k += kRowsAhead) {
        Two<T> v[2 * kRowsAhead];
#pragma unroll
        for (int j = 0; j < 2 * kRowsAhead; j++) v[j] = row(2 * k + Op::H + j);
#pragma unroll
        for (int u = 0; u < kRowsAhead; u++) step(k + u, v[2 * u], v[2 * u + 1]);
    }
    for (; k < y1; k++) step(k, row(2 * k + Op::H), row(2 * k + Op::H + 1));
}

template <class Op, int CH, class TOut>
__global__ __launch_bounds__(256) void inv_yx(TOut* __restrict__ dst, const typename Op::T* __restrict__ src, XYShape g) {
    using T = typename Op::T;
    constexpr int HP = Op::G, W = 4 * Op::G + 2;
    int k0, cnt, y0, y1, z;
    if (!g.place(k0, cnt, y0, y1, z)) return;
    const int lane = threadIdx.x & 63, mx = g.nx / 2, my = g.ny / 2;
    const int gp = min(k0 - HP + lane, mx + HP - 1);
    const int xl = ext_low1(gp, mx), xh = mx + ext_high1(gp, mx);
    const bool out = lane >= HP && lane < HP + cnt;
    const T* s = src + z * g.sSlice;
    // y row q's low and high x coefficients
    auto row = [&](int q) -> Two<T> {
        const T* r = s + q * g.sRow;
        return Two<T>{r[xl], r[xh]};
    };
    auto lo_row = [&](int k) { return row(ext_low1(k, my)); };
    auto hi_row = [&](int k) { return row(my + ext_high1(k, my)); };
    TOut* d = dst + z * g.dSlice + (long long)2 * gp * CH;
    T wl[W], wh[W];  // interleaved y pairs u - G .. u + G of the two columns
    {
        Two<T> a[2 * Op::G], b[2 * Op::G];
#pragma unroll
        for (int j = 0; j < 2 * Op::G; j++) {
            a[j] = lo_row(y0 - Op::G + j);
            b[j] = hi_row(y0 - Op::G + j);
        }
#pragma unroll
        for (int j = 0; j < 2 * Op::G; j++) {
            wl[2 * j] = a[j].a;
            wl[2 * j + 1] = b[j].a;
            wh[2 * j] = a[j].b;
            wh[2 * j + 1] = b[j].b;
        }
    }
    auto emit = [&](int y, T lo, T hi) {
        T w[4 * HP + 2], e, o;
        x_window<HP>(Two<T>{lo, hi}, w);
        synth<Op>(w, e, o);
        if (!out) return;
        TOut* r = d + y * g.dRow;
        if constexpr (CH == 1 && std::is_same<TOut, T>::value) {
            const Two<TOut> v{store_out<TOut>(e), store_out<TOut>(o)};
            __builtin_memcpy(r, &v, sizeof(v));
        } else {
            r[0] = store_out<TOut>(e);
            r[CH] = store_out<TOut>(o);
        }
    };
    auto step = [&](int u, Two<T> lo, Two<T> hi) {
        wl[W - 2] = lo.a;
        wl[W - 1] = hi.a;
        wh[W - 2] = lo.b;
        wh[W - 1] = hi.b;
        T el, ol, eh, oh;
        synth<Op>(wl, el, ol);
        synth<Op>(wh, eh, oh);
        emit(2 * u, el, eh);
        emit(2 * u + 1, ol, oh);
#pragma unroll
        for (int t = 0; t < W - 2; t++) {
            wl[t] = wl[t + 2];
            wh[t] = wh[t + 2];
        }
    };
    int u = y0;
    for (; u + kRowsAhead <= y1; u += kRowsAhead) {
        Two<T> a[kRowsAhead], b[kRowsAhead];
#pragma unroll
        for (int j = 0; j < kRowsAhead; j++) {
            a[j] = lo_row(u + Op::G + j);
            b[j] = hi_row(u + Op::G + j);
        }
#pragma unroll
        for (int j = 0; j < kRowsAhead; j++) step(u + j, a[j], b[j]);
    }
    for (; u < y1; u++) step(u, lo_row(u + Op::G), hi_row(u + Op::G));
}

// Fused dequantize + first synthesis pass of dwtFloat{2D,3D}InverseFromSymbols
// (src/cudaCompress/util/DWTFloatFromSymbolsKernels.cui:19-464): octant b = bx + 2by (+ 4bz)
// comes from the lowpass array when b == 0, else from dense symbol band hp[b-1], dequantized
// with the deadzone rule (src/cudaCompress/util/Quantize.cuh:103-110).
template <typename S>
struct SymbolFetch {
    const float* lp;
    const S* const* hp;
    long long lpRow, lpSlice;
    int hx, hy, hz;  // half sizes
    int is3d;
    float step;
    __device__ float deq(uint32_t sym) const {
        uint32_t neg = sym & 1u;
        int q = (int)((1u - 2u * neg) * ((sym + neg) / 2u));
        float sg = q < 0 ? -1.0f : (q > 0 ? 1.0f : 0.0f);
        return (float(q) + sg * 0.5f) * step;
    }
    // pointers that were read from memory: said to be global, or every load would go by the flat path
    using Symbols = const __attribute__((address_space(1))) S*;
    struct Column {
        // both are loaded (the one that is not meant, at an address that is at hand) and one is taken:
        // a branch would have every load waited for
        struct Low {
            float lp;
            S sym;
        };
        const SymbolFetch* f;
        bool from_lp;
        const float* lp;
        Symbols lo, hi;
        long long lp_stride, stride;
        __device__ Low low(int k) const { return Low{lp[k * lp_stride], lo[k * stride]}; }
        __device__ S high(int k) const { return hi[k * stride]; }
        __device__ float low_value(Low v) const { return from_lp ? v.lp : f->deq((uint32_t)v.sym); }
        __device__ float high_value(S v) const { return f->deq((uint32_t)v); }
    };
    __device__ Column column(const float*, int x, int other, const Columns&) const {
        const int y = is3d ? other : 0;
        const int bx = x >= hx, by = y >= hy, b = bx + 2 * by;
        const long long at = (long long)(y - by * hy) * hx + (x - bx * hx);
        Column c;
        c.f = this;
        c.from_lp = b == 0;
        c.lp = b == 0 ? lp + x + y * lpRow : lp;
        c.hi = (Symbols)hp[b + (is3d ? 3 : 1)] + at;
        c.lo = b == 0 ? c.hi : (Symbols)hp[b - 1] + at;
        c.lp_stride = b ? 0 : is3d ? lpSlice : lpRow;
        c.stride = is3d ? (long long)hx * hy : hx;
        return c;
    }
};

inline dim3 x_grid(int rows, int n) { return dim3(div_up(rows, 4) * div_up(n / 2, XP)); }

// Pairs a wave takes along its streaming axis: long segments read the filter's halo (4 pairs) less
// often, but a level of few columns needs short ones to fill the chip (4096 waves: 4 a SIMD).
// `columns`: waves a segment.
int segment_pairs(int m, long long columns) {
    int seg = 32;
    while (seg > 8 && columns * div_up(m, seg) < 4096) seg /= 2;
    return seg;
}
Columns columns_of(int sx, int n, int other, long long aStride, long long oStride, long long dA, long long dO) {
    Columns C{sx, n, 0, 0, (long long)sx * other, aStride, oStride, dA, dO};
    C.seg = segment_pairs(n / 2, (C.cols + 63) / 64);
    C.nseg = (int)div_up(n / 2, C.seg);
    return C;
}
dim3 columns_grid(const Columns& C) { return dim3(div_up((C.cols + 63) / 64 * C.nseg, 4)); }
// hp: halo pairs of the x filter
XYShape xy_shape(int hp, int nx, int ny, int nz, long long dRow, long long dSlice, long long sRow, long long sSlice) {
    XYShape g{nx, ny, nz, 0, 0, 0, 0, dRow, dSlice, sRow, sSlice};
    const int most = 64 - 2 * hp;
    g.tiles = (int)div_up(nx / 2, most);
    g.per = (int)div_up(nx / 2, g.tiles);
    g.seg = segment_pairs(ny / 2, (long long)g.tiles * nz);
    g.nseg = (int)div_up(ny / 2, g.seg);
    return g;
}
dim3 xy_grid(const XYShape& g) { return dim3(div_up((uint64_t)g.tiles * g.nseg * g.nz, 4)); }

// Bytes [first, last) that a pitched array of `elem`-byte elements spans.
struct Span {
    uintptr_t lo, hi;
    Span(const void* p, long long sx, long long sy, long long sz, long long row, long long slice, size_t elem)
        : lo((uintptr_t)p), hi((uintptr_t)p + elem * (size_t)((sz - 1) * slice + (sy - 1) * row + sx)) {}
    bool meets(const Span& o) const { return lo < o.hi && o.lo < hi; }
};
// The fused pass needs rows and columns of at least kLine samples (neighbouring samples stay neighbours) and output that does not meet its input.
bool xy_fits(int sx, int sy, const Span& in, const Span& out) { return sx >= kLine && sy >= kLine && !in.meets(out); }

// A column pass.  The streaming kernels write while they read, so a pass within one array takes the
// kernel that reads a column first, as far as one holds it.
template <class Op, bool LO = false>
void forward_columns(const char* name, uint64_t bytes, typename Op::T* dst, const typename Op::T* src, Columns C,
                     hipStream_t st) {
    const size_t elem = sizeof(typename Op::T);
    const long long others = C.cols / C.sx;
    const bool meets = Span(src, C.sx, C.n, others, C.aStride, C.oStride, elem)
                           .meets(Span(dst, C.sx, LO ? C.n / 2 : C.n, others, C.dA, C.dO, elem));
    if (C.n < kLine || (C.n <= kWhole && meets)) {
        C.seg = C.n / 2, C.nseg = 1;
        CCA_LAUNCH(name, bytes, (fwd_cols_whole<Op, LO>), columns_grid(C), dim3(256), 0, st, dst, src, C);
    } else {
        CCA_LAUNCH(name, bytes, (fwd_cols<Op, LO>), columns_grid(C), dim3(256), 0, st, dst, src, C);
    }
    CCA_LAUNCH_CHECK();
}
template <class Op, class Fetch>
void inverse_columns(const char* name, uint64_t bytes, typename Op::T* dst, const typename Op::T* src, Columns C,
                     Fetch fetch, const Span& in, hipStream_t st) {
    const bool meets = in.meets(Span(dst, C.sx, C.n, C.cols / C.sx, C.dA, C.dO, sizeof(typename Op::T)));
    if (C.n < kLine || (C.n <= kWhole && meets)) {
        C.seg = C.n / 2, C.nseg = 1;
        CCA_LAUNCH(name, bytes, (inv_cols_whole<Op, Fetch>), columns_grid(C), dim3(256), 0, st, dst, src, C, fetch);
    } else {
        CCA_LAUNCH(name, bytes, (inv_cols<Op, Fetch>), columns_grid(C), dim3(256), 0, st, dst, src, C, fetch);
    }
    CCA_LAUNCH_CHECK();
}
template <class Op>
void inverse_columns(const char* name, uint64_t bytes, typename Op::T* dst, const typename Op::T* src, const Columns& C,
                     hipStream_t st) {
    inverse_columns<Op>(name, bytes, dst, src, C, PlainFetch{},
                        Span(src, C.sx, C.n, C.cols / C.sx, C.aStride, C.oStride, sizeof(typename Op::T)), st);
}

void check_dims(int sx, int sy, int sz) {
    CCA_REQUIRE(sx >= 2 && sy >= 2 && sz >= 1, CC_ERR_INVALID_ARG, "DWT sizes must be >= 2 (sizeZ >= 1)");
    CCA_REQUIRE(sx % 2 == 0 && sy % 2 == 0 && (sz == 1 || sz % 2 == 0), CC_ERR_INVALID_ARG,
                "DWT sizes must be even");
    CCA_REQUIRE(sz <= 65535, CC_ERR_INVALID_ARG, "sizeZ too large for the launch grid");
}

template <int CH, bool LO = false, class TIn>
void launch_fwd97_x(float* dst, const TIn* src, int sx, int sy, int sz, int dRow, int dSlice, int sRow, int sSlice,
                    hipStream_t st) {
    const uint64_t bytes = (uint64_t)sx * sy * sz * (sizeof(TIn) + (LO ? 2 : 4));
    CCA_LAUNCH("dwt97_fwd_x", bytes, (fwd_x<Fwd97, CH, TIn, LO>), x_grid(sy * sz, sx), dim3(256), 0, st, dst, src, sx,
               sy * sz, sy, dRow, dSlice, sRow, sSlice);
}
template <int CH, class TOut>
void launch_inv97_x(TOut* dst, const float* src, int sx, int sy, int sz, int dRow, int dSlice, int sRow, int sSlice,
                    hipStream_t st) {
    CCA_LAUNCH("dwt97_inv_x", (uint64_t)sx * sy * sz * (4 + sizeof(TOut)), (inv_x<Inv97, CH, TOut>), x_grid(sy * sz, sx),
               dim3(256), 0, st, dst, src, sx, sy * sz, sy, dRow, dSlice, sRow, sSlice);
}
template <bool LO = false, class TIn>
void launch_fwd97_x_ch(int ch, float* dst, const TIn* src, int sx, int sy, int sz, int dRow, int dSlice, int sRow,
                       int sSlice, hipStream_t st) {
    switch (ch) {
        case 1: launch_fwd97_x<1, LO>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        case 2: launch_fwd97_x<2, LO>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        case 3: launch_fwd97_x<3, LO>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        default: launch_fwd97_x<4, LO>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
    }
}
template <class TOut>
void launch_inv97_x_ch(int ch, TOut* dst, const float* src, int sx, int sy, int sz, int dRow, int dSlice, int sRow,
                       int sSlice, hipStream_t st) {
    switch (ch) {
        case 1: launch_inv97_x<1>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        case 2: launch_inv97_x<2>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        case 3: launch_inv97_x<3>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
        default: launch_inv97_x<4>(dst, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st); break;
    }
}

// f(integral constant of the channel count)
template <class F>
void by_channels(int ch, F f) {
    switch (ch) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        default: f(std::integral_constant<int, 4>{}); break;
    }
}

// dwtFloatForward<T> (src/cudaCompress/util/DWTFloat.cu:85-201) for float and byte sources.
template <class TIn>
void dwt97_forward_t(float* dst, float* buf2, float* buf1, const TIn* src, int sx, int sy, int sz, int ch, int dRow,
                     int dSlice, int sRow, int sSlice, hipStream_t st);
// dwtFloatInverse<T> (DWTFloat.cu:233-322) for float and byte destinations.
template <class TOut>
void dwt97_inverse_t(TOut* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int ch, int dRow,
                     int dSlice, int sRow, int sSlice, hipStream_t st);
// dwtFloatInverseFromSymbols<T> (DWTFloat.cu:326-463) for float and byte destinations.
template <class TOut>
void dwt97_inverse_from_symbols_t(TOut* dst, float* buf2, float* buf1, const float* lowpass,
                                  const void* const* dd_highpass, int symbolSize, float step, int sx, int sy, int sz,
                                  int ch, int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st);

}  // namespace

void dwt97_forward(float* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int ch, int dRow,
                   int dSlice, int sRow, int sSlice, hipStream_t st) {
    dwt97_forward_t(dst, buf2, buf1, src, sx, sy, sz, ch, dRow, dSlice, sRow, sSlice, st);
}
void dwt97_forward_from_byte(float* dst, float* buf2, float* buf1, const uint8_t* src, int sx, int sy, int sz, int ch,
                             int dRow, int dSlice, int sRow, int sSlice, hipStream_t st) {
    dwt97_forward_t(dst, buf2, buf1, src, sx, sy, sz, ch, dRow, dSlice, sRow, sSlice, st);
}
void dwt97_inverse(float* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int ch, int dRow,
                   int dSlice, int sRow, int sSlice, hipStream_t st) {
    dwt97_inverse_t(dst, buf2, buf1, src, sx, sy, sz, ch, dRow, dSlice, sRow, sSlice, st);
}
void dwt97_inverse_to_byte(uint8_t* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int ch,
                           int dRow, int dSlice, int sRow, int sSlice, hipStream_t st) {
    dwt97_inverse_t(dst, buf2, buf1, src, sx, sy, sz, ch, dRow, dSlice, sRow, sSlice, st);
}
void dwt97_inverse_from_symbols(float* dst, float* buf2, float* buf1, const float* lowpass,
                                const void* const* dd_highpass, int symbolSize, float step, int sx, int sy, int sz,
                                int ch, int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st) {
    dwt97_inverse_from_symbols_t(dst, buf2, buf1, lowpass, dd_highpass, symbolSize, step, sx, sy, sz, ch, dRow, dSlice,
                                 lpRow, lpSlice, st);
}
void dwt97_inverse_from_symbols_to_byte(uint8_t* dst, float* buf2, float* buf1, const float* lowpass,
                                        const void* const* dd_highpass, float step, int sx, int sy, int sz, int ch,
                                        int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st) {
    dwt97_inverse_from_symbols_t(dst, buf2, buf1, lowpass, dd_highpass, 2, step, sx, sy, sz, ch, dRow, dSlice, lpRow,
                                 lpSlice, st);
}

// One level of the 9/7 analysis at double precision (no reference counterpart; the FP64 twin of
// dwtFloat3DForward / dwtFloat2DForward used to state the FP32 transform's error).  dst and src
// share the row and slice pitches and must not overlap.  3D: X src -> dst, Y dst -> buf,
// Z buf -> dst; 2D: X src -> buf, Y buf -> dst.
void dwt97_forward_f64(double* dst, double* buf, const double* src, int sx, int sy, int sz, int row, int slice,
                       hipStream_t st) {
    check_dims(sx, sy, sz);
    CCA_REQUIRE(dst && buf && src, CC_ERR_INVALID_ARG, "null DWT buffer");
    if (row <= 0) row = sx;
    if (slice <= 0) slice = sy * row;
    CCA_REQUIRE(row >= sx && slice >= sy * row, CC_ERR_INVALID_ARG, "pitches smaller than the level");
    const bool do3d = sz > 1;
    const uint64_t bytes = (uint64_t)sx * sy * sz * 16;
    double* xdst = do3d ? dst : buf;
    CCA_LAUNCH("dwt97d_fwd_x", bytes, (fwd_x<Fwd97d, 1>), x_grid(sy * sz, sx), dim3(256), 0, st, xdst, src, sx, sy * sz,
               sy, row, slice, row, slice);
    CCA_LAUNCH_CHECK();
    const Columns Y = columns_of(sx, sy, sz, row, slice, row, slice);
    forward_columns<Fwd97d>("dwt97d_fwd_y", bytes, do3d ? buf : dst, xdst, Y, st);
    if (do3d) {
        const Columns Z = columns_of(sx, sz, sy, slice, row, slice, row);
        forward_columns<Fwd97d>("dwt97d_fwd_z", bytes, dst, buf, Z, st);
    }
}

// dwtFloat2DForwardLowpassOnlyFromByte (DWTFloat.cu:18-81, :535-552; kernels in
// src/cudaCompress/util/DWTFloat2DLowpassKernels.cui): the X pass writes only the row lowpass
// halves to buf (row pitch dRow), the Y pass only the column lowpass halves to dst.  The sums are
// the same fmaf chains as the full transform, so dst equals its LL band.
void dwt97_forward_lowpass_only_from_byte(float* dst, float* buf, const uint8_t* src, int sx, int sy, int ch,
                                          int dRow, int sRow, hipStream_t st) {
    check_dims(sx, sy, 1);
    CCA_REQUIRE(ch >= 1 && ch <= 4, CC_ERR_INVALID_ARG, "srcChannelCount must be 1..4");
    CCA_REQUIRE(dst && buf && src, CC_ERR_INVALID_ARG, "null DWT buffer");
    if (dRow <= 0) dRow = sx / 2;
    if (sRow <= 0) sRow = sx * ch;
    CCA_REQUIRE(dRow >= sx / 2, CC_ERR_INVALID_ARG, "dstRowPitch must be >= sizeX / 2");
    launch_fwd97_x_ch<true>(ch, buf, src, sx, sy, 1, dRow, 0, sRow, 0, st);
    CCA_LAUNCH_CHECK();
    const Columns Y = columns_of(sx / 2, sy, 1, dRow, 0, dRow, 0);
    forward_columns<Fwd97, true>("dwt97_fwd_y_lowpass", (uint64_t)sx / 2 * sy * 6, dst, buf, Y, st);
}

// dwtIntForwardLowpassOnly (src/cudaCompress/util/DWTInt.cu:16-76, kernels in
// DWTInt2DLowpassKernels.cui): the LL band of the 2D 5/3 transform.  The reference launches
// only whole 512-column and 64-row tiles; every even size is computed here, identical where the
// reference computes.
void dwt53_forward_lowpass_only(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int dRow, int sRow,
                                hipStream_t st) {
    check_dims(sx, sy, 1);
    CCA_REQUIRE(dst && buf && src, CC_ERR_INVALID_ARG, "null DWT buffer");
    if (dRow <= 0) dRow = sx / 2;
    if (sRow <= 0) sRow = sx;
    CCA_REQUIRE(dRow >= sx / 2, CC_ERR_INVALID_ARG, "dstRowPitch must be >= sizeX / 2");
    CCA_LAUNCH("dwt53_fwd_x_lowpass", (uint64_t)sx * sy * 3, (fwd_x<Fwd53, 1, int16_t, true>), x_grid(sy, sx), dim3(256), 0,
               st, buf, src, sx, sy, sy, dRow, 0, sRow, 0);
    CCA_LAUNCH_CHECK();
    const Columns Y = columns_of(sx / 2, sy, 1, dRow, 0, dRow, 0);
    forward_columns<Fwd53, true>("dwt53_fwd_y_lowpass", (uint64_t)sx / 2 * sy * 3, dst, buf, Y, st);
}

namespace {

template <class TIn>
void dwt97_forward_t(float* dst, float* buf2, float* buf1, const TIn* src, int sx, int sy, int sz, int ch, int dRow,
                     int dSlice, int sRow, int sSlice, hipStream_t st) {
    check_dims(sx, sy, sz);
    CCA_REQUIRE(ch >= 1 && ch <= 4, CC_ERR_INVALID_ARG, "srcChannelCount must be 1..4");
    if (dRow <= 0) dRow = sx;
    if (dSlice <= 0) dSlice = sy * dRow;
    if (sRow <= 0) sRow = sx * ch;
    if (sSlice <= 0) sSlice = sy * sRow;
    const bool do3d = sz > 1;
    CCA_REQUIRE(dst && buf1 && src && (!do3d || buf2), CC_ERR_INVALID_ARG, "null DWT buffer");
    // X: src -> buf1, Y: buf1 -> (3D ? buf2 : dst), Z: buf2 -> dst (DWTFloat.cu:113-201); fused: X and Y
    // src -> (3D ? buf2 : dst)
    float* ydst = do3d ? buf2 : dst;
    const Span in(src, (long long)sx * ch, sy, sz, sRow, sSlice, sizeof(TIn)), mid(ydst, sx, sy, sz, dRow, dSlice, 4);
    if (xy_fits(sx, sy, in, mid)) {
        const XYShape g = xy_shape(Fwd97::H / 2, sx, sy, sz, dRow, dSlice, sRow, sSlice);
        by_channels(ch, [&](auto c) {
            CCA_LAUNCH("dwt97_fwd_xy", (uint64_t)sx * sy * sz * (sizeof(TIn) + 4), (fwd_xy<Fwd97, decltype(c)::value, TIn>),
                       xy_grid(g), dim3(256), 0, st, ydst, src, g);
        });
    } else {
        launch_fwd97_x_ch(ch, buf1, src, sx, sy, sz, dRow, dSlice, sRow, sSlice, st);
        CCA_LAUNCH_CHECK();
        const Columns Y = columns_of(sx, sy, sz, dRow, dSlice, dRow, dSlice);
        forward_columns<Fwd97>("dwt97_fwd_y", (uint64_t)sx * sy * sz * 8, ydst,
                   buf1, Y, st);
    }
    CCA_LAUNCH_CHECK();
    if (do3d) {
        const Columns Z = columns_of(sx, sz, sy, dSlice, dRow, dSlice, dRow);
        forward_columns<Fwd97>("dwt97_fwd_z", (uint64_t)sx * sy * sz * 8, dst,
                   buf2, Z, st);
    }
}

// Y and X synthesis of src (pitches sRow, sSlice) to dst: fused, or by way of buf1.
template <class TOut>
void inverse97_yx(TOut* dst, float* buf1, const float* src, int sx, int sy, int sz, int ch, int dRow, int dSlice,
                  long long sRow, long long sSlice, hipStream_t st) {
    const Span in(src, sx, sy, sz, sRow, sSlice, 4), to(dst, (long long)sx * ch, sy, sz, dRow, dSlice, sizeof(TOut));
    if (xy_fits(sx, sy, in, to)) {
        const XYShape g = xy_shape(Inv97::G, sx, sy, sz, dRow, dSlice, sRow, sSlice);
        by_channels(ch, [&](auto c) {
            CCA_LAUNCH("dwt97_inv_yx", (uint64_t)sx * sy * sz * (4 + sizeof(TOut)),
                       (inv_yx<Inv97, decltype(c)::value, TOut>), xy_grid(g), dim3(256), 0, st, dst, src, g);
        });
    } else {
        const Columns Y = columns_of(sx, sy, sz, sRow, sSlice, sRow, sSlice);
        inverse_columns<Inv97>("dwt97_inv_y", (uint64_t)sx * sy * sz * 8, buf1, src, Y, st);
        launch_inv97_x_ch(ch, dst, buf1, sx, sy, sz, dRow, dSlice, (int)sRow, (int)sSlice, st);
    }
    CCA_LAUNCH_CHECK();
}

template <class TOut>
void dwt97_inverse_t(TOut* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int ch, int dRow,
                     int dSlice, int sRow, int sSlice, hipStream_t st) {
    check_dims(sx, sy, sz);
    CCA_REQUIRE(ch >= 1 && ch <= 4, CC_ERR_INVALID_ARG, "dstChannelCount must be 1..4");
    if (dRow <= 0) dRow = sx * ch;
    if (dSlice <= 0) dSlice = sy * dRow;
    if (sRow <= 0) sRow = sx;
    if (sSlice <= 0) sSlice = sy * sRow;
    const bool do3d = sz > 1;
    CCA_REQUIRE(dst && buf1 && src && (!do3d || buf2), CC_ERR_INVALID_ARG, "null DWT buffer");
    // Z: src -> buf2, Y: (3D ? buf2 : src) -> buf1, X: buf1 -> dst (DWTFloat.cu:233-322); fused: Y and X
    // (3D ? buf2 : src) -> dst
    if (do3d) {
        const Columns Z = columns_of(sx, sz, sy, sSlice, sRow, sSlice, sRow);
        inverse_columns<Inv97>("dwt97_inv_z", (uint64_t)sx * sy * sz * 8, buf2, src, Z, st);
    }
    inverse97_yx(dst, buf1, do3d ? buf2 : src, sx, sy, sz, ch, dRow, dSlice, sRow, sSlice, st);
}

template <class TOut>
void dwt97_inverse_from_symbols_t(TOut* dst, float* buf2, float* buf1, const float* lowpass,
                                  const void* const* dd_highpass, int symbolSize, float step, int sx, int sy, int sz,
                                  int ch, int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st) {
    check_dims(sx, sy, sz);
    CCA_REQUIRE(ch >= 1 && ch <= 4, CC_ERR_INVALID_ARG, "dstChannelCount must be 1..4");
    CCA_REQUIRE(symbolSize == 2 || symbolSize == 4, CC_ERR_INVALID_ARG, "symbolSize must be 2 or 4");
    if (dRow <= 0) dRow = sx * ch;
    if (dSlice <= 0) dSlice = sy * dRow;
    if (lpRow <= 0) lpRow = sx;
    if (lpSlice <= 0) lpSlice = sy * lpRow;
    const bool do3d = sz > 1;
    CCA_REQUIRE(dst && buf1 && lowpass && dd_highpass && (!do3d || buf2), CC_ERR_INVALID_ARG, "null DWT buffer");
    // buffers are dense with pitch sizeX (DWTFloat.cu:355-356)
    const long long bRow = sx, bSlice = (long long)sx * sy;
    const uint64_t n = (uint64_t)sx * sy * sz;
    auto run = [&](auto sym) {
        using S = decltype(sym);
        const SymbolFetch<S> fetch{lowpass, (const S* const*)dd_highpass, lpRow, lpSlice, sx / 2, sy / 2, sz / 2,
                                   do3d ? 1 : 0, step};
        if (do3d) {
            const Columns Z = columns_of(sx, sz, sy, 0, 0, bSlice, bRow);
            inverse_columns<Inv97>("dwt97_inv_z_from_symbols", n / 8 * 4 + n / 8 * 7 * symbolSize + n * 4, buf2, lowpass, Z,
                                   fetch, Span(lowpass, sx / 2, sy / 2, sz / 2, lpRow, lpSlice, 4), st);
            inverse97_yx(dst, buf1, buf2, sx, sy, sz, ch, dRow, dSlice, bRow, bSlice, st);
            return;
        }
        // 2D: the symbols may lie in dst, so they are all read before the first row of it is written
        const Columns Y = columns_of(sx, sy, 1, 0, 0, bRow, bSlice);
        inverse_columns<Inv97>("dwt97_inv_y_from_symbols", n / 4 * 4 + n / 4 * 3 * symbolSize + n * 4, buf1, lowpass, Y,
                               fetch, Span(lowpass, sx / 2, sy / 2, 1, lpRow, 0, 4), st);
        launch_inv97_x_ch(ch, dst, buf1, sx, sy, sz, dRow, dSlice, (int)bRow, (int)bSlice, st);
        CCA_LAUNCH_CHECK();
    };
    if (symbolSize == 2) run(uint16_t{});
    else run(uint32_t{});
}

}  // namespace

void dwt53_forward(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int sz, int dRow, int dSlice,
                   int sRow, int sSlice, hipStream_t st) {
    check_dims(sx, sy, sz);
    if (dRow <= 0) dRow = sx;
    if (dSlice <= 0) dSlice = sy * dRow;
    if (sRow <= 0) sRow = sx;
    if (sSlice <= 0) sSlice = sy * sRow;
    CCA_REQUIRE(dst && buf && src, CC_ERR_INVALID_ARG, "null DWT buffer");
    const bool do3d = sz > 1;
    // X: src -> (3D ? dst : buf), Y: -> (3D ? buf : dst), Z: buf -> dst (DWTInt.cu:106-186); fused: X and
    // Y src -> (3D ? buf : dst)
    int16_t* xdst = do3d ? dst : buf;
    int16_t* ydst = do3d ? buf : dst;
    const uint64_t n = (uint64_t)sx * sy * sz;
    if (xy_fits(sx, sy, Span(src, sx, sy, sz, sRow, sSlice, 2), Span(ydst, sx, sy, sz, dRow, dSlice, 2))) {
        const XYShape g = xy_shape(Fwd53::H / 2, sx, sy, sz, dRow, dSlice, sRow, sSlice);
        CCA_LAUNCH("dwt53_fwd_xy", n * 4, (fwd_xy<Fwd53, 1, int16_t>), xy_grid(g), dim3(256), 0, st, ydst, src, g);
    } else {
        CCA_LAUNCH("dwt53_fwd_x", n * 4, (fwd_x<Fwd53, 1>), x_grid(sy * sz, sx), dim3(256), 0, st, xdst, src, sx, sy * sz,
                   sy, dRow, dSlice, sRow, sSlice);
        CCA_LAUNCH_CHECK();
        const Columns Y = columns_of(sx, sy, sz, dRow, dSlice, dRow, dSlice);
        forward_columns<Fwd53>("dwt53_fwd_y", n * 4, ydst, xdst, Y, st);
    }
    CCA_LAUNCH_CHECK();
    if (do3d) {
        const Columns Z = columns_of(sx, sz, sy, dSlice, dRow, dSlice, dRow);
        forward_columns<Fwd53>("dwt53_fwd_z", n * 4, dst, buf, Z, st);
    }
}

void dwt53_inverse(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int sz, int dRow, int dSlice,
                   int sRow, int sSlice, hipStream_t st) {
    check_dims(sx, sy, sz);
    if (dRow <= 0) dRow = sx;
    if (dSlice <= 0) dSlice = sy * dRow;
    if (sRow <= 0) sRow = sx;
    if (sSlice <= 0) sSlice = sy * sRow;
    CCA_REQUIRE(dst && buf && src, CC_ERR_INVALID_ARG, "null DWT buffer");
    const bool do3d = sz > 1;
    // Z: src -> dst, Y: (3D ? dst : src) -> buf, X: buf -> dst (DWTInt.cu:218-316), src pitches
    // for the intermediate buffers; fused: Z src -> buf, Y and X (3D ? buf : src) -> dst
    const uint64_t n = (uint64_t)sx * sy * sz;
    const Span from(src, sx, sy, sz, sRow, sSlice, 2), to(dst, sx, sy, sz, dRow, dSlice, 2);
    const Span mid(do3d ? buf : src, sx, sy, sz, sRow, sSlice, 2);
    if (xy_fits(sx, sy, mid, to) && (!do3d || !mid.meets(from))) {
        if (do3d) {
            const Columns Z = columns_of(sx, sz, sy, sSlice, sRow, sSlice, sRow);
            inverse_columns<Inv53>("dwt53_inv_z", n * 4, buf, src, Z, st);
        }
        const XYShape g = xy_shape(Inv53::G, sx, sy, sz, dRow, dSlice, sRow, sSlice);
        CCA_LAUNCH("dwt53_inv_yx", n * 4, (inv_yx<Inv53, 1, int16_t>), xy_grid(g), dim3(256), 0, st, dst, do3d ? buf : src,
                   g);
        CCA_LAUNCH_CHECK();
        return;
    }
    if (do3d) {
        const Columns Z = columns_of(sx, sz, sy, sSlice, sRow, sSlice, sRow);
        inverse_columns<Inv53>("dwt53_inv_z", n * 4, dst, src, Z, st);
    }
    const int16_t* ysrc = do3d ? dst : src;
    const Columns Y = columns_of(sx, sy, sz, sRow, sSlice, sRow, sSlice);
    inverse_columns<Inv53>("dwt53_inv_y", n * 4, buf, ysrc, Y, st);
    CCA_LAUNCH("dwt53_inv_x", n * 4, (inv_x<Inv53, 1>), x_grid(sy * sz, sx), dim3(256), 0, st, dst, buf, sx, sy * sz, sy,
               dRow, dSlice, sRow, sSlice);
    CCA_LAUNCH_CHECK();
}

}  // namespace cca
