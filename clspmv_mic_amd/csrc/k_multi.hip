// Multi-right-hand-side SpMV for gfx950: Y[:, q] += A X[:, q] for q < k
// (k <= 16) in one pass over the matrix, for DIA and CSR.
//
// X is row-major (the k values of column c are X[c*k .. c*k+k)), so the
// gather of one column brings every right-hand side's value in one or a few
// 16-byte loads: a random column costs one cache line for all k products
// instead of one line per product.  CSR runs over row blocks
// (a work-group per block of short rows or per long row).  Y is
// column-major (ldy), so each right-hand side's y stays a contiguous
// vector.  Matrix values may be FP32 or 16-bit (widened on load); sums are
// FP32 in a fixed order, FP64 for CSR rows longer than kLongRowF64; no
// atomics.

#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace clspmv {
namespace {

using namespace dev;
using launch::kDiaRun;

// Loads right-hand sides qb .. qb+Q-1 of row c of X (zero where q >= k).
template <int Q>
__device__ __forceinline__ void load_xq(const float* __restrict__ X, int c, int k, int qb, bool vec,
                                        float* xv) {
    const float* p = X + (size_t)c * k + qb;
    if (qb >= k) {  // a lane quad past k (e.g. k = 12 with KB = 16): nothing to load
#pragma unroll
        for (int q = 0; q < Q; ++q) xv[q] = 0.0f;
        return;
    }
    if constexpr (Q == 4) {
        if (vec) {  // k % 4 == 0, X 16-byte aligned
            const float4 t = *reinterpret_cast<const float4*>(p);
            xv[0] = t.x; xv[1] = t.y; xv[2] = t.z; xv[3] = t.w;
            return;
        }
    } else if constexpr (Q == 2) {
        if (vec) {  // k == 2, X 8-byte aligned
            const float2 t = *reinterpret_cast<const float2*>(p);
            xv[0] = t.x; xv[1] = t.y;
            return;
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) xv[q] = qb + q < k ? p[q] : 0.0f;
}

// DIA.  The diagonals come as segments {first diagonal, its offset, how many
// (at most W) consecutive offsets, 0} in diagonal order.  A wave owns NR
// consecutive rows; lane t takes rows R * (t / L) .. + R - 1 and right-hand
// sides Q * (t % L) .. + Q - 1 (the last lane of a group ends at k, so every
// X access is a whole Q-float piece).
//
// What bounds it: the texture addresser.  A lane reading its own X pieces for
// every diagonal sends each X row through L1 once per diagonal, 27 times on
// the 27-point stencil, 64 bytes a cycle per CU (TA busy 73 % of the time,
// 99 us on 96^3 rows at k = 16 even with that loop tuned).  So per segment the
// wave loads the X rows of its window (NR + W - 1 consecutive rows of X) and
// the segment's values once, coalesced, into its own part of LDS, and reads
// them there: R + W - 1 pieces for R * W products per lane.  The next
// segment's loads are in flight in registers meanwhile; no work-group barrier.
// LDS rows are padded by KB floats every R rows, which keeps the 16-byte reads
// of lanes R rows apart on different banks.  96^3 27-point stencil, FP32,
// k = 2 / 4 / 7 / 8 / 16: 26 / 31 / 38 / 41 / 73 us against 41 / 49 / 135 /
// 94 / 183 us for lanes loading every diagonal's X row themselves (1.7 to 3.8
// TB/s of the bytes that cannot be avoided); 5-point Laplacian on 900^2, k = 8 /
// 16: 19 / 42 against 30 / 59 us.
//
// Each column is summed alone in diagonal order, one product at a time,
// skipping columns outside x, whatever the tile: its result does not depend
// on k.
template <int Q, int L, int R, int W, class V>
__global__ __launch_bounds__(kBlock) void dia_multi_kernel(
    int rows, int cols, int len, int nseg, const int4* __restrict__ seg,
    const typename V::T* __restrict__ data, int k, const float* __restrict__ X, float* __restrict__ Y,
    int ldy) {
    typedef typename V::T T;
    constexpr int NR = kWave / L * R;                    // rows per wave
    constexpr int RW = kWave / L;                        // X rows per load instruction
    constexpr int QP = Q == 3 ? 4 : Q;                   // LDS floats per piece
    constexpr int KB = QP * L;                           // LDS floats per X row
    constexpr int CS = (R + 1) * KB;                     // LDS floats per R rows
    constexpr int NX = NR + W - 1;                       // X rows per window
    constexpr int NLD = (NX + RW - 1) / RW;              // X pieces per lane
    constexpr int ND = NR >= kWave ? NR / kWave : 1;     // values per lane and diagonal
    constexpr int DL = NR / ND;                          // lanes that load values
    typedef VecOf<float, Q> XV;
    typedef VecOf<T, ND> DV;
    typedef VecOf<float, ND> FV;
    typedef VecOf<float, R> RV;
    constexpr int kWaves = kBlock / kWave;
    __shared__ __attribute__((aligned(16))) float sx[kWaves][(NX + R - 1) / R * CS];
    __shared__ __attribute__((aligned(16))) float sd[kWaves][W * NR];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int w0 = __builtin_amdgcn_readfirstlane((xcd_tile(blockIdx.x, gridDim.x) * kWaves + wave) * NR);
    if (w0 >= rows) return;  // the whole wave
    float* xl = sx[wave];
    float* dl = sd[wave];
    const int g = lane / L, p = lane % L;
    const int q0 = p * Q, qs = min(q0, k - Q);
    float acc[R][Q];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[r][q] = 0.0f;
    const bool tail = w0 + NR > len;  // rows past the stored length
    typename XV::type xr[NLD];
    typename DV::type dr[W];
    const unsigned xo = (unsigned)(g * k + qs), xlast = (unsigned)((NX - 1) * k + qs);
    // Whether every X row of a segment's window exists.
    auto inside = [&](int off) { return (long long)w0 + off >= 0 && (long long)w0 + off + NX <= cols; };
    auto load = [&](const int4 sg) {
        if (inside(sg.y)) {
            const float* xw = X + (ptrdiff_t)(w0 + sg.y) * k;
#pragma unroll
            for (int u = 0; u < NLD; ++u) {
                const unsigned o = xo + (unsigned)(u * RW) * k;
                xr[u] = *reinterpret_cast<const typename UVec<float, Q>::type*>(
                    xw + ((u + 1) * RW <= NX ? o : min(o, xlast)));
            }
        } else {  // rows outside X re-read the first or last one and are not added
#pragma unroll
            for (int u = 0; u < NLD; ++u) {
                const int c = min(max(w0 + sg.y + g + u * RW, 0), cols - 1);
                xr[u] = *reinterpret_cast<const typename UVec<float, Q>::type*>(X + (size_t)c * k + qs);
            }
        }
        // Diagonals past the segment's re-read its last one and are not added.
        const T* dp = data + (size_t)sg.x * len + w0;
        if (!tail) {
            const int at = min(lane, DL - 1) * ND;
#pragma unroll
            for (int n = 0; n < W; ++n)
                dr[n] = __builtin_nontemporal_load(reinterpret_cast<const typename UVec<T, ND>::type*>(
                    dp + (size_t)min(n, sg.z - 1) * len + at));
        } else {
#pragma unroll
            for (int n = 0; n < W; ++n)
#pragma unroll
                for (int h = 0; h < ND; ++h)
                    DV::set(dr[n], h, dp[(size_t)min(n, sg.z - 1) * len + min(lane * ND + h, len - 1 - w0)]);
        }
    };
    int4 sg = seg[0];
    load(sg);
    for (int s = 0; s < nseg; ++s) {
        const int z = sg.z, off = sg.y;
#pragma unroll
        for (int u = 0; u < NLD; ++u) {
            const int r = g + u * RW;
            float* at = xl + r / R * CS + r % R * KB + p * QP;
            if ((u + 1) * RW <= NX || r < NX) {
                if constexpr (Q == 3) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) at[q] = xr[u][q];
                } else {
                    *reinterpret_cast<typename XV::type*>(at) = xr[u];
                }
            }
        }
        if (lane < DL) {
#pragma unroll
            for (int n = 0; n < W; ++n) {
                typename FV::type f;
#pragma unroll
                for (int h = 0; h < ND; ++h) FV::set(f, h, V::cvt(DV::get(dr[n], h)));
                *reinterpret_cast<typename FV::type*>(dl + n * NR + lane * ND) = f;
            }
        }
        wave_lds_order();
        sg = seg[min(s + 1, nseg - 1)];
        load(sg);
        // N diagonals from the segment's n0-th on; `all`: no column to skip.
        auto add = [&](auto count, auto all, int n0) {
            constexpr int N = decltype(count)::value;
            typename XV::type xv[R + N - 1];
            typename RV::type d[N];
#pragma unroll
            for (int n = 0; n < N; ++n)
                d[n] = *reinterpret_cast<const typename RV::type*>(dl + (n0 + n) * NR + g * R);
#pragma unroll
            for (int i = 0; i < R + N - 1; ++i) {
                const int r = N == W ? i : n0 + i;  // N == W: n0 is 0, the offsets are constants
                const float* at = xl + (g + r / R) * CS + r % R * KB + p * QP;
                if constexpr (Q == 3) {
                    const f32x4 t = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
                    for (int q = 0; q < Q; ++q) xv[i][q] = t[q];
                } else {
                    xv[i] = *reinterpret_cast<const typename XV::type*>(at);
                }
            }
#pragma unroll
            for (int n = 0; n < N; ++n)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const bool in =
                        decltype(all)::value || (unsigned)(w0 + off + n0 + n + g * R + r) < (unsigned)cols;
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        const float a = fmaf(RV::get(d[n], r), XV::get(xv[n + r], q), acc[r][q]);
                        acc[r][q] = in ? a : acc[r][q];
                    }
                }
        };
        using One = std::integral_constant<int, 1>;
        if (!inside(off)) {
            for (int n = 0; n < z; ++n) add(One{}, std::false_type{}, n);
        } else if (z == W) {
            add(std::integral_constant<int, W>{}, std::true_type{}, 0);
        } else {
            for (int n = 0; n < z; ++n) add(One{}, std::true_type{}, n);
        }
        wave_lds_order();
    }
    const int r0 = w0 + g * R;
    if (q0 >= k) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (qs + q < q0) continue;  // the lane before has this column
        float* yp = Y + (size_t)(qs + q) * ldy + r0;
        if (r0 + R <= rows) {
            typedef typename UVec<float, R>::type YU;
            typename RV::type v = *reinterpret_cast<const YU*>(yp);
#pragma unroll
            for (int r = 0; r < R; ++r) RV::set(v, r, RV::get(v, r) + acc[r][q]);
            *reinterpret_cast<YU*>(yp) = v;
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r0 + r < rows) yp[r] += acc[r][q];
        }
    }
}

// Accumulates a[q] += val[j] * X[col[j]][qb + q] over j = j0, j0 + step, ...
// below j1 in that order, U nonzeros in flight per lane.  Acc is float, or
// double for rows longer than kLongRowF64 (the products are exact in
// double).
template <int Q, class V, class Acc, int U>
__device__ __forceinline__ void csr_multi_run(const int* __restrict__ col,
                                              const typename V::T* __restrict__ val, int j0, int j1,
                                              int step, const float* __restrict__ X, int k, int qb,
                                              bool vec, Acc* a) {
    int j = j0;
    for (; j + (U - 1) * step < j1; j += U * step) {
        int c[U];
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = ld_stream(col + j + u * step);
            v[u] = V::ld(val + j + u * step);
        }
        float xv[U][Q];
#pragma unroll
        for (int u = 0; u < U; ++u) load_xq<Q>(X, c[u], k, qb, vec, xv[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < Q; ++q) a[q] = fma((Acc)v[u], (Acc)xv[u][q], a[q]);
    }
    for (; j < j1; j += step) {
        const int c = ld_stream(col + j);
        const float v = V::ld(val + j);
        float xv[Q];
        load_xq<Q>(X, c, k, qb, vec, xv);
#pragma unroll
        for (int q = 0; q < Q; ++q) a[q] = fma((Acc)v, (Acc)xv[q], a[q]);
    }
}

// One row longer than kAdaptiveNnz by the whole work-group: each lane
// strides the row with 4 * L nonzeros in flight (a whole work-group round
// covers kAdaptiveNnz of them), the four waves' sums are combined in a
// fixed order through LDS, and Y[:, r] is updated once per right-hand side.
template <int KB, class V, class Acc>
__device__ __forceinline__ void csr_multi_long(const typename V::T* __restrict__ val,
                                               const int* __restrict__ col, int r, int j0, int j1,
                                               const float* __restrict__ X, int k, bool vec,
                                               float* __restrict__ Y, int ldy, Acc (*part)[KB]) {
    constexpr int Q = KB < 4 ? KB : 4;
    constexpr int L = KB / Q;
    const int t = threadIdx.x;
    const int qb = (t % L) * Q;
    Acc a[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) a[q] = 0;
    csr_multi_run<Q, V, Acc, launch::kAdaptiveNnz * L / kBlock>(col, val, j0 + t / L, j1, kBlock / L, X, k, qb,
                                                                vec, a);
#pragma unroll
    for (int q = 0; q < Q; ++q)
        for (int m = kWave >> 1; m >= L; m >>= 1) a[q] += __shfl_xor(a[q], m, kWave);
    if ((t & (kWave - 1)) < L) {
#pragma unroll
        for (int q = 0; q < Q; ++q) part[t / kWave][qb + q] = a[q];
    }
    __syncthreads();
    if (t < KB && t < k) {
        Acc tot = 0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; ++w) tot += part[w][t];
        float* yp = Y + (size_t)t * ldy + r;
        if constexpr (sizeof(Acc) == sizeof(double))
            *yp = (float)((double)*yp + tot);  // one rounding of the whole row
        else
            *yp += tot;
    }
}

// CSR over row blocks (runs of at most kAdaptiveRows rows whose
// nonzeros fit kAdaptiveNnz, or one longer row).  Each lane carries
// Q = min(KB, 4) right-hand sides (one 16-byte gather of X per nonzero), and
// L = KB / Q neighbouring lanes cover the k values of one nonzero.
//
// A block of short rows is streamed: its nonzeros are cut into G = kBlock / L
// equal consecutive chunks, one per lane group, whatever the rows' lengths
// (a row-per-group split left short rows' groups idle beside one long row's
// and put the gathers of a group's rows one after another).  A group loads
// every column, value and X row of its chunk at once, then walks the chunk
// in order: a row that starts and ends inside it is summed there and added
// to Y; the part of a row that began in an earlier chunk goes to LDS (head),
// and a row that continues past the chunk is finished, after a barrier, by
// the group where it starts (its tail, then the later chunks' heads in
// order).  Each row is thus summed in nonzero order with one break per chunk
// boundary, in FP32, the same way every time.
//
// A long row: the whole work-group, the four waves' partial sums combined in
// a fixed order through LDS, in FP64 for rows longer than kLongRowF64
// (products exact, one rounding into y).
template <int KB, class V>
__global__ __launch_bounds__(kBlock) void csr_multi_kernel(
    const int* __restrict__ blocks, const int* __restrict__ rp, const int* __restrict__ col,
    const typename V::T* __restrict__ val, int k, const float* __restrict__ X, bool vec,
    float* __restrict__ Y, int ldy) {
    constexpr int Q = KB < 4 ? KB : 4;
    constexpr int L = KB / Q;
    constexpr int G = kBlock / L;                   // lane groups
    constexpr int CM = launch::kAdaptiveNnz / G;    // nonzeros per group at most
    static_assert(CM * G == launch::kAdaptiveNnz, "a block's nonzeros must split evenly over the groups");
    __shared__ float part[kBlock / kWave][KB];
    __shared__ double part64[kBlock / kWave][KB];
    __shared__ int srp[launch::kAdaptiveRows + 1];  // the block's row starts, from its first nonzero
    __shared__ float head[G][KB];                   // each chunk's part of a row begun earlier
    const int b = blockIdx.x;
    const int r0 = blocks[b], r1 = blocks[b + 1];
    const int nrows = r1 - r0;
    const int t = threadIdx.x;
    const int qb = (t % L) * Q;
    if (nrows == 1 && rp[r1] - rp[r0] > launch::kAdaptiveNnz) {
        if (rp[r1] - rp[r0] > launch::kLongRowF64)
            csr_multi_long<KB, V, double>(val, col, r0, rp[r0], rp[r1], X, k, vec, Y, ldy, part64);
        else
            csr_multi_long<KB, V, float>(val, col, r0, rp[r0], rp[r1], X, k, vec, Y, ldy, part);
        return;
    }
    const int s = rp[r0];
    const int n = rp[r1] - s;  // at most kAdaptiveNnz
    for (int i = t; i <= nrows; i += kBlock) srp[i] = rp[r0 + i] - s;
    __syncthreads();
    if (n == 0) return;  // only empty rows (the whole work-group)
    const int gi = t / L;
    const int C = (n + G - 1) / G;  // <= CM
    const int c0 = min(n, gi * C), c1 = min(n, c0 + C);
    // Every load of the chunk before its first product (slots past the
    // chunk read nonzero s and are never used).
    int cc[CM];
    float vv[CM], xv[CM][Q];
#pragma unroll
    for (int u = 0; u < CM; ++u) {
        const int j = c0 + u < c1 ? s + c0 + u : s;
        cc[u] = ld_stream(col + j);
        vv[u] = V::ld(val + j);
    }
#pragma unroll
    for (int u = 0; u < CM; ++u) load_xq<Q>(X, cc[u], k, qb, vec, xv[u]);
    float acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = 0.0f;
    auto add_y = [&](int r) {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (qb + q < k) Y[(size_t)(qb + q) * ldy + r0 + r] += acc[q];
    };
    int r = 0, rend = 0;
    bool in_head = false;  // the current row began before this chunk
    if (c0 < c1) {
        // The row holding nonzero c0: the last row starting at or before it
        // (empty rows before it start at the same place and are passed).
        int lo = 0, hi = nrows - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (srp[mid] <= c0) lo = mid;
            else hi = mid - 1;
        }
        r = lo;
        rend = srp[r + 1];
        in_head = srp[r] < c0;
#pragma unroll
        for (int u = 0; u < CM; ++u) {
            const int j = c0 + u;
            if (j < c1) {
                if (j >= rend) {  // row r ended inside the chunk
                    if (in_head) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) head[gi][qb + q] = acc[q];
                    } else {
                        add_y(r);
                    }
                    in_head = false;
                    do {
                        ++r;
                        rend = srp[r + 1];
                    } while (j >= rend);  // empty rows
#pragma unroll
                    for (int q = 0; q < Q; ++q) acc[q] = 0.0f;
                }
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[q] = fmaf(vv[u], xv[u][q], acc[q]);
            }
        }
        if (in_head) {
#pragma unroll
            for (int q = 0; q < Q; ++q) head[gi][qb + q] = acc[q];
        } else if (rend <= c1) {
            add_y(r);
        }
    }
    __syncthreads();
    // The row this chunk ends inside of and began: its tail, then the heads
    // of the later chunks it runs through, in order.
    if (c0 < c1 && !in_head && rend > c1) {
        const int last = (rend - 1) / C;  // the chunk holding the row's last nonzero
        for (int g2 = gi + 1; g2 <= last; ++g2)
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[q] += head[g2][qb + q];
        add_y(r);
    }
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

template <int Q, int L, int R, class V>
hipError_t dia_multi_tile(hipStream_t s, int rows, int cols, int len, int nseg, int w, const int4* seg,
                          const void* data, int k, const float* X, float* Y, int ldy) {
    const dim3 grid(ceil_div(rows, kBlock / L * R)), block(kBlock);
    const typename V::T* d = static_cast<const typename V::T*>(data);
    if (w == 1)
        hipLaunchKernelGGL((dia_multi_kernel<Q, L, R, 1, V>), grid, block, 0, s, rows, cols, len, nseg, seg, d, k, X,
                           Y, ldy);
    else
        hipLaunchKernelGGL((dia_multi_kernel<Q, L, R, kDiaRun, V>), grid, block, 0, s, rows, cols, len, nseg, seg, d,
                           k, X, Y, ldy);
    return hipGetLastError();
}

// Rows per lane: more of them reuse each staged X row more often but leave
// fewer waves, each with a longer chain of segments.  On the 27-point stencil
// the wider tile wins from 80^3 to 96^3 rows on (96^3, k = 4 / 8: 31 / 41 us
// against 36 / 48 us for the narrower one) and loses below (64^3: 11.2 / 13.3
// against 10.2 / 12.6 us); with few segments it never pays at k >= 2 (5-point
// Laplacian on 900^2, k = 4 / 8: 15.5 / 22.5 against 13.4 / 19.7 us).  At k > 8
// a wave has 64 / 4 lane groups, and four rows each win from 32^3 rows on
// (32^3: 9.8 us, 22^3: 10.3 against 7.9 us).
template <class V>
hipError_t dia_multi_v(hipStream_t s, int rows, int cols, int len, int nseg, int w, const int4* seg,
                       const void* data, int k, const float* X, float* Y, int ldy) {
    const bool large = rows >= (1 << 19);
    const bool deep = large && nseg >= 6;
#define CLSPMV_DIA_MULTI(Q, L, R) dia_multi_tile<Q, L, R, V>(s, rows, cols, len, nseg, w, seg, data, k, X, Y, ldy)
    switch (k) {
        case 1: return large ? CLSPMV_DIA_MULTI(1, 1, 4) : CLSPMV_DIA_MULTI(1, 1, 1);
        case 2: return deep ? CLSPMV_DIA_MULTI(2, 1, 2) : CLSPMV_DIA_MULTI(2, 1, 1);
        case 3: return deep ? CLSPMV_DIA_MULTI(3, 1, 2) : CLSPMV_DIA_MULTI(3, 1, 1);
        case 4: return deep ? CLSPMV_DIA_MULTI(4, 1, 2) : CLSPMV_DIA_MULTI(4, 1, 1);
        default: break;
    }
    if (k <= 8) return deep && w > 1 ? CLSPMV_DIA_MULTI(4, 2, 4) : CLSPMV_DIA_MULTI(4, 2, 2);
    return rows >= (1 << 15) ? CLSPMV_DIA_MULTI(4, 4, 4) : CLSPMV_DIA_MULTI(4, 4, 2);
#undef CLSPMV_DIA_MULTI
}

template <int KB, class V>
hipError_t csr_multi_kb(hipStream_t s, int nblocks, const int* blocks, const int* rp, const int* col,
                        const void* val, int k, const float* X, float* Y, int ldy) {
    constexpr int Q = KB < 4 ? KB : 4;
    const bool vec = Q > 1 && k % Q == 0 && ((uintptr_t)X % (Q * sizeof(float))) == 0;
    hipLaunchKernelGGL((csr_multi_kernel<KB, V>), dim3(nblocks), dim3(kBlock), 0, s, blocks, rp, col,
                       static_cast<const typename V::T*>(val), k, X, vec, Y, ldy);
    return hipGetLastError();
}

template <class V>
hipError_t csr_multi_v(hipStream_t s, int nblocks, const int* blocks, const int* rp, const int* col,
                       const void* val, int k, const float* X, float* Y, int ldy, int kb) {
    if (kb > 0) {  // a fixed width: the summation order of each right-hand side does not depend on k
        switch (kb) {
            case 1: return csr_multi_kb<1, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
            case 2: return csr_multi_kb<2, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
            case 4: return csr_multi_kb<4, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
            case 8: return csr_multi_kb<8, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
            case 16: return csr_multi_kb<16, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
            default: return hipErrorInvalidValue;
        }
    }
    if (k <= 1) return csr_multi_kb<1, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
    if (k <= 2) return csr_multi_kb<2, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
    if (k <= 4) return csr_multi_kb<4, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
    if (k <= 8) return csr_multi_kb<8, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
    return csr_multi_kb<16, V>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy);
}

}  // namespace

namespace launch {

hipError_t dia_multi(hipStream_t s, int rows, int cols, int len, int nseg, int w, const int4* seg,
                     int dtype, const void* data, int k, const float* X, float* Y, int ldy) {
    if (rows <= 0 || cols <= 0 || nseg <= 0 || k <= 0) return hipSuccess;
    if (k > kMultiMax) return hipErrorInvalidValue;
    switch (dtype) {
        case 0: return dia_multi_v<ValF32>(s, rows, cols, len, nseg, w, seg, data, k, X, Y, ldy);
        case 1: return dia_multi_v<ValBF16>(s, rows, cols, len, nseg, w, seg, data, k, X, Y, ldy);
        case 2: return dia_multi_v<ValF16>(s, rows, cols, len, nseg, w, seg, data, k, X, Y, ldy);
        default: return hipErrorInvalidValue;
    }
}

hipError_t csr_multi(hipStream_t s, int nblocks, const int* blocks, const int* rp, const int* col,
                     int dtype, const void* val, int k, const float* X, float* Y, int ldy, int kb) {
    if (nblocks <= 0 || k <= 0) return hipSuccess;
    if (k > kMultiMax || (kb > 0 && k > kb)) return hipErrorInvalidValue;
    switch (dtype) {
        case 0: return csr_multi_v<ValF32>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy, kb);
        case 1: return csr_multi_v<ValBF16>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy, kb);
        case 2: return csr_multi_v<ValF16>(s, nblocks, blocks, rp, col, val, k, X, Y, ldy, kb);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace launch
}  // namespace clspmv
