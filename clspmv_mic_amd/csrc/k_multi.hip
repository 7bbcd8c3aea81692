// Multi-right-hand-side SpMV for gfx950: Y[:, q] += A X[:, q] for q < k
// (k <= 16) in one pass over the matrix, for DIA and CSR.
//
// X is row-major (the k values of column c are X[c*k .. c*k+k)), so the
// gather of one column brings every right-hand side's value in one or a few
// 16-byte loads: a random column costs one cache line for all k products
// instead of one line per product.  Y is
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
    int ldy, bool accumulate) {
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
            typename RV::type v{};
            if (accumulate) v = *reinterpret_cast<const YU*>(yp);
#pragma unroll
            for (int r = 0; r < R; ++r) RV::set(v, r, RV::get(v, r) + acc[r][q]);
            *reinterpret_cast<YU*>(yp) = v;
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r0 + r < rows) yp[r] = (accumulate ? yp[r] : 0.0f) + acc[r][q];
        }
    }
}

// DIA where the chain of segments would set the time: a lane takes one row and
// right-hand sides Q * (t % L) .. + Q - 1 (the last lane of a row ends at k) and
// reads the X pieces itself, C diagonals' values and pieces in flight.  The sums
// are dia_multi_kernel's, bit for bit.
template <int Q, int L, class V>
__global__ __launch_bounds__(kBlock) void dia_multi_direct_kernel(
    int rows, int cols, int len, int ndiag, const int* __restrict__ off,
    const typename V::T* __restrict__ data, int k, const float* __restrict__ X, float* __restrict__ Y,
    int ldy, bool accumulate) {
    constexpr int C = Q == 4 ? 8 : 16;
    typedef VecOf<float, Q> XV;
    const int t = threadIdx.x;
    const int r = xcd_tile(blockIdx.x, gridDim.x) * (kBlock / L) + t / L;
    if (r >= rows) return;
    const int q0 = t % L * Q, qs = min(q0, k - Q);
    float acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = 0.0f;
    for (int j0 = 0; j0 < ndiag; j0 += C) {  // wave-uniform
        float d[C];
        typename XV::type xv[C];
        bool in[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const int j = min(j0 + u, ndiag - 1);
            d[u] = V::ld(data + (size_t)j * len + r);
            const int c = r + off[j];
            in[u] = j0 + u < ndiag && (unsigned)c < (unsigned)cols;
            xv[u] = *reinterpret_cast<const typename UVec<float, Q>::type*>(X + (size_t)(in[u] ? c : 0) * k + qs);
        }
#pragma unroll
        for (int u = 0; u < C; ++u)
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[q] = in[u] ? fmaf(d[u], XV::get(xv[u], q), acc[q]) : acc[q];
    }
    if (q0 >= k) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (qs + q < q0) continue;  // the lane before has this column
        float* yp = Y + (size_t)(qs + q) * ldy + r;
        *yp = (accumulate ? *yp : 0.0f) + acc[q];
    }
}

// Accumulates a[q] += val[j] * X[col[j]][qb + q] over j = j0, j0 + step, ...
// below j1 in that order, U nonzeros in flight per lane also in the last round
// (slots past the end re-read the last one and are not added).  Acc is float,
// or double for rows longer than kLongRowF64 (the products are exact in
// double).
template <int Q, class V, class Acc, int U>
__device__ __forceinline__ void csr_multi_run(const int* __restrict__ col,
                                              const typename V::T* __restrict__ val, int j0, int j1,
                                              int step, const float* __restrict__ X, int k, int qb,
                                              bool vec, Acc* a) {
    // (Indices from j0: the sums stay in range near 2^31 entries.)
    const int n = j1 - j0;
    col += j0;
    val += j0;
    for (int j = 0; j < n; j += U * step) {
        int c[U];
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = min(j + u * step, n - 1);
            c[u] = ld_stream(col + at);
            v[u] = V::ld(val + at);
        }
        float xv[U][Q];
#pragma unroll
        for (int u = 0; u < U; ++u) load_xq<Q>(X, c[u], k, qb, vec, xv[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + u * step < n)
#pragma unroll
                for (int q = 0; q < Q; ++q) a[q] = fma((Acc)v[u], (Acc)xv[u][q], a[q]);
    }
}

// Work-group of the CSR kernel: with 512 threads a row over kWaveNnz entries has
// 1,024 of them in flight (a 5,000-entry row sets the time of a small
// power-law matrix: 60,000 rows, k = 4: 19.7 us against 27.3 with 256 threads;
// 17.6 with the longest rows first).
constexpr int kMultiThreads = 512;

// One row longer than kWaveNnz by the whole work-group, always with four
// lanes per entry, so that a column's sum does not depend on k: each lane
// group strides the row with 8 entries in flight, the eight waves' sums are
// combined in a fixed order through LDS, and Y[:, r] is updated once per
// right-hand side.
template <class V, class Acc>
__device__ __forceinline__ void csr_multi_long(const typename V::T* __restrict__ val,
                                               const int* __restrict__ col, int r, int j0, int j1,
                                               const float* __restrict__ X, int k, bool vec,
                                               float* __restrict__ Y, int ldy, bool accumulate,
                                               Acc (*part)[launch::kMultiMax]) {
    constexpr int Q = 4, L = launch::kMultiMax / Q;
    const int t = threadIdx.x;
    const int qb = (t % L) * Q;
    Acc a[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) a[q] = 0;
    csr_multi_run<Q, V, Acc, 8>(col, val, j0 + t / L, j1, kMultiThreads / L, X, k, qb, vec, a);
#pragma unroll
    for (int q = 0; q < Q; ++q)
        for (int m = kWave >> 1; m >= L; m >>= 1) a[q] += __shfl_xor(a[q], m, kWave);
    if ((t & (kWave - 1)) < L) {
#pragma unroll
        for (int q = 0; q < Q; ++q) part[t / kWave][qb + q] = a[q];
    }
    __syncthreads();
    if (t < k) {
        Acc tot = 0;
#pragma unroll
        for (int w = 0; w < kMultiThreads / kWave; ++w) tot += part[w][t];
        float* yp = Y + (size_t)t * ldy + r;
        const float y0 = accumulate ? *yp : 0.0f;
        if constexpr (sizeof(Acc) == sizeof(double))
            *yp = (float)((double)y0 + tot);  // one rounding of the whole row
        else
            *yp = y0 + tot;
    }
}

// The value of lane P of each aligned group of L lanes (L at most 4), by a
// DPP quad permute.
template <int L, int P, class T>
__device__ __forceinline__ T group_lane(T v) {
    if constexpr (L == 1) return v;
    constexpr int ctrl = L == 4 ? P * 0x55 : P | P << 2 | (P + 2) << 4 | (P + 2) << 6;
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false));
}

// CSR: a wave per block of short rows (the wave kernel's blocks), L lanes per
// entry with Q right-hand sides each; a work-group per longer row.
//
// A block is cut into units of 8 consecutive entries, whatever the rows'
// lengths (a lane group per row would leave groups idle beside one long row
// and put a row's gathers one after another).  A lane group loads its unit's
// columns and values (each lane a part, handed round by DPP) and its 8 rows
// of X at once, then walks the unit: a row that starts in it goes to the row's
// place in LDS, the part of a row that began in an earlier unit to the unit's
// `head`.  Then each row adds the heads of the later units it runs through, in
// order, and Y is updated a column at a time, a lane per row.  A row's sum is
// thus one FP32 chain per unit and the units in order: it depends on the
// block cut alone, not on k.
//
// What bounds it: random rows of X.  A 32- or 64-byte row costs a whole
// 128-byte line once X outgrows the L2s: 72 / 62 G rows/s at 19 / 32 MB of X
// (k = 8), 58 / 54 G at 38 / 64 MB (k = 16) when nothing else runs.  Before,
// a work-group of 1024 entries waited at two barriers, each finished row was
// added to Y where it ended (a load and a store of one float per right-hand
// side, waited for) and k not a multiple of 4 gathered single floats.
// Power-law rows: 600,011 rows, BF16, k = 8 / 16: 191 / 318 -> 138 / 174 us; 1 M
// rows, FP32, k = 5 / 8 / 16: 357 / 329 / 528 -> 266 / 251 / 302 us (53 G rows/s);
// 27-point stencil 64^3, k = 8: 74 -> 31 us.
constexpr int kUnit = 8;

template <int Q, int L, class V>
__global__ __launch_bounds__(kMultiThreads) void csr_multi_kernel(
    int nlong, const int* __restrict__ longs, int nblk, const int4* __restrict__ blk,
    const int* __restrict__ rp, const int* __restrict__ col, const typename V::T* __restrict__ val, int k,
    const float* __restrict__ X, bool vec, float* __restrict__ Y, int ldy, bool accumulate) {
    typedef typename V::T T;
    constexpr int QP = Q == 3 ? 4 : Q;              // LDS floats per piece
    constexpr int KB = QP * L;                      // and per row or unit
    constexpr int AS = KB == 1 ? 1 : KB + QP;       // LDS stride of the rows
    constexpr int G = kWave / L;                    // lane groups of a wave
    constexpr int NU = launch::kWaveNnz / kUnit;    // units of a block at most
    constexpr int NE = kUnit / L;                   // entries a lane loads
    constexpr int kWaves = kMultiThreads / kWave;
    typedef VecOf<float, Q> XV;
    typedef VecOf<float, QP> PV;
    struct WaveLds {
        float acc[kWave * AS];
        float head[NU * KB];
        int rp[kWave + 4];
    };
    __shared__ __attribute__((aligned(16))) union {
        WaveLds w[kWaves];
        float part[kWaves][launch::kMultiMax];
        double part64[kWaves][launch::kMultiMax];
    } lds;
    if ((int)blockIdx.x < nlong) {  // the longest work first
        const int r = longs[blockIdx.x], j0 = rp[r], j1 = rp[r + 1];
        if (j1 - j0 > launch::kLongRowF64)
            csr_multi_long<V, double>(val, col, r, j0, j1, X, k, vec, Y, ldy, accumulate, lds.part64);
        else
            csr_multi_long<V, float>(val, col, r, j0, j1, X, k, vec, Y, ldy, accumulate, lds.part);
        return;
    }
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int b = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x - nlong, gridDim.x - nlong) * kWaves + wave);
    if (b >= nblk) return;  // the whole wave
    const int4 B = blk[b];  // {first row, rows, first entry, entries}
    const int r0 = B.x, nrows = B.y, s = B.z, n = B.w;
    WaveLds& W = lds.w[wave];
    const int gi = lane / L, p = lane % L;
    const int q0 = p * Q, qs = min(q0, k - Q);  // the last piece ends at k
    const bool act = q0 < k;
    const float* Xq = X + qs;
    typedef VecOf<int, NE> CV;
    typedef VecOf<T, NE> TV;
    typename CV::type cn;
    typename TV::type vn;
    auto load = [&](int u) {  // unit u's columns and values; the arrays are padded past the last entry
        const int at = u * kUnit + p * NE;
        cn = __builtin_nontemporal_load(reinterpret_cast<const typename UVec<int, NE>::type*>(col + s + at));
        vn = __builtin_nontemporal_load(reinterpret_cast<const typename UVec<T, NE>::type*>(val + s + at));
    };
    const int nunits = (n + kUnit - 1) / kUnit;
    if (nunits > 0) load(min(gi, nunits - 1));
    const int myrp = rp[r0 + min(lane, nrows)] - s;
    W.rp[lane] = myrp;  // entries past nrows repeat the end
    if (lane == 0) W.rp[kWave] = n;
    wave_lds_order();
    for (int u0 = 0; u0 < nunits; u0 += G) {
        const int u = u0 + gi;
        int c[kUnit];
        float v[kUnit];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int ce = CV::get(cn, e);
            const float ve = V::cvt(TV::get(vn, e));
            c[e] = group_lane<L, 0>(ce);
            v[e] = group_lane<L, 0>(ve);
            if constexpr (L >= 2) {
                c[NE + e] = group_lane<L, 1>(ce);
                v[NE + e] = group_lane<L, 1>(ve);
            }
            if constexpr (L == 4) {
                c[2 * NE + e] = group_lane<L, 2>(ce);
                v[2 * NE + e] = group_lane<L, 2>(ve);
                c[3 * NE + e] = group_lane<L, 3>(ce);
                v[3 * NE + e] = group_lane<L, 3>(ve);
            }
        }
        typename XV::type xv[kUnit];
        const bool on = u < nunits && act;
        if (on) {
#pragma unroll
            for (int e = 0; e < kUnit; ++e)
                xv[e] = *reinterpret_cast<const typename UVec<float, Q>::type*>(Xq + (size_t)c[e] * k);
        }
        if (u0 + G < nunits) load(min(u + G, nunits - 1));
        if (on) {
            const int j0 = u * kUnit, j1 = min(n, j0 + kUnit);
            // The row of the unit's first entry: the last one starting at or
            // before it.
            int r = 0;
#pragma unroll
            for (int m = kWave / 2; m >= 1; m >>= 1)
                if (r + m < nrows && W.rp[r + m] <= j0) r += m;
            int rend = W.rp[r + 1];
            bool head = W.rp[r] < j0;
            float a[QP];
#pragma unroll
            for (int q = 0; q < QP; ++q) a[q] = 0.0f;
            auto flush = [&]() {
                float* to = head ? W.head + u * KB + p * QP : W.acc + r * AS + p * QP;
                typename PV::type t;
#pragma unroll
                for (int q = 0; q < QP; ++q) PV::set(t, q, a[q]);
                *reinterpret_cast<typename PV::type*>(to) = t;
            };
#pragma unroll
            for (int e = 0; e < kUnit; ++e) {
                const int j = j0 + e;
                if (j < j1) {
                    if (j >= rend) {  // row r ended in the unit
                        flush();
                        head = false;
                        do rend = W.rp[++r + 1];
                        while (j >= rend);  // empty rows
#pragma unroll
                        for (int q = 0; q < QP; ++q) a[q] = 0.0f;
                    }
#pragma unroll
                    for (int q = 0; q < Q; ++q) a[q] = fmaf(v[e], XV::get(xv[e], q), a[q]);
                }
            }
            flush();
        }
    }
    wave_lds_order();
    // Rows that run through several units add the later ones' heads.
    for (int rr = gi; rr < nrows; rr += G) {
        const int e0 = W.rp[rr], e1 = W.rp[rr + 1];
        const int ua = e0 / kUnit, uz = (e1 - 1) / kUnit;
        if (e1 == e0 || uz == ua || !act) continue;
        float* at = W.acc + rr * AS + p * QP;
        typename PV::type t = *reinterpret_cast<typename PV::type*>(at);
        for (int u = ua + 1; u <= uz; ++u)
            t += *reinterpret_cast<const typename PV::type*>(W.head + u * KB + p * QP);
        *reinterpret_cast<typename PV::type*>(at) = t;
    }
    wave_lds_order();
    const bool empty = lane < nrows && W.rp[lane + 1] == W.rp[lane];
    if (lane < nrows && !(empty && accumulate)) {  // empty rows leave Y as it is
        float* yp = Y + r0 + lane;
        const float* ap = W.acc + lane * AS;
        const int full = (k - 1) / Q * Q, shift = full + Q - k;  // columns before the last piece, its overlap
        constexpr int KM = Q * L;
        float y[KM];
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) y[q] = accumulate ? yp[(size_t)q * ldy] : 0.0f;
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) yp[(size_t)q * ldy] = y[q] + (empty ? 0.0f : ap[q < full ? q : q + shift]);
    }
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

template <int Q, int L, int R, class V>
hipError_t dia_multi_tile(hipStream_t s, int rows, int cols, int len, int nseg, int w, const int4* seg,
                          const void* data, int k, const float* X, float* Y, int ldy, bool accumulate) {
    const dim3 grid(ceil_div(rows, kBlock / L * R)), block(kBlock);
    const typename V::T* d = static_cast<const typename V::T*>(data);
    if (w == 1)
        hipLaunchKernelGGL((dia_multi_kernel<Q, L, R, 1, V>), grid, block, 0, s, rows, cols, len, nseg, seg, d, k, X,
                           Y, ldy, accumulate);
    else
        hipLaunchKernelGGL((dia_multi_kernel<Q, L, R, kDiaRun, V>), grid, block, 0, s, rows, cols, len, nseg, seg, d,
                           k, X, Y, ldy, accumulate);
    return hipGetLastError();
}

template <int Q, int L, class V>
hipError_t dia_multi_direct(hipStream_t s, int rows, int cols, int len, int ndiag, const int* off, const void* data,
                            int k, const float* X, float* Y, int ldy, bool accumulate) {
    hipLaunchKernelGGL((dia_multi_direct_kernel<Q, L, V>), dim3(ceil_div(rows, kBlock / L)), dim3(kBlock), 0, s, rows,
                       cols, len, ndiag, off, static_cast<const typename V::T*>(data), k, X, Y, ldy, accumulate);
    return hipGetLastError();
}

// Whether the direct kernel is the better one.  The staging kernel walks the
// segments one after the other (about 0.25 us each at k = 1, 0.4 us at k = 8),
// which sets its time on few rows, and on lone diagonals each staged X row is
// read once.  Staged / direct, us:
//   runs: 27-point stencil of 60,000 rows, k = 1 / 8 / 16, 5.2 / 7.5 / 10.5 and 4.4 /
//     6.9 / 9.8; 120,000 rows 5.6 / 8.6 / 12.2 and 5.0 / 10.3 / 17.0;
//   31 lone diagonals: 60,000 rows 10.1 / 15.1 / 17.8 and 4.6 / 7.2 / 9.9; 1 M rows
//     29.5 / 67.3 / 109.5 and 21.6 / 64.4 / 123.9;
//   14: 120,000 rows, k = 2 / 4 / 8 / 16, 6.8 / 7.7 / 9.3 / 11.9 and 4.4 / 5.2 / 7.9 /
//     12.6; 650,000 rows 14.1 / 17.0 / 26.5 / 42.5 and 12.8 / 17.7 / 32.5 / 58.4;
//   three: 120,000 rows 3.5 / 4.0 / 4.8 / 6.3 and 3.9 / 3.6 / 5.0 / 7.7.
bool dia_multi_chain(int rows, int nseg, int w, int k) {
    if (w > 1) return k == 1 ? rows < 300000 || nseg >= 10 : rows < 100000;
    if (nseg >= 24) return k <= 8 || rows < 350000;
    if (k == 1) return nseg >= 7;
    if (k <= 3) return rows < 40000LL * nseg && rows < 600000;
    if (k == 4) return nseg >= 7 || rows < 250000;
    return rows < (k <= 8 && nseg >= 7 ? 200000 : 100000);
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
hipError_t dia_multi_v(hipStream_t s, int rows, int cols, int len, int ndiag, const int* off, int nseg, int w,
                       const int4* seg, const void* data, int k, const float* X, float* Y, int ldy, bool accumulate) {
    if (dia_multi_chain(rows, nseg, w, k)) {
#define CLSPMV_DIA_DIRECT(Q, L) dia_multi_direct<Q, L, V>(s, rows, cols, len, ndiag, off, data, k, X, Y, ldy, accumulate)
        switch (k) {
            case 1: return CLSPMV_DIA_DIRECT(1, 1);
            case 2: return CLSPMV_DIA_DIRECT(2, 1);
            case 3: return CLSPMV_DIA_DIRECT(3, 1);
            case 4: return CLSPMV_DIA_DIRECT(4, 1);
            default: return k <= 8 ? CLSPMV_DIA_DIRECT(4, 2) : CLSPMV_DIA_DIRECT(4, 4);
        }
#undef CLSPMV_DIA_DIRECT
    }
    const bool large = rows >= (1 << 19);
    const bool deep = large && nseg >= 6;
#define CLSPMV_DIA_MULTI(Q, L, R) dia_multi_tile<Q, L, R, V>(s, rows, cols, len, nseg, w, seg, data, k, X, Y, ldy, accumulate)
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

template <int Q, int L, class V>
hipError_t csr_multi_tile(hipStream_t s, const launch::CsrWave& W, const int* rp, const int* col, const void* val,
                          int k, const float* X, float* Y, int ldy, bool accumulate) {
    const bool vec = k % 4 == 0 && ((uintptr_t)X % 16) == 0;  // long rows: aligned 16-byte pieces
    hipLaunchKernelGGL((csr_multi_kernel<Q, L, V>), dim3(W.nlong + ceil_div(W.nblk, kMultiThreads / kWave)),
                       dim3(kMultiThreads), 0, s,
                       W.nlong, W.longs, W.nblk, W.blk, rp, col, static_cast<const typename V::T*>(val), k, X, vec, Y,
                       ldy, accumulate);
    return hipGetLastError();
}

template <class V>
hipError_t csr_multi_v(hipStream_t s, const launch::CsrWave& W, const int* rp, const int* col, const void* val, int k,
                       const float* X, float* Y, int ldy, bool accumulate) {
    switch (k) {
        case 1: return csr_multi_tile<1, 1, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        case 2: return csr_multi_tile<2, 1, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        case 3: return csr_multi_tile<3, 1, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        case 4: return csr_multi_tile<4, 1, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        default: break;
    }
    return k <= 8 ? csr_multi_tile<4, 2, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate)
                  : csr_multi_tile<4, 4, V>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
}

}  // namespace

namespace launch {

hipError_t dia_multi(hipStream_t s, int rows, int cols, int len, int ndiag, const int* off, DiaSegments S,
                     int dtype, const void* data, int k, const float* X, float* Y, int ldy, bool accumulate) {
    if (rows <= 0 || cols <= 0 || S.count <= 0 || k <= 0) return hipSuccess;
    if (k > kMultiMax) return hipErrorInvalidValue;
    switch (dtype) {
        case 0: return dia_multi_v<ValF32>(s, rows, cols, len, ndiag, off, S.count, S.width, S.seg, data, k, X, Y, ldy, accumulate);
        case 1: return dia_multi_v<ValBF16>(s, rows, cols, len, ndiag, off, S.count, S.width, S.seg, data, k, X, Y, ldy, accumulate);
        case 2: return dia_multi_v<ValF16>(s, rows, cols, len, ndiag, off, S.count, S.width, S.seg, data, k, X, Y, ldy, accumulate);
        default: return hipErrorInvalidValue;
    }
}

hipError_t csr_multi(hipStream_t s, const CsrWave& W, const int* rp, const int* col,
                     int dtype, const void* val, int k, const float* X, float* Y, int ldy, bool accumulate) {
    if (W.nblk + W.nlong <= 0 || k <= 0) return hipSuccess;
    if (k > kMultiMax) return hipErrorInvalidValue;
    switch (dtype) {
        case 0: return csr_multi_v<ValF32>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        case 1: return csr_multi_v<ValBF16>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        case 2: return csr_multi_v<ValF16>(s, W, rp, col, val, k, X, Y, ldy, accumulate);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace launch
}  // namespace clspmv
