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
// k = 2 / 4 / 7 / 8 / 16: 25 / 30 / 38 / 41 / 52 us (16: 73 over three matrices in
// turn) against 41 / 49 / 135 / 94 / 183 us for lanes loading every diagonal's X
// row themselves (1.7 to 3.8 TB/s of the bytes that cannot be avoided); 5-point
// Laplacian on 900^2, k = 8 / 16: 19 / 31 against 30 / 59 us.
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
    const unsigned w0u =
        __builtin_amdgcn_readfirstlane(((unsigned)xcd_tile(blockIdx.x, gridDim.x) * kWaves + wave) * NR);
    if (w0u >= (unsigned)rows) return;  // the whole wave
    const int w0 = (int)w0u, left = rows - w0;  // rows from the wave's first on
    float* xl = sx[wave];
    float* dl = sd[wave];
    const int g = lane / L, p = lane % L;
    const int q0 = p * Q, qs = min(q0, k - Q);
    float acc[R][Q];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[r][q] = 0.0f;
    const bool tail = len - w0 < NR;  // rows past the stored length
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
    if (q0 >= k) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (qs + q < q0) continue;  // the lane before has this column
        float* yp = Y + (size_t)(qs + q) * ldy + w0 + g * R;
        if (g * R + R <= left) {
            typedef typename UVec<float, R>::type YU;
            typename RV::type v{};
            if (accumulate) v = *reinterpret_cast<const YU*>(yp);
#pragma unroll
            for (int r = 0; r < R; ++r) RV::set(v, r, RV::get(v, r) + acc[r][q]);
            *reinterpret_cast<YU*>(yp) = v;
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (g * R + r < left) yp[r] = (accumulate ? yp[r] : 0.0f) + acc[r][q];
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
    const unsigned ru = (unsigned)xcd_tile(blockIdx.x, gridDim.x) * (kBlock / L) + t / L;
    if (ru >= (unsigned)rows) return;
    const int r = (int)ru;
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
            const unsigned c = ru + (unsigned)off[j];
            in[u] = j0 + u < ndiag && c < (unsigned)cols;
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

// The value of lane P of each aligned group of L lanes (L at most 4), by a
// DPP quad permute.
template <int L, int P, class T>
__device__ __forceinline__ T group_lane(T v) {
    if constexpr (L == 1) return v;
    constexpr int ctrl = L == 4 ? P * 0x55 : P | P << 2 | (P + 2) << 4 | (P + 2) << 6;
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false));
}

// Work-group of the CSR kernel: a row by 512 threads has up to 4,096 entries in
// flight (a 5,000-entry row sets the time of a small power-law matrix).  Rows of
// kWaveNnz + 1 to kWideRowNnz entries go to a wave each where there are enough of
// them to fill the chip (launch::CsrWave::nwide), else, and longer ones, to a
// work-group each.  Columns of neighbouring rows overlapping / anywhere, k = 1, 4
// and 16, us: 15,000 rows of 1,100 by waves 28 / 33 / 68 and 112 / 229 / 310, by
// work-groups 39 / 80 / 101 and 94 / 231 / 297; 500 rows of 700 5.3 / 6.0 / 9.9
// against 3.6 / 4.5 / 4.6; 3,000 rows of 5,000 by work-groups 25 / 35 / 74 and 98 /
// 206 / 278.
constexpr int kMultiThreads = 512;

// One row longer than kWaveNnz by a team of T threads (a wave or the
// work-group), t its thread: "slot" t of T sums entries t, t + T, ... in order,
// and the slots are added by the tree of neighbours, neighbours' neighbours, ...
// whatever k is: a lane loads its slot's entries, L lanes hand them round and
// keep the sums of their L slots for Q right-hand sides each.  Rounds past the
// row's end are skipped by the wave, entries past it re-read the last one and
// are not added.  U rounds are in flight.  Returns the wave's sums in sum.
template <int Q, int L, int T, int U, class V, class Acc>
__device__ __forceinline__ void csr_multi_row(unsigned t, int s, unsigned n, const int* __restrict__ col,
                                              const typename V::T* __restrict__ val,
                                              const float* __restrict__ Xq, int k, Acc* sum) {
    typedef VecOf<float, Q> XV;
    const unsigned p = t % L, w0 = __builtin_amdgcn_readfirstlane(t / kWave * kWave);
    // (Unsigned indices from the row's start: the sums stay in range near 2^31
    // entries.)
    col += s;
    val += s;
    Acc a[L][Q];
#pragma unroll
    for (int i = 0; i < L; ++i)
#pragma unroll
        for (int q = 0; q < Q; ++q) a[i][q] = 0;
    for (unsigned base = 0; base + w0 < n; base += U * T) {
        const int rounds = (int)((n - base - w0 + T - 1) / T);  // wave-uniform
        int c[U];
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= rounds) break;
            const unsigned at = min(base + u * T + t, n - 1);
            c[u] = ld_stream(col + at);
            v[u] = V::ld(val + at);
        }
        typename XV::type xv[U][L];
        float vs[U][L];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= rounds) break;
            int cs[L];
            cs[0] = group_lane<L, 0>(c[u]);
            vs[u][0] = group_lane<L, 0>(v[u]);
            if constexpr (L >= 2) {
                cs[1] = group_lane<L, 1>(c[u]);
                vs[u][1] = group_lane<L, 1>(v[u]);
            }
            if constexpr (L == 4) {
                cs[2] = group_lane<L, 2>(c[u]);
                vs[u][2] = group_lane<L, 2>(v[u]);
                cs[3] = group_lane<L, 3>(c[u]);
                vs[u][3] = group_lane<L, 3>(v[u]);
            }
#pragma unroll
            for (int i = 0; i < L; ++i)
                xv[u][i] = *reinterpret_cast<const typename UVec<float, Q>::type*>(Xq + (size_t)cs[i] * k);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= rounds) break;
#pragma unroll
            for (int i = 0; i < L; ++i) {
                const bool in = base + u * T + t - p + i < n;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const Acc f = fma((Acc)vs[u][i], (Acc)XV::get(xv[u][i], q), a[i][q]);
                    a[i][q] = in ? f : a[i][q];
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        Acc b = a[0][q];
        if constexpr (L == 2) b += a[1][q];
        if constexpr (L == 4) b = (b + a[1][q]) + (a[2][q] + a[3][q]);
        for (int m = L; m < kWave; m <<= 1) b += __shfl_xor(b, m, kWave);
        sum[q] = b;
    }
}

// Rounds of a long row in flight, by the registers that leave three work-groups a
// CU.  Up to kBesideNnz entries beside as many blocks of short rows, one: more
// loads in flight only slow the blocks (power-law rows, FP32, k = 4 / 8 / 16, 600,000:
// 111 / 149 / 182 -> 104 / 136 / 177 us, 1 M: 225 / 274 / 317 -> 200 / 261 / 309).  By
// themselves the rows gain from them (3,000 of 5,000 overlapping columns, k = 1 / 8:
// 38.6 / 54.4 -> 25.6 / 45.9 us; one of 1 M, k = 1: 1172 -> 312).
constexpr int kBesideNnz = 8192;
template <int Q, int L>
constexpr int kRounds = (Q >= 3 && L < 4 ? 6 : 8) / L;

// A row by the work-group (ROUNDS in flight): the eight waves' sums are combined in a fixed order
// through LDS, and Y[:, r] is updated once per right-hand side (rows summed in
// FP64 rounded once).
template <int Q, int L, int ROUNDS, class V, class Acc>
__device__ __forceinline__ void csr_multi_long(const typename V::T* __restrict__ val,
                                               const int* __restrict__ col, int r, int s, int n,
                                               const float* __restrict__ X, int k, float* __restrict__ Y, int ldy,
                                               bool accumulate, Acc (*part)[launch::kMultiMax]) {
    const int t = threadIdx.x, q0 = t % L * Q, qs = min(q0, k - Q);
    Acc sum[Q];
    csr_multi_row<Q, L, kMultiThreads, ROUNDS, V, Acc>(t, s, n, col, val, X + qs, k, sum);
    if (t % kWave < L && q0 < k) {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (qs + q >= q0) part[t / kWave][qs + q] = sum[q];
    }
    __syncthreads();
    if (t < k) {
        Acc tot = 0;
#pragma unroll
        for (int w = 0; w < kMultiThreads / kWave; ++w) tot += part[w][t];
        float* yp = Y + (size_t)t * ldy + r;
        const float y0 = accumulate ? *yp : 0.0f;
        if constexpr (sizeof(Acc) == sizeof(double))
            *yp = (float)((double)y0 + tot);
        else
            *yp = y0 + tot;
    }
}

// Entries of a unit (below).
constexpr int kUnit = 8;

// A block whose rows hold at most four entries each: a lane per row, without
// the units' pass through LDS (2 M rows of one entry, k = 1 / 2 / 4: 22.2 / 28.9 /
// 36.8 -> 11.5 / 14.6 / 22.1 us).  The sums are the units', bit for bit: a row's
// entries up to the next multiple of kUnit from the block's start in one chain,
// those after it in another.  False: some row is longer, nothing was done.
template <int Q, class V>
__device__ __forceinline__ bool csr_multi_short(int lane, int r0, int nrows, int s, int n, const int* __restrict__ rp,
                                                const int* __restrict__ col, const typename V::T* __restrict__ val,
                                                int k, const float* __restrict__ X, float* __restrict__ Y, int ldy,
                                                bool accumulate) {
    constexpr int M = 4;
    typedef VecOf<float, Q> XV;
    if (n > M * kWave) return false;
    const bool row = lane < nrows;
    const int b0 = rp[r0 + min(lane, nrows)] - s, b1 = rp[r0 + min(lane + 1, nrows)] - s, len = b1 - b0;
    if (__ballot(len > M)) return false;
    float first[Q], a[Q], y[Q];
    bool two = false;
#pragma unroll
    for (int q = 0; q < Q; ++q) first[q] = a[q] = y[q] = 0.0f;
    const bool write = row && !(len == 0 && accumulate);  // empty rows leave Y as it is
    if (write && accumulate) {
#pragma unroll
        for (int q = 0; q < Q; ++q) y[q] = Y[(size_t)q * ldy + r0 + lane];
    }
    col += s;
    val += s;
    int c[M];
    float v[M];
    typename XV::type xv[M];
#pragma unroll
    for (int e = 0; e < M; ++e) {
        if (e >= len) continue;
        c[e] = ld_stream(col + b0 + e);
        v[e] = V::ld(val + b0 + e);
    }
#pragma unroll
    for (int e = 0; e < M; ++e)
        if (e < len) xv[e] = *reinterpret_cast<const typename UVec<float, Q>::type*>(X + (size_t)c[e] * k);
#pragma unroll
    for (int e = 0; e < M; ++e) {
        if (e >= len) continue;
        if (e > 0 && (b0 + e) % kUnit == 0) {
            two = true;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                first[q] = a[q];
                a[q] = 0.0f;
            }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) a[q] = fmaf(v[e], XV::get(xv[e], q), a[q]);
    }
    if (write) {
#pragma unroll
        for (int q = 0; q < Q; ++q) Y[(size_t)q * ldy + r0 + lane] = y[q] + (two ? first[q] + a[q] : a[q]);
    }
    return true;
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
// Power-law rows: 600,011 rows, BF16, k = 8 / 16: 191 / 318 -> 132 / 172 us; 1 M
// rows, FP32, k = 5 / 8 / 16: 357 / 329 / 528 -> 247 / 260 / 300 us (52 G rows/s);
// 27-point stencil 64^3, k = 8: 74 -> 28 us.
template <int Q, int L, class V>
__global__ __launch_bounds__(kMultiThreads, L == 4 ? 4 : 6) void csr_multi_kernel(
    int nlong, int nwide, const int* __restrict__ longs, int nblk, const int4* __restrict__ blk,
    const int* __restrict__ rp, const int* __restrict__ col, const typename V::T* __restrict__ val, int k,
    const float* __restrict__ X, float* __restrict__ Y, int ldy, bool accumulate) {
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
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int q0 = lane % L * Q, qs = min(q0, k - Q);  // the last piece ends at k
    const int nlwg = nwide + (nlong - nwide + kWaves - 1) / kWaves;
    if ((int)blockIdx.x < nwide) {  // the longest work first
        const int r = longs[blockIdx.x], j0 = rp[r], n = rp[r + 1] - j0;
        auto row = [&](auto rounds) {
            constexpr int R = decltype(rounds)::value;
            if (n > launch::kLongRowF64)
                csr_multi_long<Q, L, R, V, double>(val, col, r, j0, n, X, k, Y, ldy, accumulate, lds.part64);
            else
                csr_multi_long<Q, L, R, V, float>(val, col, r, j0, n, X, k, Y, ldy, accumulate, lds.part);
        };
        if (nblk >= nwide && n <= kBesideNnz) row(std::integral_constant<int, 1>{});
        else row(std::integral_constant<int, kRounds<Q, L>>{});
        return;
    }
    if ((int)blockIdx.x < nlwg) {  // a wave per row
        const int at = nwide + ((int)blockIdx.x - nwide) * kWaves + wave;
        if (at >= nlong) return;
        const int r = longs[at], j0 = rp[r], n = rp[r + 1] - j0;
        float sum[Q], y[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) y[q] = accumulate ? Y[(size_t)(qs + q) * ldy + r] : 0.0f;
        csr_multi_row<Q, L, kWave, kRounds<Q, L>, V, float>(lane, j0, n, col, val, X + qs, k, sum);
        if (lane < L && q0 < k) {
#pragma unroll
            for (int q = 0; q < Q; ++q)
                if (qs + q >= q0) Y[(size_t)(qs + q) * ldy + r] = y[q] + sum[q];
        }
        return;
    }
    const int b = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x - nlwg, gridDim.x - nlwg) * kWaves + wave);
    if (b >= nblk) return;  // the whole wave
    const int4 B = blk[b];  // {first row, rows, first entry, entries}
    const int r0 = B.x, nrows = B.y, s = B.z, n = B.w;
    WaveLds& W = lds.w[wave];
    const int gi = lane / L, p = lane % L;
    const bool act = q0 < k;
    const float* Xq = X + qs;
    if constexpr (L == 1) {
        if (csr_multi_short<Q, V>(lane, r0, nrows, s, n, rp, col, val, k, Xq, Y, ldy, accumulate)) return;
    }
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
    constexpr int kWaves = kMultiThreads / kWave;
    const int groups = W.nwide + ceil_div(W.nlong - W.nwide, kWaves) + ceil_div(W.nblk, kWaves);
    hipLaunchKernelGGL((csr_multi_kernel<Q, L, V>), dim3(groups), dim3(kMultiThreads), 0, s, W.nlong, W.nwide, W.longs,
                       W.nblk, W.blk, rp, col, static_cast<const typename V::T*>(val), k, X, Y, ldy, accumulate);
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
