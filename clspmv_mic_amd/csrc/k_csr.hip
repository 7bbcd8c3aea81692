// CSR SpMV kernels for gfx950 (replace kernels/spmv_csr_scalar.cl and
// kernels/spmv_csr_vector.cl).
//
// csr_vector<G>: G lanes of a wave share one row (G = 1 is the scalar
//   kernel).  Lanes stride over the row, then a lane-group xor-shuffle sum
//   replaces the reference's barrier-free "volatile" LDS tree
//   (kernels/spmv_csr_vector.cl:32-38).
// csr_wave: one wave per host-built block of rows whose entries fit
//   kWaveNnz, a work-group per longer row.  Every row belongs to exactly one
//   of them, so y is written without atomics and results do not depend on
//   what else runs on the GPU.

#include "device_common.hpp"
#include "kernels.hpp"

namespace clspmv {
namespace {

using namespace dev;

template <int G>
__global__ __launch_bounds__(kBlock) void csr_vector_kernel(
    int rows, const int* __restrict__ rp, const int* __restrict__ col,
    const float* __restrict__ val, const float* __restrict__ x,
    float* __restrict__ y) {
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int row = (tile * kBlock + (int)threadIdx.x) / G;
    const int lane = threadIdx.x & (G - 1);
    if (row >= rows) return;  // a lane group always exits together
    const int s = rp[row], e = rp[row + 1];
    float a0 = 0.0f, a1 = 0.0f;
    int k = s + lane;
    // Two independent accumulators keep two gathers in flight per lane.
    for (; k + G < e; k += 2 * G) {
        const int c0 = ld_stream(col + k), c1 = ld_stream(col + k + G);
        const float v0 = ld_stream(val + k), v1 = ld_stream(val + k + G);
        a0 = fmaf(v0, x[c0], a0);
        a1 = fmaf(v1, x[c1], a1);
    }
    if (k < e) a0 = fmaf(ld_stream(val + k), x[ld_stream(col + k)], a0);
    float sum = group_sum<G>(a0 + a1);
    if (lane == 0) y[row] += sum;
}

// One row longer than kWaveNnz by the whole work-group: it strides over the
// row, U entries' loads in flight per thread also in the last round (a row of
// up to 2,048 entries is one round), each thread's sum in index order; the
// waves' sums are added in order.  Acc is double for rows longer
// than kLongRowF64 of 16-bit values: their products are exact and the row is
// rounded once, into y.
template <class V, class Acc, int kWaves>
__device__ __forceinline__ void csr_long_row(int s, int e, const int* __restrict__ col,
                                             const typename V::T* __restrict__ val,
                                             const float* __restrict__ x, float* __restrict__ y,
                                             Acc* part) {
    constexpr int U = 4, kThreads = kWave * kWaves;
    const int t = threadIdx.x;
    Acc acc = 0;
    // (Indices from the row's start: the sums stay in range near 2^31 entries.)
    const int n = e - s;
    col += s;
    val += s;
    for (int k = t; k < n; k += U * kThreads) {
        int c[U];
        float v[U], xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {  // past the end: the last entry again, not added
            const int at = min(k + u * kThreads, n - 1);
            c[u] = ld_stream(col + at);
            v[u] = V::ld(val + at);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x[c[u]];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u * kThreads < n) acc = fma((Acc)v[u], (Acc)xv[u], acc);
    }
    for (int m = kWave >> 1; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, kWave);
    if (t % kWave == 0) part[t / kWave] = acc;
    __syncthreads();
    if (t == 0) {
        Acc tot = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) tot += part[w];
        *y = sizeof(Acc) == sizeof(double) ? (float)((double)*y + (double)tot) : *y + (float)tot;
    }
}

// A row over kWaveNnz by a wave, where there are enough of them to fill the chip
// (launch::CsrWave::nwide): 30,000 rows of 513 / 15,000 of 1,100 overlapping
// columns 27 / 27.5 us, by a work-group each 35 / 31 us.  Not 16-bit values, whose
// long rows the work-groups already take in 33 / 28 us (by waves 33 / 32.6).
template <class V>
__device__ __forceinline__ float csr_wave_row(int lane, int s, int n, const int* __restrict__ col,
                                              const typename V::T* __restrict__ val, const float* __restrict__ x) {
    constexpr int U = 8;
    float acc = 0.0f;
    col += s;
    val += s;
    for (int base = 0; base < n; base += U * kWave) {
        const int rounds = (n - base + kWave - 1) / kWave;
        int c[U];
        float v[U], xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {  // past the end: the last entry again, not added
            if (u >= rounds) break;
            const int at = min(base + u * kWave + lane, n - 1);
            c[u] = ld_stream(col + at);
            v[u] = V::ld(val + at);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= rounds) break;
            xv[u] = x[c[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= rounds) break;
            acc = base + u * kWave + lane < n ? fmaf(v[u], xv[u], acc) : acc;
        }
    }
    return group_sum<kWave>(acc);
}

// What bounds it: the gathers of x, and before that the waves' chain of
// dependent loads (block, columns, x).  A wave loads the up to kWaveNnz entries
// of its block at once as 16-byte pieces (the arrays carry kWaveNnz entries
// of padding, so no load is guarded), the x values of its 8 entries per lane
// at once, and leaves the products in its own part of LDS, where lane groups
// sized to the row count sum the rows: no barrier, 32 waves per CU.  Against
// lanes striding over rows (csr_vector) and a work-group per 1024 entries
// with a barrier: 27-point stencil 77^3 52 / 31 -> 23.5 us, 5-point Laplacian
// 701^2 15 / 10.5 -> 7 us.
//
// WIN: gathers through L1 return in order behind the streams; without them
// the 27-point stencil 97^3 (24.6 M entries) ran in 31.8 us instead of 47.7.
// Where the rows of a work-group share x, it stages their chunks of x in LDS
// (launch::XStage) while the entries are in flight and gathers there, by
// 16-bit places instead of 32-bit columns (6 bytes an entry): 27-point stencil
// 77^3 23.5 -> 15.1 us (81.6 MB of HBM traffic), 47^3 7.3 -> 5.4, 5-point Laplacian
// 1000^2 11.4 -> 9.7, mesh of 700,000 rows of 25 48.2 -> 24.6 us.
//
// A skewed block (a row of 400 entries among 50 of a few) would leave the long
// row's sum to the one or two lanes its row count gives each row; rows of more
// than kWideRow entries per lane go to the whole wave instead: power-law rows,
// 30,000: 9.7 -> 5.5 us, 270,342: 36 -> 32.7 us (16 per lane: mesh of 50,009
// rows 5.8 -> 7.9 us; 32 no different; 128: 6.4 us on the 30,000 rows).
constexpr int kWideRow = 64;

// Waves of a work-group that stages no x: the fewer, the sooner a long row's
// work-group finds room, the more, the shorter its chain (2 / 4 / 8 waves:
// power-law rows 96,050 13.9 / 11.6 / 12.4 us, 1 M 105.4 / 106.2 / 107.3).
constexpr int kPlainWaves = 4;

template <class V, bool WIN, int kWaves>
__global__ __launch_bounds__(kWave* kWaves) void csr_wave_kernel(
    int nlong, int nwide, const int* __restrict__ longs, int nblk, const int4* __restrict__ blk,
    const int* __restrict__ list, const unsigned short* __restrict__ idx, int stride, int cols,
    const int* __restrict__ rp, const int* __restrict__ col,
    const typename V::T* __restrict__ val, const float* __restrict__ x, float* __restrict__ y) {
    constexpr int U = launch::kWaveNnz / kWave, P4 = kWave * 4;
    typedef typename V::T T;
    typedef typename UVec<T, 4>::type T4U;
    typedef VecOf<unsigned short, 4> I4;
    extern __shared__ __attribute__((aligned(16))) float sm[];  // x chunks, then the products of each wave
    const int nlwg = nwide + (nlong - nwide + kWaves - 1) / kWaves;
    if ((int)blockIdx.x < nwide) {  // the longest work first
        const int r = longs[blockIdx.x], s = rp[r], e = rp[r + 1];
        double* part = reinterpret_cast<double*>(sm);
        if (sizeof(T) == 2 && e - s > launch::kLongRowF64)
            csr_long_row<V, double, kWaves>(s, e, col, val, x, y + r, part);
        else
            csr_long_row<V, float, kWaves>(s, e, col, val, x, y + r, reinterpret_cast<float*>(part));
        return;
    }
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    if (sizeof(T) == 4 && (int)blockIdx.x < nlwg) {
        const int at = nwide + ((int)blockIdx.x - nwide) * kWaves + wave;
        if (at >= nlong) return;
        const int r = longs[at], s = rp[r];
        const float sum = csr_wave_row<V>(lane, s, rp[r + 1] - s, col, val, x);
        if (lane == 0) y[r] += sum;
        return;
    }
    const int wg = xcd_tile(blockIdx.x - nlwg, gridDim.x - nlwg);
    const int b = __builtin_amdgcn_readfirstlane(wg * kWaves + wave);
    if (!WIN && b >= nblk) return;
    StageX<kWave * kWaves> stage;
    if constexpr (WIN) stage.ids(list + (size_t)wg * stride, stride);
    int4 B = blk[min(b, nblk - 1)];  // {first row, rows, first entry, entries}
    if (WIN && b >= nblk) B.y = B.w = 0;
    const int nrows = B.y, s = B.z, n = B.w;
    i32x4 c[U / 4];
    typename I4::type ix[U / 4];
    typename VecOf<T, 4>::type v[U / 4];
#pragma unroll
    for (int u = 0; u < U / 4; ++u) {
        const unsigned at = u * P4 + lane * 4;
        if constexpr (WIN)
            ix[u] = __builtin_nontemporal_load(reinterpret_cast<const UVec<unsigned short, 4>::type*>((idx + s) + at));
        else
            c[u] = __builtin_nontemporal_load(reinterpret_cast<const UVec<int, 4>::type*>((col + s) + at));
        v[u] = __builtin_nontemporal_load(reinterpret_cast<const T4U*>((val + s) + at));
    }
    // Lane groups for the sums: the largest power of two with nrows groups in
    // the wave (a block holds at most kWave rows).
    const int sh = nrows > 32 ? 0 : nrows > 16 ? 1 : nrows > 8 ? 2 : nrows > 4 ? 3 : nrows > 2 ? 4 : nrows > 1 ? 5 : 6;
    const int g = 1 << sh, gl = lane & (g - 1);
    const bool live = (lane >> sh) < nrows;
    const int r = B.x + (live ? lane >> sh : 0);
    const int k0 = rp[r] - s, k1 = rp[r + 1] - s;
    const float yv = y[r];
    float* prod = sm + (WIN ? stride * launch::kXChunk : 0) + wave * launch::kWaveNnz;
    if constexpr (WIN) stage.fetch(stride, cols, x, sm);
    const unsigned last = (unsigned)stride * launch::kXChunk - 1u;
#pragma unroll
    for (int u = 0; u < U / 4; ++u) {
        if (u * P4 + lane * 4 >= n) continue;
        f32x4 p;
        if constexpr (WIN) {  // entries past the block are another work-group's: clamped, not read
#pragma unroll
            for (int h = 0; h < 4; ++h) p[h] = V::cvt(v[u][h]) * sm[min((unsigned)I4::get(ix[u], h), last)];
        } else {
            float xv[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) xv[h] = x[c[u][h]];
#pragma unroll
            for (int h = 0; h < 4; ++h) p[h] = V::cvt(v[u][h]) * xv[h];
        }
        *reinterpret_cast<f32x4*>(prod + u * P4 + lane * 4) = p;
    }
    wave_lds_order();
    float acc = 0.0f;
    // Rows much longer than the others of their block, one after the other by
    // the whole wave.
    const bool wide = k1 - k0 > kWideRow * g;
    for (unsigned long long m = __ballot(live && wide && gl == 0); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const int e = __builtin_amdgcn_readlane(k1, l);
        float a = 0.0f;
        for (int k = __builtin_amdgcn_readlane(k0, l) + lane; k < e; k += kWave) a += prod[k];
        a = group_sum<kWave>(a);
        if (lane == l) acc = a;
    }
    if (live && !wide) {
        float a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
        int k = k0 + gl;
        for (; k + 3 * g < k1; k += 4 * g) {
            acc += prod[k];
            a1 += prod[k + g];
            a2 += prod[k + 2 * g];
            a3 += prod[k + 3 * g];
        }
        for (; k < k1; k += g) acc += prod[k];
        acc = (acc + a1) + (a2 + a3);
    }
    acc = group_sum_rt(acc, g);
    if (live && gl == 0) y[r] = yv + acc;
}

template <class V>
hipError_t csr_wave_v(hipStream_t s, const launch::CsrWave& W, const int* rp, const int* col, const void* val,
                      int cols, const float* x, float* y) {
    const typename V::T* v = static_cast<const typename V::T*>(val);
    auto launch = [&](auto kernel, int waves, const launch::XStage& X) {
        const int nwide = sizeof(typename V::T) == 4 ? W.nwide : W.nlong;  // rows by a work-group each
        const dim3 grid(nwide + (W.nlong - nwide + waves - 1) / waves + (W.nblk + waves - 1) / waves),
            block(kWave * waves);
        const size_t lds = sizeof(float) * (launch::kWaveNnz * waves + launch::kXChunk * X.stride);
        hipLaunchKernelGGL(kernel, grid, block, lds, s, W.nlong, nwide, W.longs, W.nblk, W.blk, X.list, X.idx,
                           X.stride, cols, rp, col, v, x, y);
    };
    if (W.stage.list)
        launch(csr_wave_kernel<V, true, launch::kCsrWaves>, launch::kCsrWaves, W.stage);
    else
        launch(csr_wave_kernel<V, false, kPlainWaves>, kPlainWaves, launch::XStage{});
    return hipGetLastError();
}

}  // namespace

namespace launch {

hipError_t csr_vector(hipStream_t s, int rows, int lanes, const int* rp,
                      const int* col, const float* val, const float* x, float* y) {
    if (rows <= 0) return hipSuccess;
    const long long threads = (long long)rows * lanes;
    const int grid = (int)((threads + kBlock - 1) / kBlock);
#define CSRV(G)                                                                 \
    case G:                                                                     \
        hipLaunchKernelGGL(csr_vector_kernel<G>, dim3(grid), dim3(kBlock), 0, s, \
                           rows, rp, col, val, x, y);                           \
        break;
    switch (lanes) {
        CSRV(1) CSRV(2) CSRV(4) CSRV(8) CSRV(16) CSRV(32) CSRV(64)
        default: return hipErrorInvalidValue;
    }
#undef CSRV
    return hipGetLastError();
}

hipError_t csr_wave(hipStream_t s, const CsrWave& W, const int* rp, const int* col, int dtype, const void* val,
                    int cols, const float* x, float* y) {
    if (W.nblk + W.nlong <= 0) return hipSuccess;
    switch (dtype) {
        case 0: return csr_wave_v<ValF32>(s, W, rp, col, val, cols, x, y);
        case 1: return csr_wave_v<ValBF16>(s, W, rp, col, val, cols, x, y);
        case 2: return csr_wave_v<ValF16>(s, W, rp, col, val, cols, x, y);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace launch
}  // namespace clspmv
