// DIA and BDIA SpMV for gfx950 (replace kernels/spmv_dia.cl and
// kernels/spmv_bdia.cl).
//
// Storage is diagonal-major: diagonal j of row r sits at data[j*len + r], so
// each diagonal is one coalesced stream.  Offsets are wave-uniform and come
// in through scalar loads.  x is read either directly (every row's x
// elements are contiguous across the wave and reused from L1/L2) or from an
// LDS window staged once per work-group:
//   DIA : one window covering [min offset, max offset + rows of the group)
//   BDIA: one window per band (consecutive offsets), double buffered so that
//         staging band b+1 needs a single barrier.
// BDIA methods without LDS run the DIA kernels over the band's diagonals
// listed one by one (the runtime expands the band offsets at upload).
// Out-of-range columns read zero, which replaces the reference's padded
// `vec_extended` copy of x (src/spmv_cocktail.cpp:253-301).  Unlike the
// reference's gpu_bdia there is no band-count or band-width limit
// (MAX_BAND_NUM 31, MAX_BAND_WIDTH 128); bands wider than the LDS window fall
// back to direct x loads.

#include "device_common.hpp"
#include "kernels.hpp"

namespace clspmv {
namespace {

using namespace dev;

__device__ __forceinline__ float x_at(const float* __restrict__ x, int c, int cols) {
    return (unsigned)c < (unsigned)cols ? x[c] : 0.0f;
}

// ---- DIA ---------------------------------------------------------------------

// One row per lane; U diagonals per iteration with independent
// accumulators so that U data streams and U x reads are in flight per lane.
template <int U, class V>
__global__ __launch_bounds__(kBlock) void dia1_kernel(
    int rows, int cols, int len, int ndiag, const int* __restrict__ off,
    const typename V::T* __restrict__ data, const float* __restrict__ x,
    float* __restrict__ y) {
    const int r = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (r >= rows) return;
    float a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = 0.0f;
    int j = 0;
    for (; j + U <= ndiag; j += U) {
        float d[U], xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) d[u] = V::ld(data + (size_t)(j + u) * len + r);
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x_at(x, r + off[j + u], cols);
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = fmaf(d[u], xv[u], a[u]);
    }
    for (; j < ndiag; ++j) a[0] = fmaf(V::ld(data + (size_t)j * len + r), x_at(x, r + off[j], cols), a[0]);
    float sum = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) sum += a[u];
    y[r] += sum;
}

// One row per lane with every diagonal in flight at once (ndiag <= N): the
// lane issues all N data loads and x loads before its first product, so a
// wave keeps N coalesced 256-byte streams outstanding instead of U, and the
// products are then summed in diagonal order.  Slots j >= ndiag re-load the
// last diagonal (cache hits) and are not added.
template <int N, class V>
__global__ __launch_bounds__(kBlock) void dia_row_kernel(
    int rows, int cols, int len, int ndiag, const int* __restrict__ off,
    const typename V::T* __restrict__ data, const float* __restrict__ x,
    float* __restrict__ y) {
    const int r = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (r >= rows) return;
    float d[N], xv[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int jj = j < ndiag ? j : ndiag - 1;  // wave-uniform
        d[j] = V::ld(data + (size_t)jj * len + r);
        xv[j] = x_at(x, r + off[jj], cols);
    }
    float a = 0.0f;
#pragma unroll
    for (int j = 0; j < N; ++j) a = j < ndiag ? fmaf(d[j], xv[j], a) : a;
    y[r] += a;
}

// Four consecutive rows per lane over the segments of consecutive offsets
// (launch::dia_multi's; at most W diagonals each), S segments' loads in flight:
// a diagonal's four values are one load and the W + 3 x values that a
// segment's rows need are two, where dia_row_kernel issues 2 W loads per row.
// The sums are dia_row_kernel's, in diagonal order, bit for bit; x reads zero
// outside the matrix.  len must be a multiple of 4.
//
// 16-bit values only, from 15 << 16 rows and 8 M values on: 27-point stencil 101^3 /
// 128^3 14.5 / 27.3 -> 13.4 / 26.6 us, 5-point Laplacian of 2 M rows 11.0 -> 9.6,
// nine-point 13.9 -> 12.1; below, the waves are too few (27-point stencil of
// 800,000 rows 11.8 -> 12.6 us, 400,000 7.4 -> 11.1).  And few segments, or full
// runs: a wave walks them one after the other (1 M rows, 16 consecutive diagonals
// 9.5 -> 11.4 us, 19-point stencil 11.3 -> 12.4; by S = 5 lone ones, 2 M rows, 5 / 7 /
// 31 of them 11.0 / 11.1 / 31.1 -> 9.0 / 12.3 / 37.0).  FP32 values already set
// dia_row_kernel's pace (128^3 42.3 against 42.7 us, 1400^2 12.4 against 13.1).
constexpr int kQuadRows = 15 << 16;
constexpr long long kQuadValues = 8 << 20;
bool quad_segments(const launch::DiaSegments& S, int ndiag) {
    if (S.width == 1) return S.count <= 5;
    return S.count <= 3 || (S.count <= 9 && ndiag == S.width * S.count);
}
template <int W, int S, class V>
__global__ __launch_bounds__(kBlock) void dia_quad_kernel(
    int rows, int cols, int len, int nseg, const int4* __restrict__ seg,
    const typename V::T* __restrict__ data, const float* __restrict__ x, float* __restrict__ y) {
    constexpr int R = 4, NX = R + W - 1;
    typedef typename V::T T;
    const unsigned r0u = ((unsigned)xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x) * R;
    const unsigned w0u = __builtin_amdgcn_readfirstlane(r0u);
    if (w0u >= (unsigned)rows) return;  // the whole wave
    const int w0 = (int)w0u, xl = (int)(r0u - w0u), r0 = w0 + min(xl, rows - w0);
    const int dl = min(xl, len - R - w0);
    float acc[R] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < nseg; s += S) {
        float xv[S][NX];
        typename VecOf<T, R>::type d[S][W];
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const int4 sg = seg[min(s + i, nseg - 1)];
            const long long c0 = (long long)w0 + sg.y;
            if (c0 >= 0 && c0 + kWave * R + W - 1 <= cols) {
                const float* xp = x + c0;
                const f32x4 a = *reinterpret_cast<const UVec<float, 4>::type*>(xp + xl);
#pragma unroll
                for (int e = 0; e < R; ++e) xv[i][e] = a[e];
                if constexpr (W > 1) {
                    typedef VecOf<float, W - 1> XV;
                    const typename XV::type b =
                        *reinterpret_cast<const typename UVec<float, W - 1>::type*>(xp + xl + R);
#pragma unroll
                    for (int e = 0; e < W - 1; ++e) xv[i][R + e] = XV::get(b, e);
                }
            } else {
#pragma unroll
                for (int e = 0; e < NX; ++e) xv[i][e] = x_at(x, r0 + sg.y + e, cols);
            }
            // Diagonals past the segment's re-read its last one and are not added.
            const T* dp = data + (size_t)sg.x * len + w0;
#pragma unroll
            for (int n = 0; n < W; ++n)
                d[i][n] = __builtin_nontemporal_load(
                    reinterpret_cast<const typename UVec<T, R>::type*>(dp + (size_t)min(n, sg.z - 1) * len + dl));
        }
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const int z = s + i < nseg ? seg[s + i].z : 0;
#pragma unroll
            for (int n = 0; n < W; ++n)
                if (n < z)
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r] = fmaf(V::cvt(d[i][n][r]), xv[i][n + r], acc[r]);
        }
    }
    const int left = rows - w0 - xl;  // rows from the lane's first on
    if (left >= R) {
        typedef UVec<float, R>::type YU;
        f32x4 v = *reinterpret_cast<const YU*>(y + r0);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] += acc[r];
        *reinterpret_cast<YU*>(y + r0) = v;
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r < left) y[r0 + r] += acc[r];
    }
}

// Two consecutive rows per lane (64-bit data loads, len % 2 == 0), U
// diagonals per iteration.
template <int U, class V>
__global__ __launch_bounds__(kBlock) void dia2_kernel(
    int rows, int cols, int len, int ndiag, const int* __restrict__ off,
    const typename V::T* __restrict__ data, const float* __restrict__ x,
    float* __restrict__ y) {
    const int r = (xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x) * 2;
    if (r >= rows) return;
    float a0[U], a1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) a0[u] = a1[u] = 0.0f;
    int j = 0;
    for (; j + U <= ndiag; j += U) {
        float2 d[U];
        float x0[U], x1[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            d[u] = V::ld2(data + (size_t)(j + u) * len + r);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = r + off[j + u];
            x0[u] = x_at(x, c, cols);
            x1[u] = x_at(x, c + 1, cols);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a0[u] = fmaf(d[u].x, x0[u], a0[u]);
            a1[u] = fmaf(d[u].y, x1[u], a1[u]);
        }
    }
    for (; j < ndiag; ++j) {
        const float2 d = V::ld2(data + (size_t)j * len + r);
        const int c = r + off[j];
        a0[0] = fmaf(d.x, x_at(x, c, cols), a0[0]);
        a1[0] = fmaf(d.y, x_at(x, c + 1, cols), a1[0]);
    }
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        s0 += a0[u];
        s1 += a1[u];
    }
    y[r] += s0;
    if (r + 1 < rows) y[r + 1] += s1;
}

// RPT rows per lane (strided by the work-group size) with the work-group's x
// window in LDS; the host guarantees RPT*kBlock + span <= kLdsWindow.
template <int RPT, class V>
__global__ __launch_bounds__(kBlock) void dia_lds_kernel(
    int rows, int cols, int len, int ndiag, const int* __restrict__ off,
    int min_off, int span, const typename V::T* __restrict__ data,
    const float* __restrict__ x, float* __restrict__ y) {
    __shared__ float win[launch::kLdsWindow];
    const int t = threadIdx.x;
    const int r0 = xcd_tile(blockIdx.x, gridDim.x) * kBlock * RPT;
    const int ws = r0 + min_off;
    const int wn = kBlock * RPT + span;
    for (int i = t; i < wn; i += kBlock) win[i] = x_at(x, ws + i, cols);
    __syncthreads();
    float a[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) a[q] = 0.0f;
    for (int j = 0; j < ndiag; ++j) {
        const int o = off[j] - min_off;
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int rl = q * kBlock + t;
            if (r0 + rl < rows)
                a[q] = fmaf(V::ld(data + (size_t)j * len + r0 + rl), win[rl + o], a[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = r0 + q * kBlock + t;
        if (r < rows) y[r] += a[q];
    }
}

// ---- BDIA --------------------------------------------------------------------

// RPT rows per lane strided by the work-group size; per band an LDS window
// [r0 + first offset, r0 + first offset + RPT*kBlock + width - 1), double
// buffered.  The host guarantees RPT*kBlock + max band width <= kLdsWindow/2.
template <int RPT>
__global__ __launch_bounds__(kBlock) void bdia_lds_kernel(
    int rows, int cols, int len, int nband, const int* __restrict__ boff,
    const int* __restrict__ bptr, const float* __restrict__ data,
    const float* __restrict__ x, float* __restrict__ y) {
    constexpr int kHalf = launch::kLdsWindow / 2;
    __shared__ float win[2][kHalf];
    const int t = threadIdx.x;
    const int r0 = xcd_tile(blockIdx.x, gridDim.x) * kBlock * RPT;
    float a[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) a[q] = 0.0f;
    for (int b = 0; b < nband; ++b) {
        const int d0 = bptr[b], d1 = bptr[b + 1];
        const int ws = r0 + boff[b];
        const int wn = kBlock * RPT + (d1 - d0) - 1;
        float* w = win[b & 1];
        for (int i = t; i < wn; i += kBlock) w[i] = x_at(x, ws + i, cols);
        __syncthreads();
        for (int d = d0; d < d1; ++d) {
            const int k = d - d0;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int rl = q * kBlock + t;
                if (r0 + rl < rows)
                    a[q] = fmaf(ld_stream(data + (size_t)d * len + r0 + rl), w[rl + k], a[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = r0 + q * kBlock + t;
        if (r < rows) y[r] += a[q];
    }
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

}  // namespace

namespace launch {

template <class V>
hipError_t dia_typed(hipStream_t s, int rows, int cols, int len, int ndiag,
                     const int* offsets, int min_off, int max_off, DiaSegments S, int method,
                     const typename V::T* data, const float* x, float* y) {
    const int span = max_off - min_off;
    switch (method) {
        case 0: {
            // Up to 32 diagonals: all in flight (the smallest multiple of 4
            // slots that holds them); more: 8 at a time.
            const dim3 g(ceil_div(rows, kBlock)), b(kBlock);
            if constexpr (sizeof(typename V::T) == 2) {
                if (ndiag <= 32 && S.count > 0 && rows >= kQuadRows && rows * (long long)ndiag >= kQuadValues &&
                    len % 4 == 0 && quad_segments(S, ndiag)) {
                    const dim3 q(ceil_div(rows, 4 * kBlock));
                    if (S.width == 1)
                        hipLaunchKernelGGL((dia_quad_kernel<1, 5, V>), q, b, 0, s, rows, cols, len, S.count, S.seg,
                                           data, x, y);
                    else
                        hipLaunchKernelGGL((dia_quad_kernel<kDiaRun, 1, V>), q, b, 0, s, rows, cols, len, S.count,
                                           S.seg, data, x, y);
                    break;
                }
            }
            switch ((ndiag + 3) / 4) {
#define CLSPMV_DIA_ROW(Q)                                                                              \
    case Q:                                                                                           \
        hipLaunchKernelGGL((dia_row_kernel<4 * Q, V>), g, b, 0, s, rows, cols, len, ndiag, offsets, data, x, y); \
        break;
                CLSPMV_DIA_ROW(1)
                CLSPMV_DIA_ROW(2)
                CLSPMV_DIA_ROW(3)
                CLSPMV_DIA_ROW(4)
                CLSPMV_DIA_ROW(5)
                CLSPMV_DIA_ROW(6)
                CLSPMV_DIA_ROW(7)
                CLSPMV_DIA_ROW(8)
#undef CLSPMV_DIA_ROW
                default:
                    hipLaunchKernelGGL((dia1_kernel<8, V>), g, b, 0, s, rows, cols, len, ndiag, offsets, data, x, y);
            }
            break;
        }
        case 1:
            if (len % 2) return hipErrorInvalidValue;
            hipLaunchKernelGGL((dia2_kernel<4, V>), dim3(ceil_div(rows, 2 * kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, ndiag, offsets, data, x, y);
            break;
        case 2:
            if (kBlock + span > kLdsWindow) return hipErrorInvalidValue;
            hipLaunchKernelGGL((dia_lds_kernel<1, V>), dim3(ceil_div(rows, kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, ndiag, offsets, min_off, span, data, x, y);
            break;
        case 3:
            if (4 * kBlock + span > kLdsWindow) return hipErrorInvalidValue;
            hipLaunchKernelGGL((dia_lds_kernel<4, V>), dim3(ceil_div(rows, 4 * kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, ndiag, offsets, min_off, span, data, x, y);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t dia(hipStream_t s, int rows, int cols, int len, int ndiag,
               const int* offsets, int min_off, int max_off, DiaSegments S, int method, int dtype,
               const void* data, const float* x, float* y) {
    if (rows <= 0 || ndiag <= 0) return hipSuccess;
    switch (dtype) {
        case 0:
            return dia_typed<ValF32>(s, rows, cols, len, ndiag, offsets, min_off, max_off, S, method,
                                     static_cast<const float*>(data), x, y);
        case 1:
            return dia_typed<ValBF16>(s, rows, cols, len, ndiag, offsets, min_off, max_off, S, method,
                                      static_cast<const unsigned short*>(data), x, y);
        case 2:
            return dia_typed<ValF16>(s, rows, cols, len, ndiag, offsets, min_off, max_off, S, method,
                                     static_cast<const unsigned short*>(data), x, y);
        default:
            return hipErrorInvalidValue;
    }
}

hipError_t bdia(hipStream_t s, int rows, int cols, int len, int nband,
                const int* band_off, const int* bptr, int max_band_width,
                int method, const float* data, const float* x, float* y) {
    if (rows <= 0 || nband <= 0) return hipSuccess;
    const int half = kLdsWindow / 2;
    switch (method) {
        case 1:
            if (kBlock + max_band_width > half) return hipErrorInvalidValue;
            hipLaunchKernelGGL(bdia_lds_kernel<1>, dim3(ceil_div(rows, kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, nband, band_off, bptr, data, x, y);
            break;
        case 2:
            if (2 * kBlock + max_band_width > half) return hipErrorInvalidValue;
            hipLaunchKernelGGL(bdia_lds_kernel<2>, dim3(ceil_div(rows, 2 * kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, nband, band_off, bptr, data, x, y);
            break;
        case 4:
            if (4 * kBlock + max_band_width > half) return hipErrorInvalidValue;
            hipLaunchKernelGGL(bdia_lds_kernel<4>, dim3(ceil_div(rows, 4 * kBlock)), dim3(kBlock), 0, s,
                               rows, cols, len, nband, band_off, bptr, data, x, y);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace launch
}  // namespace clspmv
