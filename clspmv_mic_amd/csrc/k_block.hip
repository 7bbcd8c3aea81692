// Blocked SpMV for gfx950: BCSR (b4csr), BELL (b4ell) and SBELL layouts
// (replace kernels/spmv_bcsr.cl, kernels/spmv_bell.cl, kernels/spmv_sbell.cl).
//
// Block shapes bh x bw with bh in {1,2,4,8} and bw in {4,8}; every layout
// keeps each block's row-h, column-quad-w4 values as one 16-byte float4 and
// puts the float4s of neighbouring blocks (BCSR) or block rows (BELL/SBELL)
// next to each other, so a wave's loads of one (h, w4) plane are contiguous.
// Block columns are stored in float4 units: x is read as float4 too.
//
// BCSR: the reference spends a 128-lane work-group per block row
// (kernels/spmv_bcsr.cl:4-40); here a group of G lanes (G from the average
// number of blocks per block row) shares a block row, strides over its
// blocks and combines its bh partial sums with lane shuffles.
// BELL/SBELL and slot-major BCSR: a lane per row of a block row walks the slots.

#include "device_common.hpp"
#include "kernels.hpp"

namespace clspmv {
namespace {

using namespace dev;

template <int BH, int BW4, int G>
__global__ __launch_bounds__(kBlock) void bcsr_kernel(
    int brows, int rows, int cols, int aligned, const int* __restrict__ rp,
    const int* __restrict__ col4, const float* __restrict__ data,
    const float* __restrict__ x, bool x_aligned, float* __restrict__ y) {
    const int g = (xcd_tile(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / G;
    const int lane = threadIdx.x & (G - 1);
    if (g >= brows) return;  // lane groups exit together
    const int s = rp[g], e = rp[g + 1];
    float acc[BH];
#pragma unroll
    for (int h = 0; h < BH; ++h) acc[h] = 0.0f;
    const size_t plane = (size_t)aligned * BH;  // floats per w4 plane
    for (int j = s + lane; j < e; j += G) {
        const int c4 = ld_stream(col4 + j);
#pragma unroll
        for (int w4 = 0; w4 < BW4; ++w4) {
            const float4 xv = ld_x4(x, (c4 + w4) * 4, cols, x_aligned);
#pragma unroll
            for (int h = 0; h < BH; ++h) {
                const float4 d = ld_stream(reinterpret_cast<const float4*>(
                    data + w4 * plane + (size_t)h * aligned + (size_t)j * 4));
                acc[h] = dot4(d, xv, acc[h]);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < BH; ++h) acc[h] = group_sum<G>(acc[h]);
    // Lane h % G of the group writes output row h.
#pragma unroll
    for (int h = 0; h < BH; ++h) {
        const int r = g * BH + h;
        if (h % G == lane && r < rows) y[r] += acc[h];
    }
}

// BELL, SBELL and BCSR in the slot-major encoding: block row r's slot s has its
// block column at col[s * cs] and the float4 of (w4, h) at data[((s * BW4 + w4)
// * BH + h) * 4 cs], both from the row's own base: the layouts differ in the
// bases, the stride cs between slots and the slot count (SBELL's differs by
// slice).  A float4 load of 64 block rows is one contiguous run.
//
// What bounds it: HBM on large matrices, the chain of slots (block column, then
// x) on small ones.  A lane takes HN rows of a block row and HW waves share
// its block rows (they find the columns and x in L1); U slots' columns and
// values load at once, the next U's in flight while the present ones' x is
// fetched (two register sets taking turns; the last group loads no more than
// its slots).  By the loads that a slot has for the chip, one float4 plane per
// block row, row and column quad (figures: block rows of 12 4x4 blocks, BCSR /
// BELL / SBELL, against a lane per block row, one slot after the other; passes
// over one matrix in turn, which up to about 250 MB the memory-side cache holds:
// read from HBM each time, 131,072 block rows take the same by every walk):
//   kSplit    four waves share block rows, two to four slots at a time: 20,000
//             block rows 14.7 / 14.7 / 15.5 -> 6.5 / 6.2 / 6.7 us, 60,000 15.5 /
//             15.6 / 16.3 -> 9.9 / 9.7 / 10.1 us;
//   kAhead    a lane per block row, the next slot in flight, from kAheadPlanes on:
//             100,000 18.7 / 18.3 / 19.5 -> 14.8 / 14.8 / 15.7 us (kSplit 16.0 /
//             15.4 / 15.9), 131,072 20.3 / 20.3 / 22.0 -> 17.1 / 17.1 / 18.5
//             (kSplit 20.4 / 20.2 / 19.8; 6.76 TB/s would be 16.8);
//   kInOrder  from kInOrderPlanes on the waves cover the chain and more loads in
//             flight only slow the stream: 200,000 28.8 us (kAhead 30.4, kSplit
//             28.6), 300,000 39.3 (40.8, 41.9), 524,288 71.8 (70.9, 75.1); 55,000
//             rows of 8x8 blocks 31.1 (kSplit 39.6).  Not SBELL, whose slot
//             counts differ by lane: 524,288 73.5 ahead, 77.2 in order.
//
// Padding slots of BCSR (column -1) and slots past a lane's last load what is
// there for another (SBELL: the wave's widest block row's blocks, one address for
// all such lanes; each its own last block, power-law rows, 300,000 of 4 on average:
// slices of eight rows of 4x1 / 4x4 / 8x2 blocks 140 / 240 / 300 us, so 83 / 173 /
// 223) and are not added, so the sum is the row's blocks' in slot
// order, one float4 dot per w4.  F4ACC = true (BELL method 1, the reference's
// "_mad" variant, kernels/spmv_bell.cl:24-42): float4 accumulators reduced at
// the end.
enum Layout { kBcsrSlots, kBell, kSbell };
constexpr int kHWaves = kBlock / kWave;  // waves of a work-group
enum Walk { kSplit, kAhead, kInOrder };
constexpr long long kAheadPlanes = 3 << 17, kInOrderPlanes = 3 << 18;
template <int BH, Walk WALK>
constexpr int kShare = WALK != kSplit ? 1 : BH < kHWaves ? BH : kHWaves;  // waves sharing block rows

template <int BH, int BW4, Layout LAY, bool F4ACC, Walk WALK>
__global__ __launch_bounds__(kBlock) void block_rows_kernel(
    int brows, int rows, int cols, int cs, long long f4, int nslots, const int* __restrict__ sptr,
    const int* __restrict__ col4, const float* __restrict__ data, const float* __restrict__ x,
    bool x_aligned, float* __restrict__ y) {
    constexpr int HW = kShare<BH, WALK>;
    constexpr int HN = BH / HW;  // rows of a block per wave
    constexpr int U = WALK != kSplit ? 1 : BW4 * HN == 1 ? 4 : BW4 * HN == 2 ? 3 : 2;  // slots at a time
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int h0 = wave % HW * HN;
    const unsigned row = ((unsigned)xcd_tile(blockIdx.x, gridDim.x) * (kHWaves / HW) + wave / HW) * kWave + lane;
    const int r = launch::shadow_row(row, brows);
    int w = nslots;
    const int* cp = LAY == kSbell ? col4 : col4 + r;
    const float* dp = LAY == kSbell ? data : data + (size_t)r * 4;
    // SBELL: the first column and float of the lane's block row, and of the wave's
    // widest, whose blocks lanes past their own last one load.
    unsigned ci = 0, cw = 0;
    size_t di = 0, dw = 0;
    long long P = f4;  // floats per (slot, w4, h) plane
    if constexpr (LAY == kSbell) {  // cs: the slice height
        const int sl = r / cs, p0 = sptr[sl];
        w = (sptr[sl + 1] - p0) / cs;
        P = launch::block_plane(cs);
        ci = (unsigned)(p0 + (r - sl * cs));
        di = (size_t)p0 * BH * BW4 * 4 + (size_t)(r - sl * cs) * 4;
    }
    int wm = w;  // the most slots of the wave's block rows
    if constexpr (LAY == kSbell) {
        if (cs % 32 == 0)  // a slice per half of the wave, at most
            wm = max(__builtin_amdgcn_readlane(w, 0), __builtin_amdgcn_readlane(w, 32));
        else
            wm = wave_max(w);
    }
    wm = __builtin_amdgcn_readfirstlane(wm);
    if constexpr (LAY == kSbell) {
        const int widest = __builtin_ctzll(__ballot(w == wm));
        cw = (unsigned)__builtin_amdgcn_readlane((int)ci, widest);
        dw = (unsigned)__builtin_amdgcn_readlane((int)di, widest) |
             (size_t)(unsigned)__builtin_amdgcn_readlane((int)(di >> 32), widest) << 32;
    }
    dp += (size_t)h0 * P;
    float acc[HN];
    float4 acc4[HN];
#pragma unroll
    for (int h = 0; h < HN; ++h) {
        acc[h] = 0.0f;
        acc4[h] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    int c[2][U];
    float4 d[2][U][BW4][HN];
    auto load_slot = [&](int s, int& cc, float4 (*dd)[HN]) {
        const bool own = LAY != kSbell || s < w;
        cc = ld_stream(cp + (size_t)s * cs + (own ? ci : cw));
        const float* from = dp + (own ? di : dw);
#pragma unroll
        for (int w4 = 0; w4 < BW4; ++w4)
#pragma unroll
            for (int h = 0; h < HN; ++h)
                dd[w4][h] = ld_stream(reinterpret_cast<const float4*>(from + (((size_t)s * BW4 + w4) * BH + h) * P));
    };
    auto load = [&](int s, int b) {
#pragma unroll
        for (int u = 0; u < U; ++u) load_slot(s + u, c[b][u], d[b][u]);
    };
    auto load_part = [&](int s, int b) {  // slots below wm
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= wm) break;
            load_slot(s + u, c[b][u], d[b][u]);
        }
    };
    auto add = [&](int s, int b) {
        float4 xv[U][BW4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= wm) break;
            const int cc = LAY == kBcsrSlots ? max(c[b][u], 0) : c[b][u];
#pragma unroll
            for (int w4 = 0; w4 < BW4; ++w4) xv[u][w4] = ld_x4(x, (cc + w4) * 4, cols, x_aligned);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= wm) break;
            const bool live = LAY == kBcsrSlots ? c[b][u] >= 0 : LAY == kSbell ? s + u < w : true;
#pragma unroll
            for (int w4 = 0; w4 < BW4; ++w4)
#pragma unroll
                for (int h = 0; h < HN; ++h) {
                    const float4 dv = d[b][u][w4][h], xx = xv[u][w4];
                    if (F4ACC) {
                        acc4[h].x = live ? fmaf(dv.x, xx.x, acc4[h].x) : acc4[h].x;
                        acc4[h].y = live ? fmaf(dv.y, xx.y, acc4[h].y) : acc4[h].y;
                        acc4[h].z = live ? fmaf(dv.z, xx.z, acc4[h].z) : acc4[h].z;
                        acc4[h].w = live ? fmaf(dv.w, xx.w, acc4[h].w) : acc4[h].w;
                    } else {
                        const float a = dot4(dv, xx, acc[h]);
                        acc[h] = live ? a : acc[h];
                    }
                }
        }
    };
    if constexpr (WALK == kInOrder) {
        for (int s = 0; s < wm; ++s) {
            load(s, 0);
            add(s, 0);
        }
    } else {
        if (U <= wm) load(0, 0);
        else load_part(0, 0);
        int s = 0;
        for (; s + 3 * U <= wm; s += 2 * U) {
            load(s + U, 1);
            add(s, 0);
            load(s + 2 * U, 0);
            add(s + U, 1);
        }
        if (s + U < wm) load_part(s + U, 1);
        add(s, 0);
        if (s + 2 * U < wm) load_part(s + 2 * U, 0);
        if (s + U < wm) add(s + U, 1);
        if (s + 2 * U < wm) add(s + 2 * U, 0);
    }
#pragma unroll
    for (int h = 0; h < HN; ++h) {
        const unsigned at = (unsigned)r * BH + h0 + h;
        const float v = F4ACC ? (acc4[h].x + acc4[h].y) + (acc4[h].z + acc4[h].w) : acc[h];
        if (row < (unsigned)brows && at < (unsigned)rows) y[at] += v;
    }
}

template <int BH, int BW4, Layout LAY, bool F4ACC>
hipError_t block_rows(hipStream_t s, int brows, int rows, int cols, int cs, long long f4, int nslots, const int* sptr,
                      const int* col4, const float* data, const float* x, bool xa, float* y) {
    auto launch = [&](auto kernel, int share) {
        const int per = kBlock / share;  // block rows per work-group
        hipLaunchKernelGGL(kernel, dim3(((long long)brows + per - 1) / per), dim3(kBlock), 0, s, brows, rows, cols, cs,
                           f4, nslots, sptr, col4, data, x, xa, y);
    };
    const long long planes = (long long)brows * BH * BW4;
    if (planes < kAheadPlanes) launch(block_rows_kernel<BH, BW4, LAY, F4ACC, kSplit>, kShare<BH, kSplit>);
    else if (LAY == kSbell || planes < kInOrderPlanes) launch(block_rows_kernel<BH, BW4, LAY, F4ACC, kAhead>, 1);
    else launch(block_rows_kernel<BH, BW4, LAY, F4ACC, LAY == kSbell ? kAhead : kInOrder>, 1);
    return hipGetLastError();
}

int grid_for(long long threads) { return (int)((threads + kBlock - 1) / kBlock); }

template <int BH, int BW4>
hipError_t bcsr_shape(hipStream_t s, int brows, int rows, int cols, int lanes,
                      int aligned, const int* rp, const int* col4,
                      const float* data, const float* x, bool xa, float* y) {
    const int grid = grid_for((long long)brows * lanes);
#define BCSRG(G)                                                                    \
    case G:                                                                         \
        hipLaunchKernelGGL((bcsr_kernel<BH, BW4, G>), dim3(grid), dim3(kBlock), 0, s, \
                           brows, rows, cols, aligned, rp, col4, data, x, xa, y);   \
        break;
    switch (lanes) {
        BCSRG(1) BCSRG(2) BCSRG(4) BCSRG(8) BCSRG(16) BCSRG(32) BCSRG(64)
        default: return hipErrorInvalidValue;
    }
#undef BCSRG
    return hipGetLastError();
}

}  // namespace

namespace launch {

#define SHAPE_DISPATCH(FN, OPT, ...)                              \
    switch (bh * 10 + bw) {                                       \
        case 14: return FN<1, 1 OPT>(__VA_ARGS__);                \
        case 24: return FN<2, 1 OPT>(__VA_ARGS__);                \
        case 44: return FN<4, 1 OPT>(__VA_ARGS__);                \
        case 84: return FN<8, 1 OPT>(__VA_ARGS__);                \
        case 18: return FN<1, 2 OPT>(__VA_ARGS__);                \
        case 28: return FN<2, 2 OPT>(__VA_ARGS__);                \
        case 48: return FN<4, 2 OPT>(__VA_ARGS__);                \
        case 88: return FN<8, 2 OPT>(__VA_ARGS__);                \
        default: return hipErrorInvalidValue;                     \
    }
// The template arguments after the block shape (a macro argument with commas).
#define LAYOUT(L, F4) , L, F4

hipError_t bcsr(hipStream_t s, int brows, int rows, int cols, int bh, int bw,
                int lanes, int aligned, const int* rp, const int* col4,
                const float* data, const float* x, bool x_aligned, float* y) {
    if (brows <= 0) return hipSuccess;
    SHAPE_DISPATCH(bcsr_shape, , s, brows, rows, cols, lanes, aligned, rp, col4,
                   data, x, x_aligned, y)
}

hipError_t bcsr_slots(hipStream_t s, int brows, int rows, int cols, int bh, int bw, int hal, int nslots,
                      const int* col4, const float* data, const float* x, bool x_aligned, float* y) {
    if (brows <= 0 || nslots <= 0) return hipSuccess;
    if (hal < brows || nslots > kBcsrSlotsMax) return hipErrorInvalidValue;
    SHAPE_DISPATCH(block_rows, LAYOUT(kBcsrSlots, false), s, brows, rows, cols, hal, block_plane(hal), nslots, nullptr,
                   col4,
                   data, x, x_aligned, y)
}

hipError_t bell(hipStream_t s, int brows, int rows, int cols, int bh, int bw,
                int method, int hal, int f4, int ellnum, const int* col4,
                const float* data, const float* x, bool x_aligned, float* y) {
    if (brows <= 0 || ellnum <= 0) return hipSuccess;
    if (method == 1)
        SHAPE_DISPATCH(block_rows, LAYOUT(kBell, true), s, brows, rows, cols, hal, f4, ellnum, nullptr, col4, data, x,
                       x_aligned, y)
    SHAPE_DISPATCH(block_rows, LAYOUT(kBell, false), s, brows, rows, cols, hal, f4, ellnum, nullptr, col4, data, x,
                   x_aligned, y)
}

hipError_t sbell(hipStream_t s, int brows, int rows, int cols, int bh, int bw,
                 int slice_height, const int* sptr, const int* col4,
                 const float* data, const float* x, bool x_aligned, float* y) {
    if (brows <= 0) return hipSuccess;
    if (slice_height <= 0) return hipErrorInvalidValue;
    SHAPE_DISPATCH(block_rows, LAYOUT(kSbell, false), s, brows, rows, cols, slice_height, 0, 0, sptr, col4, data, x,
                   x_aligned, y)
}

#undef LAYOUT
#undef SHAPE_DISPATCH

}  // namespace launch
}  // namespace clspmv
