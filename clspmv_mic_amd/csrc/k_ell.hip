// ELL and SELL SpMV for gfx950 (replace kernels/spmv_ell.cl and
// kernels/spmv_sell.cl).
//
// Both formats are column-major inside a slab (ELL: one slab of
// `ell_height_aligned` rows; SELL: one slab per slice), so consecutive lanes
// own consecutive rows and every slot load is one contiguous 256-byte wave
// access.  The 4-rows-per-lane ELL variant issues 128-bit loads.

#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace clspmv {
namespace {

using namespace dev;

// One row per lane, for ELL (ptr null: every row has `w0` slots `stride` apart)
// and SELL (slices of h rows; a slot's entries are h apart).
//
// What bounds it: on large matrices HBM (padding slots are read too), on
// small ones the chain of slots: column, then x.  kSlots slots' columns and
// values load at once, and the next kSlots' are in flight while the present
// ones' x values are gathered (two register sets taking turns, nothing
// copied; the last, shorter group loads no more than its slots).  Two slots
// at a time took 9.8 / 10.4 us (ELL / SELL) on the 27-point stencil 30^3; this
// takes 3.6 / 4.3 us.
//
// WIN: the work-group stages the chunks of x that its rows touch in LDS and
// gathers there, by 16-bit places instead of 32-bit columns (launch::XStage;
// two slots to a word, so that a word is loaded as it is used: single 16-bit
// loads were widened behind a wait for the next slots').  ELL / SELL, against
// gathering from memory: 27-point stencil 60^3 8.4 / 9.1 -> 7.4 / 8.0 us, 77^3 18.3 /
// 20.5 -> 13.0 / 14.9, mesh of 100,000 rows of 25 6.0 / 6.6 -> 4.6 / 5.6, of 700,000
// 51.0 / 53.9 -> 18.8 / 21.6 us.
template <bool SELL, bool WIN, int kSlots, int kRows>
__global__ __launch_bounds__(kRows) void ell_row_kernel(
    int rows, int h, int w0, const int* __restrict__ ptr, const int* __restrict__ list, const unsigned short* __restrict__ idx,
    int stride, int cols, const int* __restrict__ col, const float* __restrict__ val, const float* __restrict__ x,
    float* __restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    const int wg = xcd_tile(blockIdx.x, gridDim.x);
    const unsigned row = (unsigned)wg * kRows + threadIdx.x;
    const int r = launch::shadow_row(row, rows);
    int w = w0;
    constexpr int kPer = WIN ? 2 : 1;  // slots per column word
    const int* cp = WIN ? reinterpret_cast<const int*>(idx) : col;
    const float* vp = val;
    StageX<kRows> stage;
    if constexpr (WIN) stage.ids(list + (size_t)wg * stride, stride);
    // SELL: the first column word and value of the lane's row, and of the wave's
    // widest; slot indices fit 31 bits with them (ptr is int).
    unsigned ci = 0, vi = 0, cw = 0, vw = 0;
    if constexpr (SELL) {
        const int sl = r / h, p0 = ptr[sl], q0 = WIN ? p0 / h : 0;
        w = WIN ? ptr[sl + 1] / h - q0 : (ptr[sl + 1] - p0) / h;
        const int i = r - sl * h;
        ci = WIN ? (unsigned)((q0 + sl) >> 1) * h + i : (unsigned)(p0 + i);
        vi = (unsigned)(p0 + i);
    } else {
        cp += r;
        vp += r;
    }
    // The widest row of the wave: its slots are walked.  A lane past its own last
    // one loads the widest row's, one address for all such lanes, and does not add
    // it: lanes re-reading each its own last slot keep as many cache lines busy as
    // live ones (power-law rows, 300,000 of 4 on average and at most 60: slices of
    // 1 / 4 / 8 / 32 rows 112 / 132 / 107 / 87 us, with the widest's 38 / 53 / 54 /
    // 71; lanes leaving the walk one by one, two slots at a time, 43 / 65 / 70 / 80).
    int wm = w;
    if constexpr (SELL) {
        if (h % 32 == 0)  // a slice per half of the wave, at most
            wm = max(__builtin_amdgcn_readlane(w, 0), __builtin_amdgcn_readlane(w, 32));
        else
            wm = wave_max(w);
    }
    wm = __builtin_amdgcn_readfirstlane(wm);
    if constexpr (SELL) {
        const int lane = __builtin_ctzll(__ballot(w == wm));
        cw = (unsigned)__builtin_amdgcn_readlane((int)ci, lane);
        vw = (unsigned)__builtin_amdgcn_readlane((int)vi, lane);
    }
    int c[2][kSlots / kPer];
    float v[2][kSlots];
    auto load_slot = [&](int s, int u, int* cc, float* vv) {
        if constexpr (SELL) {
            const bool own = s + u < w;
            if (u % kPer == 0) cc[u / kPer] = ld_stream(cp + ((own ? ci : cw) + (unsigned)((s + u) / kPer) * h));
            vv[u] = ld_stream(vp + ((own ? vi : vw) + (unsigned)(s + u) * h));
        } else {
            if (u % kPer == 0) cc[u / kPer] = ld_stream(cp + (size_t)((s + u) / kPer) * h);
            vv[u] = ld_stream(vp + (size_t)(s + u) * h);
        }
    };
    auto load = [&](int s, int* cc, float* vv) {
#pragma unroll
        for (int u = 0; u < kSlots; ++u) load_slot(s, u, cc, vv);
    };
    auto load_part = [&](int s, int* cc, float* vv) {  // slots below wm
#pragma unroll
        for (int u = 0; u < kSlots; ++u) {
            if (s + u >= wm) break;
            load_slot(s, u, cc, vv);
        }
    };
    if (kSlots <= wm) load(0, c[0], v[0]);
    else load_part(0, c[0], v[0]);
    if constexpr (WIN) stage.fetch(stride, cols, x, xs);
    const unsigned last = (unsigned)stride * launch::kXChunk - 1u;
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](auto full, int s, const int* cc, const float* vv) {  // full: all slots below wm
        float xv[kSlots];
        if constexpr (WIN) {  // entry 0 may be another work-group's: clamped, not added
#pragma unroll
            for (int u = 0; u < kSlots; ++u) {
                const unsigned i = u % 2 ? (unsigned)cc[u / 2] >> 16 : cc[u / 2] & 0xFFFFu;
                if (full || s + u < wm) xv[u] = xs[SELL ? min(i, last) : i];
            }
        } else {
#pragma unroll
            for (int u = 0; u < kSlots; ++u)
                if (full || s + u < wm) xv[u] = x[cc[u]];
        }
#pragma unroll
        for (int u = 0; u < kSlots; ++u)
            if (full || s + u < wm) {
                // Two selects: a single one is made a branch around the gather, with
                // a wait for the next slots in it.
                const bool own = !SELL || s + u < w;
                const float t = fmaf(own ? vv[u] : 0.0f, xv[u], a[u % 4]);
                a[u % 4] = own ? t : a[u % 4];
            }
    };
    constexpr std::true_type whole{};
    constexpr std::false_type part{};
    int s = 0;
    for (; s + 3 * kSlots <= wm; s += 2 * kSlots) {
        load(s + kSlots, c[1], v[1]);
        __builtin_amdgcn_sched_barrier(0);  // the next slots' loads stay ahead of the gathers' waits
        add(whole, s, c[0], v[0]);
        load(s + 2 * kSlots, c[0], v[0]);
        __builtin_amdgcn_sched_barrier(0);
        add(whole, s + kSlots, c[1], v[1]);
    }
    if (s + kSlots < wm) load_part(s + kSlots, c[1], v[1]);
    add(part, s, c[0], v[0]);
    if (s + 2 * kSlots < wm) load_part(s + 2 * kSlots, c[0], v[0]);
    if (s + kSlots < wm) add(part, s + kSlots, c[1], v[1]);
    if (s + 2 * kSlots < wm) add(part, s + 2 * kSlots, c[0], v[0]);
    if (row < (unsigned)rows) y[r] += (a[0] + a[1]) + (a[2] + a[3]);
}

// SELL with short rows: a row per lane, two slots at a time, nothing clamped.
__global__ __launch_bounds__(kBlock) void sell_short_kernel(
    int rows, int h, const int* __restrict__ ptr, const int* __restrict__ col,
    const float* __restrict__ val, const float* __restrict__ x, float* __restrict__ y) {
    const unsigned r = (unsigned)xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (r >= (unsigned)rows) return;
    const int sl = (int)r / h, i = (int)r - sl * h;
    const int p0 = ptr[sl];
    const int w = (ptr[sl + 1] - p0) / h;
    const int* c = col + p0 + i;
    const float* v = val + p0 + i;
    float a0 = 0.0f, a1 = 0.0f;
    int k = 0;
    for (; k + 1 < w; k += 2) {
        const int c0 = ld_stream(c + (size_t)k * h), c1 = ld_stream(c + (size_t)(k + 1) * h);
        a0 = fmaf(ld_stream(v + (size_t)k * h), x[c0], a0);
        a1 = fmaf(ld_stream(v + (size_t)(k + 1) * h), x[c1], a1);
    }
    if (k < w) a0 = fmaf(ld_stream(v + (size_t)k * h), x[ld_stream(c + (size_t)k * h)], a0);
    y[r] += a0 + a1;
}

// Four consecutive rows per lane; requires hal % 4 == 0.
__global__ __launch_bounds__(kBlock) void ell4_kernel(
    int rows, int hal, int ellnum, const int* __restrict__ col,
    const float* __restrict__ val, const float* __restrict__ x,
    float* __restrict__ y) {
    const int r = (xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x) * 4;
    if (r >= rows) return;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < ellnum; ++s) {
        const size_t i = (size_t)s * hal + r;
        const int4 c = ld_stream(reinterpret_cast<const int4*>(col + i));
        const float4 v = ld_stream(reinterpret_cast<const float4*>(val + i));
        a.x = fmaf(v.x, x[c.x], a.x);
        a.y = fmaf(v.y, x[c.y], a.y);
        a.z = fmaf(v.z, x[c.z], a.z);
        a.w = fmaf(v.w, x[c.w], a.w);
    }
    y[r] += a.x;
    if (r + 1 < rows) y[r + 1] += a.y;
    if (r + 2 < rows) y[r + 2] += a.z;
    if (r + 3 < rows) y[r + 3] += a.w;
}

template <bool SELL, int kSlots, int kRows>
hipError_t ell_rows_plain(hipStream_t s, int rows, int h, int w, const int* ptr, const int* col, const float* val,
                          int cols, const float* x, float* y) {
    hipLaunchKernelGGL((ell_row_kernel<SELL, false, kSlots, kRows>), dim3(((unsigned)rows + kRows - 1) / kRows), dim3(kRows), 0,
                       s, rows, h, w, ptr, nullptr, nullptr, 0, cols, col, val, x, y);
    return hipGetLastError();
}

template <bool SELL, int kSlots>
hipError_t ell_rows_staged(hipStream_t s, int rows, int h, int w, const int* ptr, launch::XStage W, const int* col,
                           const float* val, int cols, const float* x, float* y) {
    constexpr int R = launch::kEllRows;
    hipLaunchKernelGGL((ell_row_kernel<SELL, true, kSlots, R>), dim3(((unsigned)rows + R - 1) / R), dim3(R),
                       sizeof(float) * launch::kXChunk * W.stride, s, rows, h, w, ptr, W.list, W.idx, W.stride, cols,
                       col, val, x, y);
    return hipGetLastError();
}

// Staged work-groups of 512 rows leave too many CUs idle below 96 of them: the
// mesh of 20,000 rows (40 work-groups) with 12 neighbours 3.1 / 3.7 us staged, 2.8 /
// 3.3 gathered (ELL / SELL), 27-point stencil 22^3 (21) 4.0 / 4.6 and 3.4 / 4.1;
// 50,000 rows (98) of 40 4.4 / 5.4 staged, 5.7 / 6.9 gathered.
constexpr unsigned kStagedGroups = 96;

// Slots in flight, staged: eight while there are fewer than two waves per SIMD
// (131,072 rows), where the chain of slots sets the time (mesh of 100,000 rows
// of 25 4.6 against 5.2 us), four above, where more waves cover it and the
// shorter last group matters (mesh of 400,000 rows of 12, SELL, 7.4 against 8.1 us).
//
// Gathered: work-groups of one wave, which fill the CUs evenly (random columns,
// 40,000 rows, SELL, work-groups of 512 / 256 / 64 rows: 32 slots 17.6 / 9.3 /
// 8.4 us, 100 slots 66.9 / 30.4 / 24.2 us), of four waves for rows of less than
// four slots (1 M rows of one slot: 4.8 against 5.9 us).  Slots by the mean row:
// 16 from 24 slots on (100,000 rows of 32 / 100, ELL: 16.6 / 53.2 us, by eight
// 17.2 / 55.3, by four 20.6 / 66.5), eight from ten on (200,000 rows of 12 13.6
// against 14.8 us) and on few rows, else four (400,000 rows of 5: 12.0 against
// 12.6).
template <bool SELL>
hipError_t ell_rows(hipStream_t s, int rows, int h, int w, const int* ptr, long long stored, launch::XStage W,
                    const int* col, const float* val, int cols, const float* x, float* y) {
    const bool few = rows < (1 << 17);
    if (W.list && ((unsigned)rows + launch::kEllRows - 1) / launch::kEllRows >= kStagedGroups)
        return few ? ell_rows_staged<SELL, 8>(s, rows, h, w, ptr, W, col, val, cols, x, y)
                   : ell_rows_staged<SELL, 4>(s, rows, h, w, ptr, W, col, val, cols, x, y);
    const long long mean = stored / rows;
    if (mean < 4) return ell_rows_plain<SELL, 4, 256>(s, rows, h, w, ptr, col, val, cols, x, y);
    if (mean >= 24) return ell_rows_plain<SELL, 16, 64>(s, rows, h, w, ptr, col, val, cols, x, y);
    return few || mean >= 10 ? ell_rows_plain<SELL, 8, 64>(s, rows, h, w, ptr, col, val, cols, x, y)
                             : ell_rows_plain<SELL, 4, 64>(s, rows, h, w, ptr, col, val, cols, x, y);
}

}  // namespace

namespace launch {

hipError_t ell(hipStream_t s, int rows, int hal, int ellnum, int rows_per_lane, XStage W,
               const int* col, const float* val, int cols, const float* x, float* y) {
    if (rows <= 0) return hipSuccess;
    if (rows_per_lane != 4)
        return ell_rows<false>(s, rows, hal, ellnum, nullptr, (long long)rows * ellnum, W, col, val, cols, x, y);
    if (hal % 4 != 0) return hipErrorInvalidValue;
    const int lanes = (rows + 3) / 4;
    hipLaunchKernelGGL(ell4_kernel, dim3((lanes + kBlock - 1) / kBlock),
                       dim3(kBlock), 0, s, rows, hal, ellnum, col, val, x, y);
    return hipGetLastError();
}

hipError_t sell(hipStream_t s, int rows, int slice_height, const int* ptr, long long stored, XStage W,
                const int* col, const float* val, int cols, const float* x, float* y) {
    if (rows <= 0) return hipSuccess;
    if (slice_height <= 0) return hipErrorInvalidValue;
    // Up to three slots a row the walk's bookkeeping shows: 1 M rows of 1 / 2 / 3
    // slots 5.6 / 4.8 / 7.4 us by the short kernel, 5.9 / 5.6 / 7.8 by the other; of
    // 5 11.1 / 10.0.
    if (stored * 2 <= rows * 7LL) {
        hipLaunchKernelGGL(sell_short_kernel, dim3(((unsigned)rows + kBlock - 1) / kBlock), dim3(kBlock), 0, s, rows,
                           slice_height, ptr, col, val, x, y);
        return hipGetLastError();
    }
    return ell_rows<true>(s, rows, slice_height, 0, ptr, stored, W, col, val, cols, x, y);
}

}  // namespace launch
}  // namespace clspmv
