// Index and address arithmetic of kernels and the rules on a caller's pointers,
// as constexpr functions that the library and the host's tests share (no HIP
// headers).
#pragma once

namespace clspmv {
namespace launch {

// Block SpMM, tiled X whose tiles are 8-byte aligned only: byte offset of the
// 16 bytes that stage piece `piece` (right-hand sides 2 piece, 2 piece + 1 of a
// chunk of kc), counted from 8 bytes before the chunk's first right-hand side
// in the tile.  The last right-hand side of an odd kc comes with the one
// before it (with kc = 1, never the first chunk, the chunk before's last one).
// Pieces past kc feed nothing that is stored: they re-read the first two
// right-hand sides, or with kc = 1 what its only piece reads.
constexpr unsigned spmm_piece_offset(unsigned piece, unsigned kc) {
    return 2 * piece + 1 < kc ? piece * 16 + 8u : 2 * piece + 1 == kc ? piece * 16 : kc == 1 ? 0u : 8u;
}
constexpr bool spmm_piece_end(unsigned piece, unsigned kc) { return 2 * piece + 1 == kc; }

// The row that thread `row` of a grid works on: threads past the last row
// shadow it.  (row is unsigned: with rows near 2^31 the last work-group's go past
// the signed range.)
constexpr int shadow_row(unsigned row, int rows) { return row < (unsigned)rows ? (int)row : rows - 1; }

// Floats from one (slot, row, column quad) plane of a slot-major block matrix of
// `aligned` block rows to the next: a float4 per block row.
constexpr long long block_plane(int aligned) { return 4LL * aligned; }

// f(first), f(first + step), ... below n.
template <class F>
constexpr void strided(long long first, long long step, long long n, F f) {
    for (long long i = first; i < n; i += step) f(i);
}

// Whether a server's kernels write a request's device_y themselves: device memory
// of the server's own GPU.  Everything else that the runtime can copy to (another
// device's memory, with or without peer access, host memory) is left to its copy.
// known: the runtime knows the pointer.
constexpr bool kernel_writes_y(bool known, bool device_memory, int memory_device, int server_device) {
    return known && device_memory && memory_device == server_device;
}

}  // namespace launch
}  // namespace clspmv
