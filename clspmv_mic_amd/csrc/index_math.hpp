// Index and address arithmetic of kernels, as constexpr functions that the
// kernels and the host's tests share (no HIP headers).
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

}  // namespace launch
}  // namespace clspmv
