// One part of the tile GEMM's instantiations (exl3_tile.h): the formats i
// of VQ_EXL3_FORMATS with i % kTileParts == VQ_TILE_PART, dense at both
// activation precisions and, for mul1 rates, MoE.  build.py compiles this
// file once per part, in parallel.
#include "exl3_tile.h"

#ifndef VQ_TILE_PART
#error "build with -DVQ_TILE_PART=<part>"
#endif

namespace exl3 {
namespace {

template <int kBitsX2, int kCodebook, bool kMoe, bool kLo, int kBlocks>
int launch(const TileArgs& a, dim3 grid, hipStream_t stream) {
  hipLaunchKernelGGL((tile_gemm<kBitsX2, kCodebook, kMoe, kLo, kBlocks>), grid, dim3(kTileThreads), 0, stream, a);
  return vq::check_launch(kMoe ? "exl3 moe tile_gemm" : "exl3 tile_gemm");
}

template <int kBitsX2, int kCodebook>
int launch_format(bool moe, bool lo, int blocks, const TileArgs& a, dim3 grid, hipStream_t stream) {
  if (moe) {
    if constexpr (kCodebook == 2) {
      if (blocks != kTileBlocks) return vq::fail("EXL3 MoE: no tile GEMM of this height");
      if (lo) return launch<kBitsX2, kCodebook, true, true, kTileBlocks>(a, grid, stream);
      return launch<kBitsX2, kCodebook, true, false, kTileBlocks>(a, grid, stream);
    }
    return vq::fail("EXL3 MoE: no tile GEMM for this codebook");
  }
  if (lo && blocks == 2) return launch<kBitsX2, kCodebook, false, true, 2>(a, grid, stream);
  if (lo && blocks == 4) return launch<kBitsX2, kCodebook, false, true, 4>(a, grid, stream);
  if (blocks != kTileBlocks) return vq::fail("EXL3 linear: no tile GEMM of this height");
  if (lo) return launch<kBitsX2, kCodebook, false, true, kTileBlocks>(a, grid, stream);
  return launch<kBitsX2, kCodebook, false, false, kTileBlocks>(a, grid, stream);
}

}  // namespace

template <>
int tile_launch_part<VQ_TILE_PART>(int64_t bits_x2, int64_t codebook, bool moe, bool lo, int blocks,
                                   const TileArgs& a, dim3 grid, hipStream_t stream) {
#define VQ_CASE(B, C)                                                      \
  if constexpr (format_index(B, C) % kTileParts == VQ_TILE_PART) {         \
    if (bits_x2 == B && codebook == C) {                                   \
      return launch_format<B, C>(moe, lo, blocks, a, grid, stream);        \
    }                                                                      \
  }
  VQ_EXL3_FORMATS(VQ_CASE)
#undef VQ_CASE
  return vq::fail("Unsupported EXL3 rate/codebook combination");
}

}  // namespace exl3
