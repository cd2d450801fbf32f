// EXL3 many-row GEMM for gfx950: decode in registers, activations through LDS.
//
// C[r][n] = sum_k A[r][k] W[k][n] for a tile of up to 128 rows x 256 output
// columns, on v_mfma_f32_16x16x32_f16, then the output transform (unscale
// the row, H128 over each 128-column block, times svh).  Where the tiles are
// too few to fill the chip, the K range is split over workgroups: each then
// stores the unscaled sums of its inputs, which tile_output (exl3_gemm.hip)
// adds and transforms.  Serves the dense linear above 8 rows (exl3_gemm.hip) and the MoE projections of
// prefill-sized calls (exl3_moe.hip: the tile's rows are one expert's routed
// assignments).
//
// Workgroup: 4 wavefronts (one per SIMD), two workgroups per CU.  Wavefront
// w owns output columns [64 w, 64 w + 64) of the tile: four tile columns, two
// pairs.  Per 32-input step (two tile rows) each lane decodes four encoder
// lanes (two pairs x two tile rows) straight into MFMA B operands, with the
// small-M kernel's lane map: lane (g, m) = (lane >> 4, lane & 15) decodes
// encoder lane L = 4 (m & 7) + g of tile column (m >> 3) of a pair; values
// 0-3 are B column m of the pair's first MFMA (tile column m & 7), values 4-7
// of its second (tile column (m & 7) + 8), k slots {2g, 2g+1, 2g+8, 2g+9} of
// the two tile rows.  The activations are stored in that k order (every
// 32-input step: [g 0..3][8 halves]), so no weight ever moves between lanes
// or through LDS.  The A operand of a 16-row block is then, for lane (g, m),
// the 16 bytes of group g of row m: stored in LDS as [g][m] (1 KB per block),
// read with one ds_read_b128 at 16 * lane, conflict-free.
//
// Activations: each rotated input at a per-row power-of-two scale, split
// into FP16 high and low parts (t 2^e = hi + lo, ~22 bits) with both parts
// multiplied against the exact FP16 weight into one FP32 accumulator (kLo,
// the default: the activation precision of the reference's tensor-core
// kernels, csrc/exl3/dense_prefill_tc.h:5-12), or the high part alone
// (!kLo: each rotated input rounded once to FP16, half the MFMAs; an
// explicit opt-in).
//
// Pipeline, per wavefront (one barrier a step):
//   * trellis: LDS-DMA (buffer_load ... lds), 128 bits_x2 bytes per step
//     (one 1 KB load up to 4 bits per weight, two above), into a ring of 4
//     slots, issued 4 steps ahead; a step's ring words are read and decoded
//     (into registers) one step before its MFMAs;
//   * activations: LDS-DMA of the tile's 8 row blocks per step (and their
//     low parts), 2 (4) per wavefront, into 3 buffers, issued 2 steps ahead;
//     the operands of row block rb + 2 are read under the MFMAs of rb;
//   * step s: issue the activation loads of s + 2, read the words of s + 1,
//     issue the trellis load of s + 4, run the MFMAs of s with the decode of
//     s + 1 between them (the VALU work of one step under the matrix work of
//     the other), wait for this wavefront's loads of s + 1, barrier.
//   Loads past the last step reload the last step (into a buffer or slot no
//   one reads again), so the loop has no branch around a load and every wait
//   count is a constant.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "exl3_codec.h"
#include "exl3_internal.h"

namespace exl3 {

constexpr int kTileWaves = 4;
constexpr int kTileThreads = 64 * kTileWaves;
constexpr int kTileCols = 64 * kTileWaves;          // 256
constexpr int kTileRows = 128;
constexpr int kTileBlocks = kTileRows / 16;         // 16-row blocks
constexpr int kTileABufs = 3;                       // activation buffers
constexpr int kTileRing = 4;                        // trellis ring slots, and steps per loop iteration
static_assert(kTileBlocks == kTileHeight, "the plan's full height");
constexpr int kTileRedStride = kTileCols + 4;       // epilogue row stride (floats)

// The tile GEMM serves every rate: the trellis of one step of a wavefront
// (four tile columns x two tile rows, 128 bits_x2 bytes) is one 1 KB load
// up to 4 bits per weight, two above.
constexpr bool tile_rate(int64_t bits_x2) { return bits_x2 >= 2 && bits_x2 <= 16; }
constexpr int tile_slot_bytes(int bits_x2) { return bits_x2 <= 8 ? 1024 : 2048; }

struct TileArgs {
  // activation rows: row r at act + r * act_row_bytes, [high: kp halves]
  // [low: kp halves], each 32-input step in the k order above
  const uint8_t* act;
  int64_t act_row_bytes;   // 4 * kp
  int64_t act_rows;        // rows the activation buffer holds
  const int* row_exp;      // scale exponent of row r at row_exp[r * exp_stride]
  int64_t exp_stride;
  int64_t kp;
  int64_t np;
  // dense: the matrix, rows, and the output
  const uint8_t* trellis;
  const uint16_t* svh;
  int64_t tiles_n;
  int64_t rows;
  void* out;
  int out_dtype;
  int64_t logical_out;
  int tile_rows;           // rows per row tile (a multiple of 16)
  // dense, K split over gridDim.z workgroups (> 1): FP32 sums of split z's
  // inputs, unscaled, at partial + z * rows * np; null: the whole K range in
  // one workgroup, which applies the output transform itself
  float* partial;
  // MoE: the route table (header, sorted assignments, tasks) and the
  // projection of the experts' tables; FP32 outputs [assignment][np]
  const int* table;
  int64_t task_offset;     // int4 tasks at table + task_offset
  const int64_t* ptrs;
  const int64_t* meta;
  int projection;
  float* moe_out;
  const int* moe_row_exp;  // MoE: exponent of assignment a at moe_row_exp[a * exp_stride]
  int col_tiles;           // column tiles per task
  int task_group;          // tasks per group in an XCD's order (1..8)
};

typedef __attribute__((address_space(3))) void* tile_lds_ptr_t;

// f(std::integral_constant<int, i>) for i = 0 .. n - 1.
template <int n, int i = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (i < n) {
    f(std::integral_constant<int, i>{});
    static_for<n, i + 1>(f);
  }
}

// LDS reads the compiler does not see (a read it sees, of LDS that LDS-DMA
// loads write, makes it wait for every such load in flight); a value is
// ready after a tile_wait* that names it.
template <int kOffset>
__device__ __forceinline__ void tile_read16(half8_t& v, uint32_t address) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(address), "i"(kOffset));
}
template <int kOffset>
__device__ __forceinline__ void tile_read4(uint32_t& v, uint32_t address) {
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(address), "i"(kOffset));
}
// At most n LDS reads still pending (they complete in order).
template <int n>
__device__ __forceinline__ void tile_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(n));
}
// v is ready (after a tile_lgkm that covers its read).
__device__ __forceinline__ void tile_ready(half8_t& v) { asm volatile("" : "+v"(v)); }
template <int kWords>
__device__ __forceinline__ void tile_ready(uint32_t (&w)[2][2][kWords]) {
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < kWords; ++i) asm volatile("" : "+v"(w[p][h][i]));
}

// LDS of a workgroup, and the workgroups a CU holds: as many as the
// accumulators of `blocks` row blocks leave registers for, and the LDS.
constexpr int tile_lds_bytes(int blocks, int parts, int bits_x2) {
  return kTileABufs * parts * blocks * 1024 + kTileWaves * kTileRing * tile_slot_bytes(bits_x2);
}
constexpr int tile_occupancy(int blocks, int bits_x2) {
  const int registers = blocks == 4 ? 3 : 2;
  const int lds = 160 * 1024 / tile_lds_bytes(blocks, 2, bits_x2);
  return registers < lds ? registers : lds;
}

// kBlocks: the tile's 16-row blocks: 8 (up to 128 rows), or 2 and 4 for dense
// calls of up to 32 and 64 rows.  At 2 row blocks a wavefront
// and step take 0.43 us (900 cycles: the decode's 126 VALU instructions and 16
// MFMAs, which share the SIMD's issue and add up) whether one or four
// wavefronts share a SIMD; loads 5 to 8 steps ahead instead of 2 to 4
// changed nothing.
//
// At 2 row blocks (calls of 9 to 32 rows, which the small-M kernel also
// takes, in chunks) the FP32 sums are as short-chained as the small-M kernel's,
// whose workgroups hold 4 to 32 steps: the high parts' products are
// added over 4 steps, those sums over 16 steps, and those over the K range; the
// low parts', 2^-11 of the high ones, in a chain of their own.  FP32 outputs'
// error against 64 bits (2-norms), in 1e-7, the small-M kernel / these sums / one
// chain of high and low parts: 1.69 / 1.53 / 2.42 at 4096 x 14336, 2.40 / 1.57 / 4.27 at
// 8192 x 28672, 2.38 / 1.55 / 5.88 at 4096 x 151936, 1.48 / 1.49 / 1.94 at 1024 x
// 1024.  The sums take 200 registers instead of 108 (two workgroups a CU, as
// many as the splits make) and no time: 28.9 us at 20 rows of 4096 x 14336 with
// either, 158 at 4096 x 151936.
template <int kBitsX2, int kCodebook, bool kMoe, bool kLo, int kBlocks>
__global__ __launch_bounds__(kTileThreads, tile_occupancy(kBlocks, kBitsX2)) void tile_gemm(TileArgs a) {
  constexpr int kRows = 16 * kBlocks;
  constexpr int kParts = kLo ? 2 : 1;      // activation parts: high (and low)
  constexpr int kAL = kParts * kBlocks / kTileWaves;  // activation loads per wavefront and step
  static_assert(kAL >= 1 && kAL * kTileWaves == kParts * kBlocks, "whole activation loads");
  static_assert(tile_rate(kBitsX2), "a rate the tile GEMM serves");
  constexpr int kWords = LaneLoad<kBitsX2>::kWords;
  constexpr int kTileBytes = 16 * kBitsX2;
  constexpr int kRowChunk = 4 * kTileBytes;  // one tile row of a wavefront's four tile columns
  constexpr int kSlot = tile_slot_bytes(kBitsX2);
  constexpr int kTL = kSlot / 1024;          // trellis loads per wavefront and step
  constexpr int kChunkLanes = kRowChunk / 16;
  static_assert(kRowChunk % 16 == 0 && 2 * kRowChunk <= kSlot, "a step's trellis fits its slot");
  // the activation buffers, then the wavefronts' trellis rings; the epilogue
  // keeps 16 rows of sums at its start and the row table at its end
  constexpr int kABuf = kParts * kBlocks * 1024;
  constexpr int kAhead = kTileABufs - 1;  // steps the activation loads run ahead
  static_assert(kTileRing >= kAhead, "the order of the prologue's loads");
  constexpr int kABytes = kTileABufs * kABuf;
  constexpr int kTBytes = kTileWaves * kTileRing * kSlot;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kABytes + kTBytes];
  static_assert(sizeof(lds) == tile_lds_bytes(kBlocks, kParts, kBitsX2), "the LDS the occupancy counts on");
  static_assert(sizeof(lds) >= 16 * kTileRedStride * sizeof(float) + 2 * kRows * sizeof(int), "the epilogue fits");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = vq::uniform(tid >> 6);
  const int g = lane >> 4;
  const int m = lane & 15;
  const int L = 4 * (m & 7) + g;
  // Dense: grid (column tile, row tile).  MoE: a 1-D grid; workgroups are
  // dispatched to the 8 XCDs round-robin (workgroup p on XCD p % 8, its
  // p / 8-th).  XCD x runs the contiguous task range [x P, x P + P),
  // P = ceil(tasks / 8): the tasks of one expert share an XCD.  Within it,
  // groups of task_group tasks run column-major (column tile 0 of each task
  // of the group, then column tile 1, ...), so the workgroups resident at
  // once on the XCD hold a few tasks x a few column tiles at the same K
  // steps, and its L2 fetches each activation tile and each weight stripe
  // once for all of them.
  int64_t col_tile = blockIdx.x;
  int moe_task = 0;
  if constexpr (kMoe) {
    const int local = int(blockIdx.x >> 3);
    const int span = a.task_group * a.col_tiles;
    const int group = local / span;
    const int in_group = local - group * span;
    col_tile = in_group / a.task_group;
    const int idx = group * a.task_group + (in_group - int(col_tile) * a.task_group);
    const int per_xcd = (vq::uniform(a.table[2]) + 7) >> 3;
    if (idx >= per_xcd) return;
    moe_task = int(blockIdx.x & 7) * per_xcd + idx;
  }
  const int64_t col0 = col_tile * kTileCols;

  // ---- the tile's rows, matrix and scales ----
  int nrows;
  const uint8_t* trellis;
  const uint16_t* svh;
  int64_t tiles_n;
  int first = 0;
  if constexpr (kMoe) {
    // tile tasks: table[2] of them from task table[3] on
    const int task = moe_task;
    if (task >= a.table[2]) return;
    const int4 tk = reinterpret_cast<const int4*>(a.table + a.task_offset)[a.table[3] + task];
    const int expert = vq::uniform(tk.x);
    first = vq::uniform(tk.y);
    nrows = vq::uniform(tk.z);
    const int64_t* ptrs = a.ptrs + expert * 9 + a.projection * 3;
    const int64_t* meta = a.meta + expert * 12 + a.projection * 4;
    trellis = reinterpret_cast<const uint8_t*>(vq::uniform(ptrs[0]));
    svh = reinterpret_cast<const uint16_t*>(vq::uniform(ptrs[2]));
    tiles_n = vq::uniform(meta[1]) / 16;
    // an expert of another geometry or rate is never read: NaN rows
    const bool bad = vq::uniform(meta[0]) != a.kp || vq::uniform(meta[1]) != a.np ||
                     vq::uniform(meta[2]) != kBitsX2 || vq::uniform(meta[3]) != kCodebook;
    if (bad) {
      for (int r = wave; r < nrows; r += kTileWaves) {
        float* dst = a.moe_out + int64_t(a.table[4 + first + r]) * a.np + col0;
        for (int c = lane; c < kTileCols; c += 64) {
          if (col0 + c < a.np) dst[c] = __builtin_nanf("");
        }
      }
      return;
    }
  } else {
    const int64_t row0 = int64_t(blockIdx.y) * a.tile_rows;
    nrows = int(a.rows - row0 < a.tile_rows ? a.rows - row0 : a.tile_rows);
    trellis = a.trellis;
    svh = a.svh;
    tiles_n = a.tiles_n;
  }
  // the activation row of the tile's row t (rows past the tile repeat its
  // last row)
  auto row_of = [&](int t) -> int {
    t = t < nrows ? t : nrows - 1;
    if constexpr (kMoe) {
      return a.table[4 + first + t];
    } else {
      return int(int64_t(blockIdx.y) * a.tile_rows + t);
    }
  };
  // thread t < kRows keeps row t's id and exponent for the epilogue
  int my_row = 0, my_e = 0;
  if (tid < kRows) {
    my_row = row_of(tid);
    my_e = a.row_exp[int64_t(my_row) * a.exp_stride];
  }

  const int nblocks = (nrows + 15) >> 4;  // 16-row blocks with rows
  // this workgroup's K range, in steps of 32 inputs: whole 128-input blocks,
  // spread evenly over the splits
  int step0 = 0;
  int steps = int(a.kp / 32);
  if constexpr (!kMoe) {
    const int k_blocks = steps / 4;
    const int b0 = int(blockIdx.z) * k_blocks / int(gridDim.z);
    const int b1 = (int(blockIdx.z) + 1) * k_blocks / int(gridDim.z);
    step0 = 4 * b0;
    steps = 4 * (b1 - b0);
  }
  const int last = steps - 1;
  const int row_bytes = int(tiles_n * kTileBytes);
  const int64_t tc0 = col0 / 16 + 4 * wave;  // this wavefront's first tile column
  // columns past the matrix (a partial last tile) read tile column 0 again
  // and are never stored
  const int64_t tc_load = tc0 + 4 <= tiles_n ? tc0 : 0;

  // ---- loads ----
  // trellis: 16-byte chunk c = lane + 64 u of load u (chunks past the
  // step's two tile rows copy the first chunk again, into the slot's unread
  // tail); chunk c lands at byte 16 c of the slot
  const __amdgpu_buffer_rsrc_t t_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(trellis + tc_load * kTileBytes + int64_t(2 * step0) * row_bytes), 0,
      (steps * 2 - 1) * row_bytes + kRowChunk, 0x00020000);
  int t_voff[kTL];
#pragma unroll
  for (int u = 0; u < kTL; ++u) {
    const int c = lane + 64 * u;
    t_voff[u] = c < 2 * kChunkLanes ? (c / kChunkLanes) * row_bytes + 16 * (c % kChunkLanes) : 0;
  }
  // (each builtin's offsets are locals: an array element passed straight
  // to the builtin makes the host compilation drop the kernel's launch stub)
  auto load_trellis = [&](int s) {
    const int from = min(s, last);
#pragma unroll
    for (int u = 0; u < kTL; ++u) {
      const int voff = t_voff[u];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(t_rsrc, (tile_lds_ptr_t)&lds[kABytes + (wave * kTileRing + s % kTileRing) * kSlot + 1024 * u],
                                               16, voff, from * 2 * row_bytes, 0, 0);
    }
  };
  // activations: blocks 0 .. kBlocks - 1 of a buffer are the row blocks'
  // high parts, the next kBlocks their low parts (2 kp bytes on in the row);
  // this wavefront copies blocks kAL * wave + i: lane (g, m) group g of row
  // m of the block
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(a.act), 0, int(a.act_rows * a.act_row_bytes), 0x00020000);
  int a_voff[kAL];
#pragma unroll
  for (int i = 0; i < kAL; ++i) {
    const int blk = kAL * wave + i;
    a_voff[i] = int(int64_t(row_of(16 * (blk % kBlocks) + m)) * a.act_row_bytes + 16 * g + 64 * step0) +
                (blk >= kBlocks ? int(2 * a.kp) : 0);
  }
  auto load_act = [&](int s) {
    const int buf = s % kTileABufs;
    const int from = min(s, last);
#pragma unroll
    for (int i = 0; i < kAL; ++i) {
      const int voff = a_voff[i];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (tile_lds_ptr_t)&lds[buf * kABuf + (kAL * wave + i) * 1024],
                                               16, voff, from * 64, 0, 0);
    }
  };

  constexpr bool kShortChains = !kMoe && kLo && kBlocks == 2;
  constexpr int kSums = kShortChains ? kBlocks : 1;
  f32x4_t acc[kBlocks][2][2];
  f32x4_t low[kSums][2][2];               // short chains: the low parts' products
  f32x4_t sum[kSums][2][2], total[kSums][2][2];  // high parts: over 16 steps, over the K range
#pragma unroll
  for (int rb = 0; rb < kBlocks; ++rb)
#pragma unroll
    for (int p = 0; p < 2; ++p) acc[rb][p][0] = acc[rb][p][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // LDS reads in the loop go through tile_read* (outside the compiler's
  // tracking of the LDS-DMA loads, which would make each read wait for
  // every load in flight); tile_ready names the values a wait made ready.
  const uint32_t a_lane = vq::lds_address(&lds[0]) + 16 * lane;
  // ring words: tile column t = 2 p + (m >> 3) of tile row h of the slot (p
  // and h in the read's immediate offset)
  uint32_t word_addr[kWords];
  {
    int idx[kWords];
    lane_word_index<kBitsX2>(L, idx);
    const uint32_t t_base = vq::lds_address(&lds[0]) + kABytes + wave * kTileRing * kSlot + (m >> 3) * kTileBytes;
#pragma unroll
    for (int i = 0; i < kWords; ++i) word_addr[i] = t_base + 4 * idx[i];
  }
  uint32_t words[2][2][kWords];
  auto read_words = [&](auto slot) {
    constexpr int kSlotIdx = decltype(slot)::value;
    static_for<2>([&](auto p_tag) {
      static_for<2>([&](auto h_tag) {
        constexpr int p = decltype(p_tag)::value, h = decltype(h_tag)::value;
#pragma unroll
        for (int i = 0; i < kWords; ++i)
          tile_read4<kSlotIdx * kSlot + h * kRowChunk + 2 * p * kTileBytes>(words[p][h][i], word_addr[i]);
      });
    });
  };

  // decode of step words w into B operands of pair p: first / second MFMA
  auto decode_pair = [&](const uint32_t (&w)[2][2][kWords], int p, half8_t (&b)[2][2]) {
    uint32_t q0[4], q1[4];
    decode_words<kBitsX2, kCodebook>(L, w[p][0], q0);
    decode_words<kBitsX2, kCodebook>(L, w[p][1], q1);
    b[p][0] = __builtin_bit_cast(half8_t, u32x4_t{q0[0], q0[1], q1[0], q1[1]});
    b[p][1] = __builtin_bit_cast(half8_t, u32x4_t{q0[2], q0[3], q1[2], q1[3]});
  };

  half8_t b_cur[2][2];  // step s's B operands

  // step s, its trellis in ring slot kS = s % 4 (the loop runs four steps
  // an iteration: steps is a multiple of 4): the MFMAs of kRB row blocks of
  // step s on b_cur (high parts, then low parts), with the words of step
  // s + 1 read and decoded between them
  auto step = [&](int s, auto slot, auto row_blocks) __attribute__((always_inline)) {
    constexpr int kS = decltype(slot)::value;
    constexpr int kRB = decltype(row_blocks)::value;
    static_assert(kRB >= 2, "two row blocks read ahead");
    load_act(s + kAhead);
    // T(s + 1) landed: after it came the activation and trellis loads of the
    // kTileRing - 2 steps before this one, and this step's activation load
    vq::wait_vmcnt<(kTileRing - 1) * kAL + (kTileRing - 2) * kTL>();
    read_words(std::integral_constant<int, (kS + 1) % kTileRing>{});  // (past the last step: unused)
    // this step's slot (its words read and decoded a step ago) takes step s + kTileRing
    load_trellis(s + kTileRing);

    half8_t b_next[2][2];
    const uint32_t a_buf = a_lane + uint32_t(s % kTileABufs) * kABuf;
    half8_t ah[kRB], al[kRB];
    auto read_a = [&](auto rb_tag) {
      constexpr int rb = decltype(rb_tag)::value;
      tile_read16<rb * 1024>(ah[rb], a_buf);
      if constexpr (kLo) tile_read16<(kBlocks + rb) * 1024>(al[rb], a_buf);
    };
    read_a(std::integral_constant<int, 0>{});
    read_a(std::integral_constant<int, 1>{});
    static_for<kRB>([&](auto rb_tag) {
      constexpr int rb = decltype(rb_tag)::value;
      // the reads of row block rb + 1 may still be pending (the words were
      // read before row block 0's)
      tile_lgkm<rb + 1 < kRB ? kParts : 0>();
      tile_ready(ah[rb]);
      if constexpr (kLo) tile_ready(al[rb]);
      if constexpr (rb == 0) tile_ready(words);
      if constexpr (rb + 2 < kRB) read_a(std::integral_constant<int, rb + 2>{});
      if constexpr (rb == 0) {
        decode_pair(words, 0, b_next);
        decode_pair(words, 1, b_next);
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (kShortChains && kS == 0) {
            acc[rb][p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[rb], b_cur[p][j], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
          } else {
            acc[rb][p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[rb], b_cur[p][j], acc[rb][p][j], 0, 0, 0);
          }
        }
      if constexpr (kLo) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if constexpr (kShortChains) {
              low[rb][p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[rb], b_cur[p][j], low[rb][p][j], 0, 0, 0);
            } else {
              acc[rb][p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[rb], b_cur[p][j], acc[rb][p][j], 0, 0, 0);
            }
          }
      }
    });
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      b_cur[p][0] = b_next[p][0];
      b_cur[p][1] = b_next[p][1];
    }
    // A(s + 1) of this wavefront landed: after it came its step's trellis
    // load and both loads of the kAhead - 1 steps since; then every
    // wavefront's (and every read of buffer s) is done
    vq::wait_vmcnt<(kAhead - 1) * kAL + kAhead * kTL>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Row blocks past the tile's rows hold copies of its last row: a tile
  // runs the loop of its height rounded up to 2, 4, 5, 6 or 8 row blocks (3
  // or 4 in a four-block tile).  None branches around an MFMA.
  auto run = [&](auto row_blocks) __attribute__((always_inline)) {
    if constexpr (kShortChains) {
      auto four_steps = [&](int s) __attribute__((always_inline)) {
        step(s, std::integral_constant<int, 0>{}, row_blocks);
        step(s + 1, std::integral_constant<int, 1>{}, row_blocks);
        step(s + 2, std::integral_constant<int, 2>{}, row_blocks);
        step(s + 3, std::integral_constant<int, 3>{}, row_blocks);
      };
      auto each = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < kBlocks; ++rb)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            f(rb, p, 0);
            f(rb, p, 1);
          }
      };
      const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
      each([&](int rb, int p, int j) { low[rb][p][j] = sum[rb][p][j] = total[rb][p][j] = zero; });
      for (int s = 0; s < steps;) {
        const int end = min(s + 4 * kTileRing, steps);
        for (; s < end; s += kTileRing) {
          four_steps(s);
          each([&](int rb, int p, int j) { sum[rb][p][j] += acc[rb][p][j]; });
        }
        each([&](int rb, int p, int j) {
          total[rb][p][j] += sum[rb][p][j];
          sum[rb][p][j] = zero;
        });
      }
      each([&](int rb, int p, int j) { acc[rb][p][j] = total[rb][p][j] + low[rb][p][j]; });
    } else {
      for (int s = 0; s < steps; s += kTileRing) {
        step(s, std::integral_constant<int, 0>{}, row_blocks);
        step(s + 1, std::integral_constant<int, 1>{}, row_blocks);
        step(s + 2, std::integral_constant<int, 2>{}, row_blocks);
        step(s + 3, std::integral_constant<int, 3>{}, row_blocks);
      }
    }
  };
  // A wavefront whose tile columns all lie past the matrix (in the last
  // column tile of a projection whose width is no multiple of 256) only
  // loads its share of the activation tiles and meets every barrier: its
  // SIMD serves the CU's other wavefronts meanwhile.
  const bool idle = tc0 >= tiles_n;
  if (idle) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load_act(i);
    vq::wait_vmcnt<(kAhead - 1) * kAL>();  // A(0) of this wavefront landed
    __builtin_amdgcn_s_barrier();
    for (int s = 0; s < steps; ++s) {
      asm volatile("" ::: "memory");
      load_act(s + kAhead);
      vq::wait_vmcnt<(kAhead - 1) * kAL>();  // A(s + 1) of this wavefront landed
      __builtin_amdgcn_s_barrier();
    }
    asm volatile("" ::: "memory");
  } else {
    // ---- prologue: the loads of the kTileRing steps before step 0, in the
    // order those steps would issue them (each A before its step's T) ----
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < kTileRing; ++i) {
      if (i >= kTileRing - kAhead) load_act(i - (kTileRing - kAhead));
      load_trellis(i);
    }
    vq::wait_vmcnt<(kAhead - 1) * kAL + kAhead * kTL>();  // A(0) and every load before it landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_words(std::integral_constant<int, 0>{});
    tile_lgkm<0>();
    tile_ready(words);
    decode_pair(words, 0, b_cur);
    decode_pair(words, 1, b_cur);
    if constexpr (kBlocks == 8) {
      if (nblocks > 6) {
        run(std::integral_constant<int, 8>{});
      } else if (nblocks > 5) {
        run(std::integral_constant<int, 6>{});
      } else if (nblocks > 4) {
        run(std::integral_constant<int, 5>{});
      } else if (nblocks > 2) {
        run(std::integral_constant<int, 4>{});
      } else {
        run(std::integral_constant<int, 2>{});
      }
    } else if constexpr (kBlocks == 4) {
      if (nblocks > 3) {
        run(std::integral_constant<int, 4>{});
      } else {
        run(std::integral_constant<int, 3>{});
      }
    } else {
      run(std::integral_constant<int, kBlocks>{});
    }
  }

  // ---- epilogue ----
  // the clamped loads past the last step may still be landing in the LDS
  // the epilogue reuses
  vq::wait_vmcnt<0>();
  __syncthreads();
  int* row_id = reinterpret_cast<int*>(&lds[kABytes + kTBytes - 2 * kRows * sizeof(int)]);
  int* row_e = row_id + kRows;
  if (tid < kRows) {
    row_id[tid] = my_row;
    row_e[tid] = my_e;
  }
  __syncthreads();
  // Wavefront w finishes 128-column block blk = w & 1 of the tile: in each
  // row block, rows 8 (w >> 1) + 4 b + q (b = 0, 1), one per 16-lane row q
  // = lane >> 4, lane l = lane & 15 holding the block's columns 8 l .. 8 l +
  // 7, so the output H128 runs in registers and DPP (h128_rows) and each
  // lane stores its eight outputs together.  The lane's eight svh values are
  // loaded once, here (loads and stores share one in-order counter: a load
  // waited for after an output store also waits for the store).
  const int blk = wave & 1;
  const int q = lane >> 4;
  const int l = lane & 15;
  const int64_t c0 = col0 + 128 * blk + 8 * l;  // the lane's first column
  float sv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) sv[j] = c0 + j < a.np ? vq::f16_to_f32(svh[c0 + j]) : 0.0f;
  float* red = reinterpret_cast<float*>(&lds[0]);  // [16][kTileRedStride]
#pragma unroll
  for (int rb = 0; rb < kBlocks; ++rb) {
    // (row blocks past the tile's rows store nothing: the workgroup stops
    // there, all its threads together)
    if (rb > 0 && 16 * rb >= nrows) break;
    // lane (g, m) holds rows 4 g + i of the block, column m of each MFMA
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * g + i;
      const int e = row_e[16 * rb + r];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int col = 64 * wave + 32 * p + 16 * (m >> 3) + (m & 7) + 8 * j;
          red[r * kTileRedStride + col] = ldexpf(acc[rb][p][j][i], -e);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int r = 8 * (wave >> 1) + 4 * b + q;
      const int tr = 16 * rb + r;
      const float* src = red + r * kTileRedStride + 128 * blk + 8 * l;
      const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(src);
      const f32x4_t x1 = *reinterpret_cast<const f32x4_t*>(src + 4);
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float y0 = x0[j], y1 = x1[j];
        v[j] = y0;
        v[4 + j] = y1;
      }
      if constexpr (!kMoe) {
        if (a.partial) {
          // a split's sums: the output transform follows once they are added
          if (tr < nrows) {
            const int64_t row = int64_t(blockIdx.z) * a.rows + int64_t(blockIdx.y) * a.tile_rows + tr;
            vq::store8_act(a.partial, vq::kFP32, row * a.np + c0, v, a.np - c0);
          }
          continue;
        }
      }
      vq::h128_rows(v, l);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= sv[j];
      if (tr < nrows) {
        if constexpr (kMoe) {
          vq::store8_act(a.moe_out, vq::kFP32, int64_t(row_id[tr]) * a.np + c0, v, a.np - c0);
        } else {
          const int64_t row = int64_t(blockIdx.y) * a.tile_rows + tr;
          vq::store8_act(a.out, a.out_dtype, row * a.logical_out + c0, v, a.logical_out - c0);
        }
      }
    }
    __syncthreads();
  }
}

// The tile GEMM's instantiations are split over kTileParts separately
// compiled objects (exl3_tile_part.hip): format i of VQ_EXL3_FORMATS lives
// in part i % kTileParts, with its dense kernels (both precisions) and, for
// mul1 rates, its MoE kernels.
constexpr int kTileParts = 4;

// Launches tile_gemm<bits_x2, codebook, moe, lo, blocks> for a format of
// part P (a format of another part is refused).  blocks: 8, or 2 or 4 for
// dense calls on high and low parts.
template <int P>
int tile_launch_part(int64_t bits_x2, int64_t codebook, bool moe, bool lo, int blocks, const TileArgs& a,
                     dim3 grid, hipStream_t stream);

// Launches tile_gemm<bits_x2, codebook, moe, lo, blocks> from the part that
// holds it (exl3_gemm.hip).
int launch_tile_gemm(int64_t bits_x2, int64_t codebook, bool moe, bool lo, int blocks, const TileArgs& a,
                     dim3 grid, hipStream_t stream);

}  // namespace exl3
