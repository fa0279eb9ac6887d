// Parameters of the prefill GEMM (prefill_tile.h), shared by its host side and
// the translation units that instantiate it.
#pragma once

#include "call_epoch.h"
#include "nf4_common.h"

namespace lf {
namespace prefill {
constexpr int kThreads = 256;
constexpr int kBM = 256;     // most tokens per tile
constexpr int kTileN = 256;  // output features per tile
constexpr int kZSlice = 64;  // zpad columns per slice
// Tiles of more than kFewSlots slots and at most kManyRows 32-token blocks expand all
// slots into the accumulators before one rounding pass (gemm_kernel's epilogue).
constexpr int kFewSlots = 2;
constexpr int kManyRows = 4;

struct PrefillParams {
  const uint16_t* x;
  int64_t x_stride;
  int m;
  const uint8_t* q;
  ScaleSource src;
  const float* code;
  int n;
  int k;
  const uint16_t* bias;
  uint16_t* y;
  int64_t y_stride;
  const uint16_t* a_store;
  const int64_t* a_offsets;
  const uint16_t* b_store;
  const int64_t* b_offsets;
  const int32_t* b_strides;
  const int32_t* ranks;
  const float* lscales;
  const int32_t* token_slots;
  const int32_t* slice_offsets;
  int slices;
  int num_slots;      // entries of the per-slot arrays (0: not given; slots at or past it run base only)
  uint16_t* zpad;     // [m][slices * 64]
  int y_vec;          // 2: 16-byte aligned y rows, 1: 8-byte aligned, 0: neither
  uint32_t* zflags;   // [mtiles * zparts]: the call's tag once a producer's z rows are stored
  CallEpoch ce;
  int* status;  // set to 1 if a wait for z gives up (cannot happen while producers run first)
  int mtiles;
  int zparts;   // z producers per M-tile
  int zrow_parts;  // workgroups of the producers' own launch that share a unit's A rows
  int zblocks;  // producers among this launch's workgroups (0: none, or a launch of their own)
  int tile_rows;  // tokens per M-tile
  int spin_limit;  // polls of the bounded wait for a producer's flag
  int withhold;    // test hook: producers store nothing and set no flag, so consumers recompute z
};

// Launches the GEMM with tiles of 32 * RI tokens (one translation unit per few
// tile heights, so that they compile side by side).
template <int RI>
int launch_rows(const PrefillParams& p, int64_t blocks, bool lora, bool swiglu, hipStream_t stream);
// 16-row passes over a unit's A rows, at most four: workgroups that share them.
inline int z_row_parts(int slices, int max_rank) {
  const int passes = (slices * max_rank + 15) / 16;
  return passes < 4 ? passes : 4;
}
// Launches the z producers alone (mtiles * zparts * zrow_parts workgroups; zflags may be null).
int launch_z(const PrefillParams& p, hipStream_t stream);
// y += LoRA for p.m tokens from finished z rows (lora_apply_tiles.hip).
int launch_apply_z(const PrefillParams& p, hipStream_t stream);

}  // namespace prefill
}  // namespace lf
