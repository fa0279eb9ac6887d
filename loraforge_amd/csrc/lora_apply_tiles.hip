// LoRA update of a base output for more than 64 tokens, second half: y =
// bf16(y + bf16(scale_g * z B_g^T)) per routed token from finished z rows
// (the z producers of prefill_tile.h, launched before this on the stream).
//
// A workgroup owns 32 tokens x 256 features (64 per wave): it stages the
// tokens' z rows in LDS once and, per distinct slot among them, contracts
// B_g (the MFMA's A operand, so a lane holds four consecutive features of one
// token) with z on v_mfma_f32_32x32x16_bf16 and updates the slot's tokens in
// place. A token has one slot and a column one slice, so each value of y is
// read and written once. Bound by latency (z, B, then y) at a few hundred
// tokens: 32-token tiles give 320 workgroups at 500 tokens x 5120.
//
// 500 tokens x 5120 x 4096, three slices of rank 16, four adapters: z 10.0 us and this
// kernel 11.4 us (13.5 us with y read behind z B^T), the call 24.6 us (142 us as eight
// launches of the decode kernel).
#include <algorithm>

#include "prefill_tile.h"
#include "../../include/loraforge_amd.h"

namespace lf {
namespace prefill {
namespace {

constexpr int kTokens = 32;

__global__ __launch_bounds__(kThreads) void apply_z_kernel(PrefillParams p) {
  __shared__ __attribute__((aligned(16))) uint4 zs[3][kTokens * 8];  // [slice][token][8 units], unit ^ (token & 7)
  __shared__ __attribute__((aligned(16))) int tslot[kThreads];
  __shared__ int list[kMaxList + 1];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = tid & 31;
  const int h = (tid >> 5) & 1;
  const int mt = blockIdx.x % p.mtiles;
  const int nt = blockIdx.x / p.mtiles;
  const int m0 = mt * kTokens;
  const int count = min(kTokens, p.m - m0);
  const int zw = p.slices * kZSlice;
  // (Rows past M read row M - 1; rows without a slot hold no z of this call
  // and are zeroed, so that nothing stale reaches an MFMA.)
  uint4 zr[3];
  const int zrow = min(m0 + (tid >> 3), p.m - 1);
#pragma unroll
  for (int s = 0; s < 3; ++s)
    if (s < p.slices)
      zr[s] = *reinterpret_cast<const uint4*>(p.zpad + int64_t(zrow) * zw + s * kZSlice + (tid & 7) * 8);
  const int wn0 = nt * kTileN + wave * 64;
  uint16_t* yrow = p.y + int64_t(min(m0 + c, p.m - 1)) * p.y_stride + wn0;
  // (Each value of y is updated by one slot and slice, so it can be read ahead of them all.
  // N % 64 == 0: a wave's columns are all inside or all past N.)
  uint2 yold[2][4];
  if (p.y_vec && wn0 < p.n)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) yold[j][q] = *reinterpret_cast<const uint2*>(yrow + 32 * j + 8 * q + 4 * h);
  live_slots(p, m0, count, tslot, list);
  const int nd = list[kMaxList];
  if (nd == 0) return;
#pragma unroll
  for (int s = 0; s < 3; ++s)
    if (s < p.slices) zs[s][swz(tid >> 3, tid & 7)] = tslot[tid >> 3] >= 0 ? zr[s] : make_uint4(0, 0, 0, 0);
  __syncthreads();
  if (wn0 >= p.n) return;
  for (int d = 0; d < nd; ++d) {
    const int gd = list[d];
    const int rank = p.ranks[gd];
    const int br = p.b_strides[gd];
    const float scale = p.lscales[gd];
    const uint16_t* bg = p.b_store + p.b_offsets[gd];
    const int steps = (rank + 15) >> 4;
    const bool mine = tslot[c] == gd;
    uint4 bq[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint16_t* row = bg + int64_t(wn0 + 32 * j + c) * br;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < steps) bq[j][q] = keep_first(b_raw(row, br, 16 * q + 8 * h), min(br, rank) - 8 * h - 16 * q);
    }
    for (int s = 0; s < p.slices; ++s) {
      const int lo = p.slice_offsets[s];
      const int hi = p.slice_offsets[s + 1];
      if (hi <= wn0 || lo >= wn0 + 64) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16 delta;
#pragma unroll
        for (int r = 0; r < 16; ++r) delta[r] = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < steps) delta = mfma32(as_bf16x8(bq[j][q]), as_bf16x8(zs[s][swz(c, 2 * q + h)]), delta);
        if (!mine) continue;
        // delta[4 q + e]: feature wn0 + 32 j + 8 q + 4 h + e of token c.
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = 32 * j + 8 * q + 4 * h;
          const int n = wn0 + col;
          const uint32_t t01 = pack_bf16x2(delta[4 * q] * scale, delta[4 * q + 1] * scale);
          const uint32_t t23 = pack_bf16x2(delta[4 * q + 2] * scale, delta[4 * q + 3] * scale);
          uint16_t* dst = yrow + col;
          if (p.y_vec && n >= lo && n + 3 < hi) {
            const uint2 old = yold[j][q];
            *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(bf16_lo(old.x) + bf16_lo(t01), bf16_hi(old.x) + bf16_hi(t01)),
                                                        pack_bf16x2(bf16_lo(old.y) + bf16_lo(t23), bf16_hi(old.y) + bf16_hi(t23)));
          } else {
            const float t[4] = {bf16_lo(t01), bf16_hi(t01), bf16_lo(t23), bf16_hi(t23)};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e >= lo && n + e < hi) dst[e] = uint16_t(f32_to_bf16(bf16_to_f32(dst[e]) + t[e]));
          }
        }
      }
    }
  }
}

}  // namespace

int launch_apply_z(const PrefillParams& p, hipStream_t stream) {
  const int64_t blocks = int64_t(p.mtiles) * ((p.n + kTileN - 1) / kTileN);
  LF_REQUIRE(blocks < (int64_t(1) << 31), "too many tiles");
  hipLaunchKernelGGL(apply_z_kernel, dim3(unsigned(blocks)), dim3(kThreads), 0, stream, p);
  LF_HIP(hipGetLastError());
  return kOk;
}

}  // namespace prefill

// z rows lie behind the control header and the flag region: a flag word of the
// prefill GEMM may only ever hold tags, and z bits left there by a call on a
// shared workspace could equal the tag of a later one.
constexpr int64_t kZOffset = kWorkspaceHeader + kFlagRegion;

// Tokens whose z rows the workspace holds.
int64_t apply_tiles_tokens(int64_t workspace_bytes, int slices) {
  return (workspace_bytes - kZOffset) / (slices * prefill::kZSlice * 2);
}

// y += LoRA(x) for m tokens (at most apply_tiles_tokens), two launches.
int launch_lora_apply_tiles(const uint16_t* x, int64_t m, int64_t x_stride, int64_t n, int64_t k, const lf_lora* lora,
                            uint16_t* y, int64_t y_stride, void* workspace, void* stream) {
  using namespace prefill;
  LF_REQUIRE(lora->num_slots >= 0, "num_slots must not be negative");
  auto s = static_cast<hipStream_t>(stream);
  PrefillParams p{};
  p.x = x;
  p.x_stride = x_stride;
  p.m = int(m);
  p.n = int(n);
  p.k = int(k);
  p.y = y;
  p.y_stride = y_stride;
  p.y_vec = y_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7u) == 0;
  p.a_store = lora->a_store;
  p.a_offsets = lora->a_offsets;
  p.b_store = lora->b_store;
  p.b_offsets = lora->b_offsets;
  p.b_strides = lora->b_strides;
  p.ranks = lora->ranks;
  p.lscales = lora->scales;
  p.token_slots = lora->token_slots;
  p.slice_offsets = lora->slice_offsets;
  p.slices = lora->num_slices;
  p.num_slots = lora->num_slots;
  p.zpad = reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) + kZOffset);
  // z: a producer per 16-token unit of a 256-token tile, twice as many as one
  // slot would need (tokens of many slots make smaller units).
  p.tile_rows = kBM;
  p.mtiles = int((m + kBM - 1) / kBM);
  p.zparts = 2 * kBM / 16;
  p.zrow_parts = z_row_parts(p.slices, lora->max_rank);
  const int rc = launch_z(p, s);
  if (rc != kOk) return rc;
  p.tile_rows = kTokens;
  p.mtiles = int((m + kTokens - 1) / kTokens);
  return launch_apply_z(p, s);
}

}  // namespace lf
