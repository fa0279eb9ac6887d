// Prefill (M > 64 tokens): NF4 GEMM on bf16 MFMA with a multi-LoRA epilogue.
//
// Reference chain (integrations/_sglang_nf4_linear.py:116-129 for the base,
// benchmarks/qwen35_prefill_fused.py:95-171 segmented_ab_kernel for the
// LoRA part):  y = bf16(x @ dequant(W)^T) (+bias);  z = bf16(A_g x);
//              y = bf16(y + bf16(scale_g * B_g z)).
//
// The GEMM (tile::gemm_kernel) is one launch; a double-quant weight first gets
// its fp32 block scales rebuilt into the workspace, and z may have a launch of
// its own (nf4_lora_prefill.hip):
//  - z producers: z = bf16(x A_g^T) of just the tokens routed to g (gathered,
//    16 or 32 at a time, MFMA), into a slice-padded workspace zpad[m][s*64 + j] (zeros
//    past r); then the producer's flag is set to the call's tag (call_epoch.h).
//  - GEMM tiles of 32 RI tokens x 256 output features, four waves, one per
//    SIMD with up to 512 registers: a wave owns all the tile's tokens x 64
//    features, so the weights it needs are nobody else's. They are decoded in
//    registers, straight into the MFMA operand layout, and never go through
//    LDS; only x does (direct global -> LDS copies into a ring of 128-k stages).
//    v_mfma_f32_32x32x16_bf16, W as the A operand.
//  - The decode is bit-exact bf16_rne(code * scale) without a table in memory:
//    k is handed to the MFMA so that lane half h of a 128-k stage covers NF4
//    block h, so a lane's 64 weights of a stage share one scale. It rounds the 16
//    products once, keeps them as bytes in 8 registers and looks nibbles up with
//    v_perm_b32: 32 VALU instructions per 8 weights, placed behind the MFMAs.
//  - Epilogue: round, bias; with LoRA, wait for the flags of the tile's
//    producers (lower block ids or an earlier launch), stage the tile's z rows
//    per slice in LDS and, for every distinct slot in the tile, a second MFMA
//    pass z x B_g^T over the 32-token blocks holding its tokens gives the
//    delta, applied with the reference's two bf16 roundings.
//
// What bounds it (4096 x 4096 x 12288, 96 stages, RI = 8, one round; counters of
// a 344 us form): MFMA busy 66 % of 595 k cycles, the rest decode and copy
// issue; at that load the part runs at about 1.8 GHz, so the energy of the
// decode (-20 % time without it) and of the x copies (-21 % without them)
// counts as much as their cycles. Now 323 us, against 480 us with the weights
// decoded cooperatively into LDS (tile 256 x 192, LDS-bound); a library bf16
// GEMM on dequantised weights takes 313 us. Measured and rejected: the waves'
// copies in turns (uniform branches per slot, 364 us), copies earlier in the
// stage (357-389 us), K split over two groups of waves in a 64-token tile (two
// waves per SIMD: 51.6 us against 53.6 us at 128 x 24576 x 4096, slower with LoRA).
#pragma once

#include <type_traits>

#include "call_epoch.h"
#include "lds_pipeline.h"
#include "nf4_common.h"
#include "prefill_params.h"

namespace lf {

namespace prefill {
namespace {

__device__ __forceinline__ int swz(int row, int unit) { return row * 8 + (unit ^ (row & 7)); }

// Live slot of each token of [t0, t0 + count) (rank 0 or above 64: base
// only, -1), loaded by one thread per token, and the distinct live slots in
// order of first use: list[0 .. list[kMaxList]). Wave 0 extracts them with
// one ballot per distinct slot of each 64-token chunk; a slot already listed
// (checked 64 entries per ballot) is not added again.
constexpr int kMaxList = kBM;  // a tile routes to at most one slot per token
__device__ void live_slots(const PrefillParams& p, int t0, int count, int* tslot, int* list) {
  for (int t = threadIdx.x; t < kThreads; t += kThreads) {
    int g = t < count ? p.token_slots[t0 + t] : -1;
    if (p.num_slots > 0 && g >= p.num_slots) g = -1;
    const int r = g >= 0 ? p.ranks[g] : 0;
    if (r <= 0 || r > kZSlice) g = -1;  // rank 0 / contract violation: base only
    tslot[t] = g;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int nd = 0;
    for (int c = 0; c < count; c += 64) {
      const int g = c + lane < count ? tslot[c + lane] : -1;
      uint64_t left = __ballot(g >= 0);
      while (left) {
        const int gf = __builtin_amdgcn_readlane(g, __builtin_ctzll(left));
        left &= ~__ballot(g == gf);
        bool seen = false;
        for (int b = 0; b < nd && !seen; b += 64) seen = __ballot(b + lane < nd && list[b + lane] == gf) != 0;
        if (!seen) {
          if (lane == 0) list[nd] = gf;
          ++nd;
        }
      }
    }
    if (lane == 0) list[kMaxList] = nd;
  }
  __syncthreads();
}

// Raw B values kk .. kk + 7 of one row (stride br, a power of two; kk a
// multiple of 8) from a readable place: rows of stride >= 8 are 16-byte
// aligned and kk is clamped into the row; a narrower row is read whole (8,
// 4 or 2 bytes, aligned). keep_first() then keeps what belongs to B[kk..].
__device__ __forceinline__ uint4 b_raw(const uint16_t* row, int br, int kk) {
  if (br >= 8) return *reinterpret_cast<const uint4*>(row + min(kk, br - 8));
  if (br == 4) {
    const uint2 v = *reinterpret_cast<const uint2*>(row);
    return make_uint4(v.x, v.y, 0u, 0u);
  }
  if (br == 2) return make_uint4(*reinterpret_cast<const uint32_t*>(row), 0u, 0u, 0u);
  return make_uint4(row[0], 0u, 0u, 0u);
}

// The first `keep` bf16 values of v (none when keep <= 0), zeros after.
__device__ __forceinline__ uint4 keep_first(uint4 v, int keep) {
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e >= keep) w[e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// ---------------------------------------------------------------------------
// 2. GEMM + epilogue
// ---------------------------------------------------------------------------
namespace tile {

constexpr int kWaves = kThreads / 64;
constexpr int kBN = kTileN;    // output features per tile, 64 per wave
constexpr int kJ = 2;          // 32-feature fragments per wave
constexpr int kBK = 128;       // k per stage: two NF4 blocks
constexpr int kXRow = 256;     // bytes of one x row in a stage
constexpr int kSteps = 8;      // MFMA steps per stage (8 k of each block)
constexpr int kMinRing = 36 * 1024;  // the z producers' partial tiles

// x stages in LDS: as many as fit beside the packed weights and the LoRA tables.
template <int RI>
constexpr int kRing = RI <= 5 ? 3 : 2;
// x copies per wave that go out in the step that frees their slot.
template <int RI>
constexpr int kFirstCopies = RI / 2;

template <int RI>
constexpr int stage_bytes() {
  return RI * 32 * kXRow;
}

typedef const __attribute__((address_space(1))) char* GPtr;

__device__ __forceinline__ u32x4 gload16(const char* p, int off) {
  return *(const __attribute__((address_space(1))) u32x4*)((GPtr)p + off);
}
__device__ __forceinline__ float gloadf(const char* p) { return *(const __attribute__((address_space(1))) float*)(GPtr)p; }

// LDS reads the compiler does not track, with immediate offsets.
template <int kOff>
__device__ __forceinline__ u32x4 ldsr128(uint32_t addr) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(kOff));
  return v;
}

template <int RI>
struct XFrags {
  u32x4 v[RI];
};

// The x fragments of one step: 32-token fragment i at row 32 i.
template <int RI, int I = 0>
__device__ __forceinline__ void read_x(uint32_t addr, XFrags<RI>& f) {
  if constexpr (I < RI) {
    f.v[I] = ldsr128<I * 32 * kXRow>(addr);
    read_x<RI, I + 1>(addr, f);
  }
}

// Waits for the fragment reads and ties the values to the wait.
template <int RI>
__device__ __forceinline__ void wait_x(XFrags<RI>& f) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.v[0])::"memory");
#pragma unroll
  for (int i = 1; i < RI; ++i) tie(f.v[i]);
}

// Packed bytes of one stage: fragment j's lane holds the whole 64-k block
// (lane / 32) of its row.
struct Packed {
  u32x4 q[kJ][2];
};
// Block scales of two stages (first, second), a pair per fragment.
struct Scales {
  float s[kJ][2];
};

// A wave's weights. A stage's 64 rows x 64 bytes go through 4 KiB of LDS of
// the wave's own: a copy covers 16 rows, four lanes per row (a fragment
// layout load, one row per lane, takes the address unit four times as long).
// Row r's 16-byte segment s sits at s ^ (r / 4 % 4).
struct WLane {
  const char* q;           // the wave's first row (uniform)
  uint32_t off[4];         // the lane's segment in each copy
  uint32_t read;           // LDS address of the lane's first segment, fragment 0
  const char* s[kJ];       // the lane's scales at stage 0
  int smax;                // byte offset of the last scale pair of a row
};

__device__ __forceinline__ void copy_w(const WLane& w, int st, int i, char* wbuf) {
  copy16(w.q + int64_t(st) * 64 + w.off[i], wbuf + i * 1024);
}

__device__ __forceinline__ void read_w(const WLane& w, Packed& p) {
  p.q[0][0] = ldsr128<0>(w.read);
  p.q[0][1] = ldsr128<0>(w.read ^ 16u);
  p.q[1][0] = ldsr128<2048>(w.read);
  p.q[1][1] = ldsr128<2048>(w.read ^ 16u);
}

__device__ __forceinline__ void tie_w(Packed& p) {
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    tie(p.q[j][0]);
    tie(p.q[j][1]);
  }
}

// Scales of stages st and st + 1 (st even): lane half h loads blocks
// 2 st + 2 h and the next one; pair_scales() then gives each lane its block
// 2 st + h and 2 st + 2 + h. (Past the end of a row: its last pair, unused.)
__device__ __forceinline__ void load_scales(const WLane& w, int st, int h, int j, Scales& s) {
  typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
  const f32x2u v = *(const __attribute__((address_space(1))) f32x2u*)((GPtr)w.s[j] + min(st * 8 + h * 8, w.smax));
  s.s[j][0] = v.x;
  s.s[j][1] = v.y;
}
__device__ __forceinline__ void pair_scales(Scales& s, int j) {
  const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(s.s[j][0]), __float_as_uint(s.s[j][1]), false, false);
  s.s[j][0] = __uint_as_float(v[0]);
  s.s[j][1] = __uint_as_float(v[1]);
}

// The 16 values bf16_rne(code * scale) of one block, split into their low and
// high bytes for v_perm_b32 lookups: lo[i], hi[i] hold entries 4i .. 4i + 3.
struct Codes {
  uint32_t lo[4], hi[4];
};

// Entries 4i .. 4i + 3, in three phases of independent instructions.
struct CodeBuild {
  float v[4];
  uint32_t a, b;

  __device__ __forceinline__ void phase(int k, const float (&code)[16], float s, int i, Codes& t) {
    if (k == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = code[4 * i + e] * s;
    } else if (k == 1) {
      a = pack_bf16x2(v[0], v[1]);
      b = pack_bf16x2(v[2], v[3]);
    } else {
      t.lo[i] = __builtin_amdgcn_perm(b, a, 0x06040200u);
      t.hi[i] = __builtin_amdgcn_perm(b, a, 0x07050301u);
    }
  }
};

__device__ __forceinline__ void block_codes(const float (&code)[16], float s, Codes& t) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    CodeBuild build;
#pragma unroll
    for (int k = 0; k < 3; ++k) build.phase(k, code, s, i, t);
  }
}

__device__ __forceinline__ uint32_t select(uint32_t mask, uint32_t high, uint32_t low) {
  return (mask & high) | (~mask & low);
}

// Eight consecutive weights (one packed dword, high nibble first) as four
// bf16 pairs, in kPieces pieces of two independent VALU instructions whose
// inputs come from earlier pieces: one wave runs per SIMD, so an instruction
// that waits for its predecessor's result idles the issue port.
constexpr int kPieces = 14;
struct Decode {
  uint32_t a, b;            // shifted input
  uint32_t me, mo, ie, io;  // even (high) and odd (low) nibbles: upper-half masks and indexes
  uint32_t l, u;            // lookups in the lower and upper half of the codes
  uint32_t l2, u2;
  uint32_t el, eh, ol, oh;  // low and high result bytes
  uint32_t e01, e23, o01, o23;

  __device__ __forceinline__ void piece(int k, uint32_t d, const Codes& t, u32x4& r) {
    // 0xff in every byte whose nibble is 8 or more: v_perm_b32 selectors 8..11
    // replicate the signs of bits 15, 31 (second operand) and 15, 31 (first).
    constexpr uint32_t kSigns = 0x090b080au;
    if (k == 0) {
      a = d << 8;
      b = d >> 4;
    } else if (k == 1) {
      me = __builtin_amdgcn_perm(a, d, kSigns);
      ie = b & 0x07070707u;
    } else if (k == 2) {
      a = d << 4;
      b = d << 12;
    } else if (k == 3) {
      mo = __builtin_amdgcn_perm(b, a, kSigns);
      io = d & 0x07070707u;
    } else if (k == 4) {
      l = __builtin_amdgcn_perm(t.lo[1], t.lo[0], ie);
      u = __builtin_amdgcn_perm(t.lo[3], t.lo[2], ie);
    } else if (k == 5) {
      el = select(me, u, l);
      l2 = __builtin_amdgcn_perm(t.hi[1], t.hi[0], ie);
    } else if (k == 6) {
      u2 = __builtin_amdgcn_perm(t.hi[3], t.hi[2], ie);
      l = __builtin_amdgcn_perm(t.lo[1], t.lo[0], io);
    } else if (k == 7) {
      eh = select(me, u2, l2);
      u = __builtin_amdgcn_perm(t.lo[3], t.lo[2], io);
    } else if (k == 8) {
      ol = select(mo, u, l);
      l2 = __builtin_amdgcn_perm(t.hi[1], t.hi[0], io);
    } else if (k == 9) {
      u2 = __builtin_amdgcn_perm(t.hi[3], t.hi[2], io);
      e01 = __builtin_amdgcn_perm(eh, el, 0x05010400u);
    } else if (k == 10) {
      oh = select(mo, u2, l2);
      e23 = __builtin_amdgcn_perm(eh, el, 0x07030602u);
    } else if (k == 11) {
      o01 = __builtin_amdgcn_perm(oh, ol, 0x05010400u);
      o23 = __builtin_amdgcn_perm(oh, ol, 0x07030602u);
    } else if (k == 12) {
      r.x = __builtin_amdgcn_perm(o01, e01, 0x05040100u);
      r.y = __builtin_amdgcn_perm(o01, e01, 0x07060302u);
    } else {
      r.z = __builtin_amdgcn_perm(o23, e23, 0x05040100u);
      r.w = __builtin_amdgcn_perm(o23, e23, 0x07060302u);
    }
  }
};

__device__ __forceinline__ u32x4 decode8(uint32_t d, const Codes& t) {
  Decode dec;
  u32x4 r;
#pragma unroll
  for (int k = 0; k < kPieces; ++k) dec.piece(k, d, t, r);
  return r;
}

template <int RI>
struct Acc {
  f32x16 v[RI][kJ];
};

template <int RI>
__device__ __forceinline__ void contract(const u32x4 (&w)[kJ], const XFrags<RI>& x, Acc<RI>& acc) {
#pragma unroll
  for (int i = 0; i < RI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc.v[i][j] = mfma32(vec_bf16x8(w[j]), vec_bf16x8(x.v[i]), acc.v[i][j]);
}

// Copies of x stage st: chunk d * 4 + wave of 1 KiB holds rows 16 d + 4 wave ..
// + 3; a row's 16-byte unit u sits at u ^ (row & 15). All of a lane's rows are
// 16 apart, so its unit is fixed and its offsets advance by 16 rows (clamped
// to the last token's row: results past M are never stored).
struct XLane {
  uint32_t first;  // byte offset of the lane's unit in its first row
  uint32_t last;   // the same unit of row M - 1
};

template <int RI, int kCount>
__device__ __forceinline__ void copy_x(const PrefillParams& p, const XLane& xl, uint32_t row16, int st, char* stage,
                                       int wave) {
  const char* base = reinterpret_cast<const char*>(p.x) + int64_t(st) * kXRow;
#pragma unroll
  for (int d = 0; d < kCount; ++d)
    copy16(base + min(xl.first + uint32_t(d) * row16, xl.last), stage + (d * kWaves + wave) * 1024);
}

// z producers: the launch's first mtiles * zparts workgroups. The tokens of
// M-tile mt routed to live slots are sorted by slot (counting sort in LDS)
// and cut into units of up to 16 tokens of one slot (of 32 where the launch has
// fewer producers than that makes units: see produce_units); producer (mt, q) takes
// units q, q + zparts, ... For a unit it contracts just those tokens with the
// slices * r rows of A_g, 64 rows (four 16-row tiles) per pass: the four
// waves take interleaved 32-wide k steps (v_mfma_f32_16x16x32_bf16, A rows as
// the A operand, the tokens' x as the B operand, four steps of loads in
// flight; in a launch of their own eight waves, 16 rows a pass and whole row
// pieces through LDS, below), the partial tiles meet in LDS in a fixed order, and
// z = bf16(x A_g^T) is stored in the slice-padded layout zpad[t][s * 64 + j]
// (zeros for r <= j < 64). Finally the producer sets its flag
// zflags[mt * zparts + q] to the call's tag. Work follows the routed tokens:
// a dense pass over the whole tile for every slot's rows would multiply the
// LoRA FLOPs by the number of slots in the tile (Zipf routing over 128
// adapters puts dozens in one tile).
// A device-coherent (sc1) 2-byte store: performed at the level the
// consumers' sc1 z loads read, so the producer needs no L2 write-back
// (release fence) before its flag, only a wait for its stores to complete.
__device__ __forceinline__ void store_z(uint16_t* dst, uint16_t v) {
  asm volatile("global_store_short %0, %1, off sc1" : : "v"(dst), "v"(uint32_t(v)) : "memory");
}

constexpr int kUnit = 16;        // tokens per unit

// One 16-row pass of a unit through LDS: a wave's 128-k stages wave, wave + kWaves,
// ... of the unit's x rows and the A rows j0 .. j0 + 15 are copied as whole
// 256-byte row pieces (four rows a copy) into the wave's own two slots of 8 KiB,
// the next stage in flight behind the one contracted; waves do not meet.
// Row r's 16-byte unit u sits at u ^ r. Past K the last unit is repeated (a
// readable place, not contracted).
// A unit is bound by one CU's loads: fragments straight from memory (16 rows, 64
// bytes of each) take the address unit 64 cycles a load, a copy of whole 256-byte
// pieces 16. The calls that launch it, fragment loads -> copies: lora_apply 500 x
// 5120 x 4096 (three slices of rank 16) 28.7 -> 25.4 us, 1000 tokens of rank 64 80 ->
// 53 us (more workgroups than CUs, at one per CU: still the faster form), 4096 x 4096 x
// 4096 74 -> 66 us; the prefill linear 2048 x 8192 x 4096 of rank 64 170 -> 160 us.
constexpr int kZSlot = 8192;
template <int kWaves>
__device__ __forceinline__ f32x4 contract_staged(const PrefillParams& p, const uint16_t* abase, int j0, int rows, int m0,
                                                 const int* unit, int ntok, char* ring) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int stages = (p.k + kBK - 1) / kBK;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (wave >= stages) return acc;
  const char* xr[4];
  const char* ar[4];
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * i + (lane >> 4);
    xr[i] = reinterpret_cast<const char*>(p.x + int64_t(m0 + unit[min(r, ntok - 1)]) * p.x_stride);
    ar[i] = reinterpret_cast<const char*>(abase + int64_t(min(j0 + r, rows - 1)) * p.k);
    at[i] = ((lane & 15) ^ r) * 16;
  }
  char* mine = ring + wave * 2 * kZSlot;
  auto issue = [&](int st, char* slot) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int off = min(st * (kBK * 2) + at[i], p.k * 2 - 16);
      copy16(xr[i] + off, slot + i * 1024);
      copy16(ar[i] + off, slot + kZSlot / 2 + i * 1024);
    }
  };
  issue(wave, mine);
  if (wave + kWaves < stages) issue(wave + kWaves, mine + kZSlot);
  int n = 0;
  for (int st = wave; st < stages; st += kWaves, n ^= 1) {
    if (st + kWaves < stages) wait_vm<8>();  // all but the next stage's copies
    else wait_vm<0>();
    asm volatile("" ::: "memory");
    const uint32_t base = lds_addr(mine) + uint32_t(n * kZSlot + c * 256);
    u32x4 xv[4], av[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint32_t addr = base + uint32_t(((4 * v + kg) ^ c) << 4);
      xv[v] = ldsr128<0>(addr);
      av[v] = ldsr128<kZSlot / 2>(addr);
    }
    lds_wait();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      tie(xv[v]);
      tie(av[v]);
    }
    if (st + 2 * kWaves < stages) issue(st + 2 * kWaves, mine + n * kZSlot);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (st * kBK + v * 32 < p.k) acc = mfma16(vec_bf16x8(av[v]), vec_bf16x8(xv[v]), acc);
  }
  return acc;
}

// kUnitSteps: k steps of loads in flight per wave, 0: through LDS
// (contract_staged). kRowTiles: 16-row tiles of A per pass; parts: workgroups that
// share a unit's rows (this one takes the passes rp, rp + parts, ...). In the
// producers' own launch through LDS, one tile a pass, up to four workgroups a
// unit. In the GEMM launch 4 steps of four tiles (8 steps: slower by 10 %, the
// address unit takes 64 cycles for each fragment load whatever is in flight).
// That bounds a unit (64 A rows of 4096: 20 us), so where a producer has several,
// they take 32 tokens: the A fragments are loaded once for two x fragments. 2048 x
// 11008 x 4096 in 192-token tiles with three producers each, two slices of rank 32,
// SwiGLU: 238 -> 210 us (222 in 256-token tiles with 21; no adapters 186).
template <int kUnitSteps, int kRowTiles, int kThreads = prefill::kThreads>
__device__ __forceinline__ void produce_units(const PrefillParams& p, int mt, int q, int rp, int parts, int* tslot, int* list, int* order, int* cnt,
                              int* ustart, float* red, char* ring = nullptr) {
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 15;
  const int kg = lane >> 4;
  constexpr int kWaves = kThreads / 64;
  constexpr int kPassRows = 16 * kRowTiles;
  const int m0 = mt * p.tile_rows;
  const int count = min(p.tile_rows, p.m - m0);
  const int zw = p.slices * kZSlice;
  const int steps = p.k / 32;
  live_slots(p, m0, count, tslot, list);
  const int nd = list[kMaxList];
  // Counting sort of the tile's live tokens by distinct slot index.
  for (int d = tid; d <= nd; d += kThreads) cnt[d] = 0;
  __syncthreads();
  // Every producer of the tile must cut the same units, so a token's place is
  // fixed: its slot's first position plus the number of earlier tokens of the
  // same slot (ballots over tslot, not an LDS atomic's arrival order).
  int my_d = -1, my_rank = 0;
  if (tid < count && tslot[tid] >= 0) {
    const int gt = tslot[tid];
    for (int d = 0; d < nd; ++d)
      if (list[d] == gt) my_d = d;
    atomicAdd(&cnt[my_d], 1);
  }
  {
    const int gt = tid < count ? tslot[tid] : -1;
    for (int ch = 0; ch <= wave; ++ch) {
      const int other = ch * 64 + lane < count ? tslot[ch * 64 + lane] : -1;
      uint64_t left = __ballot(gt >= 0);
      while (left) {
        const int gf = __builtin_amdgcn_readlane(gt, __builtin_ctzll(left));
        left &= ~__ballot(gt == gf);
        uint64_t same = __ballot(other == gf);
        if (ch == wave) same &= (uint64_t(1) << lane) - 1;
        if (gt == gf) my_rank += __popcll(same);
      }
    }
  }
  __syncthreads();
  // (Every producer of the tile, and a consumer that recomputes, finds the same size.)
  constexpr int kTokTiles = kUnitSteps == 0 ? 1 : 2;
  int size = kUnit;
  if constexpr (kTokTiles == 2) {
    int units = 0;
    for (int d = 0; d < nd; ++d) units += (cnt[d] + kUnit - 1) / kUnit;
    if (units > p.zparts) size = 2 * kUnit;
    __syncthreads();
  }
  if (tid == 0) {
    int pos = 0, units = 0;
    for (int d = 0; d < nd; ++d) {
      const int n = cnt[d];
      cnt[d] = pos;       // first position of slot d's tokens in `order`
      ustart[d] = units;  // first unit of slot d
      pos += n;
      units += (n + size - 1) / size;
    }
    cnt[nd] = pos;
    ustart[nd] = units;
  }
  __syncthreads();
  if (my_d >= 0) order[cnt[my_d] + my_rank] = tid;  // slot d holds positions cnt[d] .. cnt[d + 1]
  __syncthreads();
  // Zero the padding columns r .. 63 of every slice of the tokens this producer serves.
  const int units = ustart[nd];
  for (int u = rp == 0 ? q : units; u < units; u += p.zparts) {
    int d = 0;
    while (ustart[d + 1] <= u) ++d;
    const int first = cnt[d] + (u - ustart[d]) * size;
    const int ntok = min(size, cnt[d + 1] - first);
    const int r = p.ranks[list[d]];
    for (int i = tid; i < ntok * zw; i += kThreads) {
      const int t = i / zw;
      const int col = i - t * zw;
      if ((col & (kZSlice - 1)) >= r) store_z(p.zpad + int64_t(m0 + order[first + t]) * zw + col, 0);
    }
  }
  for (int u = q; u < units; u += p.zparts) {
    int d = 0;
    while (ustart[d + 1] <= u) ++d;
    const int first = cnt[d] + (u - ustart[d]) * size;
    const int ntok = min(size, cnt[d + 1] - first);
    const int gd = list[d];
    const int r = p.ranks[gd];
    const int rows = p.slices * r;
    const uint16_t* abase = p.a_store + p.a_offsets[gd];
    const uint16_t* xrow[kTokTiles];
#pragma unroll
    for (int i = 0; i < kTokTiles; ++i)
      xrow[i] = p.x + int64_t(m0 + order[first + min(16 * i + c, ntok - 1)]) * p.x_stride + 8 * kg;
    const bool two = ntok > kUnit;  // (uniform)
    for (int j0 = rp * kPassRows; j0 < rows; j0 += parts * kPassRows) {
      f32x4 acc[kTokTiles][kRowTiles];
#pragma unroll
      for (int i = 0; i < kTokTiles; ++i)
#pragma unroll
        for (int jt = 0; jt < kRowTiles; ++jt) acc[i][jt] = (f32x4){0.f, 0.f, 0.f, 0.f};
      const int tiles = (min(kPassRows, rows - j0) + 15) >> 4;  // uniform
      if constexpr (kUnitSteps == 0) {
        acc[0][0] = contract_staged<kWaves>(p, abase, j0, rows, m0, order + first, ntok, ring);
      } else for (int s0 = wave; s0 < steps; s0 += kWaves * kUnitSteps) {
        // Loads of this batch's steps first (past the end: a readable step, not contracted).
        uint4 xb[kUnitSteps][kTokTiles], ab[kUnitSteps][kRowTiles];
#pragma unroll
        for (int v = 0; v < kUnitSteps; ++v) {
          const int st = min(s0 + v * kWaves, steps - 1);
#pragma unroll
          for (int i = 0; i < kTokTiles; ++i)
            if (i == 0 || two) xb[v][i] = *reinterpret_cast<const uint4*>(xrow[i] + st * 32);
#pragma unroll
          for (int jt = 0; jt < kRowTiles; ++jt)
            if (jt < tiles)
              ab[v][jt] = *reinterpret_cast<const uint4*>(abase + int64_t(min(j0 + jt * 16 + c, rows - 1)) * p.k +
                                                          st * 32 + 8 * kg);
        }
#pragma unroll
        for (int v = 0; v < kUnitSteps; ++v)
          if (s0 + v * kWaves < steps)
#pragma unroll
            for (int jt = 0; jt < kRowTiles; ++jt)
              if (jt < tiles)
#pragma unroll
                for (int i = 0; i < kTokTiles; ++i)
                  if (i == 0 || two) acc[i][jt] = mfma16(as_bf16x8(ab[v][jt]), as_bf16x8(xb[v][i]), acc[i][jt]);
      }
      // acc[i][jt][e] = this wave's partial of z[token 16 i + c][A row j0 + 16 jt + 4 kg + e].
      constexpr int kRedRow = 16 * kTokTiles + 1;
#pragma unroll
      for (int i = 0; i < kTokTiles; ++i)
#pragma unroll
        for (int jt = 0; jt < kRowTiles; ++jt)
#pragma unroll
          for (int e = 0; e < 4; ++e) red[((wave * kRowTiles + jt) * 16 + 4 * kg + e) * kRedRow + 16 * i + c] = acc[i][jt][e];
      static_assert(kUnitSteps == 0 || kWaves * kRowTiles * 16 * kRedRow * 4 <= kMinRing, "the partial tiles fit the idle x ring");
      __syncthreads();
      for (int o = tid; o < kPassRows * kUnit * kTokTiles; o += kThreads) {
        const int jr = o / (kUnit * kTokTiles);  // A row within the pass
        const int t = o % (kUnit * kTokTiles);
        const int j = j0 + jr;
        if (t < ntok && j < rows) {
          float sum = 0.f;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) sum += red[((w * kRowTiles + (jr >> 4)) * 16 + (jr & 15)) * kRedRow + t];
          const int sl = j / r;
          store_z(p.zpad + int64_t(m0 + order[first + t]) * zw + sl * kZSlice + (j - sl * r), uint16_t(f32_to_bf16(sum)));
        }
      }
      __syncthreads();  // red is reused by the next pass
    }
  }
  // Every thread's z stores have completed (sc1: at device scope) when this
  // returns (asm with a memory clobber, so the compiler keeps later stores
  // after it).
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  __syncthreads();
}

// Producer (mt, q): its units, then its flag carries the call's tag.
template <int kUnitSteps, int kRowTiles, int kThreads = prefill::kThreads>
__device__ __forceinline__ void produce_z(const PrefillParams& p, int mt, int q, int rp, int parts, uint32_t tag, int* tslot, int* list,
                                          int* order, int* cnt, int* ustart, float* red, char* ring = nullptr) {
  if (p.withhold) return;  // test hook: the tile's consumers must recompute
  produce_units<kUnitSteps, kRowTiles, kThreads>(p, mt, q, rp, parts, tslot, list, order, cnt, ustart, red, ring);
  if (threadIdx.x == 0 && p.zflags) __hip_atomic_store(p.zflags + mt * p.zparts + q, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until the z rows of M-tile mt carry the call's tag (their producers
// have lower block ids, so they were dispatched before this workgroup).
// The flags and the z rows are read with device-scope loads (coherent past
// the caches of this CU and XCD), so no acquire fence is needed: an acquire
// at device scope would invalidate the whole L2 of the XCD under the other
// workgroups' feet. Each wait is bounded (about a quarter second); a
// producer that has not set its flag by then has its units recomputed here
// (the sums of a producer in this launch, so its z bits; one of a launch of its
// own sums over eight waves, another order), the status word records it, and the
// tile's slot metadata, whose LDS the recomputation borrowed, is reloaded.
// Returns whether it recomputed anything.
__device__ bool wait_z(const PrefillParams& p, int mt, uint32_t tag, int* tslot, int* list, int* order, int* mrank,
                       int* mstride, float* mscale, int64_t* mboff, float* red, uint32_t* missing) {
  if (threadIdx.x < 2) missing[threadIdx.x] = 0;
  __syncthreads();
  if (threadIdx.x < p.zparts) {
    const uint32_t* flag = p.zflags + mt * p.zparts + threadIdx.x;
    for (int spins = 0; __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != tag; ++spins) {
      if (spins > p.spin_limit) {
        atomicOr(&missing[threadIdx.x >> 5], 1u << (threadIdx.x & 31));
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
  }
  __syncthreads();
  const uint64_t lost = uint64_t(missing[0]) | (uint64_t(missing[1]) << 32);
  if (lost == 0) return false;
  if (threadIdx.x == 0) __hip_atomic_store(p.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // (Producers of a launch of their own cut other units: then all are made again. One tile in
  // flight, fewer registers: the sums are the same.)
  for (int q = 0; q < p.zparts; ++q)
    if (p.zblocks == 0 || ((lost >> q) & 1)) produce_units<1, 1>(p, mt, q, 0, 1, tslot, list, order, mrank, mstride, red);
  int tid = threadIdx.x;
  tie(tid);  // (opaque: nothing of this rare path is kept from before the k-loop)
  for (int d = tid; d < list[kMaxList]; d += kThreads) {
    const int gg = list[d];
    mrank[d] = p.ranks[gg];
    mstride[d] = p.b_strides[gg];
    mscale[d] = p.lscales[gg];
    mboff[d] = p.b_offsets[gg];
  }
  __syncthreads();
  return true;
}

// 16 bytes of z rows in one device-scope (sc1) load, coherent past this
// XCD's L2 like the agent-scope atomics; one request instead of four.
// Untracked: the caller waits (vmcnt) and ties the value before any use.
__device__ __forceinline__ u32x4 load_z16(const uint16_t* src) {
  u32x4 v;
  asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v) : "v"(src) : "memory");
  return v;
}

// Counts the workgroup in; the last one moves the epoch on (call_epoch.h).
__device__ __forceinline__ void depart(const PrefillParams& p, uint32_t tag) {
  if (threadIdx.x < 64) {
    const uint32_t old = depart_issue(p.ce, threadIdx.x);
    depart_finish(p.ce, old, tag - 1u, threadIdx.x);
  }
}


// The tile's output as packed bf16 pairs: o.v[i][j][2 q + e / 2] of lane l
// holds token 32 i + l % 32, features wn0 + 32 j + 8 q + 4 (l / 32) + e.
template <int RI>
struct Out {
  uint32_t v[RI][kJ][8];
};

// bf16 rounding of the contraction, then of the bias add.
template <int RI>
__device__ __forceinline__ void round_bias(const PrefillParams& p, const Acc<RI>& acc, Out<RI>& o, int wn0, int h) {
#pragma unroll
  for (int j = 0; j < kJ; ++j)
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
      for (int r = 0; r < 8; ++r) o.v[i][j][r] = pack_bf16x2(acc.v[i][j][2 * r], acc.v[i][j][2 * r + 1]);
  if (p.bias) {
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int n = min(wn0 + 32 * j + 8 * (r >> 1) + 4 * h + 2 * (r & 1), p.n - 2);
        const float b0 = bf16_to_f32(p.bias[n]), b1 = bf16_to_f32(p.bias[n + 1]);
#pragma unroll
        for (int i = 0; i < RI; ++i) o.v[i][j][r] = pack_bf16x2(bf16_lo(o.v[i][j][r]) + b0, bf16_hi(o.v[i][j][r]) + b1);
      }
  }
}

// Weight row of tile row r (0 .. kBN - 1) in column tile nt. SwiGLU output:
// tile nt produces activation columns kBN/2 nt .. + kBN/2; its rows below
// kBN/2 are the gate rows of those columns, the others the matching up rows
// (n / 2 further on), so a wave's 64 rows stay contiguous.
template <bool kSwiglu>
__device__ __forceinline__ int tile_row(const PrefillParams& p, int nt, int r) {
  if constexpr (!kSwiglu) return nt * kBN + r;
  constexpr int kHalf = kBN / 2;
  return r < kHalf ? nt * kHalf + r : (p.n >> 1) + nt * kHalf + (r - kHalf);
}

// The producers as a launch of their own, ahead of the GEMM's on the same
// stream. It takes the call's tag but leaves counting in (and so moving the
// epoch on) to the GEMM launch, which finds every flag set.
// (Eight waves: their 128 KiB of copies in flight fill the CU.)
constexpr int kZThreads = 512;
#ifdef LF_PREFILL_Z_KERNEL
__global__ __launch_bounds__(kZThreads) void z_kernel(PrefillParams p) {
  __shared__ __attribute__((aligned(256))) char ring[kZThreads / 64 * 2 * kZSlot];
  __shared__ __attribute__((aligned(16))) float red[kZThreads / 64 * 16 * 17];
  __shared__ __attribute__((aligned(16))) int tslot[kBM];
  __shared__ int list[kMaxList + 1], order[kBM], cnt[kMaxList + 1], ustart[kMaxList + 1];
  const uint32_t tag = p.zflags ? __builtin_amdgcn_readfirstlane(epoch_tag(p.ce)) : 0u;
  const int unit = blockIdx.x / p.zrow_parts;
  produce_z<0, 1, kZThreads>(p, unit / p.zparts, unit % p.zparts, blockIdx.x % p.zrow_parts, p.zrow_parts, tag, tslot, list, order, cnt, ustart, red, ring);
}
#endif

// Block ids below zblocks (LoRA launches whose last round has room for them)
// produce the tiles' z rows; the others are GEMM tiles, M-tile b % mtiles on
// consecutive ids.
// The kernel's parameters through an opaque copy of the kernarg pointer:
// fields read after this are loaded where they are used instead of being held
// in scalar registers across the k-loop. (The kernel's only argument is the
// PrefillParams, at offset 0 of the kernarg segment.)
__device__ __forceinline__ const PrefillParams& reload() {
  auto q = (const __attribute__((address_space(4))) PrefillParams*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(q));
  return *(const PrefillParams*)q;
}

template <int RI, bool kLora, bool kSwiglu>
__global__ __launch_bounds__(kThreads, 1) void gemm_kernel(PrefillParams pk) {
  constexpr int kRows = RI * 32;
  constexpr int kStage = stage_bytes<RI>();
  constexpr int kR = kRing<RI>;
  // (At least what the epilogue stages there: the output tile, or z of three slices.)
  constexpr int kRingBytes = kR * kStage > kMinRing ? kR * kStage : kMinRing;
  __shared__ __attribute__((aligned(256))) char xring[kRingBytes];
  __shared__ __attribute__((aligned(256))) char wring[kWaves * 4096];  // packed weights, 4 KiB per wave
  __shared__ __attribute__((aligned(16))) int tslot[kLora ? kBM : 1];
  __shared__ int list[kLora ? kMaxList + 1 : 1];
  __shared__ int order[kLora ? kBM : 1];  // z producer: tile rows sorted by slot
  __shared__ uint32_t zmissing[2];        // producers of the tile whose flag never came
  __shared__ int mrank[kLora ? kMaxList + 1 : 1];
  __shared__ int mstride[kLora ? kMaxList + 1 : 1];
  __shared__ float mscale[kLora ? kMaxList : 1];
  __shared__ int64_t mboff[kLora ? kMaxList : 1];
  const int tid = threadIdx.x;
  int b = blockIdx.x;
  uint32_t tag = 0;
  const PrefillParams& p = pk;
  if constexpr (kLora) {
    tag = __builtin_amdgcn_readfirstlane(epoch_tag(p.ce));
    if (b < p.zblocks) {
      // (The slot metadata arrays double as the producer's sort counters; the
      // idle x ring holds the partial tiles.)
      produce_z<4, 4>(p, b / p.zparts, b % p.zparts, 0, 1, tag, tslot, list, order, mrank, mstride, reinterpret_cast<float*>(xring));
      depart(p, tag);
      return;
    }
    b -= p.zblocks;
  }
  const int mt = b % p.mtiles;
  const int nt = b / p.mtiles;
  const int m0 = mt * kRows;
  const int n0 = nt * kBN;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 31;
  const int h = lane >> 5;
  const int stages = p.k / kBK;

  // Weight addresses. (Rows past N are clamped: their results are never stored.)
  const int wn0 = tile_row<kSwiglu>(p, nt, wave * 64);
  char* wbuf = wring + wave * 4096;
  WLane wl;
  {
    const int first = min(wn0, p.n - 1);
    wl.q = reinterpret_cast<const char*>(p.q) + int64_t(first) * (p.k >> 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * i + (lane >> 2);
      wl.off[i] = uint32_t(min(wn0 + r, p.n - 1) - first) * uint32_t(p.k >> 1) + (((lane & 3) ^ ((r >> 2) & 3)) << 4);
    }
    wl.read = lds_addr(wbuf) + uint32_t(c * 64 + (((2 * h) ^ ((c >> 2) & 3)) << 4));
#pragma unroll
    for (int j = 0; j < kJ; ++j)
      wl.s[j] = reinterpret_cast<const char*>(p.src.scales) +
                int64_t(min(wn0 + 32 * j + c, p.n - 1)) * (p.k / kNf4Block) * 4;
    wl.smax = (p.k / kNf4Block - 2) * 4;
  }
  XLane xl;
  const int xrow = wave * 4 + (lane >> 4);          // the lane's first row of a copy
  const uint32_t xunit = (lane & 15) ^ xrow;        // (its rows differ by multiples of 16)
  const uint32_t rowb = uint32_t(p.x_stride) * 2u;
  xl.last = uint32_t(p.m - 1) * rowb + xunit * 16u;
  xl.first = uint32_t(min(m0 + xrow, p.m - 1)) * rowb + xunit * 16u;
  const uint32_t row16 = rowb * 16u;
  float code[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) code[i] = sload(p.code, i);

  Acc<RI> acc;
#pragma unroll
  for (int i = 0; i < RI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc.v[i][j][r] = 0.f;

  // Fragment read address: row c (+ 32 i), unit 8 h + t at (8 h + t) ^ (row & 15);
  // step t flips bits 4..6 of the stage-aligned address.
  const uint32_t xbase = lds_addr(xring) + uint32_t(c * kXRow + (((8 * h) ^ (c & 15)) << 4));
  auto load_routes = [&]() {
    // The tile's routes and slot metadata (three dependent loads), behind the
    // first copies.
    if constexpr (kLora) {
      live_slots(p, m0, min(kRows, p.m - m0), tslot, list);
      for (int d = tid; d < list[kMaxList]; d += kThreads) {
        const int gg = list[d];
        mrank[d] = p.ranks[gg];
        mstride[d] = p.b_strides[gg];
        mscale[d] = p.lscales[gg];
        mboff[d] = p.b_offsets[gg];
      }
    }
  };
  if (stages > 0) {
    Packed even, odd;  // weights of even and odd stages
    Scales cs, ns;     // scales of this pair of stages (the second one's) and of the next pair
    Codes codes[kJ], ncodes[kJ];
    const int last = stages - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_w(wl, 0, i, wbuf);
#pragma unroll
    for (int j = 0; j < kJ; ++j) load_scales(wl, 0, h, j, cs);
    copy_x<RI, 2 * RI>(p, xl, row16, 0, xring, wave);
    if constexpr (kLora) load_routes();
    wait_vm<0>();
    read_w(wl, even);
    lds_wait();
    tie_w(even);
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_w(wl, min(1, last), i, wbuf);
    if constexpr (kR > 2) copy_x<RI, 2 * RI>(p, xl, row16, min(1, last), xring + kStage, wave);
    copy_x<RI, kFirstCopies<RI>>(p, xl, row16, min(kR - 1, last), xring + (kR - 1) * kStage, wave);
    wait_vm<kFirstCopies<RI>>();
    barrier_only();
    read_w(wl, odd);
    lds_wait();
    tie_w(odd);
    XFrags<RI> xa, xb;
    u32x4 wa[kJ], wb[kJ];
    read_x<RI>(xbase, xa);
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      pair_scales(cs, j);
      block_codes(code, cs.s[j][0], codes[j]);
      wa[j] = decode8(even.q[j][0].x, codes[j]);
    }
    wait_x<RI>(xa);
    // cs: the scales of stages 2 q and 2 q + 1; ns: those of the next pair, loaded
    // in the even stage and paired in the odd one.
    auto stage = [&](int st, auto oc, Packed& cur, Packed& nxt) {
      constexpr bool kOdd = decltype(oc)::value;
      // Ring slots of stages st, st + 1 and st + kR - 1.
      const int s0 = st % kR, s1 = (st + 1) % kR, s2 = (st + kR - 1) % kR;
      const uint32_t here = xbase + uint32_t(s0) * kStage;
      const uint32_t there = xbase + uint32_t(s1) * kStage;
      char* freed = xring + s0 * kStage;
      char* other = xring + s2 * kStage;
      const int w2 = min(st + 2, last);
      const char* x1 = reinterpret_cast<const char*>(p.x) + int64_t(min(st + kR - 1, last)) * kXRow;
      const char* x2 = reinterpret_cast<const char*>(p.x) + int64_t(min(st + kR, last)) * kXRow;
      // Step t contracts the fragments read and decoded in step t - 1, and
      // reads and decodes those of step t + 1 (of the next stage at t = 7).
      // The MFMAs are the frame: behind each goes a slot of other work short
      // enough for its shadow: decode pieces, a quarter of the next block's
      // codes (steps 2..5), copies of stage + 2's weights (step 0), of x of
      // stages + kR - 1 (four steps) and + kR (step 7), and in even stages the
      // loads of the next pair's scales (step 0: a use that the compiler had to
      // wait for would also wait for the x copies behind them).
      auto step = [&](auto tc, XFrags<RI>& xc, u32x4 (&wc)[kJ], XFrags<RI>& xn, u32x4 (&wn)[kJ]) {
        constexpr int t = decltype(tc)::value;
        constexpr bool kLast = t == kSteps - 1;
        constexpr int kNext = (t + 1) % kSteps;
        if constexpr (kLast) {
          // The next stage's x, the weights after it and the next scales have
          // landed once only this stage's x copies (three stages: all behind
          // its weight copies and scale loads) or nothing (two stages) is
          // outstanding; past the barrier this stage's x is free.
          wait_vm<(kR > 2 ? 2 * RI - kFirstCopies<RI> : 0)>();
          barrier_only();
          read_x<RI>(there, xn);
          read_w(wl, cur);
#pragma unroll
          for (int j = 0; j < kJ; ++j) codes[j] = ncodes[j];
        } else {
          read_x<RI>(here ^ (kNext << 4), xn);
        }
        constexpr int kCopies = 2 * RI;
        constexpr int kFirst = kFirstCopies<RI>;
        constexpr int kEach = (kCopies - kFirst + 3) / 4;
        constexpr int kFrom = kR > 2 ? 1 : 0;  // first of the four steps
        constexpr int c0 = kLast ? 0 : (t < kFrom ? kCopies : (kFirst + (t - kFrom) * kEach < kCopies ? kFirst + (t - kFrom) * kEach : kCopies));
        constexpr int c1 = kLast ? kFirst : (c0 + kEach < kCopies ? c0 + kEach : kCopies);
        Decode dec[kJ];
        CodeBuild build[kJ];
        __builtin_amdgcn_sched_barrier(0);
        constexpr int kSlots = RI * kJ;
#pragma unroll
        for (int m = 0; m < kSlots; ++m) {
          const int i = m / kJ, j = m % kJ;
          acc.v[i][j] = mfma32(vec_bf16x8(wc[j]), vec_bf16x8(xc.v[i]), acc.v[i][j]);
          const Packed& src = kLast ? nxt : cur;
#pragma unroll
          for (int k = m * kPieces / kSlots; k < (m + 1) * kPieces / kSlots; ++k)
#pragma unroll
            for (int f = 0; f < kJ; ++f)
              dec[f].piece(k, src.q[f][kNext >> 2][kNext & 3], codes[f], wn[f]);
#pragma unroll
          for (int f = 0; f < kJ; ++f) {
            if (kOdd && t == 1 && m == 0) {
              pair_scales(ns, f);
              cs.s[f][0] = ns.s[f][0];
              cs.s[f][1] = ns.s[f][1];
            }
            if (t >= 2 && t < 6) {
#pragma unroll
              for (int k = 0; k < 3; ++k)
                if (m == f * kSlots / kJ + k * (kSlots / kJ) / 3)
                  build[f].phase(k, code, cs.s[f][kOdd ? 0 : 1], t - 2, ncodes[f]);
            }
            if (!kOdd && t == 0 && m == f) load_scales(wl, w2, h, f, ns);
          }
          if (t == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (m == k * kSlots / 4) copy_w(wl, w2, k, wbuf);
          }
#pragma unroll
          for (int d = c0; d < c1; ++d)
            if (m == (d - c0) * kSlots / (c1 > c0 ? c1 - c0 : 1))
              copy16((kLast ? x2 : x1) + min(xl.first + uint32_t(d) * row16, xl.last),
                     (kLast ? freed : other) + (d * kWaves + wave) * 1024);
          __builtin_amdgcn_sched_barrier(0);
        }
        wait_x<RI>(xn);
        if constexpr (kLast) tie_w(cur);
      };
      step(std::integral_constant<int, 0>{}, xa, wa, xb, wb);
      step(std::integral_constant<int, 1>{}, xb, wb, xa, wa);
      step(std::integral_constant<int, 2>{}, xa, wa, xb, wb);
      step(std::integral_constant<int, 3>{}, xb, wb, xa, wa);
      step(std::integral_constant<int, 4>{}, xa, wa, xb, wb);
      step(std::integral_constant<int, 5>{}, xb, wb, xa, wa);
      step(std::integral_constant<int, 6>{}, xa, wa, xb, wb);
      step(std::integral_constant<int, 7>{}, xb, wb, xa, wa);
    };
    // (An odd last stage stands alone: a way around the odd stage inside the
    // loop would make the compiler wait, at the top of every pair, for the
    // scale loads that only the odd stage consumes, and with them for the x
    // copies just issued.)
    for (int st = 0; st + 1 < stages; st += 2) {
      stage(st, std::false_type{}, even, odd);
      stage(st + 1, std::true_type{}, odd, even);
    }
    if (stages & 1) stage(last, std::false_type{}, even, odd);
    wait_vm<0>();  // the requests past the end
    barrier_only();
  }
  if constexpr (kLora) {
    if (stages == 0) load_routes();
  }
  if (p.k % kBK != 0) {
    // The last 64 k (one block): both lane halves hold it, step t contracts
    // k 16 t + 8 h .. + 8. Copies of units 8..15 repeat units 0..7.
    const uint32_t dup = (xunit & 7u) * 16u - xunit * 16u;
    const char* base = reinterpret_cast<const char*>(p.x) + int64_t(stages) * kXRow;
#pragma unroll
    for (int d = 0; d < 2 * RI; ++d)
      copy16(base + (min(xl.first + uint32_t(d) * row16, xl.last) + dup), xring + (d * kWaves + wave) * 1024);
    Packed tail;
    Codes codes[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      const int64_t row = min(wn0 + 32 * j + c, p.n - 1);
      const char* q = reinterpret_cast<const char*>(p.q) + row * (p.k >> 1) + int64_t(stages) * 64;
      tail.q[j][0] = gload16(q, 0);
      tail.q[j][1] = gload16(q, 16);
      block_codes(code, gloadf(wl.s[j] + int64_t(stages) * 8), codes[j]);
    }
    wait_vm<0>();
    barrier_only();
    const uint32_t tbase = lds_addr(xring) + uint32_t(c * kXRow + ((h ^ (c & 15)) << 4));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      XFrags<RI> x;
      read_x<RI>(tbase ^ (t << 5), x);
      u32x4 w[kJ];
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const uint32_t lo = tail.q[j][t >> 1][(2 * t) & 3], hi = tail.q[j][t >> 1][(2 * t + 1) & 3];
        w[j] = decode8(h ? hi : lo, codes[j]);
      }
      wait_x<RI>(x);
      contract<RI>(w, x, acc);
    }
    barrier_only();
  }

  // ---- epilogue: acc[i][j][4 q + e] = C[token m0 + 32 i + c][feature wn0 + 32 j + 8 q + 4 h + e]
  // (W is the MFMA's A operand, so a lane holds four consecutive features of
  // one token).
  {
  // (Likewise the lane's place, re-derived from an opaque thread id.)
  const PrefillParams& p = reload();
  int tid = threadIdx.x;
  tie(tid);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = tid & 31;
  const int h = (tid >> 5) & 1;
  Out<RI> o;
  round_bias<RI>(p, acc, o, wn0, h);
  if constexpr (kLora) {
    const int nd = list[kMaxList];
    const int zw = p.slices * kZSlice;
    // B fragments of slot d as the MFMA's A operand: feature wn0 + 32 j + c,
    // ranks 16 q + 8 h .. + 8. Requested raw from clamped, readable places and
    // masked where used: past the row stride or the rank, and past N.
    auto request_b = [&](int d, uint4 (&bq)[kJ][4]) {
      const int br = mstride[d];
      const int steps = (mrank[d] + 15) >> 4;
      const uint16_t* bg = p.b_store + mboff[d];
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const uint16_t* row = bg + int64_t(min(wn0 + 32 * j + c, p.n - 1)) * br;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < steps) bq[j][q] = b_raw(row, br, 16 * q + 8 * h);
      }
    };
    uint4 bq[kJ][4], bnext[kJ][4];
    if (nd > 0) request_b(0, bnext);
    wait_z(p, mt, tag, tslot, list, order, mrank, mstride, mscale, mboff, reinterpret_cast<float*>(xring), zmissing);
    // Every slice's z rows are staged at once (slice s at unit s * kRows * 8
    // of the idle x ring: [token][8 units], unit ^ (row & 7)), so after one
    // barrier each wave applies exactly the slices its 64 columns touch.
    static_assert(3 * kRows * 8 * 16 <= kRingBytes, "the z rows of three slices fit the x ring");
    uint4* zs_all = reinterpret_cast<uint4*>(xring);
    constexpr int kZq = kRows * 8 / kThreads;  // 16-byte z units per thread and slice
    for (int s = 0; s < p.slices; ++s) {
      u32x4 zr[kZq];
      // Every lane loads (rows past M read row M - 1, base-only rows are
      // zeroed after the wait): no branch around the untracked loads.
#pragma unroll
      for (int q = 0; q < kZq; ++q) {
        const int row = min(m0 + (tid >> 3) + (kThreads / 8) * q, p.m - 1);
        zr[q] = load_z16(p.zpad + int64_t(row) * zw + s * kZSlice + (tid & 7) * 8);
      }
      wait_vm<0>();
#pragma unroll
      for (int q = 0; q < kZq; ++q) tie(zr[q]);
#pragma unroll
      for (int q = 0; q < kZq; ++q) {
        const int row = (tid >> 3) + (kThreads / 8) * q;
        zs_all[s * kRows * 8 + swz(row, tid & 7)] =
            tslot[row] >= 0 ? make_uint4(zr[q].x, zr[q].y, zr[q].z, zr[q].w) : make_uint4(0, 0, 0, 0);
      }
    }
    __syncthreads();
    // The output pair (j, r) of the lane's token in a block: bf16(scale * delta), then the
    // sum with the rounded base. (token: all ones for a token to update.)
    auto updated = [&](uint32_t old, float d0, float d1, uint32_t token, bool inside, int lo, int hi, int j, int r) {
      const uint32_t v = pack_bf16x2(d0, d1);
      const uint32_t sum = pack_bf16x2(bf16_lo(old) + bf16_lo(v), bf16_hi(old) + bf16_hi(v));
      uint32_t take = token;
      if (!inside) {  // columns of other slices keep their value
        const int n = wn0 + 32 * j + 8 * (r >> 1) + 4 * h + 2 * (r & 1);
        take &= ((n >= lo && n < hi) ? 0xffffu : 0u) | ((n + 1 >= lo && n + 1 < hi) ? 0xffff0000u : 0u);
      }
      return select(take, sum, old);
    };
    if (RI <= kManyRows && nd > kFewSlots) {
      // Tiles of many slots: the deltas of all of a block's slots meet in the idle
      // accumulators and are rounded once. A slot's MFMAs take the z of its own tokens
      // and zeros for the others, so a token gets its own slot's sum plus exact zeros.
      // An infinity or NaN in a slot's B makes NaN of the zeros: a tile that shows one
      // is done again with a rounding pass per slot. (The masked rounding pass per slot
      // and block below is 190 VALU instructions. Tokens of 32 slots of rank 16 in turn,
      // below -> here: 512 x 4096 x 4096 in 64-token tiles 108.5 -> 84.6 us, 512 x 16384
      // x 1024 in 128-token tiles 144.8 -> 101.3 us. Taller tiles have no registers for
      // both forms: with both, few slots take 3-12 % longer.)
      for (int g = -1, d = 0; d < nd; ++d) {
        if (list[d] == tslot[tid]) g = d;
        if (d == nd - 1) order[tid] = g;
      }
      __syncthreads();
      int td[RI];         // the lane's token in each block: its slot's place in the list
      uint64_t left[RI];  // lanes whose slot is still to come
      auto pick = [&]() {
        int d = -1;
#pragma unroll
        for (int i = RI - 1; i >= 0; --i)
          if (left[i]) d = __builtin_amdgcn_readlane(td[i], __builtin_ctzll(left[i]));
        return d;
      };
      auto begin = [&]() {
#pragma unroll
        for (int i = 0; i < RI; ++i) left[i] = __ballot(td[i] >= 0);
        return pick();
      };
#pragma unroll
      for (int i = 0; i < RI; ++i) td[i] = order[32 * i + c];
      for (int s = 0; s < p.slices; ++s) {
        const int lo = p.slice_offsets[s];
        const int hi = p.slice_offsets[s + 1];
        if (hi <= wn0 || lo >= wn0 + 64) continue;  // this wave's 64 columns miss the slice
        const bool inside = lo <= wn0 && wn0 + 64 <= hi;
        const uint4* zs = zs_all + s * kRows * 8;
        int d = begin();     // (slot 0, whose B is in flight)
        bool each = false;   // a rounding pass per slot
        while (d >= 0) {
          uint32_t done = 0;  // blocks whose token has its delta
#pragma unroll
          for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int r = 0; r < 16; ++r) acc.v[i][j][r] = 0.f;
          do {
            const int slot = d;
            const int rank = mrank[slot];
            const int keep = min(mstride[slot], rank) - 8 * h;
            const int steps = (rank + 15) >> 4;
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int q = 0; q < 4; ++q) bq[j][q] = bnext[j][q];
#pragma unroll
            for (int i = 0; i < RI; ++i) left[i] &= ~__ballot(td[i] == slot);
            d = pick();
            request_b(max(d, 0), bnext);  // (after the last slot, for the next slice)
            if (rank & 15)
#pragma unroll
              for (int j = 0; j < kJ; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                  if (q < steps) bq[j][q] = keep_first(bq[j][q], keep - 16 * q);
#pragma unroll
            for (int i = 0; i < RI; ++i) {
              const bool mine = td[i] == slot;
              if (__ballot(mine) == 0) continue;  // no token of the slot in this block
              if (mine) done |= 1u << i;
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (q < steps) {
                  uint4 z = zs[swz(32 * i + c, 2 * q + h)];
                  if (!mine) z = make_uint4(0, 0, 0, 0);
#pragma unroll
                  for (int j = 0; j < kJ; ++j) acc.v[i][j] = mfma32(as_bf16x8(bq[j][q]), as_bf16x8(z), acc.v[i][j]);
                }
            }
          } while (d >= 0 && !each);
          if (!each) {
            float nan = 0.f;
#pragma unroll
            for (int i = 0; i < RI; ++i)
#pragma unroll
              for (int j = 0; j < kJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) nan = fmaf(acc.v[i][j][r], 0.f, nan);
            if (__ballot(nan != nan) != 0) {
              each = true;
              d = begin();
              continue;
            }
          }
#pragma unroll
          for (int i = 0; i < RI; ++i) {
            const uint32_t token = (done >> i) & 1 ? 0xffffffffu : 0u;
            if (__ballot(token != 0) == 0) continue;
            const float scale = mscale[max(td[i], 0)];
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int r = 0; r < 8; ++r)
                o.v[i][j][r] = updated(o.v[i][j][r], acc.v[i][j][2 * r] * scale, acc.v[i][j][2 * r + 1] * scale, token, inside, lo, hi, j, r);
          }
        }
      }
    } else {
      bool first_ready = true;  // the B of slot 0 requested above is still unused
      for (int s = 0; s < p.slices; ++s) {
        const int lo = p.slice_offsets[s];
        const int hi = p.slice_offsets[s + 1];
        if (hi <= wn0 || lo >= wn0 + 64) continue;  // this wave's 64 columns miss the slice
        const bool inside = lo <= wn0 && wn0 + 64 <= hi;
        const uint4* zs = zs_all + s * kRows * 8;
        // delta[n][m] = sum_j B_g[n][j] z[m][j], added with the reference's two
        // roundings to the tokens routed to g and the features of slice s. The
        // next slot's B is in flight while this slot's MFMAs run.
        if (!first_ready && nd > 0) request_b(0, bnext);
        first_ready = false;
        for (int d = 0; d < nd; ++d) {
#pragma unroll
          for (int j = 0; j < kJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) bq[j][q] = bnext[j][q];
          if (d + 1 < nd) request_b(d + 1, bnext);
          const int gd = list[d];
          const int rank = mrank[d];
          const int steps = (rank + 15) >> 4;
          const float scale = mscale[d];
#pragma unroll
          for (int j = 0; j < kJ; ++j) {
            // (A rank that fills its last step needs no mask; nor do rows past
            // N, whose results are never stored.)
            if (rank & 15) {
              const int keep = min(mstride[d], rank) - 8 * h;
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (q < steps) bq[j][q] = keep_first(bq[j][q], keep - 16 * q);
            }
          }
          // 32-token blocks with a token of gd, the delta of one block two
          // MFMA chains ahead of its use.
          uint32_t here = 0;
          bool mine[RI];
#pragma unroll
          for (int i = 0; i < RI; ++i) {
            mine[i] = tslot[32 * i + c] == gd;
            if (__ballot(mine[i]) != 0) here |= 1u << i;
          }
#pragma unroll
          for (int i = 0; i < RI; ++i) {
            if (((here >> i) & 1) == 0) continue;
            f32x16 delta[kJ];
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int r = 0; r < 16; ++r) delta[j][r] = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (q < steps) {
                const bf16x8 z = as_bf16x8(zs[swz(32 * i + c, 2 * q + h)]);
#pragma unroll
                for (int j = 0; j < kJ; ++j) delta[j] = mfma32(as_bf16x8(bq[j][q]), z, delta[j]);
              }
            // bf16(scale * delta), then the sum with the rounded base; other
            // slots' tokens and other slices' columns keep their value.
            const uint32_t token = mine[i] ? 0xffffffffu : 0u;
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
              for (int r = 0; r < 8; ++r)
                o.v[i][j][r] = updated(o.v[i][j][r], delta[j][2 * r] * scale, delta[j][2 * r + 1] * scale, token, inside, lo, hi, j, r);
          }
        }
      }
    }
  }
  if (kSwiglu || p.y_vec == 2) {
    // 16-byte aligned rows (always so with the SwiGLU output): the tile goes
    // through LDS (the idle x ring, rows of 512 bytes, 16-byte chunks
    // XOR-swizzled by row & 31) and leaves as whole rows.
    static_assert(kRows * 512 <= kRingBytes, "output staging fits the x ring");
    __syncthreads();  // every wave is done with the ring
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int row = 32 * i + c;
#pragma unroll
      for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int chunk = wave * 8 + 4 * j + q;
          *reinterpret_cast<uint2*>(xring + row * 512 + ((chunk ^ c) << 4) + h * 8) =
              make_uint2(o.v[i][j][2 * q], o.v[i][j][2 * q + 1]);
        }
    }
    __syncthreads();
    if constexpr (kSwiglu) {
      // Activation chunk q (8 columns) of a row: gate chunk q and up chunk
      // q + 16 of the staged row, bf16(bf16(silu(g)) * u) as lf_swiglu.
#pragma unroll 4
      for (int id = tid; id < kRows * 16; id += kThreads) {
        const int row = id >> 4;
        const int q = id & 15;
        const int m = m0 + row;
        const int n = nt * (kBN / 2) + q * 8;
        if (m < p.m && n < (p.n >> 1)) {
          const uint4 gv = *reinterpret_cast<const uint4*>(xring + row * 512 + ((q ^ (row & 31)) << 4));
          const uint4 uv = *reinterpret_cast<const uint4*>(xring + row * 512 + (((q + 16) ^ (row & 31)) << 4));
          const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w};
          const uint32_t uw[4] = {uv.x, uv.y, uv.z, uv.w};
          uint32_t o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = pack_bf16x2(silu_times(bf16_lo(gw[e]), bf16_lo(uw[e])),
                               silu_times(bf16_hi(gw[e]), bf16_hi(uw[e])));
          *reinterpret_cast<uint4*>(p.y + int64_t(m) * p.y_stride + n) = make_uint4(o[0], o[1], o[2], o[3]);
        }
      }
    } else {
#pragma unroll 8
      for (int id = tid; id < kRows * 32; id += kThreads) {
        const int row = id >> 5;
        const int q = id & 31;
        const int m = m0 + row;
        const int n = n0 + q * 8;
        if (m < p.m && n < p.n)
          *reinterpret_cast<uint4*>(p.y + int64_t(m) * p.y_stride + n) =
              *reinterpret_cast<const uint4*>(xring + row * 512 + ((q ^ (row & 31)) << 4));
      }
    }
  } else if constexpr (!kSwiglu) {
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int m = m0 + 32 * i + c;
      if (m >= p.m) continue;
#pragma unroll
      for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = wn0 + 32 * j + 8 * q + 4 * h;  // N % 64 == 0: n < N covers n + 3
          if (n >= p.n) continue;
          uint16_t* dst = p.y + int64_t(m) * p.y_stride + n;
          const uint32_t lo = o.v[i][j][2 * q];
          const uint32_t hi = o.v[i][j][2 * q + 1];
          if (p.y_vec) {
            *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
          } else {
            dst[0] = uint16_t(lo);
            dst[1] = uint16_t(lo >> 16);
            dst[2] = uint16_t(hi);
            dst[3] = uint16_t(hi >> 16);
          }
        }
    }
  }
  if constexpr (kLora) depart(p, tag);
  }
}

}  // namespace tile

}  // namespace

#ifdef LF_PREFILL_Z_KERNEL
int launch_z(const PrefillParams& p, hipStream_t stream) {
  hipLaunchKernelGGL(tile::z_kernel, dim3(p.mtiles * p.zparts * p.zrow_parts), dim3(tile::kZThreads), 0, stream, p);
  LF_HIP(hipGetLastError());
  return kOk;
}
#endif

template <int RI>
int launch_rows(const PrefillParams& p, int64_t blocks, bool lora, bool swiglu, hipStream_t stream) {
  const dim3 grid{unsigned(blocks)};
  if (swiglu) {
    if (lora) hipLaunchKernelGGL((tile::gemm_kernel<RI, true, true>), grid, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((tile::gemm_kernel<RI, false, true>), grid, dim3(kThreads), 0, stream, p);
  } else {
    if (lora) hipLaunchKernelGGL((tile::gemm_kernel<RI, true, false>), grid, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((tile::gemm_kernel<RI, false, false>), grid, dim3(kThreads), 0, stream, p);
  }
  LF_HIP(hipGetLastError());
  return kOk;
}

}  // namespace prefill
}  // namespace lf
