// Host side of the prefill GEMM (prefill_tile.h): workspace layout, the choice
// of the tile height and the launch.
#include <algorithm>

#include "prefill_params.h"
#include "nf4_common.h"
#include "../../include/loraforge_amd.h"

namespace lf {
using namespace prefill;

namespace {
int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }
}  // namespace

int device_cus();

// Workspace: the control header (call epoch), the z flags (one per producer,
// zparts per 256-token tile) at a fixed place (so a flag word only ever holds
// tags, whatever the shapes of earlier calls on the workspace), the z rows
// (m x slices x 64 bf16), then room for the fp32 block scales of a
// double-quant weight.
constexpr int64_t kMaxFlags = kFlagRegion / 4;
constexpr int kMaxZParts = 64;

// z producers per M-tile inside the GEMM launch: they run first and hold a CU
// each (one workgroup per CU), which costs nothing where the tiles' last round
// leaves CUs idle anyway. So they fill that slack (at most 64 per tile, within
// the flag region). Below 3 a tile (a unit of 16 tokens takes about a tenth of
// the tile's own time) its consumers would wait for them: 0, a launch of
// their own.
int zparts_in_slack(int64_t mtiles, int64_t tiles, int64_t cus) {
  const int64_t rem = tiles % cus;
  const int64_t slack = rem == 0 ? 0 : cus - rem;
  const int64_t parts = std::min<int64_t>(std::min<int64_t>(kMaxZParts, kMaxFlags / mtiles), slack / mtiles);
  return parts < 3 ? 0 : int(parts);
}

// Tile heights that are built, in 32-token fragments, and the time of a round
// of such tiles per 4096 of K (us; between a full chip, which runs at a lower
// clock, and a few tiles). Below 4 fragments the decode of the tile's weights
// (the same for every height) bounds it instead of the MFMAs.
struct TileCost {
  int ri;
  double us;
};
constexpr TileCost kTileCosts[] = {{8, 100.0}, {6, 82.0}, {5, 72.0}, {4, 64.0}, {3, 58.0}, {2, 52.0}};
// What a round takes beside its k-loop: start, rounding and stores, and with
// LoRA routes, z and B reads and the expand (1024 x 4096 x 1024, rank 16, heights
// 8 .. 3: 47 / 37 / 35 / 32 / 29 us, of which the k-loop is 25 .. 14).
double round_us(int ri, bool lora) { return lora ? 9.0 + 1.2 * ri : 4.0 + 0.6 * ri; }
// A round of z producers of one unit each, one workgroup per CU, in a launch of
// its own. (More than the kernel's own time, 9-10 us a round at K = 4096: at 5 + rounds x
// (2.5 + 3 K / 4096) the rule takes the launch in sixteen of four hundred drawn shapes more,
// and all of them get slower, 1292 x 13824 x 6144 245 -> 266 us.)
double z_round_us(int64_t k) { return 12.0 + 6.0 * double(k) / 4096.0; }

struct TilePlan {
  int ri;
  int64_t mtiles, tiles;
  int zparts;
  bool z_launch;  // the z producers run in a launch of their own
  double us;
};

// The tile height whose rounds of one tile per CU take the least time: 2048 x
// 11008 x 4096 (43 column tiles) runs in two rounds of 192-token tiles (186 us)
// instead of two of 256 (208 us), 300 tokens x 24576 (SwiGLU) in one round of
// 160-token tiles (77 us against 98 us), 4096 x 4096 x 1024 with LoRA in two
// of 160 tokens (64 us) instead of one of 256, whose z would be a launch of
// its own.
TilePlan tile_plan(int64_t m, int64_t n, int64_t k, int slices, int max_rank, bool lora, bool swiglu) {
  const int64_t cus = device_cus();
  const int64_t ntiles = ((swiglu ? n / 2 : n) + (swiglu ? kTileN / 2 : kTileN) - 1) / (swiglu ? kTileN / 2 : kTileN);
  TilePlan best{};
  for (const TileCost& c : kTileCosts) {
    TilePlan p{c.ri};
    p.mtiles = (m + 32 * c.ri - 1) / (32 * c.ri);
    if (p.mtiles > kMaxFlags) continue;
    p.tiles = p.mtiles * ntiles;
    p.us = double((p.tiles + cus - 1) / cus) * (c.us * double(k) / 4096.0 + round_us(c.ri, lora));
    if (lora) {
      p.zparts = zparts_in_slack(p.mtiles, p.tiles, cus);
      p.z_launch = p.zparts == 0;
      if (p.z_launch) {
        // A producer per 16 tokens, and two for the units that slot changes add.
        p.zparts = int(std::max<int64_t>(1, std::min<int64_t>(2 * c.ri + 2, kMaxFlags / p.mtiles)));
        const int64_t groups = p.mtiles * p.zparts * z_row_parts(slices, max_rank);
        p.us += z_round_us(k) * double((groups + cus - 1) / cus);
      }
    }
    if (best.ri == 0 || p.us < best.us) best = p;
  }
  return best;
}

double prefill_us(int64_t m, int64_t n, int64_t k, const lf_lora* lora, bool swiglu) {
  return tile_plan(m, n, k, lora ? lora->num_slices : 1, lora ? lora->max_rank : 1, lora != nullptr, swiglu).us;
}

int64_t prefill_workspace_bytes(int64_t m, int64_t n, int64_t k, int slices, int) {
  return kWorkspaceHeader + kFlagRegion + align256(m * slices * kZSlice * 2) + align256(n * (k / kNf4Block) * 4);
}

int launch_nf4_lora_prefill(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w,
                            const uint16_t* bias, const lf_lora* lora, uint16_t* y, int64_t y_stride,
                            void* workspace, int64_t workspace_bytes, bool swiglu, bool withhold, void* stream) {
  const int slices = lora ? lora->num_slices : 1;
  const bool dq = w->scales == nullptr;
  const int64_t need = prefill_workspace_bytes(m, w->n, w->k, slices, lora ? lora->max_rank : 1);
  LF_REQUIRE(!(lora || dq) || (workspace && workspace_bytes >= need && aligned16(workspace)),
             "workspace too small: need %lld bytes", (long long)need);
  LF_REQUIRE((m - 1) * x_stride * 2 + w->k * 2 < (int64_t(1) << 32), "x spans 4 GiB or more");
  LF_REQUIRE((m + kBM - 1) / kBM <= kMaxFlags, "prefill handles at most %lld tokens per call",
             (long long)(kMaxFlags * kBM));
  auto s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const float* scales = w->scales;
  if (dq) {
    // The GEMM streams fp32 block scales: rebuild them from the nested state
    // (the same reconstruction as the dequantisation kernel) after the z rows.
    const int64_t nblocks = w->n * (w->k / kNf4Block);
    float* rebuilt =
        reinterpret_cast<float*>(ws + kWorkspaceHeader + kFlagRegion + align256(m * slices * kZSlice * 2));
    const int rc = lf_nf4_prepare_scales_dq(w->absmax_q, w->absmax2, w->code2, w->offset, w->dq_block, rebuilt,
                                            nblocks, stream);
    if (rc != kOk) return rc;
    scales = rebuilt;
  }
  PrefillParams p{};
  p.x = x;
  p.x_stride = x_stride;
  p.m = int(m);
  p.q = w->qweight;
  p.src = ScaleSource{scales, nullptr, nullptr, nullptr, nullptr, 1};
  p.code = w->code;
  p.n = int(w->n);
  p.k = int(w->k);
  p.bias = bias;
  p.y = y;
  p.y_stride = y_stride;
  p.y_vec = (y_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0) ? 2
            : (y_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7u) == 0)  ? 1
                                                                                 : 0;
  p.slices = slices;
  if (lora) {
    p.a_store = lora->a_store;
    p.a_offsets = lora->a_offsets;
    p.b_store = lora->b_store;
    p.b_offsets = lora->b_offsets;
    p.b_strides = lora->b_strides;
    p.ranks = lora->ranks;
    p.lscales = lora->scales;
    p.token_slots = lora->token_slots;
    p.slice_offsets = lora->slice_offsets;
    LF_REQUIRE(lora->num_slots >= 0, "num_slots must not be negative");
    p.num_slots = lora->num_slots;
    p.zflags = reinterpret_cast<uint32_t*>(ws + kWorkspaceHeader);  // after the decode header
    p.zpad = reinterpret_cast<uint16_t*>(ws + kWorkspaceHeader + kFlagRegion);
    p.ce = call_epoch_of(ws);
    p.status = reinterpret_cast<int*>(ws + kStatusOffset);
  }
  p.withhold = withhold ? 1 : 0;
  p.spin_limit = withhold ? 64 : (1 << 20);
  // SwiGLU output: each tile takes kBN / 2 activation columns (their gate and
  // up rows) and stores 16-byte chunks of them.
  LF_REQUIRE(!swiglu || p.y_vec == 2, "prefill SwiGLU output needs y 16-byte aligned with row stride %% 8 == 0");
  const TilePlan plan = tile_plan(m, w->n, w->k, slices, lora ? lora->max_rank : 1, lora != nullptr, swiglu);
  p.tile_rows = 32 * plan.ri;
  p.mtiles = int(plan.mtiles);
  p.zparts = plan.zparts;
  p.zrow_parts = z_row_parts(slices, lora ? lora->max_rank : 1);
  // LoRA launches put the z producers ahead of the GEMM tiles.
  p.zblocks = lora && !plan.z_launch ? p.mtiles * p.zparts : 0;
  const int64_t blocks = plan.tiles + p.zblocks;
  LF_REQUIRE(blocks < (int64_t(1) << 31), "too many tiles");
  if (plan.z_launch) {
    const int rc = launch_z(p, s);
    if (rc != kOk) return rc;
  }
  switch (plan.ri) {
    case 2: return launch_rows<2>(p, blocks, lora, swiglu, s);
    case 3: return launch_rows<3>(p, blocks, lora, swiglu, s);
    case 4: return launch_rows<4>(p, blocks, lora, swiglu, s);
    case 5: return launch_rows<5>(p, blocks, lora, swiglu, s);
    case 6: return launch_rows<6>(p, blocks, lora, swiglu, s);
    default: return launch_rows<8>(p, blocks, lora, swiglu, s);
  }
}

}  // namespace lf
