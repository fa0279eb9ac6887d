// Host side of the prefill GEMM (prefill_tile.h): workspace layout, the choice
// of the tile height and the launch.
#include <algorithm>
#include <cmath>

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
// the flag region; 0: none fits).
int zparts_in_slack(int64_t mtiles, int64_t tiles, int64_t cus) {
  const int64_t rem = tiles % cus;
  const int64_t slack = rem == 0 ? 0 : cus - rem;
  return int(std::min<int64_t>(std::min<int64_t>(kMaxZParts, kMaxFlags / mtiles), slack / mtiles));
}

// Tile heights that are built, in 32-token fragments, and the time of a round
// of such tiles per 4096 of K (us) at rounds that are 60 % full (a fuller chip
// runs at a lower clock: 14 % over the whole range). Below 4 fragments the decode
// of the tile's weights (the same for every height) bounds it instead of the MFMAs.
struct TileCost {
  int ri;
  double us;
};
constexpr TileCost kTileCosts[] = {{8, 75.0}, {6, 60.0}, {5, 57.0}, {4, 53.0}, {3, 52.0}, {2, 41.5}};

// How a tile of `tokens` tokens may be routed over a pool of adapters: slots
// among its tokens and among 32 of them, and z units (16 tokens of one slot, or
// 32: half a unit lost to each slot). The host does not know the routes, so a plan
// is priced for two of them: each slot's tokens together (prompts one after the
// other), and all slots in turn, the less likely the more tokens a slot has.
struct Routing {
  double tokens, slots, block, units, units32;
};
double units_of(double tokens, double slots, double size) { return std::max(slots, tokens / size + slots / 2.0); }
Routing together(double tokens, double m, double pool) {
  const double slots = std::min({pool, tokens, tokens * pool / m + 1.0});
  return {tokens, slots, 1.0 + std::min(slots - 1.0, 32.0 * pool / m), units_of(tokens, slots, 16.0), units_of(tokens, slots, 32.0)};
}
Routing in_turn(double tokens, double pool) {
  const double slots = pool * tokens / (pool + tokens);
  return {tokens, slots, pool * 32.0 / (pool + 32.0), units_of(tokens, slots, 16.0), units_of(tokens, slots, 32.0)};
}
double in_turn_weight(double m, double pool) { return std::min(0.4, 17.0 * pool / m); }
constexpr int kPoolUnknown = 16;  // adapters of a call that does not say

struct TilePlan {
  int ri;
  int64_t mtiles, tiles;
  int zparts;
  bool z_launch;  // the z producers run in a launch of their own
  double us;
};

// Time of a plan's LoRA call under a routing, us.
//  - A round's fixed part (start, routes, rounding and stores; without LoRA 5 +
//    1.2 ri, see tile_plan) and the expand beyond the first slots: per slot where
//    a tile rounds once for all, else per slot and 32-token block.
//  - Producers in the GEMM launch: a unit takes 2 us and, per 4096 of K, 3.7 us
//    for each 16 A rows and, in each 64-row pass, for each 16 tokens (four waves,
//    fragment loads); units of 32 tokens where those of 16 outnumber the producers.
//    Their consumers wait for what does not end within the first round's k-loop
//    (2048 x 11008 x 4096, three slices of rank 64: 33 producers in the slack of
//    192-token tiles 408 us, 168 in that of 256-token tiles 217 us); their loads
//    cost the first tiles about 2 %.
//  - In a launch of their own (through LDS, one 16-row pass at a time).
double lora_plan_us(const TilePlan& p, double loop, int64_t cus, int64_t k, int slices, int max_rank, const Routing& r) {
  const double k4 = double(k) / 4096.0;
  const double rounds = double((p.tiles + cus - 1) / cus);
  const int row_tiles = (slices * max_rank + 15) / 16;
  const int steps = (max_rank + 15) / 16;
  const double expand = p.ri <= kManyRows ? 0.9 * std::max(0.0, r.slots - kFewSlots) * (1.0 + 0.2 * (steps - 1))
                                          : 1.05 * p.ri * std::max(0.0, r.block - 1.0) * (1.0 + 0.1 * (steps - 1));
  const double gemm = rounds * (loop + 7.5 + 2.25 * p.ri + expand);
  if (!p.z_launch) {
    const bool pairs = r.units > p.zparts;
    const int x_tiles = pairs && r.tokens > 16.0 * r.units32 ? 2 : 1;
    const double each = 2.0 + 3.7 * k4 * ((row_tiles + 3) / 4 * x_tiles + row_tiles);
    // (Units of 32 are few: of the tiles' different numbers the larger ones count.)
    const double serial = pairs ? std::max(1.0, r.units32 / p.zparts + 0.6) : std::ceil(r.units / p.zparts);
    return 1.02 * gemm + std::max(0.0, serial * each - 0.9 * loop);
  }
  const double serial = std::ceil(r.units / p.zparts);  // units of one producer
  const int parts = z_row_parts(slices, max_rank);
  const double groups = double(p.mtiles * p.zparts * parts);
  const double busy = std::min<double>(r.units, p.zparts) * double(p.mtiles * parts) / double(cus) + 1.0;
  return gemm + 4.0 + 6.0 * std::ceil(groups / double(cus)) + busy * serial * double((row_tiles + parts - 1) / parts) * (3.0 + 3.0 * k4);
}

// The tile height, and with LoRA the place of the z producers, that take the
// least time. (Against the fastest of all heights, with the producers in the slack
// or in their own launch, all units of 16 tokens: 0.4 % slower on average over 5070 drawn calls of 512..4096
// tokens in prompts, 0.1 % over 2600 of 65..512 tokens in any routing, 28 % at most;
// the rule that took the slack wherever three producers a tile fit it 1.0 and 0.3 %,
// up to 87 %, and over a grid of ranks 8..64 and 1..3 slices up to 148 %.)
TilePlan tile_plan(int64_t m, int64_t n, int64_t k, int slices, int max_rank, bool lora, bool swiglu, int num_slots) {
  const int64_t cus = device_cus();
  const int64_t ntiles = ((swiglu ? n / 2 : n) + (swiglu ? kTileN / 2 : kTileN) - 1) / (swiglu ? kTileN / 2 : kTileN);
  const double pool = num_slots > 0 ? num_slots : kPoolUnknown;
  TilePlan best{};
  for (const TileCost& c : kTileCosts) {
    TilePlan p{c.ri};
    p.mtiles = (m + 32 * c.ri - 1) / (32 * c.ri);
    if (p.mtiles > kMaxFlags) continue;
    p.tiles = p.mtiles * ntiles;
    const double rounds = double((p.tiles + cus - 1) / cus);
    const double full = double(p.tiles) / (rounds * double(cus));
    const double loop = c.us * (1.0 + 0.14 * (full - 0.6)) * double(k) / 4096.0;
    if (!lora) {
      p.us = rounds * (loop + 5.0 + 1.2 * c.ri);
      if (best.ri == 0 || p.us < best.us) best = p;
      continue;
    }
    const double tokens = double(std::min<int64_t>(32 * c.ri, m));
    const Routing routes[2] = {together(tokens, double(m), pool), in_turn(tokens, pool)};
    const double turn = in_turn_weight(double(m), pool);
    const int in_launch = zparts_in_slack(p.mtiles, p.tiles, cus);
    for (const bool launch : {false, true}) {
      p.z_launch = launch;
      // (In their own launch: a producer per 16 tokens, and two for the units that slot changes add.)
      p.zparts = launch ? int(std::max<int64_t>(1, std::min<int64_t>(2 * c.ri + 2, kMaxFlags / p.mtiles))) : in_launch;
      if (p.zparts == 0) continue;
      p.us = (1.0 - turn) * lora_plan_us(p, loop, cus, k, slices, max_rank, routes[0]) +
             turn * lora_plan_us(p, loop, cus, k, slices, max_rank, routes[1]);
      if (best.ri == 0 || p.us < best.us) best = p;
    }
  }
  return best;
}

// Time of a prefill launch for the choice between it and the decode kernels. (A
// pool counts for at most 64 slots here: of more, few have a token.)
double prefill_us(int64_t m, int64_t n, int64_t k, const lf_lora* lora, bool swiglu) {
  return tile_plan(m, n, k, lora ? lora->num_slices : 1, lora ? lora->max_rank : 1, lora != nullptr, swiglu,
                   lora ? std::min(lora->num_slots, 64) : 0)
      .us;
}

void prefill_tiles(int64_t m, int64_t n, int64_t k, const lf_lora* lora, bool swiglu, lf_plan* plan) {
  const TilePlan p = tile_plan(m, n, k, lora ? lora->num_slices : 1, lora ? lora->max_rank : 1, lora != nullptr, swiglu,
                               lora ? lora->num_slots : 0);
  plan->tile_rows = 32 * p.ri;
  plan->z_parts = p.zparts;
  plan->z_launch = p.z_launch ? 1 : 0;
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
  const TilePlan plan = tile_plan(m, w->n, w->k, slices, lora ? lora->max_rank : 1, lora != nullptr, swiglu,
                                  lora ? lora->num_slots : 0);
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
