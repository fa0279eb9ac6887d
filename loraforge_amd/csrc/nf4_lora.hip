// C-ABI entry of the fused NF4 + multi-LoRA linear: argument validation and
// dispatch between the decode kernel (M <= 64 tokens, or 64-token chunks of a
// larger batch that the prefill tiles would not spread over the chip) and the
// prefill GEMM.
#include <algorithm>
#include <mutex>

#include "nf4_common.h"
#include "../../include/loraforge_amd.h"

namespace lf {
int64_t gemv_workspace_bytes(int64_t m, int64_t n, int64_t k, int slices, int max_rank);
int launch_nf4_gemv(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w, const uint16_t* bias,
                    const lf_lora* lora, uint16_t* y, int64_t y_stride, void* workspace, int64_t workspace_bytes,
                    bool exact, bool swiglu, bool withhold, void* stream, bool residual = false);
int64_t prefill_workspace_bytes(int64_t m, int64_t n, int64_t k, int slices, int max_rank);
int launch_nf4_lora_prefill(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w,
                            const uint16_t* bias, const lf_lora* lora, uint16_t* y, int64_t y_stride,
                            void* workspace, int64_t workspace_bytes, bool swiglu, bool withhold, void* stream);
int device_cus();
bool decode_wide_fits(int64_t m, int64_t n, int64_t k, const lf_lora* lora);
bool wide_takes_dq(const lf_nf4_weight* w);
bool gemv_takes_dq(int64_t m, const lf_nf4_weight* w, const lf_lora* lora, bool exact);
int rebuild_decode_scales(const lf_nf4_weight* w, void* workspace, int64_t workspace_bytes, void* stream,
                          const float** scales);
bool lora_apply_wide_fits(int64_t m, int64_t n, int64_t k, const lf_lora* lora);
int launch_lora_apply_wide(const uint16_t* x, int64_t m, int64_t x_stride, int64_t n, int64_t k, const lf_lora* lora,
                           uint16_t* y, int64_t y_stride, void* workspace, int64_t workspace_bytes, bool withhold,
                           void* stream);
int64_t apply_tiles_tokens(int64_t workspace_bytes, int slices);
int launch_lora_apply_tiles(const uint16_t* x, int64_t m, int64_t x_stride, int64_t n, int64_t k, const lf_lora* lora,
                            uint16_t* y, int64_t y_stride, void* workspace, void* stream);
int launch_decode_wide(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w, const uint16_t* bias,
                       const lf_lora* lora, uint16_t* y, int64_t y_stride, void* workspace, int64_t workspace_bytes,
                       bool exact, bool swiglu, bool withhold, void* stream);
constexpr int64_t kDecodeMaxTokens = 64;

// Held while a call's launches go out, so that they stay together on the stream:
// the launches of one call hand z rows, rebuilt scales and the call's tag to each
// other through the workspace, and threads that share a stream share its cached
// workspace.
std::mutex& launch_lock(const void* workspace) {
  static std::mutex locks[64];
  return locks[(reinterpret_cast<uintptr_t>(workspace) >> 12) % 64];
}

double prefill_us(int64_t m, int64_t n, int64_t k, const lf_lora* lora, bool swiglu);
void prefill_tiles(int64_t m, int64_t n, int64_t k, const lf_lora* lora, bool swiglu, lf_plan* plan);

double decode_rounds(int64_t m, int64_t n) {
  const int64_t cus = device_cus();
  const int64_t groups = ((n / 32 + 7) / 8) * 8 * ((m + 31) / 32);
  return double((groups + cus - 1) / cus);
}

// What the decode kernels take, us. A call of the wide one: a start and rounds of
// 256 workgroups (32 rows x 32 tokens over the whole K), each with its own start, x
// and weight reads and, with LoRA, shrink, z wait and expand. (24576 x 64, 4096
// tokens: 384 rounds in 911 us; 8192 x 2048, 1024 tokens, three slices of rank 64: 32
// rounds in 592 us; 14 % rms over 2818 calls with adapters, 7 % over 191 without.)
double wide_us(int64_t m, int64_t n, int64_t k, const lf_lora* lora) {
  const double k4 = double(k) / 4096.0;
  if (!lora) return 2.0 + decode_rounds(m, n) * (2.3 + 5.3 * k4);
  const double rows = double(lora->num_slices) * lora->max_rank;
  return 6.3 + decode_rounds(m, n) * (3.1 + 0.062 * rows + (4.8 + 0.024 * rows) * k4);
}
// A weight's bytes (packed + fp32 scales) at about 0.8 TB/s, and about 6 us with
// LoRA (4096 x 4096: 11.9 us base only, 18.0 us with 32 rank-16 adapters).
double stream_us(int64_t n, int64_t k, const lf_lora* lora) {
  return (lora ? 6.0 : 0.0) + double(n) * double(k) * (0.5 + 4.0 / 64.0) / 0.8e6;
}
// A launch per 64-token chunk, of the wide kernel or the narrow one (14 % rms over
// 532 calls with adapters).
double chunks_us(int64_t m, int64_t n, int64_t k, const lf_lora* lora) {
  const double chunks = double((m + kDecodeMaxTokens - 1) / kDecodeMaxTokens);
  if (decode_wide_fits(kDecodeMaxTokens, n, k, lora)) return chunks * wide_us(kDecodeMaxTokens, n, k, lora);
  if (!lora) return chunks * stream_us(n, k, lora);
  const double rows = double(lora->num_slices) * lora->max_rank;
  return chunks * (5.2 + 0.114 * rows + (5.9 + 0.029 * rows) * double(k) / 4096.0 + (6.5 + 0.04 * rows) * double(n) / 4096.0);
}

// Whether a default call of M > 64 tokens may run on the decode kernels, which
// contract bf16(code) (relative error about 0.0031 against 0.0024 with the prefill
// GEMM's exact weights). The line is where these kernels undercut tiles of 256 x
// 192 at 85 us a round per 4096 of K, by 4 us a round of their own or by the weight
// bytes: it stays there however fast either becomes, so that a call keeps its
// precision.
bool may_decode(int64_t m, int64_t n, int64_t k, const lf_lora* lora) {
  const int64_t tiles = ((m + 255) / 256) * ((n + 191) / 192);
  const int64_t cus = device_cus();
  const double k4 = double(k) / 4096.0;
  const double tiles_us = double((tiles + cus - 1) / cus) * 85.0 * k4;
  if (decode_wide_fits(m, n, k, lora) && decode_rounds(m, n) * 4.0 * k4 < tiles_us) return true;
  const int64_t chunks = (m + kDecodeMaxTokens - 1) / kDecodeMaxTokens;
  return double(chunks) * stream_us(n, k, lora) < tiles_us + (lora ? 20.0 : 0.0);
}

// The kernel of a call. Above 8 tokens (2 at N >= 8192, 16 at K > 8192): the wide
// decode kernel (one launch, base linear with or without LoRA and the SwiGLU
// output) if the shape is in its range; above 64 tokens the fastest of it, the
// prefill GEMM and decode launches over 64-token chunks (each streams W again but
// uses every CU, where few tiles leave most of the chip idle), unless a flag names
// one. (256 tokens x 4096 x 4096 with 128 ragged adapters: wide 61 us, prefill 115
// us; 256 x 11008: 98 / 67 us; 4096 x 24576 x 64: 911 / 62 us.) Against the faster
// of decode and prefill over 650 shapes and routings at K >= 1024 the prices lose
// 0.3 %, over 90 drawn calls of 65..512 tokens with up to 128 adapters 1.8 %.
int kernel_of(int64_t m, int64_t n, int64_t k, const lf_lora* lora, int32_t flags) {
  const bool wide = decode_wide_fits(m, n, k, lora) && !(flags & LF_PLAN_PREFILL);
  if (m <= kDecodeMaxTokens) return wide ? LF_KERNEL_DECODE_WIDE : LF_KERNEL_DECODE;
  if (flags & LF_PLAN_DECODE_CHUNKS) return wide ? LF_KERNEL_DECODE_WIDE : LF_KERNEL_DECODE_CHUNKS;
  if ((flags & LF_PLAN_PREFILL) || !may_decode(m, n, k, lora)) return LF_KERNEL_PREFILL;
  const double prefill = prefill_us(m, n, k, lora, (flags & LF_SWIGLU_OUTPUT) != 0);
  if (wide && wide_us(m, n, k, lora) < prefill) return LF_KERNEL_DECODE_WIDE;
  return chunks_us(m, n, k, lora) < prefill ? LF_KERNEL_DECODE_CHUNKS : LF_KERNEL_PREFILL;
}
// Whether lora_apply's two launches over all tokens are cheaper than a launch
// of the decode kernel's residual form per 64 tokens. The former's time grows
// with the distinct adapters of 64 tokens: 500 tokens x 5120 x 4096 over 4
// adapters 24.6 us against 142 us, but 300 x 1024 x 1024 over 32 110 against 42
// and 300 x 4096 x 4096 over 128 210 against 82 (above 16 adapters, or a pool of
// unknown size, a launch per 64 tokens), which takes 8 us and 8 us more per
// 4096 x 4096. A launch whose blocks run in one round (N to 4096) is faster
// than that, and both sides are priced closer there (to 10 % on 256 calls of
// 65..1000 tokens), the adapters of 64 tokens as the mean of those of tokens in
// runs and in turn: 192 x 4096 x 4096 over 8 adapters of rank 16 21.5 us in
// launches against 19.2 in runs and 32.2 in turn, 128 tokens over 4 14.6 us
// against 17.9 and 20.2; from 256 over 8 (28.5 against 19.6 and 33.9) or at rank
// 64 (39.9 against 23.6 and 46.0) the two launches.
bool apply_tiles_cheaper(int64_t m, int64_t n, int64_t k, const lf_lora* lora) {
  const int slots = lora->num_slots;
  if (slots < 1 || slots > 16) return false;
  const double k4 = double(k) / 4096.0;
  const double size = k4 * double(n) / 4096.0;
  const double tiles_us = (14.0 + 4.2 * slots) * std::max(1.0, size);
  const double launches_us = double((m + kDecodeMaxTokens - 1) / kDecodeMaxTokens) * (8.0 + 8.0 * size);
  if (tiles_us >= launches_us) return false;
  if (n % 256 != 0 || n > 4096) return true;
  const double rows = double(lora->num_slices) * lora->max_rank;
  const double split = std::max(1.0, double(n) / 1024.0);  // workgroups that share a token's rows of A
  const double launch_us = 5.5 + rows * (0.11 + 0.02 * k4 * (4.0 - split));
  const int64_t rest = m % kDecodeMaxTokens;  // (to 32 tokens the narrow kernel)
  const double live = 1.0 + (slots - 1) * (0.5 + 0.5 * std::min(1.0, double(kDecodeMaxTokens) / double(m)));
  return 9.5 + k4 + (2.1 + 0.2 * k4) * live + 0.035 * rows * (1.0 + 0.25 * live) <
         double(m / kDecodeMaxTokens) * launch_us + (rest > 32 ? launch_us : rest > 0 ? 8.8 : 0.0);
}

// One decode launch of up to 64 tokens: the wide kernel for the batches and
// shapes it takes (above 8 tokens, above 2 at N >= 8192, above 16 at
// K > 8192), else the narrow one (the kernel a direct call of these rows
// would use, so each chunk of the chunked plan equals that call).
int launch_decode(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w, const uint16_t* bias,
                  const lf_lora* lora, uint16_t* y, int64_t y_stride, void* workspace, int64_t workspace_bytes,
                  bool exact, bool swiglu, bool withhold, void* stream) {
  if (decode_wide_fits(m, w->n, w->k, lora))
    return launch_decode_wide(x, m, x_stride, w, bias, lora, y, y_stride, workspace, workspace_bytes, exact, swiglu,
                              withhold, stream);
  return launch_nf4_gemv(x, m, x_stride, w, bias, lora, y, y_stride, workspace, workspace_bytes, exact, swiglu,
                         withhold, stream);
}
}  // namespace lf

extern "C" int64_t lf_nf4_lora_workspace_size(int64_t m, int64_t n, int64_t k, int32_t num_slices,
                                              int32_t max_rank) {
  if (m < 0 || n <= 0 || k <= 0 || num_slices < 1 || max_rank < 1) return -1;
  if (m <= lf::kDecodeMaxTokens) return lf::gemv_workspace_bytes(m, n, k, num_slices, max_rank);
  return lf::prefill_workspace_bytes(m, n, k, num_slices, max_rank);
}

extern "C" int lf_nf4_lora_linear(const uint16_t* x, int64_t m, int64_t x_stride, const lf_nf4_weight* w,
                                  const uint16_t* bias, const lf_lora* lora, uint16_t* y, int64_t y_stride,
                                  void* workspace, int64_t workspace_bytes, int32_t flags, void* stream) {
  LF_REQUIRE(w != nullptr, "weight descriptor required");
  LF_REQUIRE((flags & ~(LF_EXACT_WEIGHTS | LF_SWIGLU_OUTPUT | LF_PLAN_DECODE_CHUNKS | LF_PLAN_PREFILL |
                        LF_TEST_WITHHOLD_PARTIALS)) == 0,
             "unknown flags");
  LF_REQUIRE((flags & (LF_PLAN_DECODE_CHUNKS | LF_PLAN_PREFILL)) != (LF_PLAN_DECODE_CHUNKS | LF_PLAN_PREFILL),
             "LF_PLAN_DECODE_CHUNKS and LF_PLAN_PREFILL exclude each other");
  const bool withhold = (flags & LF_TEST_WITHHOLD_PARTIALS) != 0;
  const bool swiglu = (flags & LF_SWIGLU_OUTPUT) != 0;
  LF_REQUIRE(m >= 0 && m < (int64_t(1) << 31), "token count out of range");
  const int64_t n = w->n, k = w->k;
  LF_REQUIRE(n > 0 && k > 0 && n % 64 == 0 && k % 64 == 0, "weight shape must contain two positive multiples of 64");
  LF_REQUIRE(n < (int64_t(1) << 28) && k < (int64_t(1) << 28), "weight shape too large");
  if (m == 0) return lf::kOk;
  LF_REQUIRE(x && y && w->qweight && w->code, "null pointer argument");
  LF_REQUIRE(w->scales || (w->absmax_q && w->absmax2 && w->code2 && w->offset && w->dq_block > 0),
             "scales or a complete double-quant state required");
  LF_REQUIRE(lf::aligned16(x) && x_stride >= k && x_stride % 8 == 0, "x must be 16-byte aligned with row stride %% 8 == 0");
  LF_REQUIRE(lf::aligned16(w->qweight), "packed weight must be 16-byte aligned");
  LF_REQUIRE(y_stride >= (swiglu ? n / 2 : n), "output row stride must cover the output width");
  LF_REQUIRE(!swiglu || n % 64 == 0, "SwiGLU output needs N a multiple of 64");
  LF_REQUIRE(!swiglu || !lora || lora->num_slices == 2, "SwiGLU output with LoRA needs the two gate/up slices");
  if (lora) {
    LF_REQUIRE(lora->num_slices >= 1 && lora->num_slices <= 3, "num_slices must be in 1..3");
    LF_REQUIRE(lora->max_rank >= 1 && lora->max_rank <= 64, "max_rank must be in 1..64");
    LF_REQUIRE(lora->a_store && lora->a_offsets && lora->b_store && lora->b_offsets && lora->b_strides &&
                   lora->ranks && lora->scales && lora->token_slots && lora->slice_offsets,
               "incomplete LoRA descriptor");
    LF_REQUIRE(lf::aligned16(lora->a_store) && lf::aligned16(lora->b_store), "A/B stores must be 16-byte aligned");
  }
  const bool exact = (flags & LF_EXACT_WEIGHTS) != 0;
  std::lock_guard<std::mutex> together(lf::launch_lock(workspace));
  const int kernel = lf::kernel_of(m, n, k, lora, flags);
  if (kernel == LF_KERNEL_DECODE_WIDE)
    return lf::launch_decode_wide(x, m, x_stride, w, bias, lora, y, y_stride, workspace, workspace_bytes, exact,
                                  swiglu, withhold, stream);
  if (kernel == LF_KERNEL_DECODE)
    return lf::launch_decode(x, m, x_stride, w, bias, lora, y, y_stride, workspace, workspace_bytes, exact, swiglu,
                             withhold, stream);
  if (kernel == LF_KERNEL_PREFILL)
    return lf::launch_nf4_lora_prefill(x, m, x_stride, w, bias, lora, y, y_stride, workspace, workspace_bytes,
                                       swiglu, withhold, stream);
  // 64-token chunks in token order on the caller's stream; each is one decode
  // launch over its rows of x, y and the token routes. A nested state that a
  // chunk's kernel does not read itself is rebuilt to fp32 scales once, ahead
  // of the chunks.
  lf_nf4_weight wc = *w;
  if (!w->scales) {
    const int64_t last = m - (m - 1) / lf::kDecodeMaxTokens * lf::kDecodeMaxTokens;
    auto reads = [&](int64_t mc) {
      return lf::decode_wide_fits(mc, n, k, lora) ? lf::wide_takes_dq(w) : lf::gemv_takes_dq(mc, w, lora, exact);
    };
    if (!reads(lf::kDecodeMaxTokens) || !reads(last)) {
      const int rc = lf::rebuild_decode_scales(w, workspace, workspace_bytes, stream, &wc.scales);
      if (rc != lf::kOk) return rc;
    }
  }
  w = &wc;
  for (int64_t t0 = 0; t0 < m; t0 += lf::kDecodeMaxTokens) {
    const int64_t mc = std::min<int64_t>(lf::kDecodeMaxTokens, m - t0);
    lf_lora part{};
    if (lora) {
      part = *lora;
      part.token_slots = lora->token_slots + t0;
    }
    const int rc = lf::launch_decode(x + t0 * x_stride, mc, x_stride, w, bias, lora ? &part : nullptr,
                                     y + t0 * y_stride, y_stride, workspace, workspace_bytes, exact, swiglu, withhold,
                                     stream);
    if (rc != lf::kOk) return rc;
  }
  return lf::kOk;
}

extern "C" int lf_nf4_lora_plan(int64_t m, int64_t n, int64_t k, int32_t num_slices, int32_t max_rank, int32_t num_slots,
                                int32_t flags, lf_plan* plan) {
  LF_REQUIRE(plan != nullptr, "null pointer argument");
  LF_REQUIRE(m > 0 && m < (int64_t(1) << 31), "token count out of range");
  LF_REQUIRE(n > 0 && k > 0 && n % 64 == 0 && k % 64 == 0, "weight shape must contain two positive multiples of 64");
  LF_REQUIRE(n < (int64_t(1) << 28) && k < (int64_t(1) << 28), "weight shape too large");
  LF_REQUIRE(num_slices >= 0 && num_slices <= 3, "num_slices must be in 1..3, or 0 without adapters");
  LF_REQUIRE(num_slices == 0 || (max_rank >= 1 && max_rank <= 64), "max_rank must be in 1..64");
  lf_lora lora{};
  lora.num_slices = num_slices;
  lora.max_rank = max_rank;
  lora.num_slots = num_slots;
  const lf_lora* adapters = num_slices ? &lora : nullptr;
  *plan = lf_plan{};
  plan->kernel = lf::kernel_of(m, n, k, adapters, flags);
  if (plan->kernel == LF_KERNEL_PREFILL) lf::prefill_tiles(m, n, k, adapters, (flags & LF_SWIGLU_OUTPUT) != 0, plan);
  return lf::kOk;
}

extern "C" int lf_lora_apply_plan(int64_t m, int64_t n, int64_t k, int32_t num_slices, int32_t max_rank, int32_t num_slots,
                                  int32_t* two_launches) {
  LF_REQUIRE(two_launches != nullptr, "null pointer argument");
  LF_REQUIRE(m > 0 && m < (int64_t(1) << 31), "token count out of range");
  LF_REQUIRE(n > 0 && k > 0 && n % 64 == 0 && k % 64 == 0, "N and K must be positive multiples of 64");
  LF_REQUIRE(n < (int64_t(1) << 28) && k < (int64_t(1) << 28), "shape too large");
  LF_REQUIRE(num_slices >= 1 && num_slices <= 3, "num_slices must be in 1..3");
  LF_REQUIRE(max_rank >= 1 && max_rank <= 64, "max_rank must be in 1..64");
  lf_lora lora{};
  lora.num_slices = num_slices;
  lora.max_rank = max_rank;
  lora.num_slots = num_slots;
  *two_launches = m > lf::kDecodeMaxTokens && lf::apply_tiles_cheaper(m, n, k, &lora);
  return lf::kOk;
}

extern "C" int lf_nf4_lora_status(const void* workspace, void* stream, int32_t* status) {
  LF_REQUIRE(workspace && status, "null pointer argument");
  auto s = static_cast<hipStream_t>(stream);
  LF_HIP(hipMemcpyAsync(status, static_cast<const char*>(workspace) + 8, 4, hipMemcpyDeviceToHost, s));
  LF_HIP(hipStreamSynchronize(s));
  return lf::kOk;
}

extern "C" int lf_lora_apply(const uint16_t* x, int64_t m, int64_t x_stride, int64_t n, int64_t k, const lf_lora* lora,
                             uint16_t* y, int64_t y_stride, void* workspace, int64_t workspace_bytes, int32_t flags,
                             void* stream) {
  LF_REQUIRE((flags & ~LF_TEST_WITHHOLD_PARTIALS) == 0, "unknown flags");
  LF_REQUIRE(m >= 0 && m < (int64_t(1) << 31), "token count out of range");
  LF_REQUIRE(n > 0 && k > 0 && n % 64 == 0 && k % 64 == 0, "N and K must be positive multiples of 64");
  LF_REQUIRE(n < (int64_t(1) << 28) && k < (int64_t(1) << 28), "shape too large");
  if (m == 0) return lf::kOk;
  LF_REQUIRE(x && y && lora, "null pointer argument");
  LF_REQUIRE(lf::aligned16(x) && x_stride >= k && x_stride % 8 == 0, "x must be 16-byte aligned with row stride %% 8 == 0");
  LF_REQUIRE(y_stride >= n, "output row stride must cover the output width");
  LF_REQUIRE(lora->num_slices >= 1 && lora->num_slices <= 3, "num_slices must be in 1..3");
  LF_REQUIRE(lora->max_rank >= 1 && lora->max_rank <= 64, "max_rank must be in 1..64");
  LF_REQUIRE(lora->a_store && lora->a_offsets && lora->b_store && lora->b_offsets && lora->b_strides && lora->ranks &&
                 lora->scales && lora->token_slots && lora->slice_offsets,
             "incomplete LoRA descriptor");
  LF_REQUIRE(lf::aligned16(lora->a_store) && lf::aligned16(lora->b_store), "A/B stores must be 16-byte aligned");
  lf_nf4_weight shape{};
  shape.n = n;
  shape.k = k;
  const bool withhold = (flags & LF_TEST_WITHHOLD_PARTIALS) != 0;
  std::lock_guard<std::mutex> together(lf::launch_lock(workspace));
  // Above 64 tokens, where it is cheaper: shrink and expand as two launches
  // over all tokens whose z rows the workspace holds. A workspace that holds
  // fewer than 128 tokens' rows takes the launches per 64 tokens below.
  const int64_t fit = m > lf::kDecodeMaxTokens && !withhold && workspace && lf::aligned16(workspace) &&
                              lf::apply_tiles_cheaper(m, n, k, lora)
                          ? lf::apply_tiles_tokens(workspace_bytes, lora->num_slices)
                          : 0;
  if (fit >= 128) {
    const int64_t step = std::min<int64_t>(fit / 256 > 0 ? fit / 256 * 256 : fit, int64_t(1) << 20);
    for (int64_t t0 = 0; t0 < m; t0 += step) {
      lf_lora part = *lora;
      part.token_slots = lora->token_slots + t0;
      const int rc = lf::launch_lora_apply_tiles(x + t0 * x_stride, std::min<int64_t>(step, m - t0), x_stride, n, k, &part,
                                                 y + t0 * y_stride, y_stride, workspace, stream);
      if (rc != lf::kOk) return rc;
    }
    return lf::kOk;
  }
  // One launch per 64 tokens, in token order.
  for (int64_t t0 = 0; t0 < m; t0 += lf::kDecodeMaxTokens) {
    const int64_t mc = std::min<int64_t>(lf::kDecodeMaxTokens, m - t0);
    lf_lora part = *lora;
    part.token_slots = lora->token_slots + t0;
    // 33..64 tokens: the wide kernel's residual form where it fits.
    const int rc = lf::lora_apply_wide_fits(mc, n, k, &part)
                       ? lf::launch_lora_apply_wide(x + t0 * x_stride, mc, x_stride, n, k, &part, y + t0 * y_stride,
                                                    y_stride, workspace, workspace_bytes, withhold, stream)
                       : lf::launch_nf4_gemv(x + t0 * x_stride, mc, x_stride, &shape, nullptr, &part, y + t0 * y_stride,
                                             y_stride, workspace, workspace_bytes, false, false, withhold, stream, true);
    if (rc != lf::kOk) return rc;
  }
  return lf::kOk;
}
