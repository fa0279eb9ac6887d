// Standalone NF4 -> bf16 dequantisation (reference: ops/nf4.py:7-38 and
// ops/_nf4_kernels.py:44-61, the byte-pair kernel) and the double-quant scale
// reconstruction of prepare_scales (ops/nf4.py:144-147).
//
// HBM-bound: per 64-element block it reads 32 packed bytes + 4 scale bytes
// and writes 128 bytes. Each lane decodes one packed dword (8 elements) per
// step and stores 16 bytes, so every load (256 B/wave) and store (1 KiB/wave)
// instruction is fully coalesced. How it stores goes by the output's size,
// so that the product that reads the weight next gains too (of each pair: the
// call, and the call with the product of 16 tokens behind it, over weights in
// turn whose packed bytes come from HBM):
//  - to 96 MiB written through the L2 (`sc1`): the output stays in the
//    memory-side cache, and no write-back waits for the kernel's end.
//    2048 x 2048 3.5 and 13.6 us (plain stores 4.1 and 14.2, non-temporal 3.5
//    and 16.4), 8192 x 1024 6.2 and 16.8 (6.4 and 17.9, 6.1 and 18.5), 4096 x 4096
//    10.8 and 33.0 (11.3 and 30.4, 11.1 and 35.1), 11008 x 4096 24.4 and 45.0
//    (25.1 and 45.3, 26.0 and 53.9).
//  - beyond, where outputs in turn drive each other out of that cache of
//    256 MiB, non-temporal: 16384 x 4096 of one packed weight into three outputs
//    25.4 us against 37.8 (11008 x 4096 17.7 against 18.9), 24576 x 4096 nested
//    38 against 63. Its reader pays for that (24576 x 4096 54 and 97 us against
//    50 and 84 written through) up to 256 MiB and gains beyond (32832 x 4096 with
//    256 tokens 150 against 166).
// Two independent steps per lane (one: 38.4 us, four: 37.7 us at 24576 x 4096
// with fp32 scales); four for a nested state of at least 32 M elements (39.6 us
// against 44.7 us: fewer workgroups stage the 256-entry code2), two below
// (4096 x 4096 7.5 us against 7.7 us). Packed bytes at an address that is not
// 4-byte aligned, or an output that is not 16-byte aligned (a contiguous view at
// an odd offset, which the reference accepts), take the same kernel with byte
// loads and 2-byte stores.
#include <chrono>
#include <mutex>

#include "nf4_common.h"
#include "verdict_words.h"
#include "../../include/loraforge_amd.h"

namespace lf {
namespace {

constexpr int kThreads = 256;
constexpr int64_t kLargeNested = int64_t(32) << 20;  // elements: four steps per lane
constexpr int64_t kThroughMost = int64_t(48) << 20;  // elements (96 MiB): stores written through

// Packed dword w of the weight (bytes 4w..4w+3, little endian).
template <bool kAligned>
__device__ __forceinline__ uint32_t load_packed(const uint8_t* __restrict__ packed, int64_t w) {
  if constexpr (kAligned) {
    return reinterpret_cast<const uint32_t*>(packed)[w];
  } else {
    const uint8_t* p = packed + 4 * w;
    return uint32_t(p[0]) | (uint32_t(p[1]) << 8) | (uint32_t(p[2]) << 16) | (uint32_t(p[3]) << 24);
  }
}

// Elements 8w..8w+7 of the output.
template <bool kAligned, bool kThrough>
__device__ __forceinline__ void store_elements(uint16_t* __restrict__ out, int64_t w, int64_t ndwords, uint4 v) {
  if constexpr (kAligned && kThrough) {
    constexpr int kSc1 = 16;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(out, 0, int(16 * ndwords), 0x00027000);
    __builtin_amdgcn_raw_buffer_store_b128((u32x4){v.x, v.y, v.z, v.w}, rsrc, int(16 * w), 0, kSc1);
  } else if constexpr (kAligned) {
    __builtin_nontemporal_store((u32x4){v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4*>(out) + w);
  } else {
    uint16_t* p = out + 8 * w;
    const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[2 * i] = uint16_t(words[i] & 0xffffu);
      p[2 * i + 1] = uint16_t(words[i] >> 16);
    }
  }
}

// The canonical codebook (reference ops/nf4.py:120-141), which a checked call holds `code` to.
__constant__ const float kCanonical[16] = {
    -1.0f,
    -0.6961928009986877f,
    -0.5250730514526367f,
    -0.39491748809814453f,
    -0.28444138169288635f,
    -0.18477343022823334f,
    -0.09105003625154495f,
    0.0f,
    0.07958029955625534f,
    0.16093020117282867f,
    0.24611230194568634f,
    0.33791524171829224f,
    0.44070982933044434f,
    0.5626170039176941f,
    0.7229568362236023f,
    1.0f,
};

// A checked call's answer in a word of host memory: kAnswered, plus 1 for the
// canonical codebook (word null: unchecked).
constexpr uint32_t kAnswered = 2;

template <bool kDouble, bool kAligned, int kSteps, bool kThrough>
__global__ __launch_bounds__(kThreads) void nf4_dequant_kernel(const uint8_t* __restrict__ packed,
                                                               ScaleSource src, const float* __restrict__ code,
                                                               uint16_t* __restrict__ out, int64_t ndwords,
                                                               uint32_t* verdict) {
  __shared__ float table[16];
  __shared__ float code2[kDouble ? 256 : 1];
  // Packed bytes are requested first; the codebook is staged while they travel.
  const int64_t base = int64_t(blockIdx.x) * (kThreads * kSteps) + threadIdx.x;
  uint32_t words[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    const int64_t w = base + s * kThreads;
    words[s] = w < ndwords ? load_packed<kAligned>(packed, w) : 0u;
  }
  const float offset = kDouble ? *src.offset : 0.0f;
  if (threadIdx.x < 16) table[threadIdx.x] = code[threadIdx.x];
  if constexpr (kDouble) code2[threadIdx.x] = src.code2[threadIdx.x];
  __syncthreads();
  if (kDouble && verdict && blockIdx.x == 0 && threadIdx.x < 64) {
    const uint64_t same = __ballot(threadIdx.x >= 16 || table[threadIdx.x & 15] == kCanonical[threadIdx.x & 15]);
    if (threadIdx.x == 0)
      __hip_atomic_store(verdict, kAnswered | (same == ~uint64_t(0) ? 1u : 0u), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    const int64_t w = base + s * kThreads;
    if (w < ndwords) {
      // 8 elements per dword, 64 per block: block = w / 8.
      const float scale = block_scale(src, w >> 3, code2, offset);
      store_elements<kAligned, kThrough>(out, w, ndwords, decode_dword(words[s], scale, table));
    }
  }
}

__global__ __launch_bounds__(kThreads) void dq_scales_kernel(ScaleSource src, float* __restrict__ scales,
                                                             int64_t nblocks) {
  __shared__ float code2[256];
  code2[threadIdx.x] = src.code2[threadIdx.x];
  __syncthreads();
  const float offset = *src.offset;
  for (int64_t j = int64_t(blockIdx.x) * kThreads + threadIdx.x; j < nblocks;
       j += int64_t(gridDim.x) * kThreads) {
    scales[j] = block_scale(src, j, code2, offset);
  }
}

int launch_dequant(const uint8_t* qweight, const ScaleSource& src, const float* code, uint16_t* out,
                   int64_t numel, void* stream, uint32_t* verdict = nullptr) {
  LF_REQUIRE(numel > 0 && numel % (kNf4Block * kNf4Block) == 0,
             "element count must be a positive multiple of 4096");
  LF_REQUIRE(qweight && code && out, "null pointer argument");
  LF_REQUIRE((reinterpret_cast<uintptr_t>(out) & 1u) == 0, "out must be 2-byte aligned (bf16)");
  const int64_t ndwords = numel / 8;
  const int steps = !src.scales && numel >= kLargeNested ? 4 : 2;
  const int64_t grid = (ndwords + kThreads * steps - 1) / (kThreads * steps);
  LF_REQUIRE(grid < (int64_t(1) << 31), "tensor too large");
  auto s = static_cast<hipStream_t>(stream);
  const bool vec = aligned16(out) && (reinterpret_cast<uintptr_t>(qweight) & 3u) == 0;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, s, qweight, src, code, out, ndwords, verdict);
  };
  const bool through = numel <= kThroughMost;
  if (src.scales)
    launch(!vec      ? nf4_dequant_kernel<false, false, 2, false>
           : through ? nf4_dequant_kernel<false, true, 2, true>
                     : nf4_dequant_kernel<false, true, 2, false>);
  else if (steps == 2)  // (less than kThroughMost)
    launch(vec ? nf4_dequant_kernel<true, true, 2, true> : nf4_dequant_kernel<true, false, 2, false>);
  else
    launch(!vec      ? nf4_dequant_kernel<true, false, 4, false>
           : through ? nf4_dequant_kernel<true, true, 4, true>
                     : nf4_dequant_kernel<true, true, 4, false>);
  LF_HIP(hipGetLastError());
  return kOk;
}

// Words for the answers of checked calls, one for each call in flight. Pinned
// host memory of one page, kept until the process ends.
VerdictWords g_words;
std::mutex g_page_lock;
uint32_t* g_page = nullptr;

}  // namespace
}  // namespace lf

extern "C" int lf_nf4_dequant_dq_checked(const uint8_t* qweight, const uint8_t* absmax_q, const float* absmax2,
                                         const float* code2, const float* offset, int64_t dq_block, const float* code,
                                         uint16_t* out, int64_t numel, int32_t* canonical, void* stream) {
  LF_REQUIRE(absmax_q && absmax2 && code2 && offset && canonical, "double-quant state pointers required");
  LF_REQUIRE(dq_block > 0 && dq_block <= (int64_t(1) << 30), "dq_block must be positive");
  auto s = static_cast<hipStream_t>(stream);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  LF_HIP(hipStreamIsCapturing(s, &capture));
  LF_REQUIRE(capture == hipStreamCaptureStatusNone, "a checked call waits for its answer: not under graph capture");
  {
    std::lock_guard<std::mutex> guard(lf::g_page_lock);
    if (lf::g_page == nullptr) {
      void* page = nullptr;
      // (Coherent: the host polls a word while its kernel runs.)
      LF_HIP(hipHostMalloc(&page, lf::VerdictWords::kWords * sizeof(uint32_t),
                           hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
      lf::g_page = static_cast<uint32_t*>(page);
    }
  }
  const int index = lf::g_words.take();
  LF_REQUIRE(index >= 0, "%d checked calls in flight already", lf::VerdictWords::kWords);
  uint32_t* word = lf::g_page + index;
  __atomic_store_n(word, 0u, __ATOMIC_RELAXED);
  // Nothing writes the word once the call is answered, or its kernel never
  // launched or finished: then it goes back.
  const auto returned = [&](int rc) {
    lf::g_words.give(index);
    return rc;
  };
  void* device_word = nullptr;
  if (const hipError_t err = hipHostGetDevicePointer(&device_word, word, 0); err != hipSuccess)
    return returned(lf::hip_status(err, "hipHostGetDevicePointer"));
  lf::ScaleSource src{nullptr, absmax_q, absmax2, code2, offset, int(dq_block)};
  const int rc = lf::launch_dequant(qweight, src, code, out, numel, stream, static_cast<uint32_t*>(device_word));
  if (rc != lf::kOk) return returned(rc);
  // The answer comes as the kernel starts: a short look for it, then the
  // stream's own wait (work ahead of the kernel, or an error).
  const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
  uint32_t answer;
  while ((answer = __atomic_load_n(word, __ATOMIC_ACQUIRE)) == 0) {
    if (std::chrono::steady_clock::now() < until) continue;
    LF_HIP(hipStreamSynchronize(s));  // (failed: the kernel may still run, the word stays taken)
    if ((answer = __atomic_load_n(word, __ATOMIC_ACQUIRE)) == 0)
      return returned(lf::fail(lf::kHip, "the codebook check gave no answer"));
  }
  *canonical = int32_t(answer & 1);
  return returned(lf::kOk);
}

extern "C" int lf_nf4_dequant(const uint8_t* qweight, const float* scales, const float* code, uint16_t* out,
                              int64_t numel, void* stream) {
  LF_REQUIRE(scales != nullptr, "scales required");
  lf::ScaleSource src{scales, nullptr, nullptr, nullptr, nullptr, 1};
  return lf::launch_dequant(qweight, src, code, out, numel, stream);
}

extern "C" int lf_nf4_dequant_dq(const uint8_t* qweight, const uint8_t* absmax_q, const float* absmax2,
                                 const float* code2, const float* offset, int64_t dq_block, const float* code,
                                 uint16_t* out, int64_t numel, void* stream) {
  LF_REQUIRE(absmax_q && absmax2 && code2 && offset, "double-quant state pointers required");
  LF_REQUIRE(dq_block > 0 && dq_block <= (int64_t(1) << 30), "dq_block must be positive");
  lf::ScaleSource src{nullptr, absmax_q, absmax2, code2, offset, int(dq_block)};
  return lf::launch_dequant(qweight, src, code, out, numel, stream);
}

extern "C" int lf_nf4_prepare_scales_dq(const uint8_t* absmax_q, const float* absmax2, const float* code2,
                                        const float* offset, int64_t dq_block, float* scales, int64_t nblocks,
                                        void* stream) {
  LF_REQUIRE(absmax_q && absmax2 && code2 && offset && scales, "null pointer argument");
  LF_REQUIRE(dq_block > 0 && dq_block <= (int64_t(1) << 30), "dq_block must be positive");
  LF_REQUIRE(nblocks > 0, "nblocks must be positive");
  lf::ScaleSource src{nullptr, absmax_q, absmax2, code2, offset, int(dq_block)};
  const int64_t want = (nblocks + lf::kThreads - 1) / lf::kThreads;
  const int grid = int(want < 4096 ? want : 4096);
  hipLaunchKernelGGL(lf::dq_scales_kernel, dim3(grid), dim3(lf::kThreads), 0, static_cast<hipStream_t>(stream),
                     src, scales, nblocks);
  LF_HIP(hipGetLastError());
  return lf::kOk;
}
