// K0 (NF4 blockwise quantise) and K1 (standalone NF4 -> bf16 dequant) for gfx950.
//
// K0 moves 2 B in and 0.5625 B out per value; with blocksize 64 (the expert path) eight
// lanes share a block and every wave reads and writes contiguous runs.
//
// K1 is HBM-bound: 0.5 B read + 2 B written per value (plus 4 B of absmax per 64
// values).  Each thread owns 32 consecutive values: one 16-byte load of packed nibbles,
// one absmax, four 16-byte stores of bf16.  The 16-entry codebook sits in LDS; 16
// distinct entries map to 16 distinct banks, so the lookups never conflict.
#include "common.h"

namespace moe {
namespace {

constexpr int kDequantThreads = 256;
// A wave dequantises chunks of 2048 values: lane l handles the 8 values at 512*s + 8*l of
// each quarter s, so each of its four 16-byte stores is part of one contiguous 1 KB store
// of the wave (and each 4-byte load part of a contiguous 256-byte load).
constexpr int kDequantChunk = 2048;

__global__ void __launch_bounds__(kDequantThreads)
nf4_dequant_kernel(const uint8_t *__restrict__ packed, const float *__restrict__ absmax,
                   const float *__restrict__ code, uint16_t *__restrict__ out, int64_t numel,
                   int32_t blocksize) {
  __shared__ float s_code[16];
  if (threadIdx.x < 16) s_code[threadIdx.x] = code[threadIdx.x];
  __syncthreads();

  const int lane = threadIdx.x & (kWave - 1);
  const int64_t nchunk = numel / kDequantChunk;
  const int64_t waves = (int64_t)gridDim.x * (kDequantThreads / kWave);
  for (int64_t c = (int64_t)blockIdx.x * (kDequantThreads / kWave) + (threadIdx.x >> 6); c < nchunk;
       c += waves) {
    const int64_t base = c * kDequantChunk;
    uint32_t q[4];
    float a[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t v0 = base + 512 * s + 8 * lane;
      q[s] = *reinterpret_cast<const uint32_t *>(packed + v0 / 2);
      a[s] = absmax[v0 / blocksize];  // blocksize is a multiple of 32: one block per 8 values
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      uint32_t o[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint32_t byte = (q[s] >> (8 * b)) & 0xffu;
        o[b] = pack_bf16x2(s_code[byte >> 4] * a[s], s_code[byte & 15u] * a[s]);
      }
      *reinterpret_cast<uint4 *>(out + base + 512 * s + 8 * lane) = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  // Tail: fewer than one chunk left (numel is even), two values per thread of workgroup 0.
  if (blockIdx.x == 0) {
    for (int64_t i = nchunk * kDequantChunk + 2 * threadIdx.x; i < numel; i += 2 * kDequantThreads) {
      const uint32_t byte = packed[i / 2];
      out[i] = f32_to_bf16(s_code[byte >> 4] * absmax[i / blocksize]);
      out[i + 1] = f32_to_bf16(s_code[byte & 15u] * absmax[(i + 1) / blocksize]);
    }
  }
}

constexpr int kQuantThreads = 256;

// Blocksize-64 quantisation, eight lanes per block: lane l of a wave loads the 8 bf16 values
// at 8*l of the wave's 512-value chunk (one contiguous 1 KB load per wave), the block's
// absmax is the max over its 8 lanes (DPP moves), and each lane packs its 8 values into
// 4 bytes (one contiguous 256-byte store per wave).  Same arithmetic as the per-block kernel
// below: q = number of codebook midpoints strictly below y = w * (1 / absmax), in fp32.
//
// Bound: 2.56 bytes a value of HBM (31 us at the copy rate for a 14336 x 4096 projection).
// Comparing y with all 15 midpoints is 30 VALU operations a value and took 72 us; the count
// now comes from a table of 64 equal bins over [-1, 1].  A bin index is monotone in y, so
// midpoints in lower bins are below y and those in higher bins are not; a bin holds at most
// one midpoint of a codebook like NF4's (their distance is at least 2.5 bins), against which
// one comparison decides: 32 to 34 us (4.5 TB/s; 48 us while every thread built eight table
// entries and no load ran ahead).  The entry {midpoint, count below the bin} has 32 replicas
// (conflict-free ds_read_b64).  A codebook with two midpoints in a bin compares with all 15.
// So do weights with at most one chunk a wave (TABLE false): every workgroup builds the table for
// itself, half a microsecond that one chunk does not earn back (512 / 1 M / 4 M values: 3.2 / 4.0
// / 6.4 us with the table, 2.6 / 3.2 / 6.2 without; 5 M, two chunks: 6.4 and 7.2).
constexpr int kQuant64Chunk = 512;
constexpr int kQuantBins = 64;
constexpr int kQuantReps = 32;

// Bin of y: NaN and anything below -1 in the first, anything above 1 in the last.
__device__ __forceinline__ uint32_t quant_bin(float y) {
  const float t = fmaf(y, 0.5f * kQuantBins, 0.5f * kQuantBins);
  return (uint32_t)fminf(fmaxf(t, 0.0f), (float)(kQuantBins - 1));
}

template <bool BINS>
__device__ __forceinline__ uint32_t quant8(const u32x4 raw, float r, const float (&mid)[15], const float2 *bins,
                                           uint32_t rep) {
  uint32_t out = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float y = ((i & 1) ? bf16hi_to_f32(raw[i >> 1]) : bf16lo_to_f32(raw[i >> 1])) * r;
    uint32_t q = 0;
    if constexpr (BINS) {
      const float2 e = bins[quant_bin(y) * kQuantReps + rep];
      q = __builtin_bit_cast(uint32_t, e.y) + (y > e.x ? 1u : 0u);
    } else {
#pragma unroll
      for (int m = 0; m < 15; ++m) q += y > mid[m] ? 1u : 0u;
    }
    // value 2j in the high nibble of byte j
    out |= q << (8 * (i >> 1) + ((i & 1) ? 0 : 4));
  }
  return out;
}

template <bool BINS>
__device__ __forceinline__ void quant64_chunks(const uint16_t *w, int64_t nchunk, uint8_t *packed, float *absmax,
                                               const float *s_mid, const float2 *bins) {
  float mid[15];
#pragma unroll
  for (int m = 0; m < 15; ++m) mid[m] = BINS ? 0.0f : s_mid[m];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t rep = threadIdx.x & (kQuantReps - 1);
  const int64_t waves = (int64_t)gridDim.x * (kQuantThreads / kWave);
  const int64_t c0 = (int64_t)blockIdx.x * (kQuantThreads / kWave) + (threadIdx.x >> 6);
  auto load = [&](int64_t c) {
    const uint4 v = ld_stream16(w + (c < nchunk ? c : nchunk - 1) * kQuant64Chunk + 8 * lane);
    return u32x4{v.x, v.y, v.z, v.w};
  };
  // With the table two chunks per step, the next step's loads in flight under this one's
  // arithmetic (past the end: the last chunk again, unused).
  constexpr int kStep = BINS ? 2 : 1;
  u32x4 next[kStep];
  if constexpr (BINS)
    for (int u = 0; u < kStep; ++u) next[u] = load(c0 + u * waves);
  for (int64_t c = c0; c < nchunk; c += kStep * waves) {
    u32x4 raw[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      raw[u] = BINS ? next[u] : load(c);
      if constexpr (BINS) next[u] = load(c + (u + kStep) * waves);
    }
    float amax[kStep] = {};
#pragma unroll
    for (int u = 0; u < kStep; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        amax[u] = fmaxf(amax[u], fabsf(bf16lo_to_f32(raw[u][i])));
        amax[u] = fmaxf(amax[u], fabsf(bf16hi_to_f32(raw[u][i])));
      }
    lane_groups_reduce<true>(amax, 8);
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      if (u > 0 && c + u * waves >= nchunk) break;
      const int64_t v0 = (c + u * waves) * kQuant64Chunk + 8 * lane;
      if ((lane & 7) == 0) absmax[v0 / 64] = amax[u];
      const float r = amax[u] > 0.0f ? 1.0f / amax[u] : 0.0f;
      *reinterpret_cast<uint32_t *>(packed + v0 / 2) = quant8<BINS>(raw[u], r, mid, bins, rep);
    }
  }
}

template <bool TABLE>
__global__ void __launch_bounds__(kQuantThreads)
nf4_quantize64_kernel(const uint16_t *__restrict__ w, int64_t nchunk,
                      const float *__restrict__ code, uint8_t *__restrict__ packed,
                      float *__restrict__ absmax, float *__restrict__ code_out) {
  __shared__ float s_mid[15];
  __shared__ float2 s_bins[TABLE ? kQuantBins * kQuantReps : 1];
  if (threadIdx.x < 15) s_mid[threadIdx.x] = (code[threadIdx.x] + code[threadIdx.x + 1]) * 0.5f;
  if (code_out != nullptr && blockIdx.x == 0 && threadIdx.x < 16) code_out[threadIdx.x] = code[threadIdx.x];
  __syncthreads();
  if constexpr (!TABLE) {
    quant64_chunks<false>(w, nchunk, packed, absmax, s_mid, s_bins);
    return;
  }
  // One thread per bin, then the replicas.
  int crowded = 0;
  if (threadIdx.x < kQuantBins) {
    float thr = INFINITY;
    uint32_t below = 0, in = 0;
    for (int m = 0; m < 15; ++m) {
      const float x = s_mid[m];
      const uint32_t bm = quant_bin(x);
      const bool number = x == x;  // nothing is above a NaN
      below += number && bm < threadIdx.x ? 1u : 0u;
      thr = number && bm == threadIdx.x ? x : thr;
      in += number && bm == threadIdx.x ? 1u : 0u;
    }
    crowded = in > 1u;
    s_bins[threadIdx.x * kQuantReps] = make_float2(thr, __builtin_bit_cast(float, below));
  }
  const bool general = __syncthreads_or(crowded) != 0;
  for (int i = threadIdx.x; i < kQuantBins * kQuantReps; i += kQuantThreads)
    if (i % kQuantReps != 0) s_bins[i] = s_bins[i / kQuantReps * kQuantReps];
  __syncthreads();
  // Uniform over the grid: every workgroup builds the same table.
  if (general)
    quant64_chunks<false>(w, nchunk, packed, absmax, s_mid, s_bins);
  else
    quant64_chunks<true>(w, nchunk, packed, absmax, s_mid, s_bins);
}

// One thread per quantisation block: any blocksize, partial last block.
__global__ void __launch_bounds__(kQuantThreads)
nf4_quantize_kernel(const uint16_t *__restrict__ w, int64_t numel, int32_t blocksize,
                    const float *__restrict__ code, uint8_t *__restrict__ packed,
                    float *__restrict__ absmax, float *__restrict__ code_out) {
  __shared__ float s_mid[15];
  if (code_out != nullptr && blockIdx.x == 0 && threadIdx.x < 16) code_out[threadIdx.x] = code[threadIdx.x];
  if (threadIdx.x < 15) s_mid[threadIdx.x] = (code[threadIdx.x] + code[threadIdx.x + 1]) * 0.5f;
  __syncthreads();
  const int64_t nblocks = (numel + blocksize - 1) / blocksize;
  const int64_t b = (int64_t)blockIdx.x * kQuantThreads + threadIdx.x;
  if (b >= nblocks) return;
  const int64_t lo = b * blocksize;
  const int64_t hi = lo + blocksize < numel ? lo + blocksize : numel;
  float amax = 0.0f;
  for (int64_t i = lo; i < hi; ++i) amax = fmaxf(amax, fabsf(bf16_to_f32(w[i])));
  absmax[b] = amax;
  const float r = amax > 0.0f ? 1.0f / amax : 0.0f;
  for (int64_t i = lo; i < hi; i += 2) {
    int q[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float x = bf16_to_f32(w[i + j]) * r;
      int c = 0;
#pragma unroll
      for (int m = 0; m < 15; ++m) c += x > s_mid[m];
      q[j] = c;
    }
    packed[i / 2] = (uint8_t)((q[0] << 4) | q[1]);
  }
}

constexpr int kExpandThreads = 256;

// Nested (double-quantised) absmax: the fp32 block scales stored as 8-bit indices into a
// 256-entry code, with one fp32 scale per group of blocksize2 indices and a common offset.
// out[i] = code2[q[i]] * absmax2[i / blocksize2] + offset (a product, then a sum, each
// rounded in fp32 -- bitsandbytes' dequantize_blockwise of the absmax, then += offset).
__global__ void __launch_bounds__(kExpandThreads)
expand_absmax_kernel(const uint8_t *__restrict__ q, const float *__restrict__ absmax2,
                     const float *__restrict__ code2, float offset, int64_t n, int32_t blocksize2,
                     float *__restrict__ out) {
  __shared__ float s_code[256];
  s_code[threadIdx.x] = code2[threadIdx.x];
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * kExpandThreads + threadIdx.x;
  if (i >= n) return;
  const float v = s_code[q[i]] * absmax2[i / blocksize2];
  out[i] = v + offset;
}

}  // namespace
}  // namespace moe

extern "C" int moe_nf4_expand_absmax(const void *absmax_u8, const void *absmax2_f32,
                                     const void *code2_f32, float offset, int64_t n,
                                     int32_t blocksize2, void *out_f32, void *stream) {
  MOE_REQUIRE(n >= 0, "n must be non-negative (got %lld)", (long long)n);
  MOE_REQUIRE(blocksize2 > 0, "blocksize2 must be positive (got %d)", blocksize2);
  if (n == 0) return MOE_STATUS_OK;
  MOE_REQUIRE(absmax_u8 && absmax2_f32 && code2_f32 && out_f32, "null device pointer");
  const int64_t grid = (n + moe::kExpandThreads - 1) / moe::kExpandThreads;
  MOE_REQUIRE(grid <= 0x7fffffff, "n too large");
  hipLaunchKernelGGL(moe::expand_absmax_kernel, dim3((unsigned)grid), dim3(moe::kExpandThreads), 0,
                     (hipStream_t)stream, (const uint8_t *)absmax_u8, (const float *)absmax2_f32,
                     (const float *)code2_f32, offset, n, blocksize2, (float *)out_f32);
  MOE_LAUNCH_CHECK();
  return MOE_STATUS_OK;
}

extern "C" int moe_nf4_dequant_bf16(const void *packed, const void *absmax, const void *code16,
                                    void *out_bf16, int64_t numel, int32_t blocksize,
                                    void *stream) {
  MOE_REQUIRE(numel >= 0 && numel % 2 == 0, "numel must be even and non-negative (got %lld)",
              (long long)numel);
  MOE_REQUIRE(blocksize > 0 && blocksize % 32 == 0,
              "blocksize must be a positive multiple of 32 (got %d)", blocksize);
  if (numel == 0) return MOE_STATUS_OK;
  MOE_REQUIRE(packed && absmax && code16 && out_bf16, "null device pointer");
  MOE_REQUIRE(((uintptr_t)packed % 16) == 0 && ((uintptr_t)out_bf16 % 16) == 0,
              "packed and out must be 16-byte aligned");
  const int64_t nchunk = numel / moe::kDequantChunk;
  int64_t blocks = (nchunk + (moe::kDequantThreads / moe::kWave) - 1) / (moe::kDequantThreads / moe::kWave);
  const int64_t cap = (int64_t)moe::device_cu_count() * 8;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(moe::nf4_dequant_kernel, dim3((unsigned)blocks), dim3(moe::kDequantThreads),
                     0, (hipStream_t)stream, (const uint8_t *)packed, (const float *)absmax,
                     (const float *)code16, (uint16_t *)out_bf16, numel, blocksize);
  MOE_LAUNCH_CHECK();
  return MOE_STATUS_OK;
}

extern "C" int moe_nf4_quantize_bf16(const void *w_bf16, int64_t numel, int32_t blocksize,
                                     const void *code16, void *packed_out, void *absmax_out,
                                     void *stream) {
  return moe_nf4_quantize_state_bf16(w_bf16, numel, blocksize, code16, packed_out, absmax_out, nullptr,
                                     stream);
}

extern "C" int moe_nf4_quantize_state_bf16(const void *w_bf16, int64_t numel, int32_t blocksize,
                                           const void *code16, void *packed_out, void *absmax_out,
                                           void *code_out, void *stream) {
  MOE_REQUIRE(numel >= 0 && numel % 2 == 0, "numel must be even and non-negative (got %lld)",
              (long long)numel);
  MOE_REQUIRE(blocksize >= 2 && blocksize <= 4096 && blocksize % 2 == 0,
              "blocksize must be even and in [2, 4096] (got %d)", blocksize);
  if (numel == 0) return MOE_STATUS_OK;
  MOE_REQUIRE(w_bf16 && code16 && packed_out && absmax_out, "null device pointer");
  if (blocksize == 64 && numel % moe::kQuant64Chunk == 0 && ((uintptr_t)w_bf16 % 16) == 0 &&
      ((uintptr_t)packed_out % 4) == 0 && ((uintptr_t)absmax_out % 4) == 0) {
    const int64_t nchunk = numel / moe::kQuant64Chunk;
    int64_t blocks = (nchunk + (moe::kQuantThreads / moe::kWave) - 1) / (moe::kQuantThreads / moe::kWave);
    const int64_t cap = (int64_t)moe::device_cu_count() * 8;
    blocks = blocks > cap ? cap : blocks;
    const bool table = nchunk > blocks * (moe::kQuantThreads / moe::kWave);  // more than a chunk a wave
    auto kern = table ? moe::nf4_quantize64_kernel<true> : moe::nf4_quantize64_kernel<false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(moe::kQuantThreads),
                       0, (hipStream_t)stream, (const uint16_t *)w_bf16, nchunk,
                       (const float *)code16, (uint8_t *)packed_out, (float *)absmax_out,
                       (float *)code_out);
    MOE_LAUNCH_CHECK();
    return MOE_STATUS_OK;
  }
  const int64_t nblocks = (numel + blocksize - 1) / blocksize;
  const int64_t grid = (nblocks + moe::kQuantThreads - 1) / moe::kQuantThreads;
  MOE_REQUIRE(grid <= 0x7fffffff, "numel too large");
  hipLaunchKernelGGL(moe::nf4_quantize_kernel, dim3((unsigned)grid), dim3(moe::kQuantThreads), 0,
                     (hipStream_t)stream, (const uint16_t *)w_bf16, numel, blocksize,
                     (const float *)code16, (uint8_t *)packed_out, (float *)absmax_out,
                     (float *)code_out);
  MOE_LAUNCH_CHECK();
  return MOE_STATUS_OK;
}
