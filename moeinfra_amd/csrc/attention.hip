// Grouped-query causal attention of the decoder against its KV cache (the reference runs it
// as the eager attention of MixtralDecoderLayer inside Hugging Face modules,
// engine/engine.py:211-314).
//
//   attention_kernel          one workgroup per (query head, token), any head dim
//   few_attention_kernel      up to 8 tokens: several workgroups share a row's keys
//   prefill_attention_kernel  more tokens at head dim 64 or 128: 128 query rows per workgroup
//                             on the matrix cores, one pass over the keys (a few dozen tokens
//                             with a short context row by row)
// Numbers below: 32 query heads, 8 KV heads of 128, MI355X, launches back to back.
#include <type_traits>

#include "common.h"

namespace moe {
namespace {

constexpr int kAttnThreads = 256;
constexpr int kAttnMaxKeys = 8192;
constexpr int kAttnMaxHeadDim = 256;
constexpr int kAttnRowsInFlight = 8;  // cache rows per thread per pass

// Scores of the pass starting at key j0 from its loaded K rows: s_p[j] = bf16(bf16(q.k_j) *
// scaling) for the keys j < nkeys, and the running maximum.  The eight rows' lane partials
// are formed first and summed over each row's lpr lanes together (DPP within a 16-lane row).
__device__ __forceinline__ void attn_scores(const uint4 (&kv)[kAttnRowsInFlight], const float (&qf)[8],
                                            int j0, int nkeys, int rpp, int rr, int lpr, int sub,
                                            float scaling, float *s_p, float &mx) {
  float dot[kAttnRowsInFlight];
#pragma unroll
  for (int u = 0; u < kAttnRowsInFlight; ++u) {
    float kf[8];
    unpack8(kv[u], kf);
    float d = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) d = fmaf(qf[e], kf[e], d);
    dot[u] = d;
  }
  lane_groups_reduce<false>(dot, lpr);
#pragma unroll
  for (int u = 0; u < kAttnRowsInFlight; ++u) {
    const int j = j0 + u * rpp + rr;
    const float sc = bf16r(bf16r(dot[u]) * scaling);
    const bool ok = j < nkeys;
    mx = ok ? fmaxf(mx, sc) : mx;
    if (ok && sub == 0) s_p[j] = sc;
  }
}

// acc += p_j v_j over the pass's rows j < nkeys, in row order.
__device__ __forceinline__ void attn_pv(const uint4 (&vv)[kAttnRowsInFlight], int j0, int nkeys,
                                        int rpp, int rr, const float *s_p, float (&acc)[8]) {
#pragma unroll
  for (int u = 0; u < kAttnRowsInFlight; ++u) {
    const int j = j0 + u * rpp + rr;
    if (j < nkeys) {
      const float p = s_p[j];
      float vf[8];
      unpack8(vv[u], vf);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(p, vf[e], acc[e]);
    }
  }
}

// NH query heads of a KV head, one token, on kAttnThreads threads: scores of keys 0 .. pos0 + t
// (causal), bf16 scores scaled in bf16, fp32 softmax rounded to bf16, then the bf16 probabilities times V with
// fp32 accumulation.  A cache row of hd bf16 is read by hd/8 consecutive lanes, 16 bytes
// each, so the threads cover rpp = 256/(hd/8) rows per load instruction and a pass takes
// 8 such loads per thread (128 rows at hd = 128); a score is the xor-shuffle sum over its
// row's lanes.  The first pass's K and V rows are loaded together with q and the position
// (first()), before the key count is known (row indexes clamped to the cache, results of rows
// past the last key discarded), so a context of up to one pass of keys costs one memory round
// trip; later passes load rows clamped to the last key.
template <int NH>
struct AttnRow {
  const uint16_t *kbase, *vbase;
  int tid, hd, lpr, rpp, sub, rr;
  float qf[NH][8];
  uint4 kv[kAttnRowsInFlight], vv[kAttnRowsInFlight];

  __device__ __forceinline__ void load(uint4 (&dst)[kAttnRowsInFlight], const uint16_t *base, int j0, int last) {
#pragma unroll
    for (int u = 0; u < kAttnRowsInFlight; ++u)
      dst[u] = *reinterpret_cast<const uint4 *>(base + (size_t)min(j0 + u * rpp + rr, last) * hd);
  }
  __device__ __forceinline__ void place(const uint16_t *kc, const uint16_t *vc, int kvh, int hd_,
                                        int64_t max_seq, int tid_) {
    tid = tid_;
    hd = hd_;
    lpr = hd >> 3;               // lanes per row: a power of two <= 32
    rpp = kAttnThreads / lpr;    // rows per load instruction
    sub = tid & (lpr - 1);
    rr = tid / lpr;
    kbase = kc + (size_t)kvh * max_seq * hd + sub * 8;
    vbase = vc + (size_t)kvh * max_seq * hd + sub * 8;
  }
  // q (heads h .. h + NH - 1 of row t, of the KV head) and the first pass's rows, up to row `last` of the keys at kbase / vbase.
  __device__ __forceinline__ void first(const uint16_t *q, int nq, int h, int t, int last) {
#pragma unroll
    for (int n = 0; n < NH; ++n)
      unpack8(*reinterpret_cast<const uint4 *>(q + ((size_t)t * nq + h + n) * hd + sub * 8), qf[n]);
    load(kv, kbase, 0, last);
    load(vv, vbase, 0, last);
  }
  // The NH output rows over the nkeys keys at kbase / vbase, value d of row n to store(n, d, o):
  // o = sum_j p_j v_j[d], or with PART sum_j e^(s_j - mx) v_j[d], unnormalised, and the rows'
  // maxima and sums (keys that all score -inf weigh nothing: any finite reference).  s_p: NH
  // arrays of `stride` >= nkeys floats, s_red: NH per wave, s_acc: NH * kAttnThreads * 8.  The
  // barriers are the same whatever nkeys is.
  template <bool PART, typename Store>
  __device__ __forceinline__ void run(int nkeys, float scaling, float *s_p, int stride, float *s_red, float *s_acc,
                                      Store store, float (&mx)[NH], float (&sum)[NH]) {
    constexpr int kWaves = kAttnThreads / kWave;
    const int npass = kAttnRowsInFlight * rpp;
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      mx[n] = -INFINITY;
      attn_scores(kv, qf[n], 0, nkeys, rpp, rr, lpr, sub, scaling, s_p + n * stride, mx[n]);
    }
    for (int j0 = npass; j0 < nkeys; j0 += npass) {
      load(kv, kbase, j0, nkeys - 1);
#pragma unroll
      for (int n = 0; n < NH; ++n)
        attn_scores(kv, qf[n], j0, nkeys, rpp, rr, lpr, sub, scaling, s_p + n * stride, mx[n]);
    }
    // block max, then the block sum of the exponentials (each a wave reduction, then the
    // four waves' values through LDS in wave order)
    const int lane = tid & (kWave - 1), wave = tid >> 6;
    lane_groups_reduce<true>(mx, kWave);
    if (lane == 0)
      for (int n = 0; n < NH; ++n) s_red[n * kWaves + wave] = mx[n];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      mx[n] = s_red[n * kWaves];
      for (int w = 1; w < kWaves; ++w) mx[n] = fmaxf(mx[n], s_red[n * kWaves + w]);
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      const float mref = PART && mx[n] == -INFINITY ? 0.0f : mx[n];
      sum[n] = 0.0f;
      for (int j = tid; j < nkeys; j += kAttnThreads) {
        const float e = expf(s_p[n * stride + j] - mref);
        s_p[n * stride + j] = e;
        sum[n] += e;
      }
    }
    lane_groups_reduce<false>(sum, kWave);
    if (lane == 0)
      for (int n = 0; n < NH; ++n) s_red[n * kWaves + wave] = sum[n];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      sum[n] = 0.0f;
      for (int w = 0; w < kWaves; ++w) sum[n] += s_red[n * kWaves + w];
    }
    __syncthreads();
    if constexpr (!PART) {
#pragma unroll
      for (int n = 0; n < NH; ++n)
        for (int j = tid; j < nkeys; j += kAttnThreads) s_p[n * stride + j] = bf16r(s_p[n * stride + j] / sum[n]);
      __syncthreads();
    }
    // out[d] = sum_j p_j v_j[d]: thread (rr, sub) accumulates dims sub*8 .. sub*8+7 over rows
    // rr, rr + rpp, ... in order; then the rpp partial rows are summed through LDS.
    float acc[NH][8];
#pragma unroll
    for (int n = 0; n < NH; ++n) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[n][e] = 0.0f;
      attn_pv(vv, 0, nkeys, rpp, rr, s_p + n * stride, acc[n]);
    }
    for (int j0 = npass; j0 < nkeys; j0 += npass) {
      load(vv, vbase, j0, nkeys - 1);
#pragma unroll
      for (int n = 0; n < NH; ++n) attn_pv(vv, j0, nkeys, rpp, rr, s_p + n * stride, acc[n]);
    }
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      float4 *sa = reinterpret_cast<float4 *>(s_acc + n * kAttnThreads * 8 + rr * hd + sub * 8);
      sa[0] = make_float4(acc[n][0], acc[n][1], acc[n][2], acc[n][3]);
      sa[1] = make_float4(acc[n][4], acc[n][5], acc[n][6], acc[n][7]);
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NH; ++n)
      for (int d = tid; d < hd; d += kAttnThreads) {
        float o = 0.0f;
        for (int r = 0; r < rpp; ++r) o += s_acc[n * kAttnThreads * 8 + r * hd + d];
        store(n, d, o);
      }
  }
  // The whole of it: NH bf16 rows at `orow`.
  __device__ __forceinline__ void finish(int nkeys, float scaling, uint16_t *orow, float *s_p, int stride,
                                         float *s_red, float *s_acc) {
    float mx[NH], sum[NH];
    run<false>(nkeys, scaling, s_p, stride, s_red, s_acc,
               [&](int n, int d, float o) { orow[n * hd + d] = f32_to_bf16(o); }, mx, sum);
  }
};

// One workgroup per (query head, token).
__global__ void __launch_bounds__(kAttnThreads)
attention_kernel(const uint16_t *__restrict__ q, const uint16_t *__restrict__ kc,
                 const uint16_t *__restrict__ vc, int nq, int nkv, int hd,
                 const int32_t *__restrict__ pos0, int64_t max_seq, float scaling,
                 uint16_t *__restrict__ out) {
  __shared__ float s_p[kAttnMaxKeys];
  __shared__ float s_red[kAttnThreads / kWave];
  __shared__ __attribute__((aligned(16))) float s_acc[kAttnThreads * 8];
  MOE_ARGS_FIRST(MOE_LIST("+s"(nq), "+s"(nkv), "+s"(hd), "+s"(max_seq), "+s"(scaling)),
                 MOE_LIST("s"(q), "s"(kc), "s"(vc), "s"(pos0), "s"(out)));
  const int h = blockIdx.x, t = blockIdx.y;
  AttnRow<1> row;
  row.place(kc, vc, h / (nq / nkv), hd, max_seq, (int)threadIdx.x);
  row.first(q, nq, h, t, (int)max_seq - 1);
  // Keys 0 .. pos0 + t, bounded by the cache (a position past it is a caller error).
  row.finish(min(*pos0 + t + 1, (int)max_seq), scaling, out + ((size_t)t * nq + h) * hd, s_p, 0, s_red,
             s_acc);
}

// Partial results pass between workgroups, which may run on different XCDs, through
// device-scope accesses that do not stay in an XCD's L2: attn_put writes through, attn_get
// reads past stale lines.  With every shared word moved that way, arrival needs only the
// writers' stores to have completed (their vmcnt is zero before the workgroup counts itself
// in), not a write-back and invalidation of whole caches: with a device-scope fence per
// workgroup instead, one token behind 3000 keys took 67 us, more than the 54 us of the
// single-workgroup form.
__device__ __forceinline__ void attn_put(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float attn_get(const float *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether this workgroup is the last of n to arrive at *count (which it then leaves zero for
// the next launch).  What the others wrote with attn_put is there for the last one's
// attn_get.  Uniform over the workgroup; nothing here waits for another workgroup.
__device__ __forceinline__ bool attn_last_of(uint32_t *count, int n) {
  __shared__ uint32_t s_seen;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t seen =
        __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    if (seen == (uint32_t)n)
      __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_seen = seen;
  }
  __syncthreads();
  return s_seen == (uint32_t)n;
}

// A few tokens, possibly behind a long context.  attention_kernel's workgroup walks a (query
// head, token)'s keys alone; here up to kFewSplits workgroups share them, whole passes each,
// and the last to finish adds the partial outputs (fp32, unnormalised) up.  Up to kFewWhole
// keys the first workgroup does it all as attention_kernel does, bit for bit, and the others
// leave at once.
//
// Bound: latency (the keys of 3000 tokens are 12 MB, 2 us of HBM).  attention_kernel keeps 32
// of 256 CUs busy and walks 24 dependent passes there.  One token behind 400 / 1000 / 3000
// keys: 9.7 / 17.1 / 54.4 us so, 7.2 / 8.2 / 11.8 us here; 8 tokens behind 1000 / 3000: 17.6 /
// 53.1 and 15.7 / 33.6.  Behind a short context the workgroups that leave at once cost 0.25 us
// (1 / 2 / 8 tokens, nothing cached: 3.9 / 4.0 / 4.1 and 4.2 / 4.2 / 4.4 us; with the token as
// the slow grid index, behind all splits of the tokens before it, 4.3 / 5.0 / 5.1).
constexpr int kFewTokens = 8;
constexpr int kFewSplits = 16;
constexpr int kFewWhole = 384;
constexpr int kFewKeys = kAttnMaxKeys / 2;  // of one split, at two splits or more

__global__ void __launch_bounds__(kAttnThreads)
few_attention_kernel(const uint16_t *__restrict__ q, const uint16_t *__restrict__ kc,
                        const uint16_t *__restrict__ vc, int nq, int nkv, int grp, uint32_t over_nkv, int hd,
                        const int32_t *__restrict__ pos0, int64_t max_seq, float scaling,
                        uint16_t *__restrict__ out, uint32_t *__restrict__ count,
                        float *__restrict__ part) {
  __shared__ float s_p[kFewKeys];
  __shared__ float s_red[kAttnThreads / kWave];
  __shared__ __attribute__((aligned(16))) float s_acc[kAttnThreads * 8];
  MOE_ARGS_FIRST(MOE_LIST("+s"(nq), "+s"(nkv), "+s"(grp), "+s"(over_nkv), "+s"(hd), "+s"(max_seq), "+s"(scaling)),
                 MOE_LIST("s"(q), "s"(kc), "s"(vc), "s"(pos0), "s"(out), "s"(count), "s"(part)));
  // The KV head is the fast index: a group's query heads read the same cache rows, and with
  // 8 KV heads they run on one XCD.  The split is the slow one: the first splits, which have
  // work at any length, start first.
  const int g = (int)__umulhi(blockIdx.x << 1, over_nkv), kvh = (int)blockIdx.x - g * nkv;
  const int h = kvh * grp + g;
  const int t = (int)blockIdx.y, split = (int)blockIdx.z;
  const int unit = t * nq + h;
  AttnRow<1> row;
  row.place(kc, vc, kvh, hd, max_seq, (int)threadIdx.x);
  if (split == 0) row.first(q, nq, h, t, (int)max_seq - 1);  // with the position, as in attention_kernel
  const int nkeys = min(*pos0 + t + 1, (int)max_seq);
  if (nkeys <= kFewWhole) {  // uniform over the workgroup, as what follows
    if (split == 0) row.finish(nkeys, scaling, out + (size_t)unit * hd, s_p, 0, s_red, s_acc);
    return;
  }
  const int npass = kAttnRowsInFlight * row.rpp;
  const int passes = (nkeys + npass - 1) / npass;
  const int per = (passes + (int)gridDim.z - 1) / (int)gridDim.z;
  const int nact = (passes + per - 1) / per;
  if (split >= nact) return;
  const int begin = split * per * npass;
  const int n = min(nkeys - begin, per * npass);
  if (split > 0) {
    row.kbase += (size_t)begin * hd;
    row.vbase += (size_t)begin * hd;
    row.first(q, nq, h, t, n - 1);
  }
  // Partials of (token, head): [split][output of hd, maximum, sum].
  float *const ph = part + (size_t)unit * gridDim.z * (hd + 2);
  float *const mine = ph + (size_t)split * (hd + 2);
  float mx[1], sum[1];
  row.run<true>(n, scaling, s_p, 0, s_red, s_acc, [&](int, int d, float o) { attn_put(mine + d, o); }, mx, sum);
  if (threadIdx.x == 0) {
    attn_put(mine + hd, mx[0]);
    attn_put(mine + hd + 1, sum[0]);
  }
  if (!attn_last_of(count + unit, nact)) return;
  // Weights of the splits (and the sum's share of each) in LDS, then the outputs, all loads
  // of a thread in flight together.
  if (threadIdx.x < kFewSplits) {
    const bool has = (int)threadIdx.x < nact;
    const float *pm = ph + (size_t)(has ? threadIdx.x : 0) * (hd + 2) + hd;
    const float my = attn_get(pm), ly = attn_get(pm + 1);
    float m[1] = {my};
    lane_groups_reduce<true>(m, kFewSplits);
    const float w = has ? expf(my - m[0]) : 0.0f;
    float l[1] = {has ? w * ly : 0.0f};
    lane_groups_reduce<false>(l, kFewSplits);
    s_p[threadIdx.x] = w;
    s_p[kFewSplits + threadIdx.x] = l[0];
  }
  __syncthreads();
  const float l = s_p[kFewSplits];
  for (int d = threadIdx.x; d < hd; d += kAttnThreads) {
    float pv[kFewSplits];
#pragma unroll
    for (int y = 0; y < kFewSplits; ++y) pv[y] = y < nact ? attn_get(ph + (size_t)y * (hd + 2) + d) : 0.0f;
    float o = 0.0f;
#pragma unroll
    for (int y = 0; y < kFewSplits; ++y)
      if (y < nact) o = fmaf(s_p[y], pv[y], o);
    out[(size_t)unit * hd + d] = f32_to_bf16(o / l);
  }
}

// ------------------------------------------------------------------ prefill on the matrix cores
// Rows of one KV head are (token, query head of its group), r = t * group + g, so that the
// group's heads share the K and V tiles; a workgroup takes 128 consecutive rows, each of its
// waves 32, and walks the keys in tiles of 64 with a running maximum and sum per row:
//
//   S^T = K Q^T   lane (column q = l % 32) holds 16 keys of its row per 32-key half
//   O^T += V^T P^T, P = bf16(e^(s - m)), s = bf16(bf16(q.k) * scaling), sums in fp32
//
// Scores, maxima, sums and the output stay in fp32 registers; the rows' values are in
// columns, so maxima, sums and rescaling are per lane (one exchange with lane l ^ 32).  The
// P of a lane is the B operand of the second product as it stands: V^T is staged with its
// keys in the order that the first product's rows have, so no value
// crosses lanes.
//
// Bound: the serial chain of a row tile's keys.  At 1500 tokens the products are 18 GFLOP,
// about 12 us at the rate of a large GEMM; the last row tile walks 12 pairs of key tiles of
// about 2.3 us (MFMA, score rounding and exponentials, and 256 KB of LDS operand reads a
// pair), and 376 workgroups fill 256 CUs once and a half.  A second group of four waves takes
// every other tile (the chain halves; their sums meet in LDS), and where row tiles alone
// leave CUs idle, workgroups share a tile's keys through the workspace.  1500 tokens: 1022 us
// one workgroup per (head, token), 40 us here; 500 tokens behind 2000: 967 and 39 us; 40
// behind 2500: 99 and 24 us.
// Key tiles wait in registers while the previous pair is multiplied; two LDS planes per key
// group make that one barrier per pair.
//
// One pair of tiles is 8 to 10 us from end to end, most of it first use of the code and of the
// loads, more than a row takes alone (up to kFewTokens = 8 tokens keep the other form: 4.2 us
// at 7).  So a lone pair goes through group 0 without the joining of the groups (40 tokens: 9.9
// -> 8.2 us; one workgroup per row 8.5), and up to kFaRowKeys keys, where the device holds all
// units of ROWS heads of a token at once, the workgroups take those instead: 9 / 16 / 32 tokens
// 7.9 / 8.4 / 9.8 us in pairs, 4.7 / 4.9 / 7.2 one workgroup per row, 4.4 / 4.5 / 6.3 so; 32
// behind 100 / 300: 13.0 / 14.4, 9.6 / 17.2 and 9.4 / 13.3.
constexpr int kFaThreads = 512;
constexpr int kFaHalf = 256;  // threads of one key group
constexpr int kFaRows = 128;  // query rows per workgroup
constexpr int kFaKeys = 64;   // keys per tile
constexpr int kFaRowKeys = 384;  // the row instance's keys at most
constexpr float kLog2e = 1.44269504088896341f;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

__device__ __forceinline__ bf16x8 fa_op(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// LDS byte address of 16-byte piece p of K row r (HD * 2 bytes): the XOR spreads the 16 rows
// that a ds_read_b128 serves together over all banks.  Piece p of V^T row d (128 bytes, 8
// keys a piece) sits at p ^ fa_vx(d), with d >> 4 in it so that the staging's writes (HD / 16
// dims apart) spread too.  Only XORs of a lane's part with a step's constant: the loop
// computes each address in one instruction instead of holding all of them in registers.
template <int HD>
__device__ __forceinline__ uint32_t fa_kx(uint32_t r) {
  return HD == 128 ? r & 15 : (r >> 1) & 7;
}
__device__ __forceinline__ uint32_t fa_vx(uint32_t d) { return ((d >> 1) ^ (d >> 4)) & 7; }

// Whether a word of two bf16 values holds an infinity or a NaN.
__device__ __forceinline__ bool fa_nonfinite(uint32_t w) {
  return (w & 0x7f80u) == 0x7f80u || (w & 0x7f800000u) == 0x7f800000u;
}

// The rows row0 .. row_end - 1 against keys k_begin .. k_end - 1 without matrix products: a
// wave per row, 64 keys at a time (a key per lane), the same running maximum and sum.  Row
// r's unnormalised output, maximum and sum go to s_row[(r - row0) * (HD + 2) ...].
template <int HD>
__device__ __noinline__ void fa_rows_scalar(const uint16_t *q, const char *kbase, const char *vbase,
                                            int row0, int row_end, int k_begin, int k_end, int p0, int cap,
                                            int kvh, int grp, int nq, float scaling, float *s_row, int tid) {
  const int lane = tid & (kWave - 1);
  for (int r = row0 + (tid >> 6); r < row_end; r += kFaThreads / kWave) {
    const int t = r / grp, head = kvh * grp + (r - t * grp);
    const uint16_t *qrow = q + ((size_t)t * nq + head) * HD;
    const int end = min(min(p0 + t + 1, cap), k_end);
    float m = -INFINITY, l = 0.0f, o[HD / kWave];
    for (int e = 0; e < HD / kWave; ++e) o[e] = 0.0f;
    for (int k0 = k_begin; k0 < end; k0 += kWave) {
      const int j = min(k0 + lane, end - 1);
      const uint16_t *krow = reinterpret_cast<const uint16_t *>(kbase) + (size_t)j * HD;
      float d = 0.0f;
      for (int i = 0; i < HD; ++i) d = fmaf(bf16_to_f32(qrow[i]), bf16_to_f32(krow[i]), d);
      const float x = k0 + lane < end ? bf16r(bf16r(d) * scaling) : -INFINITY;
      float mx[1] = {x};
      lane_groups_reduce<true>(mx, kWave);
      const float mn = fmaxf(m, mx[0]);
      const float mref = mn == -INFINITY ? 0.0f : mn;
      const float alpha = __builtin_amdgcn_exp2f((m - mref) * kLog2e);
      const float p = __builtin_amdgcn_exp2f((x - mref) * kLog2e);
      m = mn;
      l = l * alpha + wave_sum(p);
      for (int e = 0; e < HD / kWave; ++e) o[e] *= alpha;
      const int n = min(kWave, end - k0);
      for (int i = 0; i < n; ++i) {
        const float pi = bf16r(__shfl(p, i, kWave));
        const uint16_t *vrow = reinterpret_cast<const uint16_t *>(vbase) + (size_t)(k0 + i) * HD;
        for (int e = 0; e < HD / kWave; ++e) o[e] = fmaf(pi, bf16_to_f32(vrow[e * kWave + lane]), o[e]);
      }
    }
    float *dst = s_row + (r - row0) * (HD + 2);
    for (int e = 0; e < HD / kWave; ++e) dst[e * kWave + lane] = o[e];
    if (lane == 0) {
      dst[HD] = m;
      dst[HD + 1] = l;
    }
  }
}

// Row `row`'s values back into the lanes' layout of O^T (rows without an entry: leftovers
// that are not stored).
template <int HD>
__device__ __forceinline__ void fa_load_row(const float *s_row, int row, int hh, f32x16 (&acc)[HD / 32],
                                            float &m, float &l) {
  const float *src = s_row + row * (HD + 2);
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[dt][v] = src[32 * dt + 8 * (v >> 2) + 4 * hh + (v & 3)];
  m = src[HD];
  l = src[HD + 1];
}

template <int HD, int ROWS>
__global__ void __launch_bounds__(kFaThreads, 2)
prefill_attention_kernel(const uint16_t *__restrict__ q, const uint16_t *__restrict__ kc,
                         const uint16_t *__restrict__ vc, int T, int nq, int nkv,
                         const int32_t *__restrict__ pos0, int64_t max_seq, float scaling,
                         uint16_t *__restrict__ out, uint32_t *__restrict__ count,
                         float *__restrict__ part, int splits) {
  static_assert(HD == 64 || HD == 128, "head dims of the matrix form");
  constexpr int kPieces = HD / 8;                       // 16-byte pieces per K row
  constexpr int kKRows = kFaHalf / kPieces;             // K rows per load instruction
  constexpr int kKLoads = kFaKeys / kKRows;
  constexpr int kVWords = HD / 32;                      // words per thread and V row
  constexpr int kDT = HD / 32;                          // 32-dim output tiles
  constexpr int kKPlane = kFaKeys * HD * 2, kVPlane = HD * kFaKeys * 2;  // bytes
  __shared__ __attribute__((aligned(16))) uint8_t s_kv[2][2][kKPlane + kVPlane];
  __shared__ int s_nonfinite;

  if constexpr (ROWS > 0) {
    // Two units of ROWS heads of a token a workgroup.  (Their loads are on the way when the
    // position arrives; a long context drops them.)
    constexpr int kAcc = ROWS * kAttnThreads * 8, kUnit = kAcc + ROWS * (kFaRowKeys + kAttnThreads / kWave);
    static_assert(2 * kUnit * 4 <= (int)sizeof(s_kv), "the units fit the planes");
    const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kAttnThreads);
    const int wg = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int units = nq / ROWS * T;
    const int unit = min(2 * wg + half, units - 1);  // (an odd last unit twice, the same values)
    const int t = unit / (nq / ROWS), h = (unit - t * (nq / ROWS)) * ROWS;
    AttnRow<ROWS> row;
    row.place(kc, vc, h / (nq / nkv), HD, max_seq, (int)threadIdx.x & (kAttnThreads - 1));
    row.first(q, nq, h, t, (int)max_seq - 1);
    const int p0 = min(*pos0, (int)max_seq);  // (a position past the cache is a caller error)
    if (min(p0 + T, (int)max_seq) <= kFaRowKeys) {
      if (2 * wg >= units) return;
      float *const s_acc = reinterpret_cast<float *>(&s_kv[0][0][0]) + half * kUnit;
      float *const s_p = s_acc + kAcc;
      row.finish(min(p0 + t + 1, (int)max_seq), scaling, out + ((size_t)t * nq + h) * HD, s_p, kFaRowKeys,
                 s_p + ROWS * kFaRowKeys, s_acc);
      return;
    }
  }

  const int tid = threadIdx.x & (kFaHalf - 1);
  const int lane = tid & (kWave - 1);
  const int li = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) & 3;   // row group
  const int kgrp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);       // key group
  const int grp = nq / nkv;
  const int rows = T * grp;
  // The KV head is the fast index (one head's workgroups share an XCD's L2 when nkv is a
  // multiple of 8), and the last rows, which see the most keys, start first.
  const int ntile = (rows + kFaRows - 1) / kFaRows;
  const int kvh = (int)blockIdx.x % nkv;
  const int row0 = (ntile - 1 - (int)blockIdx.x / nkv) * kFaRows;
  const int cap = (int)max_seq;

  const int r = row0 + wave * 32 + li;
  const int rc = min(r, rows - 1);
  const int t = rc / grp;
  const int head = kvh * grp + (rc - t * grp);
  // Q as the B operand: column q = li, values 16 s + 8 hh .. + 7 of its row.
  u32x4 qf[HD / 16];
  {
    const uint16_t *qrow = q + ((size_t)t * nq + head) * HD + 8 * hh;
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) qf[s] = *reinterpret_cast<const u32x4 *>(qrow + 16 * s);
  }

  // Staging: K rows kr + i * kKRows, piece kp; V rows 4 vq .. 4 vq + 3, dims vd .. + HD/16 - 1.
  // Row indexes clamp to the cache; rows past the last key are masked and zeroed.
  const char *kbase = reinterpret_cast<const char *>(kc + (size_t)kvh * max_seq * HD);
  const char *vbase = reinterpret_cast<const char *>(vc + (size_t)kvh * max_seq * HD);
  const int kp = tid % kPieces, kr = tid / kPieces;
  const int vq = tid >> 4, vd = (tid & 15) * (HD / 16);
  u32x4 kreg[kKLoads];
  uint32_t vreg[4][kVWords];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kKLoads; ++i) {
      const uint32_t j = (uint32_t)min(k0 + kr + i * kKRows, cap - 1);
      kreg[i] = *reinterpret_cast<const u32x4 *>(kbase + (j * (2 * HD) + 16 * kp));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t j = (uint32_t)min(k0 + 4 * vq + i, cap - 1);
      const char *src = vbase + (j * (2 * HD) + 2 * vd);
      if constexpr (kVWords == 4) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(src);
#pragma unroll
        for (int e = 0; e < 4; ++e) vreg[i][e] = w[e];
      } else {
        const uint2 w = *reinterpret_cast<const uint2 *>(src);
        vreg[i][0] = w.x;
        vreg[i][1] = w.y;
      }
    }
  };
  // Keys 4 vq .. + 3 of a 64-key tile sit in piece 2 (vq >> 2) + (vq & 1), half (vq >> 1) & 1
  // of a V^T row: the lanes hh of product step s then find keys 16 s + 4 hh .. + 3 and
  // 16 s + 8 + 4 hh .. + 3, which are the rows of S^T that they hold, in one 16-byte piece.
  // Rows kr + i * kKRows share kr's swizzle; dims vd + 2 e + o have fa_vx(vd) ^ e.
  const uint32_t kst = kr * (2 * HD) + 16 * (kp ^ fa_kx<HD>(kr));
  const uint32_t vst = kKPlane + vd * (2 * kFaKeys) + 8 * ((vq >> 1) & 1);
  const uint32_t vsx = 16 * ((2 * (vq >> 2) + (vq & 1)) ^ fa_vx(vd));
  auto stage = [&](uint8_t *buf) {
#pragma unroll
    for (int i = 0; i < kKLoads; ++i)
      *reinterpret_cast<u32x4 *>(buf + kst + i * kKRows * (2 * HD)) = kreg[i];
    uint32_t x = vsx;
    asm volatile("" : "+v"(x));
#pragma unroll
    for (int e = 0; e < kVWords; ++e) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const uint32_t sel = o ? 0x07060302u : 0x05040100u;  // high or low halves of two words
        const uint32_t a = __builtin_amdgcn_perm(vreg[1][e], vreg[0][e], sel);
        const uint32_t b = __builtin_amdgcn_perm(vreg[3][e], vreg[2][e], sel);
        *reinterpret_cast<uint2 *>(buf + vst + (x ^ (16 * e)) + (2 * e + o) * (2 * kFaKeys)) = make_uint2(a, b);
      }
    }
  };
  // Operand reads: K row 32 st + li, piece 2 s + hh; V^T row 32 dt + li, piece 2 s + hh.
  const uint32_t krd = li * (2 * HD), krx = 16 * (hh ^ fa_kx<HD>(li));
  const uint32_t vrd = kKPlane + li * (2 * kFaKeys), vrx = 16 * (hh ^ fa_vx(li));
  f32x16 acc[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[dt][v] = 0.0f;
  float m = -INFINITY, l = 0.0f;

  // The first split's first pair of tiles is loaded with q and the position.
  const int split = (int)blockIdx.y;
  if (ROWS == 0 && split == 0) load(kgrp * kFaKeys);
  const int p0 = *pos0;
  const int limit = min(p0 + t + 1, cap);  // keys 0 .. limit - 1 of this lane's row
  const int nkeys = min(p0 + min(row0 + kFaRows - 1, rows - 1) / grp + 1, cap);  // of the last row
  const int first = min(p0 + row0 / grp + 1, cap);                              // of the first row
  uint16_t *orow = out + ((size_t)t * nq + head) * HD;
  if (nkeys <= 0) {  // no key at all (a position below zero: caller error): zeros
    if (split == 0 && kgrp == 0 && r < rows)
      for (int d = hh * 4; d < HD; d += 8) *reinterpret_cast<uint2 *>(orow + d) = make_uint2(0u, 0u);
    return;  // uniform over the workgroup
  }
  // Pairs [it0, it1) are this split's: two at least with one or two pairs in all (32 tokens
  // behind 100 keys: 13.8 us in two splits, 12.3 in one) and from eight (40 behind 1000: 20.8
  // and 19.6), as a split's partial output costs about what a pair does.
  const int npair = (nkeys + 2 * kFaKeys - 1) / (2 * kFaKeys);
  const int per = max(npair <= 2 || npair >= 8 ? 2 : 1, (npair + splits - 1) / splits);
  const int nact = (npair + per - 1) / per;  // splits with work
  if (split >= nact) return;                 // uniform over the workgroup
  const int it0 = split * per, it1 = min(it0 + per, npair);
  const int kend = min(nkeys, it1 * 2 * kFaKeys);
  if (ROWS > 0 || split > 0) load((2 * it0 + kgrp) * kFaKeys);
  bool nonfinite = false;
  if (threadIdx.x == 0) s_nonfinite = 0;  // (the first pair's barrier follows)
  const int nfull = min(max(max(first, 0) / (2 * kFaKeys), it0), it1);
  const bool lone = it1 - it0 == 1 && nfull == it0;
  // One pair of tiles.  EDGE: some row of the workgroup stops inside the pair.
  auto pair = [&](int it, auto edge_c) __attribute__((always_inline)) {
    constexpr bool kEdge = decltype(edge_c)::value;
    int k0 = (2 * it + kgrp) * kFaKeys;
    uint8_t *buf = s_kv[(it - it0) & 1][kgrp];
    uint32_t kx = krx, vx = vrx;
    asm volatile("" : "+v"(kx), "+v"(vx));
    if constexpr (kEdge) {
      // Rows past the last key hold anything: zeros, so that their zero probabilities stay
      // out.  A row that stops early meets V rows that it does not see in the same way: an
      // infinity or NaN among the tile's is noted, and the workgroup starts over below.
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < kVWords; ++e) {
          vreg[i][e] = k0 + 4 * vq + i < kend ? vreg[i][e] : 0u;
          nonfinite |= fa_nonfinite(vreg[i][e]);
        }
    }
    // Plane `buf` was last read two pairs ago, before the previous pair's barrier.
    stage(buf);
    __syncthreads();
    if (it + 1 < it1) load(k0 + 2 * kFaKeys);
    auto tile = [&]() __attribute__((always_inline)) {
      f32x16 sc[2];
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[st][v] = 0.0f;
#pragma unroll
      for (int s = 0; s < HD / 16; ++s) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const u32x4 a = *reinterpret_cast<const u32x4 *>(buf + krd + (kx ^ (32 * s)) + 32 * st * (2 * HD));
          sc[st] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_op(a), fa_op(qf[s]), sc[st], 0, 0, 0);
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          float x = bf16r(bf16r(sc[st][v]) * scaling);
          if constexpr (kEdge) x = k0 + 32 * st + 8 * (v >> 2) + 4 * hh + (v & 3) < limit ? x : -INFINITY;
          sc[st][v] = x;
          mx = fmaxf(mx, x);
        }
      mx = op_xor32<true>(mx);
      const float mn = fmaxf(m, mx);
      // Before a row's first key (none of its keys so far above -inf): any finite reference.
      const float mref = mn == -INFINITY ? 0.0f : mn;
      if (__any(mn > m)) {
        const float alpha = __builtin_amdgcn_exp2f((m - mref) * kLog2e);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[dt][v] *= alpha;
        m = mn;
      }
      u32x4 pf[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int v = 8 * (s & 1) + 2 * j;
          // (The difference first: mref * kLog2e alone overflows from 2.36e38.)
          const float e0 = __builtin_amdgcn_exp2f((sc[s >> 1][v] - mref) * kLog2e);
          const float e1 = __builtin_amdgcn_exp2f((sc[s >> 1][v + 1] - mref) * kLog2e);
          l += e0 + e1;
          pf[s][j] = pack_bf16x2(e0, e1);
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) {
          const u32x4 a = *reinterpret_cast<const u32x4 *>(
              buf + vrd + (vx ^ (16 * ((2 * s) ^ ((2 * dt) & 7)))) + 32 * dt * (2 * kFaKeys));
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_op(a), fa_op(pf[s]), acc[dt], 0, 0, 0);
        }
    };
    if constexpr (!kEdge) {
      tile();
    } else {
      // A workgroup with this one pair: group 0 takes both tiles (nothing to join), else each
      // group its own.
      k0 = (2 * it + (lone ? 0 : kgrp)) * kFaKeys;
      buf = s_kv[(it - it0) & 1][lone ? 0 : kgrp];
#pragma unroll 1
      for (int n = lone ? 2 - 2 * kgrp : 1; n > 0 && k0 < kend; --n) {
        tile();
        k0 += kFaKeys;
        buf += kKPlane + kVPlane;
      }
    }
  };
  // Pairs that every row sees whole, then the (at most two or so) where rows stop: apart, so
  // that the long loop has no masks and keeps all its values in registers.
  for (int it = it0; it < nfull; ++it) pair(it, std::false_type{});
  for (int it = nfull; it < it1; ++it) pair(it, std::true_type{});
  if (nonfinite) s_nonfinite = 1;
  __syncthreads();  // (also the barrier before the planes are reused)
  if (s_nonfinite != 0) {
    // Row by row, a wave per row and a key per lane, so that each row reads the V rows that
    // it sees and no others.
    fa_rows_scalar<HD>(q, kbase, vbase, row0, min(row0 + kFaRows, rows), it0 * 2 * kFaKeys, kend, p0, cap,
                       kvh, grp, nq, scaling, reinterpret_cast<float *>(&s_kv[0][0][0]), (int)threadIdx.x);
    __syncthreads();
    fa_load_row<HD>(reinterpret_cast<float *>(&s_kv[0][0][0]), wave * 32 + li, hh, acc, m, l);
    __syncthreads();
    if (kgrp == 1) {
      m = -INFINITY;
      l = 0.0f;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = 0.0f;
    }
  } else {
    l = op_xor32<false>(l);
  }
  // Key group 1's maxima, sums and output join group 0's through LDS, four words of a lane at
  // [row group][quad][lane].
  if (!lone) {
    float4 *const s_o = reinterpret_cast<float4 *>(&s_kv[0][0][0]);
    static_assert(4 * (4 * kDT + 1) * kWave * 16 <= (int)sizeof(s_kv), "partial outputs fit the planes");
    float4 *const mine = s_o + wave * (4 * kDT + 1) * kWave + lane;
    if (kgrp == 1) {
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; v += 4)
          mine[(4 * dt + v / 4) * kWave] = make_float4(acc[dt][v], acc[dt][v + 1], acc[dt][v + 2], acc[dt][v + 3]);
      mine[4 * kDT * kWave] = make_float4(m, l, 0.0f, 0.0f);
    }
    __syncthreads();
    // From here on key group 1's waves only keep the barriers.
    if (kgrp == 0) {
      const float4 ml = mine[4 * kDT * kWave];
      const float mn = fmaxf(m, ml.x);
      const float mref = mn == -INFINITY ? 0.0f : mn;
      const float a0 = __builtin_amdgcn_exp2f((m - mref) * kLog2e);
      const float a1 = __builtin_amdgcn_exp2f((ml.x - mref) * kLog2e);
      m = mn;
      l = l * a0 + ml.y * a1;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
          const float4 o = mine[(4 * dt + v / 4) * kWave];
          acc[dt][v] = acc[dt][v] * a0 + o.x * a1;
          acc[dt][v + 1] = acc[dt][v + 1] * a0 + o.y * a1;
          acc[dt][v + 2] = acc[dt][v + 2] * a0 + o.z * a1;
          acc[dt][v + 3] = acc[dt][v + 3] * a0 + o.w * a1;
        }
    }
  }
  if (nact > 1) {
    // Partial results to the workspace, word w of a lane at [w][lane] of its wave's block;
    // the split that finishes a row tile last adds them up, in split order whichever it is
    // (its own too is read back), and writes the rows.
    constexpr int kWords = (16 * kDT + 2) * kWave;
    const int unit = (int)blockIdx.x;
    float *const pu = part + ((size_t)unit * splits * 4 + wave) * kWords + lane;
    const bool live = kgrp == 0 && row0 + wave * 32 < rows;  // waves without rows have nothing
    if (live) {
      float *const pw = pu + (size_t)split * 4 * kWords;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) attn_put(pw + (16 * dt + v) * kWave, acc[dt][v]);
      attn_put(pw + 16 * kDT * kWave, m);
      attn_put(pw + (16 * kDT + 1) * kWave, l);
    }
    if (!attn_last_of(count + unit, nact)) return;  // uniform over the workgroup
    if (!live) return;
    m = -INFINITY;
    l = 0.0f;
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[dt][v] = 0.0f;
    for (int y = 0; y < nact; ++y) {
      const float *pw = pu + (size_t)y * 4 * kWords;
      const float m1 = attn_get(pw + 16 * kDT * kWave), l1 = attn_get(pw + (16 * kDT + 1) * kWave);
      const float mn = fmaxf(m, m1);
      const float mref = mn == -INFINITY ? 0.0f : mn;
      const float a0 = __builtin_amdgcn_exp2f((m - mref) * kLog2e);
      const float a1 = __builtin_amdgcn_exp2f((m1 - mref) * kLog2e);
      m = mn;
      l = l * a0 + l1 * a1;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = acc[dt][v] * a0 + attn_get(pw + (16 * dt + v) * kWave) * a1;
    }
  }
  if (kgrp == 0 && r < rows) {
    const float inv = limit > 0 ? 1.0f / l : 0.0f;
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; v += 4)
        *reinterpret_cast<uint2 *>(orow + 32 * dt + 2 * v + 4 * hh) =
            make_uint2(pack_bf16x2(acc[dt][v] * inv, acc[dt][v + 1] * inv),
                       pack_bf16x2(acc[dt][v + 2] * inv, acc[dt][v + 3] * inv));
  }
}

}  // namespace
}  // namespace moe

namespace moe {
namespace {

constexpr int64_t kAttnCounterBytes = 4096;  // arrival counters at the start of the workspace
constexpr int64_t kAttnUnitsMax = kAttnCounterBytes / 4;

// Launch plan of a call: which kernel, its splits of the keys, and the workspace it needs.
struct AttnPlan {
  bool matrix;     // prefill_attention_kernel
  int rows;        // its instance that takes short contexts by rows (heads a unit; 0: none)
  int64_t units;   // workgroups per split
  int splits;
  int64_t bytes;   // workspace (0: none)
};

AttnPlan attn_plan(int64_t T, int32_t nq, int32_t nkv, int32_t hd, int64_t max_seq, bool ws) {
  AttnPlan p{false, 0, nq, 1, 0};
  const int64_t rows = T * (nq / nkv);
  const int64_t fit = 2 * (int64_t)device_cu_count();  // (head, token) units at a time
  // Without a workspace no keys are shared, and a row tile's one workgroup has a longer chain
  // than the rows' own while those run all at once (9 tokens behind 1000 keys: 26 us, 22 with a
  // workgroup per row; 8 heads of 64, 16 tokens: 20 and 11; 64 tokens of 32 heads: 30 and 75).
  if (T > kFewTokens && (hd == 64 || hd == 128) && (ws || nq * T > fit)) {
    p.matrix = true;
    p.rows = nq * T <= fit ? 1 : nq / nkv % 2 == 0 && nq / 2 * T <= fit ? 2 : 0;
    p.units = (rows + kFaRows - 1) / kFaRows * nkv;
    // Row tiles alone do not fill the chip: share a tile's keys, down to two pairs of key
    // tiles per split.
    if (ws && p.units <= device_cu_count() / 2 && p.units <= kAttnUnitsMax) {
      const int64_t s = device_cu_count() / p.units;
      const int64_t most = (max_seq + 4 * kFaKeys - 1) / (4 * kFaKeys);
      p.splits = (int)(s < most ? s : most);
      if (p.splits > 1) p.bytes = kAttnCounterBytes + p.units * p.splits * 4 * (hd / 2 + 2) * kWave * 4;
    }
  } else if (T <= kFewTokens && ws && max_seq > kFewWhole && (hd == 64 || hd == 128 || hd == 256)) {
    // Two workgroups per CU: those that leave at once behind a short context cost 0.25 us (half as
    // many splits 0.2, and 12.3 instead of 11.8 us behind 3000 keys).
    const int64_t pass = kAttnRowsInFlight * (kAttnThreads / (hd / 8));
    const int64_t most = (max_seq + pass - 1) / pass;
    int64_t s = 2 * (int64_t)device_cu_count() / (nq * T);
    s = s < most ? s : most;
    p.splits = (int)(s < 1 ? 1 : s < kFewSplits ? s : kFewSplits);
    if (nq * T > kAttnUnitsMax) p.splits = 1;
    if (p.splits > 1) p.bytes = kAttnCounterBytes + nq * T * p.splits * (hd + 2) * 4;
  }
  return p;
}

bool attn_sizes_ok(int64_t T, int32_t nq, int32_t nkv, int32_t hd, int64_t max_seq) {
  return T >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0 && hd > 0 && hd <= kAttnMaxHeadDim &&
         kAttnThreads % hd == 0 && hd % 8 == 0 && max_seq > 0 && max_seq <= kAttnMaxKeys;
}

}  // namespace
}  // namespace moe

extern "C" int64_t moe_attention_workspace_bytes(int64_t T, int32_t n_q_heads, int32_t n_kv_heads,
                                                 int32_t head_dim, int64_t max_seq) {
  if (!moe::attn_sizes_ok(T, n_q_heads, n_kv_heads, head_dim, max_seq)) return -1;
  if (T == 0) return 0;
  int64_t most = 0;
  auto take = [&](int64_t t) {
    const int64_t b = moe::attn_plan(t, n_q_heads, n_kv_heads, head_dim, max_seq, true).bytes;
    most = b > most ? b : most;
  };
  for (int64_t t = 1; t <= T && t <= moe::kFewTokens; ++t) take(t);
  // More tokens: the plan depends on the row tiles only, and only few of them split.
  const int32_t grp = n_q_heads / n_kv_heads;
  for (int64_t tiles = 1; tiles * n_kv_heads <= moe::device_cu_count() / 2; ++tiles) {
    const int64_t t = (tiles - 1) * moe::kFaRows / grp + 1;  // the fewest tokens with these tiles
    const int64_t tt = t > moe::kFewTokens ? t : moe::kFewTokens + 1;
    if (tt <= T) take(tt);
  }
  return most;
}

extern "C" int moe_attention_ws_bf16(const void *q, const void *k_cache, const void *v_cache,
                                     int64_t T, int32_t n_q_heads, int32_t n_kv_heads,
                                     int32_t head_dim, const void *pos0_i32, int64_t max_seq,
                                     float scaling, void *out, void *workspace,
                                     int64_t workspace_bytes, void *stream) {
  MOE_REQUIRE(T >= 0 && n_q_heads > 0 && n_kv_heads > 0 && n_q_heads % n_kv_heads == 0,
              "query heads must be a multiple of the KV heads");
  MOE_REQUIRE(head_dim > 0 && head_dim <= moe::kAttnMaxHeadDim && moe::kAttnThreads % head_dim == 0 &&
                  head_dim % 8 == 0,
              "head dim must divide %d and be a multiple of 8 (got %d)", moe::kAttnThreads, head_dim);
  MOE_REQUIRE(max_seq > 0 && max_seq <= moe::kAttnMaxKeys, "max_seq must be in [1, %d]",
              moe::kAttnMaxKeys);
  if (T == 0) return MOE_STATUS_OK;
  MOE_REQUIRE(q && k_cache && v_cache && pos0_i32 && out, "null pointer");
  MOE_REQUIRE(((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0,
              "q and the KV cache must be 16-byte aligned");
  moe::AttnPlan p = moe::attn_plan(T, n_q_heads, n_kv_heads, head_dim, max_seq, workspace != nullptr);
  if (workspace != nullptr) {
    MOE_REQUIRE(workspace_bytes >= p.bytes, "workspace too small: need %lld bytes, got %lld",
                (long long)p.bytes, (long long)workspace_bytes);
    MOE_REQUIRE((uintptr_t)workspace % 16 == 0, "workspace must be 16-byte aligned");
  }
  hipStream_t s = (hipStream_t)stream;
  const uint16_t *qp = (const uint16_t *)q, *kp = (const uint16_t *)k_cache, *vp = (const uint16_t *)v_cache;
  const int32_t *pp = (const int32_t *)pos0_i32;
  uint16_t *op = (uint16_t *)out;
  uint32_t *count = (uint32_t *)workspace;
  float *part = workspace ? (float *)((char *)workspace + moe::kAttnCounterBytes) : nullptr;
  // The matrix form's 8-byte stores need `out` aligned, its row index 31 bits.
  const bool matrix = p.matrix && (uintptr_t)out % 8 == 0 &&
                      T * (int64_t)(n_q_heads / n_kv_heads) <= 0x7fffffff - moe::kFaRows && p.units <= 0x7fffffff;
  if (matrix) {
    auto kern = head_dim == 64 ? (p.rows == 0   ? moe::prefill_attention_kernel<64, 0>
                                  : p.rows == 1 ? moe::prefill_attention_kernel<64, 1>
                                                : moe::prefill_attention_kernel<64, 2>)
                               : (p.rows == 0   ? moe::prefill_attention_kernel<128, 0>
                                  : p.rows == 1 ? moe::prefill_attention_kernel<128, 1>
                                                : moe::prefill_attention_kernel<128, 2>);
    // The row instances: a workgroup for every two units at least.
    const int64_t row_wgs = p.rows > 0 ? (n_q_heads / p.rows * T + 1) / 2 : 0;
    const int64_t row_y = (row_wgs + p.units - 1) / p.units;
    const unsigned y = (unsigned)(row_y > p.splits ? row_y : p.splits);
    hipLaunchKernelGGL(kern, dim3((unsigned)p.units, y), dim3(moe::kFaThreads), 0, s, qp, kp, vp, (int)T,
                       n_q_heads, n_kv_heads, pp, max_seq, scaling, op, count, part, p.splits);
  } else if (!p.matrix && p.splits > 1) {
    // grp = nq / nkv and x / nkv = (x * over_nkv) >> 31 (exact: x < nq <= kAttnUnitsMax), so that
    // no division stands before the kernel's first loads.
    const uint32_t over_nkv = (uint32_t)((((int64_t)1 << 31) + n_kv_heads - 1) / n_kv_heads);
    hipLaunchKernelGGL(moe::few_attention_kernel, dim3((unsigned)n_q_heads, (unsigned)T, (unsigned)p.splits),
                       dim3(moe::kAttnThreads), 0, s, qp, kp, vp, n_q_heads, n_kv_heads,
                       n_q_heads / n_kv_heads, over_nkv, head_dim, pp, max_seq, scaling, op, count, part);
  } else {
    hipLaunchKernelGGL(moe::attention_kernel, dim3((unsigned)n_q_heads, (unsigned)T),
                       dim3(moe::kAttnThreads), 0, s, qp, kp, vp, n_q_heads, n_kv_heads, head_dim, pp,
                       max_seq, scaling, op);
  }
  MOE_LAUNCH_CHECK();
  return MOE_STATUS_OK;
}

extern "C" int moe_attention_bf16(const void *q, const void *k_cache, const void *v_cache, int64_t T,
                                  int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                                  const void *pos0_i32, int64_t max_seq, float scaling, void *out,
                                  void *stream) {
  return moe_attention_ws_bf16(q, k_cache, v_cache, T, n_q_heads, n_kv_heads, head_dim, pos0_i32, max_seq,
                               scaling, out, nullptr, 0, stream);
}
