// Similarities and top-k for few queries: one streaming pass over the
// documents, no score matrix.
//
// Bound: reading the documents (4 d bytes each) from HBM. Before, a call ran
// the fp32-MFMA product on 64-row tiles (one query cost what 64 do, 109 us
// for 100 000 x 768), wrote the scores and selected from them in two more
// passes (40 + 10 us). Here a wave takes 16 documents against up to 32 queries
// (QB column blocks of v_mfma_f32_16x16x4_f32) with its document values loaded
// from global memory straight into operand registers, two groups of eight
// 16-byte loads in flight per lane; the queries sit in LDS. Every workgroup
// keeps its documents' scores in LDS and reduces them to its best k per
// query by rank counting (a serial argmax per result took 1 us each); a
// second kernel merges those. 100 000 x 768, one query, top 10:
// 148 -> 75 us per call (62 us at the rate of a large copy); 16 queries 155
// -> 83, 32 queries 160 -> 130; 1 000 x 768, one query: 38 -> 12.
//
// Sums: four consecutive k per MFMA group, two accumulators (even and odd
// 16-wide steps) added at the end. Order: (score descending, index
// ascending); NaN is never selected, slots past the non-NaN scores get index
// -1 and value NaN.
#include <algorithm>
#include <cstdint>

#include "fa_internal.h"
#include "device_math.h"

namespace fa {
namespace {

constexpr int kFewSteps = 8;    // 16-wide steps per load group
constexpr int kFewMaxDocs = 128;  // documents per workgroup, at most: a 16-row block for each wave

struct FewParams {
  const float* q;     // [nq x d]
  const float* docs;  // [nd x d]
  int64_t nd;
  int d, nq, per, k;  // per: documents per workgroup (16 per wave and round)
  uint2* cand;        // candidates (key, index) [nq][workgroups][k]
};

// Orders floats as unsigned integers; 0 for NaN (below every number).
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t u = __float_as_uint(v + 0.f);  // -0 -> +0
  return v != v ? 0u : (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k ^ 0x80000000u : ~k);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
// Largest value over the wave, in every lane (the butterfly of wave_sum).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  v = max((uint32_t)a[0], (uint32_t)a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max((uint32_t)b[0], (uint32_t)b[1]);
  v = max(v, dpp_u32<0x128>(v));
  v = max(v, dpp_u32<0x124>(v));
  v = max(v, dpp_u32<0x122>(v));
  v = max(v, dpp_u32<0x121>(v));
  return v;
}

// Rank of entry i among the first n of keys (LDS, padded to whole groups of
// four with zeros): the entries before it in the order (key descending,
// position ascending). No chain between entries.
__device__ __forceinline__ int rank_of(const uint32_t* keys, int n, int i, uint32_t key) {
  int r = 0;
  for (int j = 0; j < n; j += 4) {
    const uint4 v = *reinterpret_cast<const uint4*>(keys + j);
    // an equal key ranks before only at a lower position: v + 1 > key (no key is ~0)
    r += v.x + (j < i ? 1u : 0u) > key;
    r += v.y + (j + 1 < i ? 1u : 0u) > key;
    r += v.z + (j + 2 < i ? 1u : 0u) > key;
    r += v.w + (j + 3 < i ? 1u : 0u) > key;
  }
  return r;
}

// A value that at least k of the 64 lanes' m reach and few more: the least m
// with fewer than k greater ones. sm: 64 words of LDS of the wave's own.
__device__ __forceinline__ uint32_t kth_of_lanes(uint32_t m, int k, int lane, uint32_t* sm) {
  sm[lane] = m;
  __builtin_amdgcn_wave_barrier();
  int above = 0;
#pragma unroll
  for (int j = 0; j < 64; j += 4) {
    const uint4 v = *reinterpret_cast<const uint4*>(sm + j);
    above += (v.x > m) + (v.y > m) + (v.z > m) + (v.w > m);
  }
  __builtin_amdgcn_wave_barrier();
  return ~wave_max_u32(above < k ? ~m : 0u);
}

template <int QB>
__global__ __launch_bounds__(512) void score_few_kernel(FewParams p) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int waves = 8;
  const int lq = lane & 15, g = lane >> 4;
  const int d = p.d, ldq = d + 4;  // rows four banks apart
  // documents in blocks of 16 per wave; with fewer than 128 per workgroup KW
  // waves share a block, each a part of K
  const int KW = kFewMaxDocs / p.per;
  constexpr int sst = kFewMaxDocs + 4;  // score rows: KW parts of `per` documents
  float* qs = sm;
  float* sc = sm + (int64_t)p.nq * ldq;
  uint2* out = reinterpret_cast<uint2*>(sc + (int64_t)p.nq * sst);  // [nq][k] (key, index)
  for (int i = threadIdx.x; i < p.nq * (d / 4); i += blockDim.x) {
    const int r = i / (d / 4), c = i - r * (d / 4);
    *reinterpret_cast<f32x4*>(qs + r * ldq + 4 * c) = *reinterpret_cast<const f32x4*>(p.q + (int64_t)r * d + 4 * c);
  }
  for (int i = threadIdx.x; i < p.nq * p.k; i += blockDim.x) out[i] = make_uint2(0u, 0x7FFFFFFFu);
  const int64_t r0 = (int64_t)blockIdx.x * p.per;
  const int n = (int)min((int64_t)p.per, p.nd - r0);
  const int nb = (n + 15) / 16;
  const int kw = wave % KW, bw = wave / KW, bstep = waves / KW;
  const int mine = nb > bw ? (nb - bw + bstep - 1) / bstep : 0;  // blocks bw, bw + bstep, ...
  const int all = d / 16, s_lo = kw * all / KW, steps = (kw + 1) * all / KW - s_lo;
  const int groups = (steps + kFewSteps - 1) / kFewSteps;
  const int total = mine * groups;
  // group t of the wave: steps [8 gi, 8 gi + 8) of its part of block t /
  // groups (steps past the part's end repeat its last one; their products
  // are skipped)
  auto load = [&](f32x4 (&a)[kFewSteps], int t) {
    const int b = t / groups, gi = t - b * groups;
    const float* row = p.docs + min(r0 + 16 * (bw + b * bstep) + lq, p.nd - 1) * d + 16 * s_lo + 4 * g;
#pragma unroll
    for (int u = 0; u < kFewSteps; u++)
      a[u] = *reinterpret_cast<const f32x4*>(row + 16 * min(gi * kFewSteps + u, steps - 1));
  };
  // queries past nq repeat the last one (their results are not used)
  const float* qrow[QB];
#pragma unroll
  for (int j = 0; j < QB; j++) qrow[j] = qs + min(16 * j + lq, p.nq - 1) * ldq + 16 * s_lo + 4 * g;
  f32x4 acc[QB][2];
  auto compute = [&](const f32x4 (&a)[kFewSteps], int t) {
    const int b = t / groups, gi = t - b * groups;
    if (gi == 0) {
#pragma unroll
      for (int j = 0; j < QB; j++) acc[j][0] = acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kFewSteps; u++) {
      const int s = gi * kFewSteps + u;
      if (s < steps) {
#pragma unroll
        for (int j = 0; j < QB; j++) {
          const f32x4 bq = *reinterpret_cast<const f32x4*>(qrow[j] + 16 * s);
#pragma unroll
          for (int c = 0; c < 4; c++)
            acc[j][u & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][c], bq[c], acc[j][u & 1], 0, 0, 0);
        }
      }
    }
    if (gi == groups - 1) {  // lane: query lq, documents 4g .. 4g + 3 of the block
#pragma unroll
      for (int j = 0; j < QB; j++)
        if (16 * j + lq < p.nq)
          *reinterpret_cast<f32x4*>(sc + (16 * j + lq) * sst + kw * p.per + 16 * (bw + b * bstep) + 4 * g) =
              acc[j][0] + acc[j][1];
    }
  };
  f32x4 a0[kFewSteps], a1[kFewSteps];
  if (total > 0) load(a0, 0);
  __syncthreads();  // the queries are in LDS
  for (int t = 0; t < total; t += 2) {
    load(a1, min(t + 1, total - 1));
    compute(a0, t);
    load(a0, min(t + 2, total - 1));
    if (t + 1 < total) compute(a1, t + 1);
  }
  if (KW > 1 && total == 0) {  // a part of K without steps, or no block: zero partials
    for (int b = bw; b < nb; b += bstep)
      for (int q = 0; q < p.nq; q++)
        if (lane < 16) sc[q * sst + kw * p.per + 16 * b + lane] = 0.f;
  }
  __syncthreads();
  // keys in place of the (summed) scores, zeros up to whole groups of four
  uint32_t* keys = reinterpret_cast<uint32_t*>(sc);
  for (int q0 = 0; q0 < p.nq; q0 += 4) {
    const int q = q0 + (threadIdx.x >> 7), j = threadIdx.x & 127;
    float v = 0.f;
    if (q < p.nq && j < n) {
      v = sc[q * sst + j];
      for (int w = 1; w < KW; w++) v += sc[q * sst + w * p.per + j];
    }
    __syncthreads();  // a part's place may be another thread's to write
    if (q < p.nq) keys[q * sst + j] = j < n ? order_key(v) : 0u;
  }
  __syncthreads();
  // queries over the waves: two documents per lane, a bound from the lanes'
  // better ones, the documents from it on (about k) packed and ranked
  __shared__ __attribute__((aligned(16))) uint32_t pack[waves][kFewMaxDocs];
  for (int q = wave; q < p.nq; q += waves) {
    const uint32_t k0 = keys[q * sst + lane], k1 = keys[q * sst + 64 + lane];
    const uint32_t bound = max(1u, kth_of_lanes(max(k0, k1), p.k, lane, pack[wave]));
    const uint64_t b0 = __ballot(k0 >= bound), b1 = __ballot(k1 >= bound);
    const int c0 = __popcll(b0), m = c0 + __popcll(b1);
    const uint64_t below = (1ull << lane) - 1;
    const int p0 = __popcll(b0 & below), p1 = c0 + __popcll(b1 & below);
    pack[wave][lane] = 0;
    pack[wave][64 + lane] = 0;
    __builtin_amdgcn_wave_barrier();
    if (k0 >= bound) pack[wave][p0] = k0;
    if (k1 >= bound) pack[wave][p1] = k1;
    __builtin_amdgcn_wave_barrier();
    if (k0 >= bound) {
      const int r = rank_of(pack[wave], m, p0, k0);
      if (r < p.k) out[q * p.k + r] = make_uint2(k0, (uint32_t)(r0 + lane));
    }
    if (k1 >= bound) {
      const int r = rank_of(pack[wave], m, p1, k1);
      if (r < p.k) out[q * p.k + r] = make_uint2(k1, (uint32_t)(r0 + 64 + lane));
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  for (int i = threadIdx.x; i < p.nq * p.k; i += blockDim.x) {
    const int q = i / p.k, r = i - q * p.k;
    p.cand[((int64_t)q * gridDim.x + blockIdx.x) * p.k + r] = out[i];
  }
}

// One workgroup per query: the best k of its nc candidates (key, index). The
// 64 maxima over the lanes' columns of candidates give a bound: their k-th
// largest is at most the k-th of all, so only candidates from it on (about k
// of them) are kept in LDS and ranked there. More than kFewKeep of them (many
// equal scores) are taken one at a time instead.
constexpr int kFewMergeWaves = 16, kFewKeep = 1024;
__global__ __launch_bounds__(64 * kFewMergeWaves) void score_few_merge_kernel(const uint2* __restrict__ cand, int nc,
                                                                              int k, int32_t* __restrict__ oidx,
                                                                              float* __restrict__ oval) {
  __shared__ uint32_t colmax[kFewMergeWaves][64];
  __shared__ __attribute__((aligned(16))) uint32_t lanes[64];
  __shared__ __attribute__((aligned(16))) uint64_t kept[kFewKeep];  // key, ~index
  __shared__ uint32_t wkey[kFewMergeWaves], widx[kFewMergeWaves];
  __shared__ uint32_t bound, count;
  constexpr int N = 8, NT = 64 * kFewMergeWaves;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint2* cq = cand + (int64_t)blockIdx.x * nc;
  uint2 mine[N];  // the first N * NT candidates stay in registers
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < N; i++) {
    mine[i] = i * NT + tid < nc ? cq[i * NT + tid] : make_uint2(0u, 0u);
    m = max(m, mine[i].x);
  }
  for (int c = N * NT + tid; c < nc; c += NT) m = max(m, cq[c].x);
  // (columns turned per wave: a candidate list has its best entries at every
  // k-th place)
  colmax[wave][(lane + 5 * wave) & 63] = m;
  if (tid == 0) count = 0;
  if (tid < k) {
    oidx[(int64_t)blockIdx.x * k + tid] = -1;
    if (oval) oval[(int64_t)blockIdx.x * k + tid] = NAN;
  }
  __syncthreads();
  if (wave == 0) {
    m = colmax[0][lane];
#pragma unroll
    for (int w = 1; w < kFewMergeWaves; w++) m = max(m, colmax[w][lane]);
    m = kth_of_lanes(m, k, lane, lanes);
    if (lane == 0) bound = m;
  }
  __syncthreads();
  const uint32_t lo = max(bound, 1u);
  auto keep = [&](uint2 v) {
    if (v.x >= lo) {
      const uint32_t at = atomicAdd(&count, 1u);
      if (at < kFewKeep) kept[at] = (uint64_t)v.x << 32 | (uint32_t)~v.y;
    }
  };
#pragma unroll
  for (int i = 0; i < N; i++) keep(mine[i]);
  for (int c = N * NT + tid; c < nc; c += NT) keep(cq[c]);
  __syncthreads();
  const int n = (int)count;
  if (n <= kFewKeep) {
    // ranked by (key, index) themselves: the order in which they were kept varies
    if (tid < n) {
      const uint64_t e = kept[tid];
      int r = 0;
#pragma unroll 8
      for (int j = 0; j < n; j++) r += kept[j] > e;
      if (r < k) {
        oidx[(int64_t)blockIdx.x * k + r] = (int32_t)~(uint32_t)e;
        if (oval) oval[(int64_t)blockIdx.x * k + r] = key_value((uint32_t)(e >> 32));
      }
    }
    return;
  }
  // one at a time: the best candidate after the last one taken
  uint32_t lk = 0xFFFFFFFFu;
  int32_t li = -1;
  for (int r = 0; r < k; r++) {
    uint32_t bk = 0;
    uint32_t bi = 0;  // ~index
    for (int c = tid; c < nc; c += NT) {
      const uint2 v = cq[c];
      if (v.x == 0 || v.x > lk || (v.x == lk && (int32_t)v.y <= li)) continue;
      if (v.x > bk || (v.x == bk && ~v.y > bi)) {
        bk = v.x;
        bi = ~v.y;
      }
    }
    const uint32_t wk = wave_max_u32(bk), wi = wave_max_u32(bk == wk ? bi : 0u);
    if (lane == 0) {
      wkey[wave] = wk;
      widx[wave] = wi;
    }
    __syncthreads();
    bk = 0;
    bi = 0;
    for (int w = 0; w < kFewMergeWaves; w++)
      if (wkey[w] > bk || (wkey[w] == bk && widx[w] > bi)) {
        bk = wkey[w];
        bi = widx[w];
      }
    __syncthreads();
    if (bk == 0) return;
    lk = bk;
    li = (int32_t)~bi;
    if (tid == 0) {
      oidx[(int64_t)blockIdx.x * k + r] = li;
      if (oval) oval[(int64_t)blockIdx.x * k + r] = key_value(bk);
    }
  }
}

// Documents per workgroup: the fewest of 16, 32, 64 and 128 that leave at most
// about four workgroups per CU, so that a small corpus still spreads over the
// CUs; from 65 537 documents on 128, a whole block for each wave, and the
// workgroups (and the candidates of the merge) grow with the corpus.
int few_docs(int64_t nd) {
  int per = 16;
  while (per < kFewMaxDocs && (nd + per - 1) / per > 1024) per *= 2;
  return per;
}

size_t few_lds(int nq, int d, int k) { return (size_t)nq * (((size_t)d + 4 + kFewMaxDocs + 4) * 4 + (size_t)k * 8); }

}  // namespace

// Where the streaming pass is not the faster one, though it could run: its
// merge reads the candidates, k of every 128 documents, with one workgroup per
// query (0.5 to 1.5 us per thousand, more with more queries), which rows of at
// least 256 columns hide behind their own bytes; and more than 16 queries
// against a handful of documents pay for a second query block. Us, product and
// streaming: 2 000 000 x 64, 32 queries, k = 32: 528 and 1 014; the same of one
// query: 483 and 533, k = 1: 396 and 335; 500 000 x 64, 16 queries, k = 32: 205 and
// 172, 32 queries: 211 and 235; 6 000 000 x 16, 16 queries, k = 10: 970 and 1 044;
// 2 000 000 x 128, 32 queries, k = 10: 701 and 650, k = 32: 770 and 1 072; 500 000 x
// 256, 32 queries, k = 32: 410 and 288; 50 x 128, 32 queries, k = 1: 15 and 19,
// k = 10: 19 and 20, 300 documents, k = 10: 27 and 21.
static bool score_few_pays(int64_t nq, int64_t nd, int d, int topk) {
  if (nq >= 16 && topk < 4 && nd < 256 && d < 512) return false;
  const int64_t cands = (nd + kFewMaxDocs - 1) / kFewMaxDocs * topk;
  return d >= 256 || cands <= (d >= 128 ? 200000 : nq <= 16 ? 128000 : 40000);
}

bool score_few_ok(const float* q, int64_t nq, const float* docs, int64_t nd, int d, int topk) {
  return nq >= 1 && nq <= kScoreFewMax && topk >= 1 && topk <= 32 && d % 16 == 0 &&
         ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(docs)) & 15) == 0 &&
         few_lds((int)nq, d, topk) <= 150 * 1024 &&
         (nd + kFewMaxDocs - 1) / kFewMaxDocs * topk < (1LL << 30) && nd <= INT32_MAX &&
         score_few_pays(nq, nd, d, topk);
}

size_t score_few_scratch(int64_t nq, int64_t nd, int topk) {
  const int per = few_docs(nd);
  return (size_t)nq * ((nd + per - 1) / per) * topk * 8;
}

int launch_score_few(fa_ctx* ctx, const float* q, int64_t nq, const float* docs, int64_t nd, int d, int topk,
                     int32_t* idx, float* val, void* scratch, hipStream_t s) {
  if (!score_few_ok(q, nq, docs, nd, d, topk))
    return set_error(ctx, FA_ERR_ARG, "Similarities: %lld queries x %lld x %d, k=%d not for the streaming kernel",
                     (long long)nq, (long long)nd, d, topk);
  const int per = few_docs(nd);
  const int64_t nwg = (nd + per - 1) / per;
  FewParams p;
  p.q = q; p.docs = docs; p.nd = nd; p.d = d; p.nq = (int)nq;
  p.per = per; p.k = topk;
  p.cand = static_cast<uint2*>(scratch);
  const size_t lds = few_lds(p.nq, d, topk);
  if (nq <= 16)
    hipLaunchKernelGGL(score_few_kernel<1>, dim3((unsigned)nwg), dim3(512), lds, s, p);
  else
    hipLaunchKernelGGL(score_few_kernel<2>, dim3((unsigned)nwg), dim3(512), lds, s, p);
  hipLaunchKernelGGL(score_few_merge_kernel, dim3((unsigned)nq), dim3(64 * kFewMergeWaves), 0, s, p.cand,
                     (int)(nwg * topk), topk, idx, val);
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

}  // namespace fa
