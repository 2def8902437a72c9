// The tensor.AttentionScaled drop-in at head_dim 64, 128 and 256 on the 16-bit
// MFMA with fp32 accuracy, for any operands: attention_dense_kernel
// (attention.hip) runs the same products on the fp32 MFMA, a sixteenth of
// that rate, and stays for small calls, few queries and head_dim 512
// (attention_split_pays). 8 x 8 heads x 512 x 512, head_dim 64: 55 -> 36 us per call
// (10 of them the image pass); 32 x 3 x 256 x 256 on one kv head, head_dim 256, padded:
// 95 -> 65. What bounds it now: at head_dim 64 the MFMAs (busy 0.45 of the time)
// and the softmax between them; at 256 one workgroup per CU, two waves per SIMD
// that wait half their cycles at the two barriers of a stage (MFMAs busy 0.25).
// The error against float64 is below the fp32 kernel's (5.0e-7 -> 3.7e-7 and 3.6e-7
// -> 2.5e-7), whose sums take more roundings.
//
// Queries, keys, values and probabilities are three exact bf16 terms each
// (split8), a product the six MFMAs whose terms' orders add up to at most two
// (what is dropped, mid . lo and lo . lo, is below 2^-25 of the product). bf16 has
// float32's range, so elements of one row may be of any magnitude beside each
// other, and a masked key may hold any finite value without touching its
// neighbours. (Two fp16 terms for the scores, scaled by a power of two per
// row, took three MFMAs but lost the small elements of a row beside a large one.)
//
// split_kv_kernel writes, per (batch, kv head, tile of 32 keys), a key image
// [term][key][HD] and a value image [term][dim][32 slots], in the order in
// which the attention's direct global->LDS loads and operand reads take them:
// 16-byte chunk c of key k at c ^ (k mod 16) (head_dim 64: c ^ (k / 2 mod 8)), slot 8g + 4h + r of a dim holding key 16h + 4g + r,
// chunk g of dim d at g ^ (d / 2 mod 4), both free of bank conflicts (d / 4 mod 4
// had a third of the value reads in conflict). Heads that share one key/value
// head share its images.
//
// attention_split_kernel: a workgroup of W waves takes 16 W queries of one
// (batch, head), a wave 16 (v_mfma_f32_16x16x32): S^T = K . Q^T puts a query's
// scores in the four lanes that share l % 16, and its probabilities are then
// the B operand of O^T += V^T . P^T as they are. Per stage of SK keys (64 at
// head_dim 64): [barrier: this stage's keys and the previous stage's values
// landed] load this stage's values and the next keys (with one key buffer they
// load after a second barrier: head_dim 256 has room for no more, and four-wave
// workgroups of the others fit a CU twice with one); scores; P.V of the previous
// stage; softmax. P.V one stage behind leaves the values a whole stage to land
// (2 048 queries and keys, 3 heads of 256: 211 -> 192 us per call). The row maximum
// is lazy: the offset moves when a stage's maximum exceeds it by more than 8.
#include <algorithm>
#include <cstdlib>

#include "fa_internal.h"
#include "device_math.h"

namespace fa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitTau = 8.f;

template <int HD>
__device__ __forceinline__ int key_chunk(int key, int c) {
  return HD == 64 ? c ^ ((key >> 1) & 7) : c ^ (key & 15);
}
__device__ __forceinline__ int slot_chunk(int dim, int g) { return g ^ ((dim >> 1) & 3); }

// Eight values as three bf16 terms, each packed as the 16 bytes it takes in an
// image or an operand: hi the nearest bf16, mid that of the rest, lo the rest
// of that, both rests exact in float32 and lo in bf16. Rounded terms leave
// signed rests of half the size that cut ones (split3) leave: the dropped
// products are a sixteenth of theirs and carry no bias.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&t)[3]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f32x2 r = {x[2 * i], x[2 * i + 1]};
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
      t[j][i] = w;
      r.x -= __uint_as_float(w << 16);
      r.y -= __uint_as_float(w & 0xFFFF0000u);
    }
  }
}

struct SplitKvParams {
  const float *k, *v;
  int64_t k_sb, k_sh, v_sb, v_sh;
  int Hk, S, tiles;  // kv heads with images of their own; tiles per (batch, kv head)
  uint16_t *kimg, *vimg;
};

template <int HD>
__global__ __launch_bounds__(256) void split_kv_kernel(SplitKvParams p) {
  constexpr int VST = HD + 4;
  __shared__ __attribute__((aligned(16))) float Vt[32 * VST];
  const int64_t at = blockIdx.x;  // (batch * Hk + kv head) * tiles + tile
  const int64_t bh = at / p.tiles;
  const int t0 = (int)(at - bh * p.tiles) * 32, n = p.S - t0;  // n <= 0: a padding tile
  const int b = (int)(bh / p.Hk), h = (int)(bh - (int64_t)b * p.Hk);
  const float* kb = p.k + b * p.k_sb + h * p.k_sh;
  const float* vb = p.v + b * p.v_sb + h * p.v_sh;
  uint16_t* ko = p.kimg + at * (3 * 32 * HD);
  uint16_t* vo = p.vimg + at * (3 * 32 * HD);
  constexpr int CH = HD / 8;          // chunks (threads) per key
  constexpr int KPP = 256 / CH;       // keys per pass
  const int c = threadIdx.x % CH;
  float x[32 / KPP][8], y[32 / KPP][8];
#pragma unroll
  for (int i = 0; i < 32 / KPP; i++) {
    const int key = threadIdx.x / CH + i * KPP;
    const int64_t row = (int64_t)min(t0 + key, p.S - 1) * HD + 8 * c;
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(kb + row + e), w = *reinterpret_cast<const f32x4*>(vb + row + e);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        x[i][e + q] = key < n ? a[q] : 0.f;
        y[i][e + q] = key < n ? w[q] : 0.f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 32 / KPP; i++) {
    const int key = threadIdx.x / CH + i * KPP;
    u32x4 t[3];
    split8(x[i], t);
    uint16_t* o16 = ko + key * HD + key_chunk<HD>(key, c) * 8;
#pragma unroll
    for (int j = 0; j < 3; j++) *reinterpret_cast<u32x4*>(o16 + j * 32 * HD) = t[j];
#pragma unroll
    for (int e = 0; e < 8; e += 4)
      *reinterpret_cast<f32x4*>(&Vt[key * VST + 8 * c + e]) = f32x4{y[i][e], y[i][e + 1], y[i][e + 2], y[i][e + 3]};
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HD * 4 / 256; i++) {
    const int u = threadIdx.x + 256 * i, d = u >> 2, g = u & 3;
    float x8[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x8[e] = Vt[((e >> 2) * 16 + 4 * g + (e & 3)) * VST + d];
    u32x4 t[3];
    split8(x8, t);
    uint16_t* o = vo + d * 32 + slot_chunk(d, g) * 8;
#pragma unroll
    for (int j = 0; j < 3; j++) *reinterpret_cast<u32x4*>(o + j * 32 * HD) = t[j];
  }
}

struct SplitParams {
  const float *q, *k, *v, *mask;
  const uint16_t *kimg, *vimg;
  float* out;
  int H, Hk, T, S, tiles, qblocks;
  int64_t q_sb, q_sh, k_sb, k_sh, v_sb, v_sh, m_sb, m_sh, m_sr, m_sc;
  float scale;
};

// Workgroup barriers after the wave's vector loads and LDS accesses, and after
// its LDS accesses alone.
__device__ __forceinline__ void split_barrier() {
  __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ void split_lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ float lanes4_max(float x) {  // lanes l, l ^ 16, l ^ 32, l ^ 48
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float lanes4_sum(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The wave's 16 queries on the fp32 MFMA with operands straight from memory,
// those in `redo` stored: for queries whose split result is not finite. An
// infinity has no finite second term, so the split gives NaN where the
// operands themselves give an infinity, or a weight of 0. The organisation is
// attention_dense_kernel's without its staging: 16 keys a step, S^T = K . Q^T,
// O^T += V^T . P^T. One query at a time in vector code took 42 ms where one key
// of each head is infinite (32 x 8 heads x 512 x 1 024, head_dim 64) against
// 0.86 here (0.25 with finite operands, 0.36 on attention_dense_kernel).
template <int HD, bool MASK>
__device__ __forceinline__ void plain_queries(const SplitParams& p, int b, int h, int q0, uint64_t redo, int lane) {
  const int lq = lane & 15, g = lane >> 4;
  const int qi = q0 + lq, qc = min(qi, p.T - 1);
  const float* qr = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qc * HD + 4 * g;
  const float* kb = p.k + b * p.k_sb + h * p.k_sh + 4 * g;
  const float* vb = p.v + b * p.v_sb + h * p.v_sh + lq;
  const float* mrow = MASK ? p.mask + b * p.m_sb + h * p.m_sh + (int64_t)qc * p.m_sr : nullptr;
  f32x4 q[HD / 16], o[HD / 16];  // dims 16 s + 4 g .. + 3 of query lq
#pragma unroll
  for (int s = 0; s < HD / 16; s++) {
    q[s] = *reinterpret_cast<const f32x4*>(qr + 16 * s);
    o[s] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m = -1e30f, l = 0.f;
  for (int j0 = 0; j0 < p.S; j0 += 16) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};  // keys j0 + 4 g + r against query lq
    const float* kr = kb + (int64_t)min(j0 + lq, p.S - 1) * HD;
#pragma unroll
    for (int c = 0; c < HD / 16; c++) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(kr + 16 * c);
#pragma unroll
      for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], q[c][e], s, 0, 0, 0);
    }
    float w[4], top = -1e30f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = j0 + 4 * g + r;
      w[r] = s[r] * p.scale;
      if constexpr (MASK) w[r] += mrow[(int64_t)min(j, p.S - 1) * p.m_sc];
      if (j < p.S) top = fmaxf(top, w[r]);
    }
    const float mn = fmaxf(m, lanes4_max(top));
    const float alpha = exp_flush(m - mn);
    m = mn;
    l *= alpha;
#pragma unroll
    for (int c = 0; c < HD / 16; c++) o[c] *= alpha;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      w[r] = j0 + 4 * g + r < p.S ? exp_flush(w[r] - mn) : 0.f;
      l += w[r];
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = j0 + 4 * g + r;
      const float* vr = vb + (int64_t)min(j, p.S - 1) * HD;
#pragma unroll
      for (int c = 0; c < HD / 16; c++) {
        const float v = vr[16 * c];
        o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(j < p.S ? v : 0.f, w[r], o[c], 0, 0, 0);
      }
    }
  }
  const float inv = 1.f / lanes4_sum(l);
  if (!(redo >> lq & 1)) return;
  float* orow = p.out + (((int64_t)b * p.H + h) * p.T + qi) * HD + 4 * g;
#pragma unroll
  for (int c = 0; c < HD / 16; c++) *reinterpret_cast<f32x4*>(orow + 16 * c) = o[c] * inv;
}

template <int HD, int W, bool MASK>
__global__ __launch_bounds__(64 * W, 2) void attention_split_kernel(SplitParams p) {
  constexpr int SK = HD == 64 ? 64 : 32;  // keys per stage
  constexpr int NT = SK / 32;             // tiles per stage
  constexpr int NC = HD / 32, NDB = HD / 16;
  constexpr int IMG = 3 * 32 * HD;        // 16-bit values of a tile's key or value image
  static_assert(NT * IMG % (64 * W * 8) == 0, "whole loads");
  constexpr bool KD = HD < 256 && W == 8;  // two key buffers (72 KB with one, 96 with two)
  __shared__ __attribute__((aligned(16))) uint16_t K0[NT * IMG], K1[KD ? NT * IMG : 8], V0[NT * IMG], V1[NT * IMG];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lq = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x / p.qblocks, qblk = blockIdx.x % p.qblocks;
  const int b = bh / p.H, h = bh % p.H;
  const int64_t img = ((int64_t)b * p.Hk + (p.Hk == 1 ? 0 : h)) * p.tiles;
  const uint16_t* kimg = p.kimg + img * IMG;
  const uint16_t* vimg = p.vimg + img * IMG;
  const int stages = (p.S + SK - 1) / SK;

  auto load = [&](const uint16_t* src, uint16_t* dst, int st) {
#pragma unroll
    for (int i = 0; i < NT * IMG / 8 / 64 / W; i++)
      __builtin_amdgcn_global_load_lds(src + (int64_t)st * NT * IMG + ((i * W + wave) * 64 + lane) * 8,
                                       (__attribute__((address_space(3))) void*)(dst + (i * W + wave) * 512), 16, 0, 0);
  };
  load(kimg, K0, 0);

  // the wave's queries: their terms in registers
  const int qi = (qblk * W + wave) * 16 + lq;
  const bool qvalid = qi < p.T;
  const int qc = min(qi, p.T - 1);
  bf16x8 qt[NC][3];
  {
    const float* qr = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qc * HD + 8 * g;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(qr + 32 * c + e);
#pragma unroll
        for (int u = 0; u < 4; u++) x[e + u] = a[u];
      }
      u32x4 t[3];
      split8(x, t);
#pragma unroll
      for (int j = 0; j < 3; j++) qt[c][j] = __builtin_bit_cast(bf16x8, t[j]);
    }
  }
  const float* mrow = MASK ? p.mask + b * p.m_sb + h * p.m_sh + (int64_t)qc * p.m_sr : nullptr;

  f32x4 oacc[NDB];  // O^T: dims 16 db + 4 g + r of query lq
#pragma unroll
  for (int db = 0; db < NDB; db++) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -1e30f, l_part = 0.f;

  bf16x8 pt[NT][3];   // the previous stage's probability terms
  bool live = false;  // whether any of them is not 0
  auto pv = [&](const uint16_t* Vc) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int db = 0; db < NDB; db++) {
        const int dim = 16 * db + lq;
        const uint16_t* vr = Vc + t * IMG + dim * 32 + slot_chunk(dim, g) * 8;
        const bf16x8 v0 = *reinterpret_cast<const bf16x8*>(vr);
        const bf16x8 v1 = *reinterpret_cast<const bf16x8*>(vr + 32 * HD);
        const bf16x8 v2 = *reinterpret_cast<const bf16x8*>(vr + 64 * HD);
        f32x4 o = oacc[db];
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v2, pt[t][0], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v0, pt[t][2], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v1, pt[t][1], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v1, pt[t][0], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v0, pt[t][1], o, 0, 0, 0);
        oacc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v0, pt[t][0], o, 0, 0, 0);
      }
  };
  // a stage's mask values: keys 4g .. + 3 of the tiles' halves
  float mn_[NT][8];
  auto fetch = [&](int st) {
    if constexpr (MASK) {
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int j = st * SK + 32 * t + 16 * (e >> 2) + 4 * g + (e & 3);
          mn_[t][e] = mrow[(int64_t)min(j, p.S - 1) * p.m_sc];
        }
    }
  };
  fetch(0);
  auto stage = [&](int st, const uint16_t* Kc, uint16_t* Kn, uint16_t* Vn, const uint16_t* Vp) {
    split_barrier();  // this stage's keys, the last one's values landed; every wave is done with the last stage
    // the mask values loaded during the last stage: taken here, where the
    // barrier has waited for them. A use after the loads below would wait for
    // those too (the compiler does not count direct loads in order).
    float mv[NT][8];
    if constexpr (MASK) {
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          asm volatile("" : "+v"(mn_[t][e]));
          mv[t][e] = mn_[t][e];
        }
    }
    fetch(min(st + 1, stages - 1));
    load(vimg, Vn, st);
    if constexpr (KD) load(kimg, Kn, min(st + 1, stages - 1));
    f32x4 sacc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
        // hi . hi and the smaller terms in sums of their own: a sum of all of them
        // is rounded at full size six times per chunk
        f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, y = s;
        const int key = 16 * kb + lq;
        const uint16_t* kr = Kc + t * IMG + key * HD;
#pragma unroll
        for (int c = 0; c < NC; c++) {
          const int pos = key_chunk<HD>(key, 4 * c + g) * 8;
          const bf16x8 k0 = *reinterpret_cast<const bf16x8*>(kr + pos);
          const bf16x8 k1 = *reinterpret_cast<const bf16x8*>(kr + 32 * HD + pos);
          const bf16x8 k2 = *reinterpret_cast<const bf16x8*>(kr + 64 * HD + pos);
          y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k2, qt[c][0], y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qt[c][2], y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qt[c][1], y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qt[c][0], y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qt[c][1], y, 0, 0, 0);
          s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qt[c][0], s, 0, 0, 0);
        }
        sacc[t][kb] = s + y;
      }
    if constexpr (!KD) {
      split_lds_barrier();  // every wave has read the keys
      load(kimg, Kn, min(st + 1, stages - 1));
    }
    if (live) pv(Vp);
    float w[NT][8];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        w[t][e] = sacc[t][e >> 2][e & 3] * p.scale;
        if constexpr (MASK) w[t][e] += mv[t][e];
      }
    if (st * SK + SK > p.S) {  // the last stage: no keys past S
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (st * SK + 32 * t + 16 * (e >> 2) + 4 * g + (e & 3) >= p.S) w[t][e] = -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int e = 0; e < 8; e++) tmax = fmaxf(tmax, w[t][e]);
    tmax = lanes4_max(tmax);
    const bool need = tmax > m_run + kSplitTau;
    const float mn = need ? tmax : m_run;
    if (__any(need)) {
      const float alpha = exp_flush(m_run - mn);  // 0 for the first stage
      l_part *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; db++) oacc[db] *= alpha;
    }
    m_run = mn;
    // a stage whose every weight flushes to 0 (padding, outside a window)
    // adds nothing: no weights, no P.V, unless a score is NaN (which the
    // maximum passes over)
    live = __any(tmax - mn >= -87.f);
    if (!live) {
      bool nan = false;
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 8; e++) nan = nan || w[t][e] != w[t][e];
      live = __any(nan);
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
      if (!live) break;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        x[e] = exp_flush(w[t][e] - mn);
        l_part += x[e];
      }
      u32x4 y[3];
      split8(x, y);
#pragma unroll
      for (int j = 0; j < 3; j++) pt[t][j] = __builtin_bit_cast(bf16x8, y[j]);
    }
  };
  for (int st = 0; st < stages; st += 2) {
    stage(st, K0, KD ? K1 : K0, V0, V1);
    if (st + 1 < stages) stage(st + 1, KD ? K1 : K0, K0, V1, V0);
  }
  split_barrier();  // the last values (no load may still be writing LDS when the workgroup ends)
  if (live) pv((stages & 1) ? V0 : V1);

  const float l_tot = lanes4_sum(l_part);
  const float inv = 1.f / l_tot;
  float seen = 0.f;  // NaN if any output is not finite
  float* orow = p.out + ((int64_t)bh * p.T + qi) * HD + 4 * g;
#pragma unroll
  for (int db = 0; db < NDB; db++) {
    const f32x4 o = oacc[db] * inv;
#pragma unroll
    for (int r = 0; r < 4; r++) seen = fmaf(o[r], 0.f, seen);
    if (qvalid) *reinterpret_cast<f32x4*>(orow + 16 * db) = o;
  }
  // (a query whose weights are all 0, masked entirely, is NaN either way)
  uint64_t redo = __ballot(qvalid && seen != seen && l_tot != 0.f);
  redo = (redo | redo >> 16 | redo >> 32 | redo >> 48) & 0xFFFFu;  // queries of the wave
  if (redo) {
    __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0): the stores above, which other lanes write over
    plain_queries<HD, MASK>(p, b, h, (qblk * W + wave) * 16, redo, lane);
  }
}

struct SplitSizes {
  int Hk, tiles;
  int64_t blocks;  // key or value images
  size_t bytes;    // of the key images, and of the value images
};
SplitSizes split_sizes(const AttnGenericArgs& a) {
  SplitSizes z;
  z.Hk = a.k_sh == 0 && a.v_sh == 0 ? 1 : a.H;
  const int sk = a.D == 64 ? 64 : 32;
  z.tiles = (a.S + sk - 1) / sk * (sk / 32);
  z.blocks = (int64_t)a.B * z.Hk * z.tiles;
  z.bytes = (size_t)z.blocks * 3 * 32 * a.D * 2;
  return z;
}

template <int HD, int W>
void launch_split(const SplitParams& p, int64_t grid, hipStream_t s) {
  if (p.mask)
    hipLaunchKernelGGL((attention_split_kernel<HD, W, true>), dim3((unsigned)grid), dim3(64 * W), 0, s, p);
  else
    hipLaunchKernelGGL((attention_split_kernel<HD, W, false>), dim3((unsigned)grid), dim3(64 * W), 0, s, p);
}

// The rule: the 16-bit path where the time it saves on the keys exceeds what
// it adds, from both kernels' times at 156 shapes (1 to 1 024 queries, 32 to
// 4 096 keys, 1 to 64 batches of 1 to 8 heads, with and without a shared
// key/value head). It adds a launch, a longer prologue and the images, which
// cost their 18 bytes per key element whatever the queries are (6 TB/s while
// they stay in the last-level cache, 4 beyond). It saves microseconds per key
// that grow with the 64-query blocks once those are more than one per CU (at
// head_dim 256 the fp32 kernel slows down from half the CUs on). Below 192 keys
// and 0.1 GFLOP (0.5 at 256) the fp32 kernel stays in any case. Us, fp32 and
// 16-bit: 8 heads x 1 024 x 1 024, 64: 72 and 34; 51 x 8 x 1 x 1 024, 64: 103 and
// 159; the same on one shared head: 102 and 63; 2 x 8 x 128 x 256, 256: 35 and 43;
// 32 x 3 x 256 x 256, 256: 87 and 65; 4 x 3 x 1 024 x 1 024, 256: 194 and 118; 8 x 8 x
// 32 x 256, 256: 34 and 45; 26 x 8 x 1 x 1 024, 128: 113 and 170.
// (FA_ATTN_SPLIT=0 turns it off, for comparisons.)
bool attention_split_pays(const AttnGenericArgs& a, const SplitSizes& z) {
  if (a.S < 192 || 4.0 * a.B * a.H * (double)a.T * a.S * a.D < (a.D == 256 ? 5e8 : 1e8)) return false;
  const double blocks = (double)a.B * a.H * ((a.T + 63) / 64);
  const double image = 18.0 * a.D * a.B * z.Hk * (double)a.S;
  double key, fixed;  // us saved per key, us added per call
  if (a.D == 64) {
    key = blocks <= 256 ? 0.04 : std::max(0.055, 9.5e-5 * blocks);
    fixed = 7.5;
  } else if (a.D == 128) {
    key = blocks <= 256 ? 0.058 : std::max(0.095, 1.4e-4 * blocks);
    fixed = 6.5;
  } else {
    key = blocks <= 128 ? 0.0236 : blocks <= 256 ? 0.085 : std::max(0.11, 4.2e-4 * blocks);
    fixed = 12.;
  }
  return key * a.S >= fixed + image / (image < 2e8 ? 6e6 : 4e6);
}

}  // namespace

bool attention_split_ok(const AttnGenericArgs& a) {
  static const bool off = [] {
    const char* e = std::getenv("FA_ATTN_SPLIT");
    return e && e[0] == '0';
  }();
  if (off || !attention_dense_ok(a) || (a.D != 64 && a.D != 128 && a.D != 256)) return false;
  if (!(a.scale > 0.f) || a.S <= 0 || a.T <= 0) return false;
  const SplitSizes z = split_sizes(a);
  // images of at most 8 GiB: keys broadcast over a batch are written once per
  // entry, and the context keeps the buffer
  if (2 * z.bytes > (8ULL << 30) || !attention_split_pays(a, z)) return false;
  return z.blocks < INT32_MAX && (int64_t)a.B * a.H * ((a.T + 63) / 64) < INT32_MAX;
}

int launch_attention_split(fa_ctx* ctx, const AttnGenericArgs& a, hipStream_t s) {
  if (!attention_split_ok(a)) return set_error(ctx, FA_ERR_UNSUPPORTED, "Attention: no split path for these operands");
  const SplitSizes z = split_sizes(a);
  DevBuf& buf = ctx->slot(slots::S_ATTN);
  if (const int rc = buf.ensure(ctx, 2 * z.bytes)) return rc;
  SplitKvParams kv;
  kv.k = a.k; kv.v = a.v; kv.k_sb = a.k_sb; kv.k_sh = a.k_sh; kv.v_sb = a.v_sb; kv.v_sh = a.v_sh;
  kv.Hk = z.Hk; kv.S = a.S; kv.tiles = z.tiles;
  kv.kimg = buf.as<uint16_t>();
  kv.vimg = reinterpret_cast<uint16_t*>(buf.as<char>() + z.bytes);
  SplitParams p;
  p.q = a.q; p.k = a.k; p.v = a.v; p.mask = a.mask; p.kimg = kv.kimg; p.vimg = kv.vimg; p.out = a.out;
  p.H = a.H; p.Hk = z.Hk; p.T = a.T; p.S = a.S; p.tiles = z.tiles;
  p.q_sb = a.q_sb; p.q_sh = a.q_sh; p.k_sb = a.k_sb; p.k_sh = a.k_sh; p.v_sb = a.v_sb; p.v_sh = a.v_sh;
  p.m_sb = a.m_sb; p.m_sh = a.m_sh; p.m_sr = a.m_sr; p.m_sc = a.m_sc;
  p.scale = a.scale;
  // 64 queries per workgroup while those are at most one per CU, else 128 (at
  // head_dim 64 and 128 only where they fill their last one to more than half:
  // there two 64-query workgroups share a CU, at 256 a CU holds one of either).
  // Us with 64 and 128 queries, 512 keys: 64 heads x 256, head_dim 64: 24 and 29,
  // 256: 68 and 86; 64 x 512, 64: 32 and 31, 256: 124 and 91; 64 x 320, 64: 29 and
  // 30, 256: 121 and 86; 64 x 700, 64: 44 and 51, 128: 75 and 85, 256: 179 and 161.
  const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const int64_t bh = (int64_t)a.B * a.H;
  const bool half = (a.T + 127) / 128 * 128 - a.T >= 64;
  const int W = bh * ((a.T + 63) / 64) > cus && (a.D == 256 || !half) ? 8 : 4;
  p.qblocks = (a.T + 16 * W - 1) / (16 * W);
  const dim3 gk((unsigned)z.blocks), bk(256);
  switch (a.D) {
    case 64:
      hipLaunchKernelGGL(split_kv_kernel<64>, gk, bk, 0, s, kv);
      if (W == 8) launch_split<64, 8>(p, bh * p.qblocks, s);
      else launch_split<64, 4>(p, bh * p.qblocks, s);
      break;
    case 128:
      hipLaunchKernelGGL(split_kv_kernel<128>, gk, bk, 0, s, kv);
      if (W == 8) launch_split<128, 8>(p, bh * p.qblocks, s);
      else launch_split<128, 4>(p, bh * p.qblocks, s);
      break;
    default:
      hipLaunchKernelGGL(split_kv_kernel<256>, gk, bk, 0, s, kv);
      if (W == 8) launch_split<256, 8>(p, bh * p.qblocks, s);
      else launch_split<256, 4>(p, bh * p.qblocks, s);
      break;
  }
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

}  // namespace fa
