// Products of the encoder on the fp16 MFMA with fp32 accuracy:
// C = epilogue(A . W^T) with A fp32 values held as two fp16 terms (split2,
// device_math.h) and W bf16-exact weights held in fp16.
//
// A value a, scaled by a power of two that keeps its product's whole operand
// inside fp16's range, is stored by the kernel that produces it as
// hi = fp16(a) and lo = fp16((a - hi) * 2^11): within 2^-23 of a (a - hi is
// exact; lo rounds one value in four), the same 4 bytes as the float. lo
// carries its own 2^11 so that it stays a normal fp16 number down to 2^-25 of
// the largest value. A weight w times its matrix's power of two is exact in
// fp16 (checked when the model is finalized; otherwise the model keeps the
// three-term bf16 products of gemm.hip); w * 2^-11, the lo terms' factor, is
// rounded where w is below 2^-21 of its matrix's largest, and prepare_h2
// (model.cpp) holds what that and the operands' range add below a sixteenth of a
// float32 rounding in every row. Two v_mfma_f32_32x32x16_f16 per operand pair,
// hi . w and lo . (w * 2^-11), accumulate in fp32; the epilogue takes the
// powers of two back out. Against the exact three-term bf16 split this is two
// thirds of the MFMA work, no split in the product (each value is split once,
// where it is made, instead of once per column tile), and fewer fp32 roundings
// per sum, which is what the error against float64 comes from: two layers of
// 30 x 60..150 tokens 7.9e-7 by three terms and 6.8e-7, of 19 tokens 4.3e-7 and
// 3.8e-7, the 24-layer forward of 19 tokens 6.6e-7 and 4.1e-7.
//
// What bounds the large tiles: their MFMA pipes are busy 0.45 to 0.56 of the time
// (rocprofv3; LDS without a bank conflict), a wave waits a third of its cycles
// at the slab barriers, and the clock falls under the load: 32 768 x 2 304 x 768
// takes 453 thousand cycles in 252 to 275 us, 1.7 of 2.4 GHz, 0.92 PF/s executed.
//
// Layout of a split operand: row-major like the float matrix it replaces,
// with each 8 values as 16 bytes of hi then 16 bytes of lo.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "fa_internal.h"
#include "device_math.h"
#include "gemm_common.h"

namespace fa {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

struct H2Params {
  int64_t m, n, k;
  const uint16_t* a;  // split rows
  int64_t lda;        // values per row
  const uint16_t* b;  // fp16 [n x k]
  int64_t ldb;
  float* c;
  int64_t ldc;        // values per row
  float c_scale;      // accumulator -> value
  float out_scale;    // value -> stored split value (SPLIT)
  const float* mul;   // Generic: act(c) * mul
  int64_t ldm;
  int act;
  int tiles_m, tiles_n;
  int nk;             // slabs of a K part
  int64_t c_split;    // K part blockIdx.y writes c + blockIdx.y * c_split
};

template <int BM_, int BN_, int WM_, int WN_, int ST_, int MINW_>
struct HTile {
  static constexpr int BM = BM_, BN = BN_, BK = 32, WM = WM_, WN = WN_, ST = ST_, MINW = MINW_;
  static constexpr int NT = WM * WN * 64;
  static constexpr int TM = BM / WM, TN = BN / WN;
  static constexpr int FM = TM / 32, FN = TN / 32;
  static constexpr int NA = BM * 8 / NT, NB = BN * 4 / NT;  // 16-byte pieces per thread and slab
  static_assert(TM % 32 == 0 && TN % 32 == 0 && NA * NT == BM * 8 && NB * NT == BN * 4, "tile shape");
};

// LDS slots (16 bytes) of a slab: A row r's eight pieces (hi and lo of four
// 8-value chunks) at 8r + (j ^ (r >> 1)), W row r's four at 4r + (j ^ (r >> 2)).
// The 16 rows that 16 lanes read at once then take 16 different bank groups,
// and the slots are in the order in which the direct loads fill them (lane l
// of a wave at base + 16 l): each lane fetches the piece that belongs there.
__device__ __forceinline__ int a_slot(int r, int j) { return 8 * r + (j ^ ((r >> 1) & 7)); }
__device__ __forceinline__ int b_slot(int r, int j) { return 4 * r + (j ^ ((r >> 2) & 3)); }

// Workgroup barrier after all but the newest `left` direct loads of the wave
// have landed and its LDS reads are done.
template <int left>
__device__ __forceinline__ void h2_barrier() {
  __builtin_amdgcn_s_waitcnt((left & 15) | (7 << 4) | ((left >> 4) << 14));
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Writes one value, or (SPLIT) its two terms.
template <bool SPLIT>
__device__ __forceinline__ void put(float* row, int64_t col, float v, float out_scale, bool ok) {
  if constexpr (SPLIT) store_split1(row, col, v * out_scale, ok);
  else if (ok) row[col] = v;
}

__device__ __forceinline__ float h2_generic(const H2Params& p, float v, int64_t row, int64_t col, bool ok) {
  if (p.act == FA_ACT_GELU) v = gelu_sigmoid(v);
  if (p.mul) v = v * (ok ? p.mul[row * p.ldm + col] : 0.f);
  return v;
}

template <class TL, Epi EPI, bool SPLIT>
__global__ __launch_bounds__(TL::NT, TL::MINW) void gemm_h2_kernel(H2Params p) {
  constexpr int BM = TL::BM, BN = TL::BN, NT = TL::NT, FM = TL::FM, FN = TL::FN, NA = TL::NA, NB = TL::NB;
  constexpr int ST = TL::ST, LOADS = NA + NB;
  static_assert((ST == 2 || ST == 3) && NA <= 8 && NB <= 8, "two or three slabs in LDS, few pieces per thread");
  static_assert(!SPLIT || EPI != Epi::None, "split results come from an epilogue");
  __shared__ __attribute__((aligned(16))) uint16_t A0[BM * 64], B0[BN * 32], A1[BM * 64], B1[BN * 32];
  __shared__ __attribute__((aligned(16))) uint16_t A2[ST == 3 ? BM * 64 : 8], B2[ST == 3 ? BN * 32 : 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const int64_t M = p.m, N = p.n;
  const int tile = xcd_tile(p.tiles_m, p.tiles_n);
  const int64_t m0 = (int64_t)(tile / p.tiles_n) * BM, n0 = (int64_t)(tile % p.tiles_n) * BN;
  const int nk = p.nk;
  const int64_t k_off = (int64_t)blockIdx.y * nk * 32;

  const uint16_t* ga[8];  // NA, NB used (with dependent bounds here clang drops the host stub)
  const uint16_t* gb[8];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int idx = i * NT + tid, row = idx >> 3, j = (idx & 7) ^ ((row >> 1) & 7);
    ga[i] = p.a + (min(m0 + row, M - 1) * p.lda + k_off) * 2 + j * 8;
  }
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const int idx = i * NT + tid, row = idx >> 2, j = (idx & 3) ^ ((row >> 2) & 3);
    gb[i] = p.b + min(n0 + row, N - 1) * p.ldb + k_off + j * 8;
  }
  auto load = [&](uint16_t* As, uint16_t* Bs, int kt) {
#pragma unroll
    for (int i = 0; i < NA; i++)
      __builtin_amdgcn_global_load_lds(ga[i] + (int64_t)kt * 64,
                                       (__attribute__((address_space(3))) void*)(As + (i * NT + wave * 64) * 8), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < NB; i++)
      __builtin_amdgcn_global_load_lds(gb[i] + (int64_t)kt * 32,
                                       (__attribute__((address_space(3))) void*)(Bs + (i * NT + wave * 64) * 8), 16, 0, 0);
  };

  const int arow = wm * TL::TM + (lane & 31), brow = wn * TL::TN + (lane & 31), h = lane >> 5;
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  auto compute = [&](const uint16_t* As, const uint16_t* Bs) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      f16x8 hi[FM], lo[FM], w[FN], w2[FN];
#pragma unroll
      for (int i = 0; i < FM; i++) {
        hi[i] = *reinterpret_cast<const f16x8*>(As + a_slot(arow + 32 * i, 2 * (2 * s + h)) * 8);
        lo[i] = *reinterpret_cast<const f16x8*>(As + a_slot(arow + 32 * i, 2 * (2 * s + h) + 1) * 8);
      }
#pragma unroll
      for (int j = 0; j < FN; j++) {
        w[j] = *reinterpret_cast<const f16x8*>(Bs + b_slot(brow + 32 * j, 2 * s + h) * 8);
        w2[j] = w[j] * (_Float16)0x1p-11f;
      }
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[i], w2[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[i], w[j], acc[i][j], 0, 0, 0);
    }
  };

  if constexpr (ST == 2) {
    load(A0, B0, 0);
    h2_barrier<0>();
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      load(A1, B1, min(kt + 1, nk - 1));
      compute(A0, B0);
      h2_barrier<0>();
      load(A0, B0, min(kt + 2, nk - 1));
      compute(A1, B1);
      h2_barrier<0>();
    }
    if (kt < nk) compute(A0, B0);
  } else {
    load(A0, B0, 0);
    load(A1, B1, min(1, nk - 1));
    h2_barrier<LOADS>();
    int kt = 0;
    for (; kt + 3 <= nk; kt += 3) {
      load(A2, B2, min(kt + 2, nk - 1));
      compute(A0, B0);
      h2_barrier<LOADS>();
      load(A0, B0, min(kt + 3, nk - 1));
      compute(A1, B1);
      h2_barrier<LOADS>();
      load(A1, B1, min(kt + 4, nk - 1));
      compute(A2, B2);
      h2_barrier<LOADS>();
    }
    if (kt < nk) compute(A0, B0);
    if (kt + 1 < nk) {
      h2_barrier<0>();
      compute(A1, B1);
    }
  }
  // no direct load may still be writing LDS when the workgroup ends
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));

  // Epilogue. Lane l holds column l%32 and rows 8*(r/4) + 4*(l/32) + r%4 of
  // each block; a row's address is a wave-uniform base plus the lane's
  // 32-bit offset, and a wave whose sub-tile lies inside C stores without
  // bounds tests.
  constexpr bool kGe = EPI == Epi::GeGLU;
  const int64_t NO = kGe ? N / 2 : N;  // columns of C
  const int lcol = lane & 31, lrow4 = (lane >> 5) * 4;
  const int64_t r0 = m0 + wm * TL::TM, c0 = (n0 + wn * TL::TN) / (kGe ? 2 : 1);
  constexpr int CB = kGe ? FN / 2 : FN;  // column blocks of C per wave
  static_assert(!kGe || FN % 2 == 0, "GeGLU pairs column blocks");
  const bool inside = r0 + TL::TM <= M && c0 + CB * 32 <= NO;
  char* base = reinterpret_cast<char*>(p.c + (int64_t)blockIdx.y * p.c_split) + r0 * p.ldc * 4 + c0 * 4;
  const uint32_t ldc4 = (uint32_t)p.ldc * 4;
  const uint32_t voff = lrow4 * ldc4 + (SPLIT ? (uint32_t)split1_off(lcol) : lcol * 4);
  const float up_scale = p.c_scale * (SPLIT ? p.out_scale : 1.f);  // powers of two
  auto value = [&](int i, int j, int r) -> float {
    if constexpr (kGe) {
      return gelu_sigmoid(acc[i][2 * j][r] * p.c_scale) * (acc[i][2 * j + 1][r] * up_scale);
    } else if constexpr (EPI == Epi::Generic) {
      const int64_t row = r0 + i * 32 + (r >> 2) * 8 + lrow4 + (r & 3), col = c0 + j * 32 + lcol;
      const float v = h2_generic(p, acc[i][j][r] * p.c_scale, row, col, row < M && col < NO);
      return SPLIT ? v * p.out_scale : v;
    } else {
      return acc[i][j][r] * p.c_scale;
    }
  };
#pragma unroll
  for (int j = 0; j < CB; j++)
#pragma unroll
    for (int i = 0; i < FM; i++) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        char* at = base + (uint64_t)((uint32_t)(i * 32 + (r >> 2) * 8 + (r & 3)) * (uint64_t)ldc4) + j * 128;
        uint32_t w;
        if constexpr (SPLIT) w = split1_pair(value(i, j, r));
        else w = __float_as_uint(value(i, j, r));
        if (inside || (r0 + i * 32 + (r >> 2) * 8 + lrow4 + (r & 3) < M && c0 + j * 32 + lcol < NO))
          *reinterpret_cast<uint32_t*>(at + voff) = w;
      }
    }
}

// ---------------------------------------------------------------------------
// Few rows (a query, a batch of short sentences): a workgroup of eight waves
// computes one 32 x 64 tile of C, wave w taking the w-th of eight equal runs
// of the tile's K slabs with its operands loaded from global memory straight
// into MFMA registers (nothing is shared between waves), the eight partial
// tiles added through LDS in wave order; the organisation and the narrow
// GeGLU tiles (NB = 1: 16 features, their gate rows in columns 0-15 and up
// rows in 16-31) are those of gemm_x3_small_kernel, without its split.
constexpr int kSmallNW = 8;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <Epi EPI, bool SPLIT, int NB>
__global__ __launch_bounds__(kSmallNW * 64) void gemm_h2_small_kernel(H2Params p) {
  static_assert(NB == 2 || (NB == 1 && EPI == Epi::GeGLU), "narrow tiles: GeGLU only");
  constexpr int NW = kSmallNW;
  // the waves' partial tiles: with two column blocks four rows of a lane beside
  // each other (16-byte accesses), with one a row at a time
  constexpr int RV = NB == 2 ? 4 : 1;
  __shared__ __attribute__((aligned(16))) float red[NW][NB][16 / RV][64][RV];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t M = p.m, N = p.n;
  const int64_t m0 = (int64_t)(blockIdx.x / p.tiles_n) * 32;
  const int64_t n0 = (int64_t)(blockIdx.x % p.tiles_n) * 32 * NB;
  const int nk = p.nk;
  const int s0 = (int)((int64_t)wave * nk / NW), s1 = (int)((int64_t)(wave + 1) * nk / NW);
  const int64_t k_off = (int64_t)blockIdx.y * nk * 32 + (lane >> 5) * 8;
  const uint16_t* arow = p.a + (min(m0 + (lane & 31), M - 1) * p.lda + k_off) * 2;
  const int64_t bn = NB == 2 ? n0 + (lane & 31) : (n0 / 64) * 64 + (n0 / 2) % 32 + (lane & 15) + ((lane & 16) ? 32 : 0);
  const uint16_t* b0 = p.b + min(bn, N - 1) * p.ldb + k_off;
  const uint16_t* b1 = p.b + min(n0 + 32 + (lane & 31), N - 1) * p.ldb + k_off;

  // hi . w and lo . w in sums of their own: one sum for both is rounded twice
  // per step at full size (24 layers of 19 tokens: error against 64 bits 6.7e-7
  // with one, 4.3e-7 with two, 6.6e-7 by the three-term bf16 products)
  f32x16 acc[NB], low[NB];
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[j][r] = low[j][r] = 0.f;
  struct Regs {
    u32x4 a[4];  // hi, lo of the slab's two k-steps
    u32x4 b[2 * NB];
  };
  auto load = [&](Regs& g, int kt) {
#pragma unroll
    for (int st = 0; st < 2; st++) {
      const int64_t o = (int64_t)kt * 32 + 16 * st;
      g.a[2 * st] = *reinterpret_cast<const u32x4*>(arow + 2 * o);
      g.a[2 * st + 1] = *reinterpret_cast<const u32x4*>(arow + 2 * o + 8);
      g.b[NB * st] = *reinterpret_cast<const u32x4*>(b0 + o);
      if constexpr (NB == 2) g.b[2 * st + 1] = *reinterpret_cast<const u32x4*>(b1 + o);
    }
  };
  auto compute = [&](const Regs& g) {
#pragma unroll
    for (int st = 0; st < 2; st++) {
      const f16x8 hi = __builtin_bit_cast(f16x8, g.a[2 * st]), lo = __builtin_bit_cast(f16x8, g.a[2 * st + 1]);
#pragma unroll
      for (int j = 0; j < NB; j++)
        low[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            lo, __builtin_bit_cast(f16x8, g.b[NB * st + j]) * (_Float16)0x1p-11f, low[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NB; j++)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, __builtin_bit_cast(f16x8, g.b[NB * st + j]), acc[j], 0, 0, 0);
    }
  };
  if (s0 < s1) {
    Regs ra, rb;
    load(ra, s0);
    int kt = s0;
    for (; kt + 2 < s1; kt += 2) {  // the next slab's loads are issued before the current slab's MFMAs
      load(rb, kt + 1);
      compute(ra);
      load(ra, kt + 2);
      compute(rb);
    }
    if (kt + 1 < s1) {
      load(rb, kt + 1);
      compute(ra);
      compute(rb);
    } else {
      compute(ra);
    }
  }
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][j][r / RV][lane][r % RV] = acc[j][r] + low[j][r];
  __syncthreads();

  // C element (j, r, l): row 8*(r/4) + 4*(l/32) + r%4, column 32*j + l%32.
  // Neighbouring threads hold neighbouring columns of a row (put's pairs);
  // every thread takes part in each step.
  float* C = p.c + (int64_t)blockIdx.y * p.c_split;
  if constexpr (EPI == Epi::GeGLU) {
    const int64_t F = N / 2;
    constexpr int FW = NB == 1 ? 16 : 32;  // features of the tile
    constexpr int V = NB;                  // rows per thread
    static_assert(16 * 2 * FW == V * NW * 64, "one step");
    const int r0 = tid / (2 * FW) * V, lq = tid % (2 * FW);
    const int l = (lq % FW) + (lq / FW) * 32;  // gate lane; its up value: lane + 16 of block 0, or block 1
    float g[V], u[V];
#pragma unroll
    for (int i = 0; i < V; i++) g[i] = u[i] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int i = 0; i < V; i++) {
        g[i] += red[w][0][r0 / RV][l][(r0 + i) % RV];
        u[i] += NB == 1 ? red[w][0][r0 / RV][(l + 16) & 63][0] : red[w][NB - 1][r0 / RV][l][(r0 + i) % RV];
      }
#pragma unroll
    for (int i = 0; i < V; i++) {
      const int r = r0 + i;
      const int64_t row = m0 + (r >> 2) * 8 + (l >> 5) * 4 + (r & 3);
      const int64_t fcol = n0 / 2 + (lq % FW);
      const float v = gelu_sigmoid(g[i] * p.c_scale) * (u[i] * p.c_scale);
      put<SPLIT>(C + row * p.ldc, fcol, v, p.out_scale, row < M && fcol < F);
    }
  } else {
    static_assert(NB * 16 * 64 == 4 * NW * 64, "four rows per thread");
    const int j = tid >> 8, q = (tid >> 6) & 3, l = lane;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) v += *reinterpret_cast<const f32x4*>(red[w][j][q][l]);
    const int64_t col = n0 + 32 * j + (l & 31);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int64_t row = m0 + 8 * q + (l >> 5) * 4 + c;
      const bool ok = row < M && col < N;
      float x = v[c] * p.c_scale;
      if constexpr (EPI == Epi::Generic) x = h2_generic(p, x, row, col, ok);
      put<SPLIT>(C + row * p.ldc, col, x, p.out_scale, ok);
    }
  }
}

// ---- weights -----------------------------------------------------------------
__global__ __launch_bounds__(256) void h2_absmax_kernel(const uint16_t* __restrict__ w, int64_t n,
                                                        uint32_t* __restrict__ out) {
  uint32_t m = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    m = max(m, (uint32_t)(w[i] & 0x7FFFu));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(out, m);
}

__global__ __launch_bounds__(256) void h2_row_norms_kernel(const uint16_t* __restrict__ w, int64_t rows, int64_t cols,
                                                           const float* __restrict__ t, float* __restrict__ norms) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  double s = 0.;  // (squares of small weights leave float32's range)
  for (int64_t c = lane; c < cols; c += 64) {
    const double x = (double)__uint_as_float((uint32_t)w[row * cols + c] << 16) * (t ? (double)t[c] : 1.);
    s = fma(x, x, s);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) norms[row] = (float)sqrt(s);
}

__global__ __launch_bounds__(256) void h2_convert_kernel(const uint16_t* __restrict__ w, int64_t n, float scale,
                                                         uint16_t* __restrict__ dst, uint32_t* __restrict__ bad) {
  bool off = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float x = __uint_as_float((uint32_t)w[i] << 16) * scale;
    const _Float16 h = (_Float16)x;
    off |= (float)h != x;
    if (dst) dst[i] = __builtin_bit_cast(uint16_t, h);
  }
  if (bad && off) atomicOr(bad, 1u);
}

// ---- launches -----------------------------------------------------------------
using H128x128 = HTile<128, 128, 4, 2, 3, 4>;  // eight 32x64 waves, three slabs (72 KB): two workgroups per CU
using H64x128 = HTile<64, 128, 2, 2, 3, 3>;    // four 32x64 waves, three slabs (48 KB): three per CU
using H128x256 = HTile<128, 256, 2, 4, 2, 4>;  // eight 64x64 waves, two slabs (64 KB): two per CU

enum class HTileId { h128x128 = 0, h64x128, h128x256, small, kCount };
const char* const kHTileNames[] = {"128x128", "64x128", "128x256", "small"};

// FA_GEMM_HTILE=<name> forces a tile (tuning).
int forced_htile() {
  static int v = [] {
    const char* e = std::getenv("FA_GEMM_HTILE");
    if (!e) return -1;
    for (int i = 0; i < (int)HTileId::kCount; i++)
      if (std::strcmp(e, kHTileNames[i]) == 0) return i;
    return -1;
  }();
  return v;
}

// Tile by the workgroups each would launch. Us per launch, K = 768 (o: K parts
// included), small, 64x128, 128x128 and 128x256:
//  - small while its 32 x 64 tiles have a CU each (40 rows of q|k|v 8.0, 9.4,
//    10.6; of gate|up 9.1, 12.9, 14.7; 200 rows 10.9, 12.8, 15.2 and 11.4, 13.4,
//    15.7; 256 rows of gate|up 14.4, 13.2, 15.8: level);
//  - GeGLU on 128x256 from four per CU (32 768 rows -, 301, 258, 251; 24 576: 223,
//    193, 195; 16 384: 143, 127, 139: the line lies low), or where they fill one
//    and a quarter to two rounds that 128x128 does not fit into (5 504: 55, 53, 51;
//    6 912: 63, 57, 55);
//  - 64x128 where 128x128 leaves most CUs with one or less (512 rows of q|k|v 13.0
//    and 14.9; 1 280: 13.8 and 15.4; 1 792: 16.3 and 15.9) or would begin a third
//    round of two per CU (o at 5 504: 24.9 and 26.1);
//  - launches beside other groups' (shared): 128x128 unless it fills less than
//    half the CUs; the other streams fill what it leaves.
HTileId pick_htile(int64_t m, int64_t n, int ksplit, Epi epi, int cus, bool shared) {
  if (((m + 31) / 32) * ((n + 63) / 64) * ksplit <= cus) return HTileId::small;
  const int64_t t128 = ((m + 127) / 128) * ((n + 127) / 128) * ksplit;
  const int64_t t256 = ((m + 127) / 128) * ((n + 255) / 256) * ksplit;
  if (epi == Epi::GeGLU && (t256 >= 4LL * cus || (t256 > cus + cus / 4 && t256 <= 2LL * cus && t128 > 2LL * cus)))
    return HTileId::h128x256;
  if (shared) return 2 * t128 < cus ? HTileId::h64x128 : HTileId::h128x128;
  if (4 * t128 <= 5LL * cus || (t128 > 2LL * cus && 4 * t128 <= 9LL * cus)) return HTileId::h64x128;
  return HTileId::h128x128;
}

template <class TL, Epi EPI, bool SPLIT>
void launch_h2(H2Params p, int ksplit, hipStream_t s) {
  p.tiles_m = (int)((p.m + TL::BM - 1) / TL::BM);
  p.tiles_n = (int)((p.n + TL::BN - 1) / TL::BN);
  hipLaunchKernelGGL((gemm_h2_kernel<TL, EPI, SPLIT>), dim3(p.tiles_m * p.tiles_n, ksplit), dim3(TL::NT), 0, s, p);
}

template <Epi EPI, bool SPLIT>
void launch_h2_small(H2Params p, int ksplit, int cus, hipStream_t s) {
  p.tiles_m = (int)((p.m + 31) / 32);
  if constexpr (EPI == Epi::GeGLU) {
    // 16-feature tiles while they fit one per CU: twice the workgroups, each
    // loading half the weight rows
    if (p.tiles_m * (p.n / 32) <= cus) {
      p.tiles_n = (int)(p.n / 32);
      hipLaunchKernelGGL((gemm_h2_small_kernel<EPI, SPLIT, 1>), dim3(p.tiles_m * p.tiles_n, 1), dim3(kSmallNW * 64),
                         0, s, p);
      return;
    }
  }
  p.tiles_n = (int)((p.n + 63) / 64);
  hipLaunchKernelGGL((gemm_h2_small_kernel<EPI, SPLIT, 2>), dim3(p.tiles_m * p.tiles_n, ksplit), dim3(kSmallNW * 64),
                     0, s, p);
}

template <Epi EPI, bool SPLIT>
void dispatch_h2(HTileId t, const H2Params& p, int ksplit, int cus, hipStream_t s) {
  switch (t) {
    case HTileId::small: launch_h2_small<EPI, SPLIT>(p, ksplit, cus, s); break;
    case HTileId::h64x128: launch_h2<H64x128, EPI, SPLIT>(p, ksplit, s); break;
    case HTileId::h128x256:
      if constexpr (EPI == Epi::GeGLU) launch_h2<H128x256, EPI, SPLIT>(p, ksplit, s);
      else launch_h2<H128x128, EPI, SPLIT>(p, ksplit, s);
      break;
    default: launch_h2<H128x128, EPI, SPLIT>(p, ksplit, s); break;
  }
}

}  // namespace

bool gemm_h2_enabled() {
  static const bool v = [] {
    const char* e = std::getenv("FA_GEMM_H2");
    return !(e && e[0] == '0') && !gemm_f32_mfma_forced() && !std::getenv("FA_GEMM_XTILE");
  }();
  return v;
}

int launch_gemm_h2(fa_ctx* ctx, const GemmH2Args& g, hipStream_t s) {
  if (g.m == 0 || g.n == 0) return FA_OK;
  const int ks = std::max(g.ksplit, 1);
  if (g.m < 0 || g.n < 0 || g.k <= 0 || g.k % (32 * ks) != 0 || g.lda % 8 != 0 || g.ldb % 8 != 0 || g.lda < g.k ||
      g.ldb < g.k || g.ldc >= (1LL << 26))
    return set_error(ctx, FA_ERR_ARG, "MatMul: split product m=%lld n=%lld k=%lld lda=%lld ldb=%lld K parts %d",
                     (long long)g.m, (long long)g.n, (long long)g.k, (long long)g.lda, (long long)g.ldb, ks);
  if ((reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b)) & 15)
    return set_error(ctx, FA_ERR_ARG, "MatMul: split product needs 16-byte aligned operands");
  if (g.epi == Epi::GeGLU && g.n % 64 != 0)
    return set_error(ctx, FA_ERR_ARG, "GeGLU product needs n (2F) divisible by 64, got %lld", (long long)g.n);
  const bool split = g.out_scale != 0.f;
  if (split && (g.epi == Epi::None || (g.epi == Epi::GeGLU ? g.n / 2 : g.n) % 8 != 0))
    return set_error(ctx, FA_ERR_ARG, "MatMul: split results need an epilogue and whole groups of eight columns");
  if (ks > 1 && (g.epi != Epi::None || g.c_split < g.m * g.ldc))
    return set_error(ctx, FA_ERR_ARG, "MatMul: K parts need no epilogue and disjoint partial outputs");
  if (((g.m + 31) / 32) * ((g.n + 31) / 32) > INT32_MAX / 4) return set_error(ctx, FA_ERR_ARG, "MatMul: too many tiles");
  H2Params p;
  std::memset(&p, 0, sizeof p);
  p.m = g.m; p.n = g.n; p.k = g.k;
  p.a = reinterpret_cast<const uint16_t*>(g.a); p.lda = g.lda;
  p.b = g.b; p.ldb = g.ldb; p.c = g.c; p.ldc = g.ldc;
  p.c_scale = g.c_scale; p.out_scale = g.out_scale;
  p.mul = g.mul; p.ldm = g.ldm; p.act = g.act;
  p.nk = (int)(g.k / 32 / ks);
  p.c_split = ks > 1 ? g.c_split : 0;
  const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  HTileId t = (HTileId)forced_htile();
  if ((int)t < 0) t = pick_htile(g.m, g.n, ks, g.epi, cus, g.shared);
  switch (g.epi) {
    case Epi::None: dispatch_h2<Epi::None, false>(t, p, ks, cus, s); break;
    case Epi::Generic:
      if (split) dispatch_h2<Epi::Generic, true>(t, p, ks, cus, s);
      else dispatch_h2<Epi::Generic, false>(t, p, ks, cus, s);
      break;
    case Epi::GeGLU:
      if (split) dispatch_h2<Epi::GeGLU, true>(t, p, ks, cus, s);
      else dispatch_h2<Epi::GeGLU, false>(t, p, ks, cus, s);
      break;
  }
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

int launch_h2_absmax(fa_ctx* ctx, const uint16_t* w, int64_t n, uint32_t* max_bits, hipStream_t s) {
  if (n <= 0) return FA_OK;
  const unsigned grid = (unsigned)std::min<int64_t>(256, (n + 255) / 256);
  hipLaunchKernelGGL(h2_absmax_kernel, dim3(grid), dim3(256), 0, s, w, n, max_bits);
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

int launch_h2_row_norms(fa_ctx* ctx, const uint16_t* w, int64_t rows, int64_t cols, const float* t, float* norms,
                        hipStream_t s) {
  if (rows <= 0) return FA_OK;
  hipLaunchKernelGGL(h2_row_norms_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, w, rows, cols, t,
                     norms);
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

int launch_h2_convert(fa_ctx* ctx, const uint16_t* w, int64_t n, float scale, uint16_t* dst, uint32_t* bad,
                      hipStream_t s) {
  if (n <= 0) return FA_OK;
  const unsigned grid = (unsigned)std::min<int64_t>(1024, (n + 255) / 256);
  hipLaunchKernelGGL(h2_convert_kernel, dim3(grid), dim3(256), 0, s, w, n, scale, dst, bad);
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

}  // namespace fa
