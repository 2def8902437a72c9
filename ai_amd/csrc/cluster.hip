// k-means and nearest-centre search over embedding rows on gfx950: the
// drop-in for fiber/ai's cluster package (cluster/cluster.go:17-146).
//
// Nearest = one fp32-MFMA product sim = x . centres^T [n x k] (the GEMM of
// gemm.hip) + a per-row first-max argmax (tensor/reduce.go:269-297).
//
// KMeans keeps every step on the device; the host only draws the random
// numbers (Go's math/rand/v2 PCG, whose draws do not depend on the data, so
// all of them are drawn up front) and reads the per-iteration change count
// and centre sizes for the early stop and the empty-centre restarts.
//   k-means++ (cluster.go:51-85): per new centre, kpp_weights_kernel scores
//     every row against the newest centre, keeps the best similarity,
//     writes the float64 weight (1 - best)^2 and sums the weights in blocks
//     of 256; kpp_pick_kernel (one workgroup) scans the
//     block sums, scales the uniform draw by the total, finds the block and
//     then the row where the running subtraction crosses zero, and copies
//     that row into the centre list.
//   Lloyd rounds (cluster.go:86-129): nearest_kernel, or the sim product and
//     argmax_rows_kernel (assignment, similarity), count_kernel (per-chunk centre counts and
//     change counts), a stable counting sort of the row indices by centre
//     (chunk_scan_kernel, offsets_kernel, scatter_kernel), then
//     colsum_kernel adds each centre's rows in increasing row order, one
//     lane per (centre, column): the same float32 additions in the same
//     order as the reference's loop, so the centre sums are bit-identical
//     given the same assignment. Empty centres restart on the worst-fitting
//     row (worst_kernel, in increasing centre order), and
//     normalize_rows_kernel renormalises.
#include <cmath>
#include <cstring>
#include <vector>

#include "device_math.h"
#include "fa_internal.h"

namespace fa {
namespace {

constexpr int kRowWG = 256;        // one wave per row, 4 rows per workgroup
constexpr int kChunk = 256;        // rows per counting-sort chunk (one per thread of count_kernel)
constexpr int kCntWindow = 8192;   // centres per LDS counter window
constexpr int kSumBlock = 256;     // weights per partial sum of the k-means++ pick
constexpr int kColTile = 64;       // rows per load group of colsum_kernel (one per lane)

inline unsigned row_blocks(int64_t n) { return (unsigned)((n + 3) / 4); }

// cluster.Normalize (cluster.go:17-28): x / sqrt(sum x^2), a zero norm
// replaced by 1 (zero rows stay zero). In place allowed (out == x).
__global__ __launch_bounds__(kRowWG) void normalize_rows_kernel(const float* x, int64_t n, int d, float* out) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n) return;
  const float* xr = x + row * d;
  float* orow = out + row * d;
  float ss = 0.f;
  constexpr int kHeld = 16;  // up to 1 024 columns: the row's loads all in flight (40 x 768: 8.0 -> 3.2 us)
  if (d <= 64 * kHeld) {
    float v[kHeld];
#pragma unroll
    for (int i = 0; i < kHeld; i++) v[i] = lane + 64 * i < d ? xr[lane + 64 * i] : 0.f;
#pragma unroll
    for (int i = 0; i < kHeld; i++) ss += v[i] * v[i];
    float nrm = sqrtf(wave_sum(ss));
    if (nrm == 0.f) nrm = 1.f;
#pragma unroll
    for (int i = 0; i < kHeld; i++)
      if (lane + 64 * i < d) orow[lane + 64 * i] = v[i] / nrm;
    return;
  }
  for (int j = lane; j < d; j += 64) {
    const float v = xr[j];
    ss += v * v;
  }
  float nrm = sqrtf(wave_sum(ss));
  if (nrm == 0.f) nrm = 1.f;
  for (int j = lane; j < d; j += 64) orow[j] = xr[j] / nrm;
}

// First-max argmax of each row of sim [n x k] with the sequential rule of
// (*Tensor).Argmax: the first index holding the maximum; NaN never wins
// except at index 0, where the sequential scan starts.
__global__ __launch_bounds__(kRowWG) void argmax_rows_kernel(const float* __restrict__ sim, int64_t n, int k,
                                                             int32_t* __restrict__ assign,
                                                             float* __restrict__ simil) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n) return;
  const float* sr = sim + row * k;
  float bv = -INFINITY;
  int bi = INT32_MAX;
  for (int j = lane; j < k; j += 64) {
    const float v = sr[j];
    if (v > bv) {
      bv = v;
      bi = j;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane != 0) return;
  if (bi == INT32_MAX || isnan(sr[0])) bi = 0;
  assign[row] = bi;
  simil[row] = sr[bi];
}

// Product and first-max argmax in one pass for up to 64 centres (d % 8 == 0,
// 16-byte aligned rows): bound by reading x once (154 MB at 50 000 x 768,
// 31 us at a large copy's rate; the fp32 MFMAs take as long). A wave takes 32
// rows, their values loaded from global memory straight into the operand
// registers of v_mfma_f32_32x32x2_f32 (two groups of eight 16-byte loads in
// flight per lane); the centres pass through LDS 128 columns at a time,
// shared by the workgroup's four waves. Operands and order of the additions are
// gemm_kernel's, so the similarities are the same bits as the product's (a
// row between two centres falls to the same one). Lane l holds centre 32 b +
// l%32 (block b) against rows 8 (r/4) + 4 (l/32) + r%4: a row's argmax is a
// maximum over blocks and five exchanges, then the lowest index that has it.
// 67 us at 50 000 x 768 and 40 centres against 61 + 12 for the product and the
// argmax of its stored rows: the MFMA pipes set it (391 workgroups of four
// waves leave some SIMDs two waves of 32 rows, 47 us of fp32 MFMAs).
constexpr int kNearCols = 128, kNearSteps = 8, kNearMax = 64;
typedef float f32x16 __attribute__((ext_vector_type(16)));

// max / min over lanes l ^ 1, 2, 4, 8, 16: the 32 lanes of a half wave
template <class F>
__device__ __forceinline__ uint32_t half_wave(uint32_t v, F f) {
  auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = f((uint32_t)a[0], (uint32_t)a[1]);
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, false));
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, false));
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xF, 0xF, false));
  v = f(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xF, 0xF, false));
  return v;
}

template <int CB>
__global__ __launch_bounds__(256) void nearest_kernel(const float* __restrict__ x, int64_t n, int d,
                                                      const float* __restrict__ centres, int k,
                                                      int32_t* __restrict__ assign, float* __restrict__ simil) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int LD = kNearCols + 4;  // rows four banks apart
  __shared__ __attribute__((aligned(16))) float cs[32 * CB * LD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lq = lane & 31, h = lane >> 5;
  const int64_t row0 = ((int64_t)blockIdx.x * 4 + wave) * 32;
  const float* xr = x + min(row0 + lq, n - 1) * d + 4 * h;
  const int steps = d / 8;
  f32x16 acc[CB];
#pragma unroll
  for (int b = 0; b < CB; b++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[b][r] = 0.f;
  auto load = [&](f4 (&a)[kNearSteps], int s0) {
#pragma unroll
    for (int u = 0; u < kNearSteps; u++) a[u] = *reinterpret_cast<const f4*>(xr + 8 * min(s0 + u, steps - 1));
  };
  auto compute = [&](const f4 (&a)[kNearSteps], int s0, int c0) {
#pragma unroll
    for (int u = 0; u < kNearSteps; u++) {
      if (s0 + u < steps) {
        f4 c[CB];
#pragma unroll
        for (int b = 0; b < CB; b++)
          c[b] = *reinterpret_cast<const f4*>(cs + (32 * b + lq) * LD + 8 * (s0 + u) - c0 + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int b = 0; b < CB; b++)
            acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][e], c[b][e], acc[b], 0, 0, 0);
      }
    }
  };
  // the next columns of the centres load into registers while the current
  // ones are used (centres past k repeat the last, columns past d its last)
  constexpr int NC = 32 * CB * (kNearCols / 4) / 256;
  f4 pre[NC];
  auto fetch = [&](int c0) {
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int at = threadIdx.x + 256 * i, r = at / (kNearCols / 4), c = at % (kNearCols / 4);
      pre[i] = *reinterpret_cast<const f4*>(centres + (int64_t)min(r, k - 1) * d + min(c0 + 4 * c, d - 4));
    }
  };
  f4 a0[kNearSteps], a1[kNearSteps];
  fetch(0);
  load(a0, 0);
  for (int c0 = 0; c0 < d; c0 += kNearCols) {
    __syncthreads();  // the previous columns were read
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int at = threadIdx.x + 256 * i;
      *reinterpret_cast<f4*>(cs + at / (kNearCols / 4) * LD + at % (kNearCols / 4) * 4) = pre[i];
    }
    __syncthreads();
    const int s0 = c0 / 8;
    fetch(c0 + kNearCols);
    load(a1, s0 + kNearSteps);
    compute(a0, s0, c0);
    load(a0, s0 + 2 * kNearSteps);
    if (s0 + kNearSteps < steps) compute(a1, s0 + kNearSteps, c0);
  }
#pragma unroll
  for (int r = 0; r < 16; r++) {
    // floats as ordered integers; 0 for NaN and for centres past k
    uint32_t key = 0, idx = 0xFFFFFFFFu;
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const float v = acc[b][r];
      const uint32_t u = __float_as_uint(v + 0.f);
      const uint32_t o = v != v || 32 * b + lq >= k ? 0u : (u & 0x80000000u) ? ~u : (u | 0x80000000u);
      if (o > key) {
        key = o;
        idx = 32 * b + lq;
      }
    }
    const uint32_t top = half_wave(key, [](uint32_t p, uint32_t q) { return max(p, q); });
    const uint32_t at = half_wave(key == top ? idx : 0xFFFFFFFFu, [](uint32_t p, uint32_t q) { return min(p, q); });
    const float first = __shfl(acc[0][r], 32 * h, 64);  // centre 0
    const int64_t row = row0 + (r >> 2) * 8 + 4 * h + (r & 3);
    // no number above -inf, or NaN at index 0 where the sequential scan
    // starts: index 0
    const bool zero = at == 0xFFFFFFFFu || top == 0x007FFFFFu || isnan(first);
    if (row < n && lq == (zero ? 0 : (int)(at & 31))) {
      assign[row] = zero ? 0 : (int)at;
      simil[row] = zero ? first : (CB == 2 && at >= 32 ? acc[CB - 1][r] : acc[0][r]);
    }
  }
}

// Per chunk of kChunk rows: rows per centre (chunk_cnt[c][ch], centre-major)
// and rows whose centre differs from the previous round's
// (chunk_changed[ch]); then the previous assignment is brought up to date.
__global__ __launch_bounds__(kChunk) void count_kernel(const int32_t* __restrict__ cur, int32_t* __restrict__ prev,
                                                       int64_t n, int k, int nchunks, int32_t* __restrict__ chunk_cnt,
                                                       int32_t* __restrict__ chunk_changed) {
  __shared__ int32_t cnt[kCntWindow];
  __shared__ int32_t nchanged;
  const int t = threadIdx.x;
  const int64_t ch = blockIdx.x;
  const int64_t row = ch * kChunk + t;
  const int a = row < n ? cur[row] : -1;
  if (t == 0) nchanged = 0;
  __syncthreads();
  if (row < n && prev[row] != a) atomicAdd(&nchanged, 1);
  for (int w0 = 0; w0 < k; w0 += kCntWindow) {
    const int w1 = min(k, w0 + kCntWindow);
    for (int c = t; c < w1 - w0; c += kChunk) cnt[c] = 0;
    __syncthreads();
    if (a >= w0 && a < w1) atomicAdd(&cnt[a - w0], 1);
    __syncthreads();
    for (int c = t; c < w1 - w0; c += kChunk) chunk_cnt[(int64_t)(w0 + c) * nchunks + ch] = cnt[c];
    __syncthreads();
  }
  if (row < n) prev[row] = a;
  if (t == 0) chunk_changed[ch] = nchanged;
}

// k-means++ step over all rows: s = x[i] . c, best[i] = max(best[i], s),
// w[i] = float64(1 - best[i])^2 (cluster.go:62-72), and part[b] = the sum of
// w[b * kSumBlock ...] in a fixed tree order. One workgroup of 16 waves per
// kSumBlock rows, each wave four rows at a time (bound by reading x: 25 us at
// 50 000 x 768; the block sums were a launch of their own, 4.7 us and a gap
// per centre).
constexpr int kKppWaves = 16;
__global__ __launch_bounds__(64 * kKppWaves) void kpp_weights_kernel(const float* __restrict__ x, int64_t n, int d,
                                                                     const float* __restrict__ c, float* best,
                                                                     double* w, double* __restrict__ part) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  __shared__ double buf[kSumBlock];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * kSumBlock;
  const bool vec = (d & 3) == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(c)) & 15) == 0;
  constexpr int U = 4;
  for (int i = wave * U; i < kSumBlock; i += kKppWaves * U) {
    float s[U] = {0.f, 0.f, 0.f, 0.f};
    const float* xr[U];
#pragma unroll
    for (int u = 0; u < U; u++) xr[u] = x + min(r0 + i + u, n - 1) * d;
    if (vec) {
      for (int j = lane; j < d / 4; j += 64) {
        const f4 b = reinterpret_cast<const f4*>(c)[j];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const f4 a = reinterpret_cast<const f4*>(xr[u])[j];
          s[u] += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
        }
      }
    } else {
      for (int j = lane; j < d; j += 64) {
#pragma unroll
        for (int u = 0; u < U; u++) s[u] += xr[u][j] * c[j];
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) s[u] = wave_sum(s[u]);
    if (lane < U) {
      const int64_t row = r0 + i + lane;
      const float v = lane == 0 ? s[0] : lane == 1 ? s[1] : lane == 2 ? s[2] : s[3];
      double om = 0.0;
      if (row < n) {
        float b = best[row];
        if (v > b) b = v;
        best[row] = b;
        om = (double)(1.f - b);
        om = om * om;
        w[row] = om;
      }
      buf[i + lane] = om;
    }
  }
  __syncthreads();
  const int t = threadIdx.x;
  for (int o = kSumBlock / 2; o > 0; o >>= 1) {
    if (t < o) buf[t] += buf[t + o];
    __syncthreads();
  }
  if (t == 0) part[blockIdx.x] = buf[0];
}

// k-means++ pick (cluster.go:73-82): pick = u * total; the chosen row is
// the first i where pick - w[0] - ... - w[i] <= 0 (n-1 when rounding leaves
// it positive). The block partial sums' inclusive prefix locates the
// crossing block, whose weights are then walked one by one. The row is
// copied to centre_out.
// kPickThreads: 256 for up to 65 536 rows (one tile of partial sums, four
// waves at each barrier), else 1 024.
template <int kPickThreads>
__global__ __launch_bounds__(kPickThreads) void kpp_pick_kernel(const double* __restrict__ w, int64_t n,
                                                                const double* __restrict__ part, int nparts, double u,
                                                                const float* __restrict__ x, int d,
                                                                float* __restrict__ centre_out, int32_t* chosen) {
  __shared__ double scan[kPickThreads];
  __shared__ double wblk[kSumBlock];
  __shared__ double carry, total_s;
  __shared__ int first_blk;
  __shared__ int64_t pick_idx;
  const int t = threadIdx.x;
  if (t == 0) {
    carry = 0;
    first_blk = INT32_MAX;
  }
  __syncthreads();
  // total: inclusive scan of the partials in tiles of kPickThreads (pass 1)
  for (int base = 0; base < nparts; base += kPickThreads) {
    scan[t] = base + t < nparts ? part[base + t] : 0.0;
    __syncthreads();
    for (int o = 1; o < kPickThreads; o <<= 1) {
      const double add = t >= o ? scan[t - o] : 0.0;
      __syncthreads();
      scan[t] += add;
      __syncthreads();
    }
    if (t == 0) carry += scan[kPickThreads - 1];
    __syncthreads();
  }
  if (t == 0) total_s = carry;
  __syncthreads();
  const double pick = u * total_s;
  // pass 2: the first block whose inclusive prefix reaches pick (one tile of
  // partials: the scan of pass 1 is still in LDS)
  const bool one_tile = nparts <= kPickThreads;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nparts; base += kPickThreads) {
    if (!one_tile) {
      scan[t] = base + t < nparts ? part[base + t] : 0.0;
      __syncthreads();
      for (int o = 1; o < kPickThreads; o <<= 1) {
        const double add = t >= o ? scan[t - o] : 0.0;
        __syncthreads();
        scan[t] += add;
        __syncthreads();
      }
    }
    if (base + t < nparts && pick - (carry + scan[t]) <= 0) atomicMin(&first_blk, base + t);
    __syncthreads();
    if (first_blk != INT32_MAX) break;
    if (t == 0) carry += scan[kPickThreads - 1];
    __syncthreads();
  }
  __syncthreads();
  const int fb = first_blk;
  // the prefix before block fb, in the order pass 2 formed it
  if (fb != INT32_MAX && t == 0) {
    const int tile = fb / kPickThreads * kPickThreads;
    total_s = carry + (fb > tile ? scan[fb - tile - 1] : 0.0);
  }
  const int64_t b0 = fb != INT32_MAX ? (int64_t)fb * kSumBlock : n;
  if (t < kSumBlock) wblk[t] = b0 + t < n ? w[b0 + t] : 0.0;
  __syncthreads();
  if (t == 0) {
    int64_t idx = n - 1;
    if (fb != INT32_MAX) {
      double p = pick - total_s;
      // 16 weights read ahead of their subtractions (past the rows: zeros,
      // which leave p as it is)
      int at = kSumBlock;
      for (int j = 0; j < kSumBlock && at == kSumBlock; j += 16) {
        double v[16];
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] = wblk[j + e];
#pragma unroll
        for (int e = 0; e < 16; e++) {
          p -= at == kSumBlock ? v[e] : 0.0;
          if (p <= 0 && at == kSumBlock) at = j + e;
        }
      }
      int64_t i = min(n, b0 + at);
      if (at == kSumBlock)  // rounding: keep walking
        for (; i < n; i++) {
          p -= w[i];
          if (p <= 0) break;
        }
      if (i < n) idx = i;
    }
    pick_idx = idx;
    *chosen = (int32_t)idx;
  }
  __syncthreads();
  const float* src = x + pick_idx * d;
  for (int j = t; j < d; j += kPickThreads) centre_out[j] = src[j];
}

// chunk_cnt[c][ch] (rows of chunk ch assigned to c) -> exclusive prefix over
// chunks; sizes[c] = total. One workgroup per centre.
__global__ __launch_bounds__(256) void chunk_scan_kernel(int32_t* chunk_cnt, int nchunks, int32_t* sizes) {
  __shared__ int32_t buf[256];
  __shared__ int32_t carry;
  const int t = threadIdx.x;
  int32_t* row = chunk_cnt + (int64_t)blockIdx.x * nchunks;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nchunks; base += 256) {
    const int32_t v = base + t < nchunks ? row[base + t] : 0;
    buf[t] = v;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
      const int32_t add = t >= o ? buf[t - o] : 0;
      __syncthreads();
      buf[t] += add;
      __syncthreads();
    }
    if (base + t < nchunks) row[base + t] = carry + buf[t] - v;
    __syncthreads();
    if (t == 0) carry += buf[255];
    __syncthreads();
  }
  if (t == 0) sizes[blockIdx.x] = carry;
}

// offsets[c] = sizes[0] + ... + sizes[c-1]; summary = the sizes and the sum of
// the chunks' change counts, what the host reads per round. One workgroup.
__global__ __launch_bounds__(1024) void offsets_kernel(const int32_t* sizes, int k, int32_t* offsets,
                                                       const int32_t* chunk_changed, int nchunks, int32_t* summary) {
  __shared__ int32_t buf[1024];
  __shared__ int32_t carry;
  const int t = threadIdx.x;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < k; base += 1024) {
    const int32_t v = base + t < k ? sizes[base + t] : 0;
    buf[t] = v;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {  // inclusive Hillis-Steele scan
      const int32_t add = t >= o ? buf[t - o] : 0;
      __syncthreads();
      buf[t] += add;
      __syncthreads();
    }
    if (base + t < k) {
      offsets[base + t] = carry + buf[t] - v;
      summary[base + t] = v;
    }
    __syncthreads();
    if (t == 0) carry += buf[1023];
    __syncthreads();
  }
  int32_t s = 0;
  for (int ch = t; ch < nchunks; ch += 1024) s += chunk_changed[ch];
  buf[t] = s;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o) buf[t] += buf[t + o];
    __syncthreads();
  }
  if (t == 0) summary[k] = buf[0];
}

// Stable scatter of row indices by centre: list[offsets[a] + (rows of a in
// earlier chunks) + (rows of a earlier in this chunk)] = row. One wave per
// chunk walks its rows in order 64 at a time; the rank among equal lanes
// comes from shuffles, the running count per centre from LDS (centre
// windows of kCntWindow).
__global__ __launch_bounds__(64) void scatter_kernel(const int32_t* __restrict__ assign, int64_t n, int k,
                                                     int nchunks, const int32_t* __restrict__ offsets,
                                                     const int32_t* __restrict__ chunk_pre, int32_t* __restrict__ list) {
  __shared__ int32_t cnt[kCntWindow];
  const int lane = threadIdx.x;
  const int64_t ch = blockIdx.x;
  const int64_t r0 = ch * kChunk;
  for (int w0 = 0; w0 < k; w0 += kCntWindow) {
    const int w1 = min(k, w0 + kCntWindow);
    for (int c = lane; c < w1 - w0; c += 64) cnt[c] = 0;
    __syncthreads();
    for (int sub = 0; sub < kChunk; sub += 64) {
      const int64_t row = r0 + sub + lane;
      int a = row < n ? assign[row] : -1;
      if (a < w0 || a >= w1) a = -1;
      // the lanes with the same centre, bit by bit (an absent row is a
      // value of its own)
      const uint32_t key = a < 0 ? (uint32_t)(w1 - w0) : (uint32_t)(a - w0);
      uint64_t same = ~0ull;
      for (int b = 0; (w1 - w0) >> b; b++) {
        const uint64_t m = __ballot((key >> b) & 1);
        same &= (key >> b) & 1 ? m : ~m;
      }
      const uint64_t below = (1ull << lane) - 1;
      const int rank = __popcll(same & below), later = __popcll(same & ~below) - 1;
      if (a >= 0) list[offsets[a] + chunk_pre[(int64_t)a * nchunks + ch] + cnt[a - w0] + rank] = (int32_t)row;
      __syncthreads();
      if (a >= 0 && later == 0) cnt[a - w0] += rank + 1;
      __syncthreads();
    }
  }
}

// sums[c][j] = sum over c's rows in increasing row order of x[row][j],
// accumulated in float32 from 0 (cluster.go:100-112). One wave per (centre,
// 64 columns). Latency bound (a lane's additions are one chain, and k * d / 64
// waves are about two per CU): groups of kColTile rows, the next group's
// loads in flight while the current one is added, and a group's row indices one
// per lane (69 -> 50 us at 50 000 x 768 and 40 centres against 32 rows loaded,
// then added).
__global__ __launch_bounds__(64) void colsum_kernel(const float* __restrict__ x, int d,
                                                    const int32_t* __restrict__ list,
                                                    const int32_t* __restrict__ offsets,
                                                    const int32_t* __restrict__ sizes, float* __restrict__ sums) {
  const int c = blockIdx.x;
  const int j = blockIdx.y * 64 + threadIdx.x;
  const int32_t* rows = list + offsets[c];
  const int m = sizes[c];
  float acc = 0.f;
  if (m > 0) {
    const float* xc = x + min(j, d - 1);
    // lane u holds the group's u-th row (past the last: the last again; its
    // value is not added)
    auto index = [&](int p) { return rows[min(p + (int)threadIdx.x, m - 1)]; };
    auto load = [&](float (&v)[kColTile], int32_t iv) {
#pragma unroll
      for (int u = 0; u < kColTile; u++) v[u] = xc[(int64_t)__builtin_amdgcn_readlane(iv, u) * d];
    };
    auto add = [&](const float (&v)[kColTile], int p) {
      if (p + kColTile <= m) {
#pragma unroll
        for (int u = 0; u < kColTile; u++) acc += v[u];
      } else {
#pragma unroll
        for (int u = 0; u < kColTile; u++)
          if (p + u < m) acc += v[u];
      }
    };
    float va[kColTile], vb[kColTile];
    int32_t ia = index(0), ib = index(kColTile);
    load(va, ia);
    for (int p = 0; p < m; p += 2 * kColTile) {
      ia = index(p + 2 * kColTile);
      load(vb, ib);
      add(va, p);
      ib = index(p + 3 * kColTile);
      load(va, ia);
      if (p + kColTile < m) add(vb, p + kColTile);
    }
  }
  if (j < d) sums[(int64_t)c * d + j] = acc;
}

// Empty-centre restart (cluster.go:113-124): worst = the first index of the
// minimum similarity (index 0 when no element compares below simil[0]);
// its row becomes the centre's sum and its similarity is set to 1.
__global__ __launch_bounds__(1024) void worst_kernel(float* simil, int64_t n, const float* __restrict__ x, int d,
                                                     float* __restrict__ sums_row) {
  __shared__ float sv[1024];
  __shared__ int64_t si[1024];
  const int t = threadIdx.x;
  float bv = INFINITY;
  int64_t bi = INT64_MAX;
  for (int64_t i = t; i < n; i += 1024) {
    const float v = simil[i];
    if (v < bv) {
      bv = v;
      bi = i;
    }
  }
  sv[t] = bv;
  si[t] = bi;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o) {
      const float ov = sv[t + o];
      const int64_t oi = si[t + o];
      if (ov < sv[t] || (ov == sv[t] && oi < si[t])) {
        sv[t] = ov;
        si[t] = oi;
      }
    }
    __syncthreads();
  }
  const int64_t worst = (si[0] == INT64_MAX || isnan(simil[0])) ? 0 : si[0];
  __syncthreads();
  if (t == 0) simil[worst] = 1.f;
  const float* src = x + worst * d;
  for (int j = t; j < d; j += 1024) sums_row[j] = src[j];
}

__global__ void fill_f32_kernel(float* p, int64_t n, float v) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace
}  // namespace fa

// ---- host side -----------------------------------------------------------------

namespace fa {
namespace {

// Go's math/rand/v2 generator as cluster.KMeans seeds it
// (rand.New(rand.NewPCG(seed, seed^0x9e3779b97f4a7c15)), cluster.go:47):
// a 128-bit LCG (pcg-cpp's default multiplier and increment) whose new
// state goes through the DXSM output function; IntN is Lemire's
// multiply-shift with rejection (a mask for powers of two), Float64 the top
// 53 bits of a draw over 2^53.
struct GoPCG {
  uint64_t hi, lo;
  uint64_t Uint64() {
    typedef unsigned __int128 u128;
    const u128 mul = ((u128)2549297995355413924ULL << 64) | 4865540595714422341ULL;
    const u128 inc = ((u128)6364136223846793005ULL << 64) | 1442695040888963407ULL;
    const u128 s = ((((u128)hi) << 64) | lo) * mul + inc;
    hi = (uint64_t)(s >> 64);
    lo = (uint64_t)s;
    uint64_t h = hi;
    h ^= h >> 32;
    h *= 0xda942042e4dd58b5ULL;
    h ^= h >> 48;
    return h * (lo | 1);
  }
  uint64_t IntN(uint64_t n) {
    typedef unsigned __int128 u128;
    if ((n & (n - 1)) == 0) return Uint64() & (n - 1);
    u128 m = (u128)Uint64() * n;
    if ((uint64_t)m < n) {
      const uint64_t thresh = (0 - n) % n;
      while ((uint64_t)m < thresh) m = (u128)Uint64() * n;
    }
    return (uint64_t)(m >> 64);
  }
  double Float64() { return (double)(Uint64() << 11 >> 11) / 9007199254740992.0; }
};

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

int check_rows(fa_ctx* ctx, const char* op, int64_t n, int64_t d) {
  if (n < 0 || d < 0 || n > INT32_MAX || d > INT32_MAX)
    return set_error(ctx, FA_ERR_ARG, "%s: shape [%lld x %lld] outside this build's int32 row/column range", op,
                     (long long)n, (long long)d);
  return FA_OK;
}

int launch_normalize(fa_ctx* ctx, const float* x, int64_t n, int d, float* out) {
  if (n == 0 || d == 0) return FA_OK;
  hipLaunchKernelGGL(normalize_rows_kernel, dim3(row_blocks(n)), dim3(kRowWG), 0, ctx->stream, x, n, d, out);
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

// sim = x . c^T [n x k] on the fp32 MFMA GEMM.
int launch_sim(fa_ctx* ctx, const float* x, int64_t n, const float* c, int64_t k, int d, float* sim) {
  GemmArgs g;
  g.m = n;
  g.n = k;
  g.k = d;
  g.a = x;
  g.lda = d;
  g.b = c;
  g.ldb = d;
  g.b_dtype = FA_DT_F32;
  g.b_layout = FA_B_NK;
  g.c = sim;
  g.ldc = k;
  return launch_gemm(ctx, g, ctx->stream);
}

// assign, simil of every row: fused, or the product into sim [n x k] and the
// argmax of its rows, for more than 64 centres, other widths or alignments, and
// where it is the faster one: up to a round of its 64-row tiles (the fused
// kernel's 128-row workgroups leave half the CUs idle there), and with two
// blocks of centres where those fill an odd number of rounds, so that the fused
// kernel's last one is at most half full, until the bytes of the similarities
// weigh more. Us at 768 columns, product and fused: 40 centres, 1 000 rows 21 and
// 34, 16 000: 26 and 35, 28 000: 40 and 36, 42 000: 55 and 64, 50 000: 70 and 64,
// 80 000: 90 and 94, 200 000: 404 and 227; 4 centres, 1 000: 21 and 23, 28 000: 40
// and 24. At 256: 40 centres, 1 000: 11 and 15, 42 000: 29 and 26; 4 centres 11
// and 10.
bool nearest_fused_ok(fa_ctx* ctx, const float* x, int64_t n, const float* c, int64_t k, int d) {
  if (k > kNearMax || d % 8 != 0 || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(c)) & 15) != 0)
    return false;
  const int64_t round = 64LL * (ctx->cu_count > 0 ? ctx->cu_count : 256);
  if (k <= 32 && d <= 256) return true;
  if (n <= round) return false;
  return k <= 32 || d <= 256 || (n - 1) / round % 2 == 1 || n > 8 * round;
}
int launch_nearest(fa_ctx* ctx, const float* x, int64_t n, const float* c, int64_t k, int d, float* sim,
                   int32_t* assign, float* simil) {
  if (nearest_fused_ok(ctx, x, n, c, k, d)) {
    const dim3 grid((unsigned)((n + 127) / 128)), block(256);
    if (k <= 32) hipLaunchKernelGGL(nearest_kernel<1>, grid, block, 0, ctx->stream, x, n, d, c, (int)k, assign, simil);
    else hipLaunchKernelGGL(nearest_kernel<2>, grid, block, 0, ctx->stream, x, n, d, c, (int)k, assign, simil);
  } else {
    if (const int rc = launch_sim(ctx, x, n, c, k, d, sim)) return rc;
    hipLaunchKernelGGL(argmax_rows_kernel, dim3(row_blocks(n)), dim3(kRowWG), 0, ctx->stream, (const float*)sim, n,
                       (int)k, assign, simil);
  }
  FA_CHECK_LAUNCH(ctx);
  return FA_OK;
}

}  // namespace
}  // namespace fa

using fa::set_error;
using namespace fa::slots;

extern "C" {

int fa_cluster_normalize_dev(fa_ctx* ctx, const float* x, int64_t n, int32_t d, float* out) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "Normalize", n, d))) return rc;
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "cluster");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  return fa::launch_normalize(ctx, x, n, d, out);
}

int fa_cluster_normalize(fa_ctx* ctx, const float* x, int64_t n, int32_t d, float* out) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "Normalize", n, d))) return rc;
  if (n == 0 || d == 0) return FA_OK;
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "cluster");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  void* dx;
  const size_t bytes = (size_t)n * d * 4;
  if ((rc = fa::stage_h2d(ctx, S_CL_X, x, bytes, &dx))) return rc;
  if ((rc = fa::launch_normalize(ctx, (const float*)dx, n, d, (float*)dx))) return rc;
  FA_HIP_CHECK(ctx, hipMemcpyAsync(out, dx, bytes, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return FA_OK;
}

int fa_cluster_nearest_dev(fa_ctx* ctx, const float* x, int64_t n, const float* centres, int64_t k, int32_t d,
                           int32_t* index, float* similarity) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "Nearest", n, d))) return rc;
  if (k <= 0 || k > INT32_MAX)
    return set_error(ctx, FA_ERR_ARG, "Argmax: cannot reduce empty dimension 1 of shape [%lld %lld]", (long long)n,
                     (long long)k);
  if (d <= 0) return set_error(ctx, FA_ERR_ARG, "Nearest: rows of length %d", d);
  if (n == 0) return FA_OK;
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "Nearest");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  fa::DevBuf& ws = ctx->slot(S_CL_WORK);
  if (!fa::nearest_fused_ok(ctx, x, n, centres, k, d) && (rc = ws.ensure(ctx, (size_t)n * k * 4))) return rc;
  return fa::launch_nearest(ctx, x, n, centres, k, d, ws.as<float>(), index, similarity);
}

int fa_cluster_nearest(fa_ctx* ctx, const float* x, int64_t n, const float* centres, int64_t k, int32_t d,
                       int32_t* index, float* similarity) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "Nearest", n, d))) return rc;
  if (k <= 0 || k > INT32_MAX)
    return set_error(ctx, FA_ERR_ARG, "Argmax: cannot reduce empty dimension 1 of shape [%lld %lld]", (long long)n,
                     (long long)k);
  if (d <= 0) return set_error(ctx, FA_ERR_ARG, "Nearest: rows of length %d", d);
  if (n == 0) return FA_OK;
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "Nearest");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  void *dx, *dc;
  if ((rc = fa::stage_h2d(ctx, S_CL_X, x, (size_t)n * d * 4, &dx))) return rc;
  if ((rc = fa::stage_h2d(ctx, S_CL_C, centres, (size_t)k * d * 4, &dc))) return rc;
  fa::DevBuf& ob = ctx->slot(S_CL_OUT);
  if ((rc = ob.ensure(ctx, (size_t)n * 8))) return rc;
  int32_t* di = ob.as<int32_t>();
  float* ds = (float*)(di + n);
  if ((rc = fa_cluster_nearest_dev(ctx, (const float*)dx, n, (const float*)dc, k, d, di, ds))) return rc;
  FA_HIP_CHECK(ctx, hipMemcpyAsync(index, di, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipMemcpyAsync(similarity, ds, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return FA_OK;
}

int fa_cluster_kmeans_dev(fa_ctx* ctx, const float* x, int64_t n, int32_t d, int32_t k, int32_t iters,
                          uint64_t seed, float* centres, int32_t* assignment, float* similarity, int32_t* sizes,
                          int32_t* iterations) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "KMeans", n, d))) return rc;
  if (k <= 0 || k > n) return set_error(ctx, FA_ERR_ARG, "cluster: k must be between 1 and the number of rows");
  if (d <= 0) return set_error(ctx, FA_ERR_ARG, "KMeans: rows of length %d", d);
  if (!iterations) return set_error(ctx, FA_ERR_ARG, "KMeans: iterations is NULL");
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "cluster");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int nchunks = (int)((n + fa::kChunk - 1) / fa::kChunk);

  // workspace: raw centres, sums [k x d]; best [n]; w [n] f64; partial
  // sums of w; sim [n x k]; chunk counts [nchunks x k]; chunk change counts;
  // offsets [k]; list [n]; previous assignment [n]; changed; chosen [k]
  const int nparts = (int)((n + fa::kSumBlock - 1) / fa::kSumBlock);
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t o = off;
    off += fa::align256(bytes);
    return o;
  };
  const size_t o_raw = take((size_t)k * d * 4), o_sums = take((size_t)k * d * 4), o_best = take((size_t)n * 4),
               o_w = take((size_t)n * 8), o_part = take((size_t)nparts * 8), o_sim = take(fa::nearest_fused_ok(ctx, x, n, centres, k, d) ? 0 : (size_t)n * k * 4),
               o_cnt = take((size_t)nchunks * k * 4), o_chg = take((size_t)nchunks * 4), o_offs = take((size_t)k * 4),
               o_list = take((size_t)n * 4), o_prev = take((size_t)n * 4), o_summary = take(((size_t)k + 1) * 4),
               o_chosen = take((size_t)k * 4);
  fa::DevBuf& ws = ctx->slot(S_CL_WORK);
  if ((rc = ws.ensure(ctx, off))) return rc;
  char* base = ws.as<char>();
  float* raw = (float*)(base + o_raw);
  float* sums = (float*)(base + o_sums);
  float* best = (float*)(base + o_best);
  double* w = (double*)(base + o_w);
  double* part = (double*)(base + o_part);
  float* sim = (float*)(base + o_sim);
  int32_t* cnt = (int32_t*)(base + o_cnt);
  int32_t* chg = (int32_t*)(base + o_chg);
  int32_t* offs = (int32_t*)(base + o_offs);
  int32_t* list = (int32_t*)(base + o_list);
  int32_t* prev = (int32_t*)(base + o_prev);
  int32_t* summary = (int32_t*)(base + o_summary);
  int32_t* chosen = (int32_t*)(base + o_chosen);

  // k-means++ seeding (cluster.go:47-85); every draw up front
  fa::GoPCG rng{seed, seed ^ 0x9e3779b97f4a7c15ULL};
  const int64_t first = (int64_t)rng.IntN((uint64_t)n);
  std::vector<double> u((size_t)k, 0.0);
  for (int r = 1; r < k; r++) u[r] = rng.Float64();
  FA_HIP_CHECK(ctx, hipMemcpyAsync(raw, x + first * d, (size_t)d * 4, hipMemcpyDeviceToDevice, st));
  hipLaunchKernelGGL(fa::fill_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, best, n, -1.f);
  FA_CHECK_LAUNCH(ctx);
  for (int r = 1; r < k; r++) {
    hipLaunchKernelGGL(fa::kpp_weights_kernel, dim3((unsigned)nparts), dim3(64 * fa::kKppWaves), 0, st, x, n, (int)d,
                       (const float*)(raw + (size_t)(r - 1) * d), best, w, part);
    FA_CHECK_LAUNCH(ctx);
    if (nparts <= 256)
      hipLaunchKernelGGL(fa::kpp_pick_kernel<256>, dim3(1), dim3(256), 0, st, (const double*)w, n,
                         (const double*)part, nparts, u[r], x, (int)d, raw + (size_t)r * d, chosen + r);
    else
      hipLaunchKernelGGL(fa::kpp_pick_kernel<1024>, dim3(1), dim3(1024), 0, st, (const double*)w, n,
                         (const double*)part, nparts, u[r], x, (int)d, raw + (size_t)r * d, chosen + r);
    FA_CHECK_LAUNCH(ctx);
  }
  if ((rc = fa::launch_normalize(ctx, raw, k, d, centres))) return rc;

  // Lloyd rounds (cluster.go:86-129)
  FA_HIP_CHECK(ctx, hipMemsetAsync(assignment, 0, (size_t)n * 4, st));
  FA_HIP_CHECK(ctx, hipMemsetAsync(prev, 0, (size_t)n * 4, st));
  FA_HIP_CHECK(ctx, hipMemsetAsync(similarity, 0, (size_t)n * 4, st));
  FA_HIP_CHECK(ctx, hipMemsetAsync(sizes, 0, (size_t)k * 4, st));
  std::vector<int32_t> host((size_t)k + 1);
  int it_done = 0;
  for (int it = 1; it <= iters; it++) {
    it_done = it;
    if ((rc = fa::launch_nearest(ctx, x, n, centres, k, d, sim, assignment, similarity))) return rc;
    hipLaunchKernelGGL(fa::count_kernel, dim3((unsigned)nchunks), dim3(fa::kChunk), 0, st,
                       (const int32_t*)assignment, prev, n, (int)k, nchunks, cnt, chg);
    FA_CHECK_LAUNCH(ctx);
    hipLaunchKernelGGL(fa::chunk_scan_kernel, dim3((unsigned)k), dim3(256), 0, st, cnt, nchunks, sizes);
    FA_CHECK_LAUNCH(ctx);
    hipLaunchKernelGGL(fa::offsets_kernel, dim3(1), dim3(1024), 0, st, (const int32_t*)sizes, (int)k, offs,
                       (const int32_t*)chg, nchunks, summary);
    FA_CHECK_LAUNCH(ctx);
    hipLaunchKernelGGL(fa::scatter_kernel, dim3((unsigned)nchunks), dim3(64), 0, st, (const int32_t*)assignment, n,
                       (int)k, nchunks, (const int32_t*)offs, (const int32_t*)cnt, list);
    FA_CHECK_LAUNCH(ctx);
    hipLaunchKernelGGL(fa::colsum_kernel, dim3((unsigned)k, (unsigned)((d + 63) / 64)), dim3(64), 0, st, x, (int)d,
                       (const int32_t*)list, (const int32_t*)offs, (const int32_t*)sizes, sums);
    FA_CHECK_LAUNCH(ctx);
    FA_HIP_CHECK(ctx, hipMemcpyAsync(host.data(), summary, ((size_t)k + 1) * 4, hipMemcpyDeviceToHost, st));
    FA_HIP_CHECK(ctx, hipStreamSynchronize(st));
    for (int c = 0; c < k; c++) {
      if (host[c] != 0) continue;
      hipLaunchKernelGGL(fa::worst_kernel, dim3(1), dim3(1024), 0, st, similarity, n, x, (int)d,
                         sums + (size_t)c * d);
      FA_CHECK_LAUNCH(ctx);
    }
    if ((rc = fa::launch_normalize(ctx, sums, k, d, centres))) return rc;
    if (host[k] == 0 && it > 1) break;
  }
  *iterations = it_done;
  return FA_OK;
}

int fa_cluster_kmeans(fa_ctx* ctx, const float* x, int64_t n, int32_t d, int32_t k, int32_t iters, uint64_t seed,
                      float* centres, int32_t* assignment, float* similarity, int32_t* sizes, int32_t* iterations) {
  if (!ctx) return set_error(ctx, FA_ERR_ARG, "cluster: ctx is NULL");
  int rc;
  if ((rc = fa::check_rows(ctx, "KMeans", n, d))) return rc;
  if (k <= 0 || k > n) return set_error(ctx, FA_ERR_ARG, "cluster: k must be between 1 and the number of rows");
  if (d <= 0) return set_error(ctx, FA_ERR_ARG, "KMeans: rows of length %d", d);
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "cluster");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  void* dx;
  if ((rc = fa::stage_h2d(ctx, S_CL_X, x, (size_t)n * d * 4, &dx))) return rc;
  fa::DevBuf& ob = ctx->slot(S_CL_OUT);
  const size_t cb = fa::align256((size_t)k * d * 4), nb = fa::align256((size_t)n * 4);
  if ((rc = ob.ensure(ctx, cb + 2 * nb + (size_t)k * 4))) return rc;
  char* o = ob.as<char>();
  float* dcent = (float*)o;
  int32_t* dassign = (int32_t*)(o + cb);
  float* dsim = (float*)(o + cb + nb);
  int32_t* dsizes = (int32_t*)(o + cb + 2 * nb);
  int32_t it = 0;
  if ((rc = fa_cluster_kmeans_dev(ctx, (const float*)dx, n, d, k, iters, seed, dcent, dassign, dsim, dsizes, &it)))
    return rc;
  FA_HIP_CHECK(ctx, hipMemcpyAsync(centres, dcent, (size_t)k * d * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipMemcpyAsync(assignment, dassign, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipMemcpyAsync(similarity, dsim, (size_t)n * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipMemcpyAsync(sizes, dsizes, (size_t)k * 4, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  if (iterations) *iterations = it;
  return FA_OK;
}

}  // extern "C"
