// The EmbeddingGemma encoder on one GPU: bf16-resident weights, packed
// variable-length token rows, and the forward pass
//   gather*sqrt(d) -> 24 x [qkv GEMM, qk-norm+RoPE, attention, o GEMM,
//   post-norm+residual(+next pre-norm), gate|up GEMM with GeGLU epilogue,
//   down GEMM, post-norm+residual(+next pre-norm)] -> mean pool -> Dense head
//   -> L2
// following models/gemma/embed.go:160-240,381-475 and model.go:76-232.
// Variant 2 (EmbeddingGemma 2, embed.go:247-377) adds per-layer head dims
// and key/value heads, the v norm, the per-layer inputs (one projection of
// the scaled embeddings, normalised per layer), each layer's
// per-layer-input block (gate GEMM with GELU and the layer's input in the
// epilogue, projection GEMM, post-norm + residual, times the layer scalar)
// and the embedding projection of the pooled vector.
//
// Layout in HBM (M = sum of valid lengths; padding rows are never stored):
//   x   [M, d] fp32   residual stream
//   xn  [M, d] fp32   RMSNorm(x; 1+g) feeding the next product (the
//                     reference folds 1+g into the weights and applies the
//                     row scale in the product's epilogue, model.go:210-222,
//                     embed.go:193-197; the values agree to rounding)
//   qkv [M, (H+2Hkv)*D] fp32   q | k | v per token, normed and rotated in place
//   att [M, H*D] fp32, o [M, d] fp32, gu [M, F] fp32
// Weights: [out, in] bf16 as in the checkpoint; q|k|v stacked into one
// [(H+2Hkv)*D, d] matrix, gate and up interleaved in 32-row groups into one
// [2F, d] matrix (see gemm.hip), 1+w norm vectors in fp32.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "fa_internal.h"
#include "plan.h"

namespace fa {

namespace {

constexpr int64_t kAttnSplitRows = 1024;  // key-split attention only for batches up to this many tokens

bool bf16_exact(float f, uint16_t* out) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if (u & 0xFFFFu) return false;
  *out = (uint16_t)(u >> 16);
  return true;
}

// A weight matrix [rows, cols] in HBM: bf16 values as stored in the
// checkpoint (terms = 1), or, once any of its float32 values is not
// bf16-exact, three bf16 planes hi, mid, lo of the float32 values (terms = 3,
// rows*cols elements apart; hi + mid + lo is the value exactly), which the
// products take through the six-term split kernel.
struct Mat {
  uint16_t* p = nullptr;
  int64_t rows = 0, cols = 0;
  int terms = 1;
  int64_t plane() const { return rows * cols; }
  // the values times h_scale in fp16 (prepare_h2), for the products on split
  // activations
  uint16_t* h = nullptr;
  float h_scale = 1.f;
};

struct Layer {
  int D = 0, Hkv = 0, width = 0;  // head dim, key/value heads, q|k|v width (H+2Hkv)*D
  bool sliding = true;
  const float *cos_t = nullptr, *sin_t = nullptr;  // RoPE tables of this layer's base and D
  Mat wqkv;   // [(H+2Hkv)*D, d]
  Mat wo;     // [d, H*D]
  Mat wgu;    // [2F, d], 32-row groups gate/up alternating
  Mat wdown;  // [d, F]
  float *g_in = nullptr, *g_post_attn = nullptr, *g_pre_ffn = nullptr, *g_post_ffn = nullptr;
  float *g_q = nullptr, *g_k = nullptr;
  // variant 2: per-layer-input block and layer scalar
  Mat wple_gate;  // [P, d]
  Mat wple_proj;  // [d, P]
  float* g_ple_post = nullptr;
  float scalar = 1.f;
  // prepare_h2: the powers of two by which the split operands of this
  // layer's products are scaled (normed inputs of q|k|v and gate|up,
  // attention output, GeGLU output; variant 2: the residual stream before
  // the per-layer-input block and the block's gated input)
  float s_in = 0, s_att = 0, s_ffn = 0, s_gu = 0, s_x = 0, s_ple = 0;
  // and of the tile attention's q and key images (its value images: s_att)
  float s_q = 0, s_k = 0;
};

struct KernelStat {
  int64_t launches = 0;
  double ms = 0, flops = 0, bytes = 0;
};

struct PendingEvent {
  hipEvent_t a, b;
  int kind;
  double flops, bytes;
};

}  // namespace
}  // namespace fa

struct fa_model {
  fa_ctx* ctx = nullptr;
  fa_gemma_config cfg{};
  int variant = 0;
  int max_width = 0, max_hd = 0;  // widest q|k|v row, widest attention output H*D
  int P = 0, E = 0;               // variant 2: per-layer input width, embedding projection width
  fa::Mat wple_model;             // variant 2: [layers*P, d]
  float* g_ple_norm = nullptr;    // variant 2: [P]
  fa::Mat wemb_proj;              // variant 2: [E, d]
  std::vector<void*> allocations;
  fa::Mat embed;
  std::vector<fa::Layer> layers;
  float* g_final = nullptr;
  std::vector<fa::Mat> dense;
  std::vector<int> dense_in, dense_out, dense_act;  // dense_act: FA_ACT_NONE or FA_ACT_TANH
  float *cos_local = nullptr, *sin_local = nullptr, *cos_global = nullptr, *sin_global = nullptr;
  int d_local = 0, d_global = 0;  // head dims of the sliding and the full layers
  std::set<std::string> seen;
  bool finalized = false;
  // the layers' products run on split activations (prepare_h2): every layer
  // matrix is exact in fp16 and every operand's range is known
  bool h2 = false;
  // the split-fp16 tile attention can run (prepare_h2: every head_dim-256
  // layer's q, keys and values have a known range)
  bool tiles = false;
  float s_x0 = 0;  // variant 2: scale of the scaled embeddings
  // workspace
  fa::DevBuf ws, plan_dev;
  int64_t ws_rows = 0, ws_seqs = 0;
  int32_t* plan_host = nullptr;  // pinned
  size_t plan_host_ints = 0;
  hipEvent_t plan_done = nullptr;
  bool plan_pending = false;
  // streams of micro-batches 1.. (micro-batch 0 runs on the context's
  // stream), the fork event and one join event per extra stream
  hipStream_t mb_stream[fa::kMaxMicrobatches] = {};
  hipEvent_t ev_fork = nullptr, ev_join[fa::kMaxMicrobatches] = {};
  std::vector<int> seq_order;                 // plan scratch
  std::vector<int> plan_layer_D, plan_layer_Hkv;  // plan inputs: each layer's head dim, kv heads
  fa::DevBuf ids_dev, out_dev;
  // pinned staging of the host entry points' ids and results (asynchronous
  // copies; the entry points synchronise before returning)
  void* io_host = nullptr;
  size_t io_host_bytes = 0;
  // profiling
  bool profiling = false;
  std::vector<hipEvent_t> event_pool;
  std::vector<fa::PendingEvent> pending;
  fa::KernelStat stats[FA_K_COUNT];
};

namespace fa {
namespace {

int alloc_dev(fa_model* m, size_t bytes, void** out) {
  hipError_t e = hipMalloc(out, bytes ? bytes : 1);
  if (e != hipSuccess) return set_error(m->ctx, FA_ERR_OOM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
  m->allocations.push_back(*out);
  return FA_OK;
}

// Frees one of the model's allocations (a matrix promoted to three planes).
void free_dev(fa_model* m, void* ptr) {
  for (auto& a : m->allocations)
    if (a == ptr) {
      (void)hipFree(a);
      a = m->allocations.back();
      m->allocations.pop_back();
      return;
    }
}

// B operand of a product over w's rows [row0, ...): one bf16 plane or three.
void set_b(GemmArgs& g, const Mat& w, int64_t row0 = 0) {
  g.b = w.p + row0 * w.cols;
  g.ldb = w.cols;
  g.b_terms = w.terms;
  g.b_plane = w.plane();
}

// 2-norms of the rows of matrices (a three-plane one's hi plane, within 1 % of
// the whole), each column weighted by t (all ones if empty).
struct RowNorms {
  struct Job {
    const Mat* w;
    std::vector<float> t;
    std::vector<float> out;
  };
  std::vector<Job> jobs;
  int add(const Mat& w, std::vector<float> t = {}) {
    jobs.push_back({&w, std::move(t), {}});
    return (int)jobs.size() - 1;
  }
  int run(fa_ctx* ctx, hipStream_t s) {
    size_t nt = 0, rows = 0;
    for (auto& j : jobs) {
      nt += j.t.size();
      rows += j.w->rows;
    }
    std::vector<float> t, host(rows);
    for (auto& j : jobs) t.insert(t.end(), j.t.begin(), j.t.end());
    DevBuf buf;
    int rc = buf.ensure(ctx, (nt + rows) * 4);
    auto work = [&]() -> int {
      if (nt) FA_HIP_CHECK(ctx, hipMemcpyAsync(buf.ptr, t.data(), nt * 4, hipMemcpyHostToDevice, s));
      size_t at = 0, out = nt;
      for (auto& j : jobs) {
        const float* jt = j.t.empty() ? nullptr : buf.as<float>() + at;
        if (const int r = launch_h2_row_norms(ctx, j.w->p, j.w->rows, j.w->cols, jt, buf.as<float>() + out, s)) return r;
        at += j.t.size();
        out += j.w->rows;
      }
      FA_HIP_CHECK(ctx, hipMemcpyAsync(host.data(), buf.as<float>() + nt, rows * 4, hipMemcpyDeviceToHost, s));
      FA_HIP_CHECK(ctx, hipStreamSynchronize(s));
      return FA_OK;
    };
    if (!rc) rc = work();
    buf.release();
    if (rc) return rc;
    size_t at = 0;
    for (auto& j : jobs) {
      j.out.assign(host.begin() + at, host.begin() + at + j.w->rows);
      at += j.w->rows;
    }
    return FA_OK;
  }
};

// Decides whether the layers' products can run on split activations
// (gemm_h2.hip) and the head_dim-256 layers on the tile attention, and
// prepares both: m->h2, m->tiles.
//
// Each split operand needs a bound, from which its power of two is taken (the
// bound just below 2^15). A normed row has 2-norm at most sqrt(d) before its
// gains g, so a product with weights w of it is at most sqrt(d) |w o g|, the
// gains taken into the row's norm (gains and weights may make up for each
// other); attention outputs are convex combinations of values; |gelu(a) b| <=
// |a| |b|; the residual stream is a sum of normed rows.
//
// A bound far above the values themselves costs them their low bits: an
// element of the products' operands is off by 2^-36 of the scaled range where
// that is more than 2^-23 of it, and one of the attention's, whose lo terms
// have no scale of their own, by 2^-25. What that adds to an output is the
// row's norm times it, to be held against the output itself, the row's norm
// with each column weighted by its operand's typical size: the gain for a
// normed row, the same with one in 32 for attention outputs (averaged over
// keys), a quarter of the two factors' product for GeGLU. It has to stay below
// 2^-28 (attention 2^-26) in every row: a sixteenth of a float32 rounding,
// which leaves room for operands that far below their typical size (evenly
// sized gains and weights come to 2^-40 to 2^-45, and 2^-34). The same for the
// weights: w 2^-11, the factor of the lo terms, is rounded to 2^-24 of the
// scaled range where w is below 2^-21 of its matrix's largest.
//
// Models that do not hold this keep the three-term products, or the fp32
// attention, as do those with non-finite weights; the products also need
// every layer matrix bf16-exact (terms == 1) and exact in fp16 after one power
// of two for the matrix (its largest value just below 2^15). Only then are the
// fp16 copies made.
int range_h2(fa_model* m, std::vector<Mat*>& mats) {
  fa_ctx* ctx = m->ctx;
  const fa_gemma_config& c = m->cfg;
  const bool v2 = m->variant == 2;
  const int d = c.hidden_size, H = c.num_attention_heads, F = c.intermediate_size, P = m->P;
  for (auto& L : m->layers) {
    mats.insert(mats.end(), {&L.wqkv, &L.wo, &L.wgu, &L.wdown});
    if (v2) mats.insert(mats.end(), {&L.wple_gate, &L.wple_proj});
  }
  if (v2) mats.push_back(&m->wple_model);
  bool ok = gemm_h2_enabled();
  for (Mat* w : mats) ok = ok && w->terms == 1 && w->cols % 32 == 0;
  // largest |w| of each matrix (and of the embedding table)
  const size_t nm = mats.size();
  DevBuf tmp;
  const size_t head = (2 * (nm + 1) + 63) / 64 * 64;
  int rc = tmp.ensure(ctx, head * 4);
  std::vector<uint32_t> host(head);
  hipStream_t s = ctx->stream;
  uint32_t* bits = tmp.as<uint32_t>();
  auto largest = [&]() -> int {
    int r;
    if ((r = launch_zero(ctx, bits, head * 4, s))) return r;
    for (size_t i = 0; i < nm; i++)
      if ((r = launch_h2_absmax(ctx, mats[i]->p, mats[i]->plane(), bits + i, s))) return r;
    if ((r = launch_h2_absmax(ctx, m->embed.p, m->embed.plane(), bits + nm, s))) return r;
    FA_HIP_CHECK(ctx, hipMemcpyAsync(host.data(), bits, head * 4, hipMemcpyDeviceToHost, s));
    FA_HIP_CHECK(ctx, hipStreamSynchronize(s));
    return FA_OK;
  };
  if (!rc) rc = largest();
  auto value = [&](size_t i) {
    const uint32_t u = host[i] << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
  };
  // the power of two that takes bound b just below 2^15; 0 if there is none
  auto pow2_for = [](double b) -> float {
    if (!(b > 0) || !std::isfinite(b)) return 0.f;
    const int e = 14 - std::ilogb(b * 1.0001);
    return e < -100 || e > 100 ? 0.f : std::ldexp(1.f, e);
  };
  ok = ok && !rc;
  for (size_t i = 0; i < nm && ok; i++) {
    const float mx = value(i);
    mats[i]->h_scale = mx == 0.f ? 1.f : pow2_for(mx);
    ok = mats[i]->h_scale != 0.f;
    if (ok) rc = launch_h2_convert(ctx, mats[i]->p, mats[i]->plane(), mats[i]->h_scale, nullptr, bits + nm + 1 + i, s);
    if (rc) ok = false;
  }
  if (ok) {
    std::vector<uint32_t> bad(nm);
    if (hipMemcpyAsync(bad.data(), bits + nm + 1, nm * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      rc = set_error(ctx, FA_ERR_HIP, "gemma: reading the weights' range failed");
    for (uint32_t b : bad) ok = ok && b == 0;
  }
  tmp.release();
  if (rc) return rc;

  // gains, as absolute values (a non-finite one: no bound, nothing is split)
  typedef std::vector<float> Vec;
  bool finite = true;
  auto gains = [&](const float* dev, int n) {
    Vec v(n);
    finite = finite && hipMemcpy(v.data(), dev, (size_t)n * 4, hipMemcpyDeviceToHost) == hipSuccess;
    for (float& x : v) {
      finite = finite && std::isfinite(x);
      x = std::fabs(x);
    }
    return v;
  };
  auto norm = [](const Vec& v) {
    double t = 0;
    for (float x : v) t += (double)x * x;
    return std::sqrt(t);
  };
  auto top = [](const Vec& v) {  // +inf if one is not finite
    double t = 0;
    for (float x : v) t = std::isfinite(x) ? std::max(t, (double)x) : INFINITY;
    return t;
  };
  const double rd = std::sqrt((double)d);
  struct Range {  // a layer's operands: typical sizes, and jobs of the two passes below
    Vec g_in, g_ffn, g_q, g_k, att, gu, x, xb, ple;
    int qkv, qkv_g, o, o_t, gu_, gu_g, down, down_t, gate, gate_t, gate_b, proj, proj_t;
  };
  std::vector<Range> rs(m->layers.size());
  RowNorms first, second;
  const Vec g_ple = v2 ? gains(m->g_ple_norm, P) : Vec();
  // variant 2's products also read the residual stream: per column, a bound
  // and the typical square
  Vec xb(v2 ? d : 0, (float)(value(nm) * 1.01 * rd)), x2(v2 ? d : 0);
  const int emb = v2 ? first.add(m->embed) : 0, model_w = v2 ? first.add(m->wple_model) : 0;
  for (size_t l = 0; l < rs.size(); l++) {
    Layer& L = m->layers[l];
    Range& r = rs[l];
    r.g_in = gains(L.g_in, d);
    r.g_ffn = gains(L.g_pre_ffn, d);
    r.g_q = gains(L.g_q, L.D);
    r.g_k = gains(L.g_k, L.D);
    r.qkv = first.add(L.wqkv);
    r.qkv_g = first.add(L.wqkv, r.g_in);
    r.o = first.add(L.wo);
    r.gu_ = first.add(L.wgu);
    r.gu_g = first.add(L.wgu, r.g_ffn);
    r.down = first.add(L.wdown);
    if (!v2) continue;
    const Vec ga = gains(L.g_post_attn, d), gf = gains(L.g_post_ffn, d), gp = gains(L.g_ple_post, d);
    for (int j = 0; j < d; j++) {
      xb[j] += (float)(rd * (ga[j] + gf[j]));
      x2[j] += ga[j] * ga[j] + gf[j] * gf[j];
    }
    r.xb = xb;
    for (int j = 0; j < d; j++) r.x.push_back(std::sqrt(x2[j]));
    const float sc = std::fabs(L.scalar);
    for (int j = 0; j < d; j++) {
      xb[j] = (float)((xb[j] + rd * gp[j]) * sc);
      x2[j] = (x2[j] + gp[j] * gp[j]) * sc * sc;
    }
    r.gate = first.add(L.wple_gate);
    r.gate_t = first.add(L.wple_gate, r.x);
    r.gate_b = first.add(L.wple_gate, r.xb);
    r.proj = first.add(L.wple_proj);
  }
  if ((rc = first.run(ctx, s))) return rc;
  if (!finite) return FA_OK;
  auto out1 = [&](int j) -> const Vec& { return first.jobs[j].out; };
  for (size_t l = 0; l < rs.size(); l++) {
    Layer& L = m->layers[l];
    Range& r = rs[l];
    const Vec &nv = out1(r.qkv_g), &ng = out1(r.gu_g);
    L.s_in = pow2_for(rd * top(r.g_in));
    L.s_ffn = pow2_for(rd * top(r.g_ffn));
    double att = v2 ? std::sqrt((double)L.D) : 0, gu = 0;
    for (int h = 0; h < H; h++)
      for (int i = 0; i < L.D; i++) {
        const float n = v2 ? 1.f : nv[(size_t)(H + L.Hkv + h / (H / L.Hkv)) * L.D + i];
        if (!v2) att = std::isfinite(n) ? std::max(att, 1.01 * rd * n) : INFINITY;
        r.att.push_back(n / 32);
      }
    for (int f = 0; f < F; f++) {
      const int64_t row = f / 32 * 64 + f % 32;  // gate rows first in each 64-row group, then up
      const double p = (double)ng[row] * ng[row + 32];
      gu = std::isfinite(p) ? std::max(gu, 1.02 * d * p) : INFINITY;
      r.gu.push_back((float)(p / 4));
    }
    L.s_att = pow2_for(att);
    L.s_gu = pow2_for(gu);
    r.o_t = second.add(L.wo, r.att);
    r.down_t = second.add(L.wdown, r.gu);
    if (!v2) continue;
    double ple = 0;
    for (int p = 0; p < P; p++) {
      const double b = rd * out1(r.gate_b)[p] * std::sqrt((double)P) * g_ple[p];  // sum |w x| <= sqrt(d) |w o xb|
      ple = std::isfinite(b) ? std::max(ple, 1.01 * b) : INFINITY;
      r.ple.push_back(out1(r.gate_t)[p] * g_ple[p] / 4);
    }
    L.s_x = pow2_for(top(r.xb));
    L.s_ple = pow2_for(ple);
    r.proj_t = second.add(L.wple_proj, r.ple);
  }
  if ((rc = second.run(ctx, s))) return rc;
  auto out2 = [&](int j) -> const Vec& { return second.jobs[j].out; };

  // whether a product whose operand carries scale a and has typical sizes t
  // holds the limit in every row: plain and typical row norms n, nt
  auto holds = [&](const Mat& w, const Vec& n, const Vec& nt, const Vec& t, float a) {
    if (a == 0.f) return false;
    const double act = 0x1p-36 / a, wt = 0x1p-25 / w.h_scale * norm(t);
    for (size_t i = 0; i < n.size(); i++)
      if (nt[i] != 0.f && !(act * n[i] + wt <= 0x1p-28 * nt[i])) return false;
    return true;
  };
  bool tiles = true;
  for (size_t l = 0; l < rs.size(); l++) {
    Layer& L = m->layers[l];
    const Range& r = rs[l];
    ok = ok && holds(L.wqkv, out1(r.qkv), out1(r.qkv_g), r.g_in, L.s_in) &&
         holds(L.wo, out1(r.o), out2(r.o_t), r.att, L.s_att) &&
         holds(L.wgu, out1(r.gu_), out1(r.gu_g), r.g_ffn, L.s_ffn) &&
         holds(L.wdown, out1(r.down), out2(r.down_t), r.gu, L.s_gu);
    if (v2)
      ok = ok && holds(L.wple_gate, out1(r.gate), out1(r.gate_t), r.x, L.s_x) &&
           holds(L.wple_proj, out1(r.proj), out2(r.proj_t), r.ple, L.s_ple);
    if (L.D != 256) continue;
    // a rotated row keeps its norm; its dims j and j + 128 share their gains
    L.s_q = pow2_for(16 * top(r.g_q));
    L.s_k = pow2_for(16 * top(r.g_k));
    if (L.s_q == 0 || L.s_k == 0 || L.s_att == 0) {
      tiles = false;
      continue;
    }
    double qq = 0, kk = 0, qk = 0;
    for (int j = 0; j < 128; j++) {
      const double q2 = (double)r.g_q[j] * r.g_q[j] + (double)r.g_q[j + 128] * r.g_q[j + 128];
      const double k2 = (double)r.g_k[j] * r.g_k[j] + (double)r.g_k[j + 128] * r.g_k[j + 128];
      qq += q2;
      kk += k2;
      qk += q2 * k2 / 2;
    }
    tiles = tiles && 0x1p-25 * (std::sqrt(kk) / L.s_q + std::sqrt(qq) / L.s_k) <= 0x1p-26 * std::sqrt(qk);
    for (size_t i = 0; i < out1(r.o).size(); i++)  // (the values are not averaged yet: 32 r.att)
      tiles = tiles && (out2(r.o_t)[i] == 0.f || 0x1p-25 / L.s_att * out1(r.o)[i] <= 0x1p-26 * 32 * out2(r.o_t)[i]);
  }
  if (v2) {
    // the embeddings as an operand: a token's values have rms |its row|, and
    // its result is normed, so the least row sets the limit, down to where the
    // norm's eps outweighs the result (|w| |row| / sqrt(d) < sqrt(eps))
    m->s_x0 = pow2_for(value(nm) * 1.01 * rd);
    float least = INFINITY;
    const double w_top = top(out1(model_w));
    const float from = w_top > 0 ? (float)(rd * std::sqrt((double)c.rms_norm_eps) / w_top) : 0.f;
    for (float n : out1(emb))
      if (n != 0.f) least = std::min(least, std::max(n, from));
    ok = ok && (least == INFINITY || holds(m->wple_model, out1(model_w), out1(model_w), Vec(d, 1.f), m->s_x0 * least));
  }
  m->tiles = tiles;
  if (!ok) return FA_OK;
  for (Mat* w : mats) {
    if (!w->h) {
      void* np = nullptr;
      if ((rc = alloc_dev(m, (size_t)w->plane() * 2, &np))) return rc;
      w->h = (uint16_t*)np;
    }
    if ((rc = launch_h2_convert(ctx, w->p, w->plane(), w->h_scale, w->h, nullptr, s))) return rc;
  }
  FA_HIP_CHECK(ctx, hipStreamSynchronize(s));
  m->h2 = true;
  return FA_OK;
}

// The copies are for speed: where they, or the scratch of the checks, find no
// memory, the model keeps the three-term products of the matrices it holds.
int prepare_h2(fa_model* m) {
  m->h2 = m->tiles = false;
  std::vector<Mat*> mats;
  int rc = range_h2(m, mats);
  if (rc == FA_ERR_OOM) {
    (void)hipGetLastError();
    rc = FA_OK;
  }
  if (!m->h2)
    for (Mat* w : mats)
      if (w->h) {
        free_dev(m, w->h);
        w->h = nullptr;
      }
  return rc;
}

// Fills the operands of a product on split activations: A scaled by a_scale.
void set_h2(GemmH2Args& g, const Mat& w, float a_scale) {
  g.b = w.h;
  g.ldb = w.cols;
  g.c_scale = 1.f / (a_scale * w.h_scale);
}

hipEvent_t take_event(fa_model* m) {
  if (!m->event_pool.empty()) {
    hipEvent_t e = m->event_pool.back();
    m->event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

// Token count from which a batch runs as micro-batches on several streams;
// FA_MICROBATCH=0 turns that off, FA_MICROBATCH=<rows> sets the threshold.
int64_t microbatch_min_rows() {
  static const int64_t v = [] {
    const char* e = std::getenv("FA_MICROBATCH");
    if (!e) return (int64_t)2048;
    const long long n = std::atoll(e);
    return n <= 0 ? INT64_MAX : (int64_t)n;
  }();
  return v;
}

// Number of micro-batches (2..kMaxMicrobatches; FA_MICROBATCH_GROUPS). Three
// measured best on MI355X at 5 517, 11 550 and 32 768 tokens (C2: 6.41 ms
// per forward on one stream, 5.49 with two groups, 5.43 with three, 5.92
// with four) and within 3 % of best at 17 923.
// FA_ATTN_KEY_PARTS=<1..8> forces the key runs of the short-batch attention
// (tuning); 0 when unset.
int attention_key_parts_forced() {
  static const int v = [] {
    const char* e = std::getenv("FA_ATTN_KEY_PARTS");
    if (!e) return 0;
    return std::max(1, std::min(std::atoi(e), kMaxKeyParts));
  }();
  return v;
}

// FA_ATTN_SHORT=0: the q/k norm pass and the fp32 attention for short
// sequences too; also with forced key runs.
bool attention_short_enabled() {
  static const bool on = [] {
    const char* e = std::getenv("FA_ATTN_SHORT");
    return !(e && e[0] == '0');
  }();
  return on && attention_key_parts_forced() == 0;
}

// FA_ATTN_ROWS=64|128 forces the tile attention's rows per item (tuning);
// 0 when unset.
int attention_rows_forced() {
  static const int v = [] {
    const char* e = std::getenv("FA_ATTN_ROWS");
    if (!e) return 0;
    const int r = std::atoi(e);
    return r == 64 || r == 128 ? r : 0;
  }();
  return v;
}

// FA_ATTN_XCD=1|0 forces the XCD-local attention item order on or off
// (tuning); 0 when unset (chosen per group).
int attention_xcd_forced() {
  static const int v = [] {
    const char* e = std::getenv("FA_ATTN_XCD");
    if (!e) return 0;
    return e[0] == '0' ? -1 : 1;
  }();
  return v;
}

// K parts of the N = hidden products (o, down) for a few-row batch whose
// small-M tiles, times four parts, still fit one per CU (FA_SMALL_KSPLIT=2
// or 4, default 4). A small-M workgroup's time is its operand loads: with
// four parts each loads half the bytes of two (at 128 rows: o 8.5 -> 7.4
// us, down 9.8 -> 8.4 us per launch; C1 1.30 -> 1.28 ms per forward, 64
// tokens 1.25 -> 1.22 ms on MI355X), for two more partial planes read by
// the residual step.
int small_ksplit() {
  static const int v = [] {
    const char* e = std::getenv("FA_SMALL_KSPLIT");
    if (!e) return 4;
    return std::atoi(e) >= 4 ? 4 : 2;
  }();
  return v;
}

// K parts of a few-row batch's q|k|v product on the fp32 attention path,
// added by the q/k norm pass (FA_QKV_KSPLIT=1 or 2, default 2): 160 instead
// of 80 workgroups at 128 rows, each loading half the operands (11.1 ->
// 9.0 us per launch; C1 1.28 -> 1.24 ms, 64 tokens 1.22 -> 1.17 ms per
// forward on MI355X), for one more read of the product in the norm pass.
int qkv_ksplit() {
  static const int v = [] {
    const char* e = std::getenv("FA_QKV_KSPLIT");
    if (!e) return 2;
    return std::atoi(e) >= 2 ? 2 : 1;
  }();
  return v;
}

// FA_TILE_MIN_ROWS=<tokens>: the tile attention from more tokens than this
// (tuning; 1 024 when unset).
int64_t tile_min_rows() {
  static const int64_t v = [] {
    const char* e = std::getenv("FA_TILE_MIN_ROWS");
    if (!e) return (int64_t)1024;
    return (int64_t)std::max(0LL, std::atoll(e));
  }();
  return v;
}

// FA_MICROBATCH_GROUPS=<2..4> forces the group count (tuning); 0 when unset.
int microbatch_count_forced() {
  static const int v = [] {
    const char* e = std::getenv("FA_MICROBATCH_GROUPS");
    if (!e) return 0;
    return std::max(2, std::min(std::atoi(e), kMaxMicrobatches));
  }();
  return v;
}

// Group count by the batch, from sweeps of 2, 3 and 4 groups on MI355X (ms
// per forward of the 24-layer model): three for most batches (32 x 64..256
// tokens: 4.45 with two or three, 4.59 with four; 256 x 16..128: 11.83, 11.61
// and 11.68), two where the mean key count per token (sum L^2 / sum L) is at
// least 1 024 (8 x 1 024..2 048: 10.36, 10.41 and 10.35) and from 24 576
// tokens (64 x 512: 24.48, 24.73 and 24.56), where each group's launches
// fill the chip. Not four: a process has four hardware queues, so with
// another stream in use (a framework's own) the fourth group waits behind
// one of the others (two layers of 8 x 1 024..2 048: 1.49 ms with four
// groups, 1.18 with two).
int microbatch_count(int64_t tokens, double sum_l2) {
  if (const int f = microbatch_count_forced()) return f;
  return tokens >= 24576 || sum_l2 >= 1024.0 * (double)tokens ? 2 : 3;
}

// HBM bytes of one residual_norm launch: the product's K parts and x
// read, x written, and the next norm's input written when there is a next
// norm.
double resnorm_bytes(int64_t rows, int64_t d, int parts, const float* g_next) {
  return (double)rows * d * 4.0 * (2.0 + parts + (g_next ? 1.0 : 0.0));
}

// Brackets one launch with events when profiling.
struct Probe {
  fa_model* m;
  hipEvent_t a = nullptr;
  int kind;
  double flops, bytes;
  Probe(fa_model* mm, int k, double f, double b) : m(mm), kind(k), flops(f), bytes(b) {
    if (m->profiling) {
      a = take_event(m);
      if (a) (void)hipEventRecord(a, m->ctx->stream);
    }
  }
  void done() {
    if (!a) return;
    hipEvent_t b = take_event(m);
    if (!b) return;
    (void)hipEventRecord(b, m->ctx->stream);
    m->pending.push_back({a, b, kind, flops, bytes});
    a = nullptr;
  }
};

int collect_stats(fa_model* m) {
  if (m->pending.empty()) return FA_OK;
  FA_HIP_CHECK(m->ctx, hipStreamSynchronize(m->ctx->stream));
  for (auto& p : m->pending) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      KernelStat& s = m->stats[p.kind];
      s.launches++;
      s.ms += ms;
      s.flops += p.flops;
      s.bytes += p.bytes;
    }
    m->event_pool.push_back(p.a);
    m->event_pool.push_back(p.b);
  }
  m->pending.clear();
  return FA_OK;
}

// The pinned staging buffer of the host entry points, grown to at least bytes.
int io_staging(fa_model* m, size_t bytes, char** out) {
  if (bytes > m->io_host_bytes) {
    if (m->io_host) (void)hipHostFree(m->io_host);
    m->io_host = nullptr;
    m->io_host_bytes = 0;
    FA_HIP_CHECK(m->ctx, hipHostMalloc(&m->io_host, bytes, hipHostMallocDefault));
    m->io_host_bytes = bytes;
  }
  *out = static_cast<char*>(m->io_host);
  return FA_OK;
}

// Host-side check of a host batch: lengths in 1..T and every valid id inside
// the vocabulary (an out-of-range id would read outside the table).
int check_ids(fa_model* m, const int32_t* ids, const int32_t* lengths, int B, int T) {
  const int V = m->cfg.vocab_size;
  for (int b = 0; b < B; b++) {
    if (lengths[b] < 1 || lengths[b] > T)
      return set_error(m->ctx, FA_ERR_ARG, "gemma: length[%d] = %d outside 1..T=%d", b, lengths[b], T);
    for (int t = 0; t < lengths[b]; t++) {
      const int32_t id = ids[(size_t)b * T + t];
      if (id < 0 || id >= V)
        return set_error(m->ctx, FA_ERR_ARG, "gemma: token id %d at [%d,%d] outside 0..%d", id, b, t, V - 1);
    }
  }
  return FA_OK;
}

int parse_layer(const std::string& s, int nl, int* l, std::string* rest) {
  if (s.rfind("layers.", 0) != 0) return -1;
  size_t dot = s.find('.', 7);
  if (dot == std::string::npos) return -1;
  char* end = nullptr;
  long v = std::strtol(s.c_str() + 7, &end, 10);
  if (end != s.c_str() + dot || v < 0 || v >= nl) return -1;
  *l = (int)v;
  *rest = s.substr(dot + 1);
  return 0;
}

}  // namespace
}  // namespace fa

using fa::set_error;

extern "C" {

int fa_gemma_create(fa_ctx* ctx, const fa_gemma_config* cfg, fa_model** out) {
  if (!ctx || !cfg || !out) return set_error(ctx, FA_ERR_ARG, "gemma: NULL argument");
  *out = nullptr;
  const fa_gemma_config& c = *cfg;
  if (c.hidden_size <= 0 || c.num_hidden_layers <= 0 || c.num_attention_heads <= 0 || c.num_key_value_heads <= 0 ||
      c.head_dim <= 0 || c.intermediate_size <= 0 || c.vocab_size <= 0)
    return set_error(ctx, FA_ERR_ARG, "gemma: config sizes must be positive");
  if (c.variant != 0 && c.variant != 2) return set_error(ctx, FA_ERR_ARG, "gemma: variant %d not 0 or 2", c.variant);
  const bool v2 = c.variant == 2;
  if (c.hidden_size % 256 != 0 || c.hidden_size > 1024)
    return set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: hidden_size %d not in {256,512,768,1024}", c.hidden_size);
  if (c.num_hidden_layers > FA_GEMMA_MAX_LAYERS)
    return set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: %d layers, at most %d", c.num_hidden_layers, FA_GEMMA_MAX_LAYERS);
  if (!v2 && c.head_dim != 256) return set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: head_dim %d != 256", c.head_dim);
  if (c.intermediate_size % 32 != 0)
    return set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: intermediate_size %d not a multiple of 32", c.intermediate_size);
  if (c.n_dense < 0 || c.n_dense > 4) return set_error(ctx, FA_ERR_ARG, "gemma: n_dense %d outside 0..4", c.n_dense);
  if (c.max_tokens <= 0) return set_error(ctx, FA_ERR_ARG, "gemma: max_tokens must be positive");
  if (!v2 && c.query_pre_attn_scalar <= 0) return set_error(ctx, FA_ERR_ARG, "gemma: query_pre_attn_scalar must be > 0");
  if (v2 && (c.hidden_size_per_layer_input <= 0 || c.hidden_size_per_layer_input % 32 != 0))
    return set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: hidden_size_per_layer_input %d not a positive multiple of 32",
                     c.hidden_size_per_layer_input);
  if (v2 && c.embedding_dim <= 0) return set_error(ctx, FA_ERR_ARG, "gemma: embedding_dim must be positive");
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  fa_model* m = new fa_model();
  m->ctx = ctx;
  m->cfg = c;
  m->variant = c.variant;
  if (m->cfg.sliding_window_pattern <= 0) m->cfg.sliding_window_pattern = 6;
  const int d = c.hidden_size, H = c.num_attention_heads, F = c.intermediate_size, NL = c.num_hidden_layers;
  m->layers.resize(NL);
  int rc = FA_OK;
  for (int l = 0; l < NL && !rc; l++) {
    fa::Layer& L = m->layers[l];
    L.D = v2 && c.layer_head_dim[l] > 0 ? c.layer_head_dim[l] : c.head_dim;
    L.Hkv = v2 && c.layer_kv_heads[l] > 0 ? c.layer_kv_heads[l] : c.num_key_value_heads;
    L.sliding = v2 ? c.layer_sliding[l] != 0 : (l + 1) % m->cfg.sliding_window_pattern != 0;  // config.go:213-225
    L.width = (H + 2 * L.Hkv) * L.D;
    int& dt = L.sliding ? m->d_local : m->d_global;
    if (L.D != 256 && L.D != 512)
      rc = set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: layer %d head_dim %d not 256 or 512", l, L.D);
    else if (H % L.Hkv != 0)
      rc = set_error(ctx, FA_ERR_ARG, "gemma: layer %d: %d heads not a multiple of %d kv heads", l, H, L.Hkv);
    else if (dt != 0 && dt != L.D)
      rc = set_error(ctx, FA_ERR_UNSUPPORTED, "gemma: layer %d head_dim %d differs from other %s layers' %d", l, L.D,
                     L.sliding ? "sliding" : "full-attention", dt);
    dt = L.D;
    m->max_width = std::max(m->max_width, L.width);
    m->max_hd = std::max(m->max_hd, H * L.D);
  }
  if (rc) {
    delete m;
    return rc;
  }
  m->P = v2 ? c.hidden_size_per_layer_input : 0;
  m->E = v2 ? c.embedding_dim : 0;
  void* p;
  auto A = [&](size_t bytes) -> void* {
    if (rc) return nullptr;
    rc = fa::alloc_dev(m, bytes, &p);
    return rc ? nullptr : p;
  };
  auto M_ = [&](int64_t rows, int64_t cols) {
    fa::Mat w;
    w.rows = rows;
    w.cols = cols;
    w.p = (uint16_t*)A((size_t)rows * cols * 2);
    return w;
  };
  m->embed = M_(c.vocab_size, d);
  for (auto& L : m->layers) {
    L.wqkv = M_(L.width, d);
    L.wo = M_(d, (int64_t)H * L.D);
    L.wgu = M_(2LL * F, d);
    L.wdown = M_(d, F);
    L.g_in = (float*)A(d * 4);
    L.g_post_attn = (float*)A(d * 4);
    L.g_pre_ffn = (float*)A(d * 4);
    L.g_post_ffn = (float*)A(d * 4);
    L.g_q = (float*)A(L.D * 4);
    L.g_k = (float*)A(L.D * 4);
    if (v2) {
      L.wple_gate = M_(m->P, d);
      L.wple_proj = M_(d, m->P);
      L.g_ple_post = (float*)A(d * 4);
    }
  }
  m->g_final = (float*)A(d * 4);
  if (v2) {
    m->wple_model = M_((int64_t)NL * m->P, d);
    m->g_ple_norm = (float*)A(m->P * 4);
    m->wemb_proj = M_(m->E, d);
  }
  int in = v2 ? m->E : d;
  for (int i = 0; i < c.n_dense; i++) {
    if (c.dense_out[i] <= 0) rc = set_error(ctx, FA_ERR_ARG, "gemma: dense_out[%d] = %d", i, c.dense_out[i]);
    if (c.dense_act[i] != FA_ACT_NONE && c.dense_act[i] != FA_ACT_TANH)
      rc = set_error(ctx, FA_ERR_ARG, "gemma: dense_act[%d] = %d (identity or tanh)", i, c.dense_act[i]);
    m->dense_in.push_back(in);
    m->dense_out.push_back(c.dense_out[i]);
    m->dense_act.push_back(c.dense_act[i]);
    m->dense.push_back(M_(c.dense_out[i], in));
    in = c.dense_out[i];
  }
  if (m->d_local) {
    const size_t tab = (size_t)c.max_tokens * (m->d_local / 2) * 4;
    m->cos_local = (float*)A(tab);
    m->sin_local = (float*)A(tab);
  }
  if (m->d_global) {
    const size_t tab = (size_t)c.max_tokens * (m->d_global / 2) * 4;
    m->cos_global = (float*)A(tab);
    m->sin_global = (float*)A(tab);
  }
  for (auto& L : m->layers) {
    L.cos_t = L.sliding ? m->cos_local : m->cos_global;
    L.sin_t = L.sliding ? m->sin_local : m->sin_global;
  }
  if (!rc && (hipEventCreateWithFlags(&m->plan_done, hipEventDisableTiming) != hipSuccess ||
              hipEventCreateWithFlags(&m->ev_fork, hipEventDisableTiming) != hipSuccess))
    rc = set_error(ctx, FA_ERR_HIP, "hipEventCreate failed");
  for (int i = 1; i < fa::kMaxMicrobatches && !rc; i++) {
    if (hipEventCreateWithFlags(&m->ev_join[i], hipEventDisableTiming) != hipSuccess)
      rc = set_error(ctx, FA_ERR_HIP, "hipEventCreate failed");
    else if (hipStreamCreateWithFlags(&m->mb_stream[i], hipStreamNonBlocking) != hipSuccess)  // default priority
      rc = set_error(ctx, FA_ERR_HIP, "hipStreamCreate failed");
  }
  if (rc) {
    fa::model_release(m);
    return rc;
  }
  fa::register_model(m, ctx);
  *out = m;
  return FA_OK;
}

void fa_gemma_destroy(fa_model* m) {
  // unknown, already closed with its context, or at exit: nothing to do
  if (!m || !fa::unregister_model(m)) return;
  fa::model_release(m);
}

}  // extern "C"

void fa::model_release(fa_model* m) {
  (void)hipSetDevice(m->ctx->device);
  (void)hipStreamSynchronize(m->ctx->stream);
  for (hipStream_t st : m->mb_stream)
    if (st) (void)hipStreamSynchronize(st);
  for (void* p : m->allocations) (void)hipFree(p);
  m->ws.release();
  m->plan_dev.release();
  m->ids_dev.release();
  m->out_dev.release();
  if (m->plan_host) (void)hipHostFree(m->plan_host);
  if (m->io_host) (void)hipHostFree(m->io_host);
  if (m->plan_done) (void)hipEventDestroy(m->plan_done);
  if (m->ev_fork) (void)hipEventDestroy(m->ev_fork);
  for (int i = 0; i < fa::kMaxMicrobatches; i++) {
    if (m->ev_join[i]) (void)hipEventDestroy(m->ev_join[i]);
    if (m->mb_stream[i]) (void)hipStreamDestroy(m->mb_stream[i]);
  }
  for (auto& p : m->pending) {
    m->event_pool.push_back(p.a);
    m->event_pool.push_back(p.b);
  }
  for (hipEvent_t e : m->event_pool) (void)hipEventDestroy(e);
  delete m;
}

extern "C" {

int fa_gemma_set_weight(fa_model* m, const char* name, int dtype, const int64_t* shape, int32_t ndim,
                        const void* data) {
  if (!m || !name || !data || (ndim > 0 && !shape)) return set_error(m ? m->ctx : nullptr, FA_ERR_ARG, "gemma: NULL argument");
  fa_ctx* ctx = m->ctx;
  if (dtype != FA_DT_F32 && dtype != FA_DT_BF16) return set_error(ctx, FA_ERR_ARG, "gemma: weight %s: dtype %d", name, dtype);
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "gemma");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  const fa_gemma_config& c = m->cfg;
  const bool v2 = m->variant == 2;
  const int d = c.hidden_size, H = c.num_attention_heads, F = c.intermediate_size, P = m->P;
  const std::string s(name);
  auto shape_is = [&](std::initializer_list<int64_t> want) {
    if ((size_t)ndim != want.size()) return false;
    int i = 0;
    for (int64_t w : want)
      if (shape[i++] != w) return false;
    return true;
  };
  auto shape_str = [&]() {
    std::string r = "[";
    for (int i = 0; i < ndim; i++) r += (i ? "," : "") + std::to_string(shape[i]);
    return r + "]";
  };
  // matrix [rows, cols] -> rows of dst (row stride cols); source row r goes to
  // destination row dst_row(r), copied in runs of consecutive rows. bf16 data
  // and bf16-exact float32 data keep one bf16 plane; float32 data with any
  // other value turns dst into three planes (hi, mid, lo: the same split as
  // the kernels' split3), the rows written before kept as hi with zero mid
  // and lo.
  auto put_matrix = [&](fa::Mat& dst, int64_t rows, int64_t cols, auto&& dst_row) -> int {
    const size_t n = (size_t)rows * cols;
    std::vector<uint16_t> tmp;
    const uint16_t* src16 = (const uint16_t*)data;
    bool exact = true;
    if (dtype == FA_DT_F32) {
      tmp.resize(n);
      const float* src = (const float*)data;
      for (size_t i = 0; i < n && exact; i++) exact = fa::bf16_exact(src[i], &tmp[i]);
      if (!exact) {
        tmp.resize(3 * n);
        for (size_t i = 0; i < n; i++) {
          uint32_t u;
          std::memcpy(&u, &src[i], 4);
          const uint32_t hi = u & 0xFFFF0000u;
          float fh, r1;
          std::memcpy(&fh, &hi, 4);
          r1 = src[i] - fh;  // exact in float32
          uint32_t u1;
          std::memcpy(&u1, &r1, 4);
          const uint32_t mid = u1 & 0xFFFF0000u;
          float fm, r2;
          std::memcpy(&fm, &mid, 4);
          r2 = r1 - fm;  // at most 8 significant bits: exact in bf16
          uint32_t u2;
          std::memcpy(&u2, &r2, 4);
          tmp[i] = (uint16_t)(hi >> 16);
          tmp[n + i] = (uint16_t)(mid >> 16);
          tmp[2 * n + i] = (uint16_t)(u2 >> 16);
        }
      }
      src16 = tmp.data();
    }
    // the six-term kernel of a three-plane matrix takes whole 32-wide K slabs
    // (the one-plane case has the fp32-MFMA kernel for other widths): refuse
    // here rather than at the first embed
    if (!exact && cols % 32 != 0)
      return set_error(ctx, FA_ERR_UNSUPPORTED,
                       "gemma: weight %s: a float32 matrix with values bfloat16 cannot hold needs an input width "
                       "that is a multiple of 32, got %lld",
                       name, (long long)cols);
    if (!exact && dst.terms == 1) {
      // promote to three planes: the rows set so far become hi, mid = lo = 0
      void* np = nullptr;
      int rc2 = fa::alloc_dev(m, (size_t)3 * dst.plane() * 2, &np);
      if (rc2) return rc2;
      FA_HIP_CHECK(ctx, hipMemcpy(np, dst.p, (size_t)dst.plane() * 2, hipMemcpyDeviceToDevice));
      FA_HIP_CHECK(ctx, hipMemset((uint16_t*)np + dst.plane(), 0, (size_t)2 * dst.plane() * 2));
      fa::free_dev(m, dst.p);
      dst.p = (uint16_t*)np;
      dst.terms = 3;
    }
    const int src_terms = exact ? 1 : 3;
    std::vector<uint16_t> zeros;
    for (int t = 0; t < dst.terms; t++) {
      const uint16_t* from = src16 + (t < src_terms ? (size_t)t * n : 0);
      if (t >= src_terms) {  // rows of an exact matrix in a three-plane one: zero mid and lo
        if (zeros.empty()) zeros.assign(n, 0);
        from = zeros.data();
      }
      uint16_t* plane = dst.p + (size_t)t * dst.plane();
      for (int64_t r0 = 0; r0 < rows;) {
        int64_t r1 = r0 + 1;
        while (r1 < rows && dst_row(r1) == dst_row(r1 - 1) + 1) r1++;
        FA_HIP_CHECK(ctx, hipMemcpy(plane + (size_t)dst_row(r0) * cols, from + (size_t)r0 * cols,
                                    (size_t)(r1 - r0) * cols * 2, hipMemcpyHostToDevice));
        r0 = r1;
      }
    }
    return FA_OK;
  };
  auto identity = [](int64_t r) { return r; };
  auto put_norm = [&](float* dst, int64_t n) -> int {
    std::vector<float> v(n);
    for (int64_t i = 0; i < n; i++) {
      float w;
      if (dtype == FA_DT_BF16) {
        uint32_t u = (uint32_t)((const uint16_t*)data)[i] << 16;
        std::memcpy(&w, &u, 4);
      } else {
        w = ((const float*)data)[i];
      }
      v[i] = v2 ? w : w + 1.0f;  // Gemma 3's (1 + w); EmbeddingGemma 2 uses w itself (model.go:128-140)
    }
    FA_HIP_CHECK(ctx, hipMemcpy(dst, v.data(), n * 4, hipMemcpyHostToDevice));
    return FA_OK;
  };
  int rc = FA_OK;
  int l;
  std::string rest;
  if (s == "embed_tokens.weight") {
    if (!shape_is({c.vocab_size, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_matrix(m->embed, c.vocab_size, d, identity);
  } else if (s == "norm.weight") {
    if (!shape_is({d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_norm(m->g_final, d);
  } else if (v2 && s == "ple.per_layer_model_projection.weight") {
    if (!shape_is({(int64_t)c.num_hidden_layers * P, d}))
      return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_matrix(m->wple_model, (int64_t)c.num_hidden_layers * P, d, identity);
  } else if (v2 && s == "ple.per_layer_projection_norm.weight") {
    if (!shape_is({P})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_norm(m->g_ple_norm, P);
  } else if (v2 && s == "embedding_projection.weight") {
    if (!shape_is({m->E, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_matrix(m->wemb_proj, m->E, d, identity);
  } else if (s.rfind("dense.", 0) == 0 && s.size() > 6) {
    char* end = nullptr;
    long i = std::strtol(s.c_str() + 6, &end, 10);
    if (i < 0 || i >= c.n_dense || std::string(end) != ".linear.weight")
      return set_error(ctx, FA_ERR_ARG, "gemma: weight \"%s\" not found", name);
    if (!shape_is({m->dense_out[i], m->dense_in[i]}))
      return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
    rc = put_matrix(m->dense[i], m->dense_out[i], m->dense_in[i], identity);
  } else if (fa::parse_layer(s, c.num_hidden_layers, &l, &rest) == 0) {
    fa::Layer& L = m->layers[l];
    const int D = L.D, Hkv = L.Hkv;
    if (rest == "input_layernorm.weight" || rest == "post_attention_layernorm.weight" ||
        rest == "pre_feedforward_layernorm.weight" || rest == "post_feedforward_layernorm.weight") {
      if (!shape_is({d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      float* dst = rest[0] == 'i' ? L.g_in : rest[1] == 'o' ? (rest[5] == 'a' ? L.g_post_attn : L.g_post_ffn) : L.g_pre_ffn;
      rc = put_norm(dst, d);
    } else if (rest == "self_attn.q_norm.weight" || rest == "self_attn.k_norm.weight") {
      if (!shape_is({D})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_norm(rest[10] == 'q' ? L.g_q : L.g_k, D);
    } else if (rest == "self_attn.q_proj.weight") {
      if (!shape_is({H * D, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wqkv, H * D, d, identity);
    } else if (rest == "self_attn.k_proj.weight") {
      if (!shape_is({Hkv * D, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wqkv, Hkv * D, d, [o = (int64_t)H * D](int64_t r) { return o + r; });
    } else if (rest == "self_attn.v_proj.weight") {
      if (!shape_is({Hkv * D, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wqkv, Hkv * D, d, [o = (int64_t)(H + Hkv) * D](int64_t r) { return o + r; });
    } else if (rest == "self_attn.o_proj.weight") {
      if (!shape_is({d, H * D})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wo, d, H * D, identity);
    } else if (rest == "mlp.gate_proj.weight" || rest == "mlp.up_proj.weight") {
      if (!shape_is({F, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      const int64_t off = rest[4] == 'g' ? 0 : 32;  // gate rows first in each 64-row group, then up
      rc = put_matrix(L.wgu, F, d, [off](int64_t r) { return (r / 32) * 64 + off + (r % 32); });
    } else if (rest == "mlp.down_proj.weight") {
      if (!shape_is({d, F})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wdown, d, F, identity);
    } else if (v2 && rest == "ple_block.per_layer_input_gate.weight") {
      if (!shape_is({P, d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wple_gate, P, d, identity);
    } else if (v2 && rest == "ple_block.per_layer_projection.weight") {
      if (!shape_is({d, P})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_matrix(L.wple_proj, d, P, identity);
    } else if (v2 && rest == "ple_block.post_per_layer_input_norm.weight") {
      if (!shape_is({d})) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      rc = put_norm(L.g_ple_post, d);
    } else if (v2 && rest == "layer_scalar") {
      // one value (model.go:183-188); the checkpoint stores it with shape [1]
      if (!(shape_is({1}) || ndim == 0)) return set_error(ctx, FA_ERR_ARG, "gemma: %s shape %s", name, shape_str().c_str());
      if (dtype == FA_DT_BF16) {
        const uint32_t u = (uint32_t)((const uint16_t*)data)[0] << 16;
        std::memcpy(&L.scalar, &u, 4);
      } else {
        L.scalar = ((const float*)data)[0];
      }
    } else {
      return set_error(ctx, FA_ERR_ARG, "gemma: weight \"%s\" not found", name);
    }
  } else {
    return set_error(ctx, FA_ERR_ARG, "gemma: weight \"%s\" not found", name);
  }
  if (rc) return rc;
  m->seen.insert(s);
  m->finalized = false;
  return FA_OK;
}

int fa_gemma_finalize(fa_model* m) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  fa_ctx* ctx = m->ctx;
  const fa_gemma_config& c = m->cfg;
  const size_t expected = m->variant == 2 ? 5 + (size_t)c.n_dense + 17 * (size_t)c.num_hidden_layers
                                          : 2 + (size_t)c.n_dense + 13 * (size_t)c.num_hidden_layers;
  if (m->seen.size() != expected)
    return set_error(ctx, FA_ERR_STATE, "gemma: %zu of %zu weights set", m->seen.size(), expected);
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "gemma");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  std::vector<int32_t> pos(c.max_tokens);
  for (int t = 0; t < c.max_tokens; t++) pos[t] = t;
  std::vector<float> cs, sn;
  const double local = c.rope_local_base_freq != 0 ? c.rope_local_base_freq : 10000.0;
  const double global = c.rope_theta != 0 ? c.rope_theta : 10000.0;
  if (m->d_local) {
    fa::rope_tables_host(local, pos.data(), c.max_tokens, m->d_local, cs, sn);
    FA_HIP_CHECK(ctx, hipMemcpy(m->cos_local, cs.data(), cs.size() * 4, hipMemcpyHostToDevice));
    FA_HIP_CHECK(ctx, hipMemcpy(m->sin_local, sn.data(), sn.size() * 4, hipMemcpyHostToDevice));
  }
  if (m->d_global) {
    fa::rope_tables_host(global, pos.data(), c.max_tokens, m->d_global, cs, sn);
    FA_HIP_CHECK(ctx, hipMemcpy(m->cos_global, cs.data(), cs.size() * 4, hipMemcpyHostToDevice));
    FA_HIP_CHECK(ctx, hipMemcpy(m->sin_global, sn.data(), sn.size() * 4, hipMemcpyHostToDevice));
  }
  {
    const int rc_ = fa::prepare_h2(m);
    if (rc_) return rc_;
  }
  m->finalized = true;
  return FA_OK;
}

}  // extern "C"

namespace fa {
namespace {

// The forward pass over device-resident ids. With hidden == nullptr: every
// layer, pooling, the head and L2 into d_out [B x dim]. With hidden != nullptr
// (encode): the packed rows [M x d] of the final hidden states (n_layers < 0)
// or of the residual stream after the first n_layers layers into hidden;
// d_out and dim are unused.
int forward(fa_model* m, const int32_t* d_ids, const int32_t* lengths, int32_t B, int32_t T, int32_t dim,
            float* d_out, int n_layers, float* hidden) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  fa_ctx* ctx = m->ctx;
  const fa_gemma_config& c = m->cfg;
  if (!m->finalized) return set_error(ctx, FA_ERR_STATE, "gemma: embed before every weight was set (finalize)");
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "gemma");
    if (rc_) return rc_;
  }
  if (B < 0 || T < 0) return set_error(ctx, FA_ERR_ARG, "gemma: negative batch shape [%d x %d]", B, T);
  if (B == 0) return FA_OK;
  if (!d_ids || !lengths || !(hidden ? hidden : d_out)) return set_error(ctx, FA_ERR_ARG, "gemma: NULL buffer");
  if (T > c.max_tokens) return set_error(ctx, FA_ERR_ARG, "gemma: T=%d exceeds max_tokens %d", T, c.max_tokens);
  const bool v2 = m->variant == 2;
  const int d = c.hidden_size, H = c.num_attention_heads, F = c.intermediate_size, NL = c.num_hidden_layers,
            P = m->P;
  if (hidden && n_layers > NL)
    return set_error(ctx, FA_ERR_ARG, "gemma: encode after %d layers, the model has %d", n_layers, NL);
  const bool final_states = !hidden || n_layers < 0;
  const int n_run = final_states ? NL : n_layers;
  const int full = c.n_dense > 0 ? m->dense_out.back() : (v2 ? m->E : d);
  if (dim <= 0) dim = full;
  if (dim > full) return set_error(ctx, FA_ERR_ARG, "gemma: Dim(%d) outside 1..%d", dim, full);
  // ---- plan (host): cu_seqlens, micro-batch groups, attention work items ----
  int64_t M = 0;
  double sum_l2 = 0;
  for (int b = 0; b < B; b++) {
    if (lengths[b] < 1 || lengths[b] > T)
      return set_error(ctx, FA_ERR_ARG, "gemma: length[%d] = %d outside 1..T=%d", b, lengths[b], T);
    M += lengths[b];
    sum_l2 += (double)lengths[b] * lengths[b];
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  // Micro-batches: with enough tokens the sequences are cut into groups of
  // about equal token count (contiguous rows) whose layers run on separate
  // streams, so that one group's kernels occupy the CUs the others leave
  // idle (the last round of GEMM tiles and attention items, the norms'
  // low-occupancy phases). Not while profiling: the probes time one stream.
  // Group g holds sequences [gb[g], gb[g+1]).
  int gb[fa::kMaxMicrobatches + 1] = {0, B};
  int groups = 1;
  if (M >= fa::microbatch_min_rows() && !m->profiling)
    groups = fa::plan_groups(lengths, B, M, fa::microbatch_count(M, sum_l2), gb);
  // each layer's attention path, the items and their key runs
  std::vector<int>& layer_D = m->plan_layer_D;
  std::vector<int>& layer_Hkv = m->plan_layer_Hkv;
  layer_D.resize(m->layers.size());
  layer_Hkv.resize(m->layers.size());
  for (size_t l = 0; l < m->layers.size(); l++) {
    layer_D[l] = m->layers[l].D;
    layer_Hkv[l] = m->layers[l].Hkv;
  }
  fa::AttnPlanIn pin;
  pin.lengths = lengths; pin.B = B; pin.T = T; pin.H = H;
  pin.layer_D = layer_D.data(); pin.layer_Hkv = layer_Hkv.data();
  pin.n_layers = (int)m->layers.size(); pin.n_run = n_run;
  pin.groups = groups; pin.gb = gb; pin.cus = cus;
  pin.tile_keys = fa::attention_tiles_keys(); pin.varlen_qblock = fa::attention_varlen_qblock();
  pin.max_key_parts = fa::kMaxKeyParts; pin.split_rows = fa::kAttnSplitRows;
  pin.forced_key_parts = fa::attention_key_parts_forced();
  pin.forced_rows = fa::attention_rows_forced();
  pin.forced_xcd = fa::attention_xcd_forced();
  pin.tile_min_rows = fa::tile_min_rows();
  pin.tiles_allowed = m->tiles;
  fa::AttnPlan ap;
  fa::plan_attention(pin, ap);
  const int64_t n_items_t = ap.n_items_t, n_items = ap.n_items_t + ap.n_items_v, n_tiles = ap.n_tiles;
  const int hkv_t = ap.hkv_t, kparts_t = ap.kparts_t, kparts_v = ap.kparts_v, waves_t = ap.waves_t;
  const int tkeys = pin.tile_keys;
  // plan buffer: cu_seqlens, items, first tile per sequence, then (16-byte
  // aligned) each item's extent (its sequence's first packed row, length and
  // first tile) and each key tile's (its first packed row, keys, first key's
  // position), which the attention and the key/value image kernels read
  // beside the item or tile (no dependent load through a sequence table)
  const size_t ext_off = (2 * (size_t)(B + 1) + 3 * (size_t)n_items + 3) & ~(size_t)3;
  const size_t plan_ints = ext_off + 4 * (size_t)(n_items + n_tiles);
  if (m->plan_pending) {
    FA_HIP_CHECK(ctx, hipEventSynchronize(m->plan_done));  // previous upload has read the pinned buffer
    m->plan_pending = false;
  }
  if (plan_ints > m->plan_host_ints) {
    if (m->plan_host) (void)hipHostFree(m->plan_host);
    m->plan_host = nullptr;
    size_t n = plan_ints * 2;
    FA_HIP_CHECK(ctx, hipHostMalloc((void**)&m->plan_host, n * 4, hipHostMallocDefault));
    m->plan_host_ints = n;
  }
  int32_t* cu_h = m->plan_host;
  int32_t* items_h = m->plan_host + (B + 1);
  int32_t* cut_h = items_h + 3 * n_items;
  cu_h[0] = 0;
  cut_h[0] = 0;
  for (int b = 0; b < B; b++) {
    cu_h[b + 1] = cu_h[b] + lengths[b];
    cut_h[b + 1] = cut_h[b] + (ap.any_tiles ? (lengths[b] + tkeys - 1) / tkeys : 0);
  }
  fa::plan_items(pin, ap, items_h, m->seq_order);
  {
    int32_t* ext_h = m->plan_host + ext_off;
    for (int64_t i = 0; i < n_items; i++) {
      const int b = items_h[3 * i];
      ext_h[4 * i] = cu_h[b];
      ext_h[4 * i + 1] = lengths[b];
      ext_h[4 * i + 2] = cut_h[b];
      ext_h[4 * i + 3] = 0;
    }
    int32_t* text_h = ext_h + 4 * n_items;
    for (int b = 0; b < B; b++)
      for (int q = cut_h[b]; q < cut_h[b + 1]; q++) {
        const int t0 = tkeys * (q - cut_h[b]);
        text_h[4 * q] = cu_h[b] + t0;
        text_h[4 * q + 1] = std::min(tkeys, lengths[b] - t0);
        text_h[4 * q + 2] = t0;
        text_h[4 * q + 3] = 0;
      }
  }
  const int64_t* group_items_t = ap.group_items_t;
  const int64_t* group_items_v = ap.group_items_v;
  int rc;
  if ((rc = m->plan_dev.ensure(ctx, plan_ints * 4 + (size_t)M * 8))) return rc;
  int32_t* cu_d = m->plan_dev.as<int32_t>();
  int32_t* items_d = cu_d + (B + 1);
  const int32_t* ext_d = cu_d + ext_off;  // [n_items][4], 16-byte aligned
  const int32_t* text_d = ext_d + 4 * n_items;  // [n_tiles][4]
  int32_t* row_src_d = cu_d + plan_ints;   // [M] b*T + t
  int32_t* pos_d = row_src_d + M;          // [M] t
  FA_HIP_CHECK(ctx, hipMemcpyAsync(cu_d, m->plan_host, plan_ints * 4, hipMemcpyHostToDevice, ctx->stream));
  FA_HIP_CHECK(ctx, hipEventRecord(m->plan_done, ctx->stream));
  m->plan_pending = true;
  // ---- workspace ----
  // o has room for two partial products of the K-split o/down GEMMs
  // variant 2 adds the per-layer inputs [M, layers*P]; its [M, P] gate
  // output reuses gu (free after the down product)
  const int ksplit = fa::gemm_ksplit();
  // a few-row batch on one stream may split those products in four
  const bool few_rows = groups == 1 && ksplit > 1 && ((M + 31) / 32) * ((d + 63) / 64) * 4 <= cus;
  const int ks_max = few_rows ? std::max(ksplit, fa::small_ksplit()) : ksplit;
  const int64_t ncols = 2LL * d + m->max_width + m->max_hd + (int64_t)ks_max * d + std::max(F, P) +
                        (v2 ? (int64_t)NL * P : 0);
  int maxw = std::max(d, std::max(full, v2 ? m->E : d));
  for (int o : m->dense_out) maxw = std::max(maxw, o);
  const int kparts_max = std::max(kparts_t, kparts_v);
  const int64_t part_floats = kparts_max > 1 ? fa::attention_part_floats(kparts_max, M, H, m->max_hd / H) : 0;
  // key/value tile images: [tile][Hkv][key | value][2 * 32 * 256] fp16
  const size_t img_bytes = (size_t)n_tiles * hkv_t * 2 * (2 * 32 * 256) * 2;
  const size_t f32_bytes = ((size_t)M * ncols + (size_t)B * (d + 2 * (size_t)maxw) + (size_t)part_floats) * 4 + 256;
  const size_t img_off = (f32_bytes + 255) & ~(size_t)255;
  const size_t ws_bytes = img_off + img_bytes + 4096;
  if ((rc = m->ws.ensure(ctx, ws_bytes))) return rc;
  uint16_t* img = reinterpret_cast<uint16_t*>(m->ws.as<char>() + img_off);
  float* x = m->ws.as<float>();
  float* xn = x + M * d;
  float* qkv = xn + M * d;
  float* att = qkv + M * m->max_width;
  float* o = att + M * m->max_hd;
  float* gu = o + (int64_t)ks_max * M * d;
  float* ple = gu + M * std::max(F, P);
  float* pooled = ple + (v2 ? M * NL * P : 0);
  float* hbuf0 = pooled + (size_t)B * d;
  float* hbuf1 = hbuf0 + (size_t)B * maxw;
  float* attn_part = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(hbuf1 + (size_t)B * maxw) + 255) &
                                              ~(uintptr_t)255);
  hipStream_t s = ctx->stream;
  // products on split activations: xn, att and gu hold split terms (the last
  // layer's xn, the final hidden states, stays in floats)
  const bool h2 = m->h2;
  // One product: g as launch_gemm takes it, or on A's split terms (at a, its
  // values times a_scale; out_scale != 0: the result split too)
  auto product = [&](const fa::GemmArgs& g, const float* a, const fa::Mat& w, float a_scale, float out_scale, int kind,
                     double flops, hipStream_t st) -> int {
    fa::Probe pr(m, kind, flops, 0);
    int r;
    if (h2) {
      fa::GemmH2Args q;
      q.m = g.m; q.n = g.n; q.k = g.k; q.a = a; q.lda = g.lda; q.c = g.c; q.ldc = g.ldc;
      fa::set_h2(q, w, a_scale);
      q.out_scale = out_scale; q.epi = g.epi; q.act = g.act; q.mul = g.mul; q.ldm = g.ldm;
      q.ksplit = g.ksplit; q.c_split = g.c_split; q.shared = g.shared;
      r = fa::launch_gemm_h2(ctx, q, st);
    } else {
      r = fa::launch_gemm(ctx, g, st);
    }
    if (r) return r;
    pr.done();
    return FA_OK;
  };
  // ---- row plan on device ----
  if ((rc = fa::launch_row_plan(ctx, cu_d, B, T, M, row_src_d, pos_d, s))) return rc;
  const float eps = c.rms_norm_eps;
  const float emb_scale = (float)std::sqrt((double)d);  // embed.go:176
  // model.go:100; variant 2 does not scale the scores (model.go:105-110)
  const float att_scale = v2 ? 1.f : (float)(1.0 / std::sqrt(c.query_pre_attn_scalar));
  // window bound (config.go:331-339): variant 2 reads an inclusive radius
  const int wbound = v2 ? c.sliding_window + 1 : c.use_bidirectional ? c.sliding_window / 2 + 1 : c.sliding_window;
  {
    fa::Probe pr(m, FA_K_GATHER, 0, (double)M * (2.0 * d + 8.0 * d + 4));
    if ((rc = fa::launch_embed_gather(ctx, d_ids, row_src_d, m->embed.p, m->embed.terms == 3 ? m->embed.plane() : 0,
                                      c.vocab_size, M, d, emb_scale, m->layers[0].g_in, eps, x, xn, s,
                                      h2 && n_run > 0 ? m->layers[0].s_in : 0.f, h2 && v2 ? qkv : nullptr, m->s_x0)))
      return rc;
    pr.done();
  }
  if (v2) {
    // per-layer inputs: RMSNorm(x0 . W_ple^T * hidden^-1/2) per layer (embed.go:274-279)
    {
      fa::GemmArgs g;
      g.m = M; g.n = (int64_t)NL * P; g.k = d; g.a = x; g.lda = d; fa::set_b(g, m->wple_model); g.c = ple;
      g.ldc = (int64_t)NL * P;
      // (split: the scaled embeddings' terms, in q|k|v's buffer until the layers run)
      if ((rc = product(g, qkv, m->wple_model, m->s_x0, 0.f, FA_K_GEMM_PLE, 2.0 * M * NL * P * d, s))) return rc;
    }
    fa::Probe pr(m, FA_K_PLE_NORM, 0, (double)M * NL * P * 8.0);
    if ((rc = fa::launch_ple_norm(ctx, ple, M, NL, P, (float)(1 / std::sqrt((double)d)), m->g_ple_norm, eps, s)))
      return rc;
    pr.done();
  }
  // The fp32 path's layers of head_dim 256 take their q/k norm into the
  // attention (FA_ATTN_SHORT=0 and forced key runs: the separate passes) where
  // every sequence is short and the items are one round of workgroups. A few
  // sequences above 32 tokens stay with the separate passes, whose key runs
  // spread them over more CUs. Us per forward, separate and fused: 1 x 16 907
  // and 844, 1 x 32 1 026 and 1 004, 1 x 48 1 014 and 1 057, 1 x 64 1 031 and
  // 1 101, 4 x 64 (24 items) 1 346 and 1 362, 8 x 64 (48) 1 582 and 1 558, 16 x
  // 64 1 827 and 1 758, 85 x 12 1 716 and 1 642, 80 x 32 (240) 2 533 and 2 526.
  const int32_t longest = *std::max_element(lengths, lengths + B);
  const bool short_seqs = fa::attention_short_enabled() && ap.n_items_v <= cus &&
                          (longest <= 32 || (longest <= fa::kAttnShortKeys && ap.n_items_v >= 48));
  // one layer over rows [r0, r0 + rows) (the sequences of one group, whose
  // attention items are items_t[0, n_it_t) for a tile layer, items_v[0,
  // n_it_v) otherwise) on stream st
  auto run_layer = [&](int l, int b0, int b1, const int32_t* items_t, int64_t n_it_t, const int32_t* items_v,
                       int64_t n_it_v, hipStream_t st) -> int {
    const int64_t r0 = cu_h[b0], rows = cu_h[b1] - r0;
    const fa::Layer& L = m->layers[l];
    const int D = L.D, Hkv = L.Hkv;
    const bool sliding = L.sliding;
    const bool tiles = ap.layer_tiles(D);
    const bool shrt = !tiles && D == 256 && short_seqs;
    // The N = hidden products (o, down, per-layer-input projection) split K
    // in two when their 128x128 tiles, counted over the concurrent groups,
    // give the CUs fewer than two each (C2: one stream 5 517 rows, or three
    // groups of about 1 840: 4 % faster split); with more tiles the second
    // partial's writes and reads cost more than the fill gains (C5's three
    // groups of about 5 970 rows: 4.7 % faster unsplit).
    const int64_t n_tiles = ((rows + 127) / 128) * ((d + 127) / 128) * groups;
    const int ks = n_tiles < 2LL * cus ? ks_max : 1;
    // per product: the most parts (ks, halved as needed) that divide K into
    // whole 32-wide slabs
    auto parts = [&](int64_t K) {
      int k = ks;
      while (k > 1 && K % (32 * k) != 0) k /= 2;
      return k;
    };
    const int ks_o = parts(H * D), ks_down = parts(F), ks_ple = parts(P);
    const float* o2_o = ks_o > 1 ? o + M * d + r0 * d : nullptr;
    const float* o2_dn = ks_down > 1 ? o + M * d + r0 * d : nullptr;
    const float* o2_pl = ks_ple > 1 ? o + M * d + r0 * d : nullptr;
    float* const xr = x + r0 * d;
    float* const xnr = xn + r0 * d;
    // per-group regions of the buffers whose row width changes with the
    // layer (EmbeddingGemma 2's head dims) or the product (gate|up vs the
    // per-layer-input gate): groups on other streams may be at other
    // layers, so each writes only inside [r0, r0 + rows) x the widest row
    float* const qkvr = qkv + r0 * m->max_width;
    float* const attr = att + r0 * m->max_hd;
    float* const gur = gu + r0 * std::max(F, P);
    float* const or_ = o + r0 * d;
    int rc;
    // a few-row batch on the fp32 attention path splits the q|k|v product
    // in K: its second part goes to o's planes (free until the o product)
    // and the q/k norm pass adds it
    const bool qkv_split = few_rows && !tiles && fa::qkv_ksplit() > 1 && d % 64 == 0 &&
                           (int64_t)ks_max * d >= m->max_width;
    const float* qkv2 = qkv_split ? o : nullptr;
    {
      fa::GemmArgs g;
      g.shared = groups > 1;
      g.m = rows; g.n = L.width; g.k = d; g.a = xnr; g.lda = d; fa::set_b(g, L.wqkv); g.c = qkvr; g.ldc = L.width;
      if (qkv_split) {
        g.ksplit = 2;
        g.c_split = o - qkvr;
      }
      if ((rc = product(g, g.a, L.wqkv, L.s_in, 0.f, FA_K_GEMM_QKV, 2.0 * rows * L.width * d, st))) return rc;
    }
    if (tiles) {
      // read k and v (4 bytes per element); write their images (4 bytes per
      // element each, tiles padded to 32 tokens); q is normed and rotated
      // by the attention as it loads it
      const int64_t ntl = cut_h[b1] - cut_h[b0];
      // (variant 2 norms the values too: each value half-block also reads
      // the other half of its keys' values for the sum of squares)
      fa::Probe pr(m, FA_K_QKNORM_ROPE, 0,
                   (double)rows * (v2 ? 3 : 2) * Hkv * 4.0 * D + (double)ntl * Hkv * 2 * 2 * 32 * 256 * 2);
      if ((rc = fa::launch_kv_tiles(ctx, qkvr, r0, H, Hkv, L.g_k, eps, L.cos_t, L.sin_t, text_d, cut_h[b0],
                                    (int32_t)ntl, img, st, v2, L.s_k, L.s_att)))
        return rc;
      pr.done();
    } else if (!shrt) {
      fa::Probe pr(m, FA_K_QKNORM_ROPE, 0, (double)rows * (H + (v2 ? 2 : 1) * Hkv) * D * 8.0);
      // a group of one sequence: row i is token i, no position table
      const int32_t* gpos = b1 - b0 == 1 ? nullptr : pos_d + r0;
      if ((rc = fa::launch_qknorm_rope(ctx, qkvr, rows, H, Hkv, D, L.g_q, L.g_k, eps, gpos, L.cos_t, L.sin_t,
                                       st, v2, qkv2)))
        return rc;
      pr.done();
    }
    {
      fa::AttnVarlenArgs a;
      a.qkv = qkvr; a.out = attr; a.row0 = r0;
      a.item_ext = ext_d + 4 * ((items_v - items_d) / 3);
      a.H = H; a.Hkv = Hkv; a.D = D; a.scale = att_scale;
      a.window = (sliding && c.sliding_window > 0) ? wbound : 0;
      a.split = h2 ? L.s_att : 0.f;
      if (kparts_v > 1) {
        a.kparts = kparts_v; a.rows = rows; a.part = attn_part;
      }
      double pairs = 0;
      if (m->profiling) {
        for (int b = 0; b < B; b++) {
          const double Lb = lengths[b];
          if (a.window > 0 && Lb > a.window) {
            // sum over i of |{j : |i-j| < w}| = L(2w-1) - w(w-1)
            pairs += Lb * (2.0 * a.window - 1) - (double)a.window * (a.window - 1);
          } else {
            pairs += Lb * Lb;
          }
        }
      }
      fa::Probe pr(m, FA_K_ATTENTION, pairs * 4.0 * H * D, 0);
      if (tiles) {
        fa::AttnTilesArgs at;
        at.qkv = qkvr; at.img = img; at.out = attr; at.row0 = r0;
        at.item_ext = ext_d + 4 * ((items_t - items_d) / 3);
        at.H = H; at.Hkv = Hkv; at.window = a.window; at.scale = a.scale;
        at.gq = L.g_q; at.eps = eps; at.cos_t = L.cos_t; at.sin_t = L.sin_t; at.waves = waves_t;
        at.split = a.split;
        at.q_scale = L.s_q; at.k_scale = L.s_k; at.v_scale = L.s_att;
        if (kparts_t > 1) {
          at.kparts = kparts_t; at.rows = M; at.nrows = rows; at.part = attn_part;
        }
        if ((rc = fa::launch_attention_tiles(ctx, at, items_t, (int32_t)n_it_t, st))) return rc;
      } else if (shrt) {
        fa::AttnShortArgs as;
        as.qkv = qkvr; as.qkv2 = qkv2; as.out = attr; as.H = H; as.Hkv = Hkv; as.window = a.window; as.scale = a.scale;
        as.split = a.split; as.eps = eps; as.row0 = r0; as.item_ext = a.item_ext;
        as.gq = L.g_q; as.gk = L.g_k; as.cos_t = L.cos_t; as.sin_t = L.sin_t; as.norm_v = v2;
        if ((rc = fa::launch_attention_short(ctx, as, items_v, (int32_t)n_it_v, st))) return rc;
      } else {
        if ((rc = fa::launch_attention_varlen_items(ctx, a, items_v, (int32_t)n_it_v, st))) return rc;
      }
      pr.done();
    }
    {
      fa::GemmArgs g;
      g.shared = groups > 1;
      g.m = rows; g.n = d; g.k = H * D; g.a = attr; g.lda = H * D; fa::set_b(g, L.wo); g.c = or_;
      g.ldc = d; g.ksplit = ks_o; g.c_split = M * d;
      if ((rc = product(g, g.a, L.wo, L.s_att, 0.f, FA_K_GEMM_O, 2.0 * rows * d * H * D, st))) return rc;
    }
    {
      fa::Probe pr(m, FA_K_RESIDUAL_NORM, 0, fa::resnorm_bytes(rows, d, ks_o, L.g_pre_ffn));
      if ((rc = fa::launch_residual_norm(ctx, or_, xr, xnr, rows, d, L.g_post_attn, L.g_pre_ffn, eps, st, o2_o, 1.f,
                                         ks_o - 1, M * d, h2 ? L.s_ffn : 0.f)))
        return rc;
      pr.done();
    }
    {
      fa::GemmArgs g;
      g.shared = groups > 1;
      g.m = rows; g.n = 2 * F; g.k = d; g.a = xnr; g.lda = d; fa::set_b(g, L.wgu); g.c = gur; g.ldc = F;
      g.epi = fa::Epi::GeGLU;
      if ((rc = product(g, g.a, L.wgu, L.s_ffn, L.s_gu, FA_K_GEMM_GATEUP, 2.0 * rows * 2 * F * d, st))) return rc;
    }
    {
      fa::GemmArgs g;
      g.shared = groups > 1;
      g.m = rows; g.n = d; g.k = F; g.a = gur; g.lda = F; fa::set_b(g, L.wdown); g.c = or_; g.ldc = d;
      g.ksplit = ks_down; g.c_split = M * d;
      if ((rc = product(g, g.a, L.wdown, L.s_gu, 0.f, FA_K_GEMM_DOWN, 2.0 * rows * d * F, st))) return rc;
    }
    // the last layer's "next norm" is the final RMSNorm (embed.go:237): xn = h
    const float* g_next = (l + 1 < NL) ? m->layers[l + 1].g_in : m->g_final;
    const float s_next = h2 && l + 1 < NL ? m->layers[l + 1].s_in : 0.f;
    {
      // variant 2: the per-layer-input block reads x itself, so no norm here
      fa::Probe pr(m, FA_K_RESIDUAL_NORM, 0, fa::resnorm_bytes(rows, d, ks_down, v2 ? nullptr : g_next));
      if ((rc = fa::launch_residual_norm(ctx, or_, xr, xnr, rows, d, L.g_post_ffn, v2 ? nullptr : g_next, eps, st,
                                         o2_dn, 1.f, ks_down - 1, M * d, v2 ? (h2 ? L.s_x : 0.f) : s_next)))
        return rc;
      pr.done();
    }
    if (v2) {
      // x = (x + RMSNorm(gelu(x . Wg^T) * ple_l . Wp^T; g)) * scalar (embed.go:359-371)
      {
        fa::GemmArgs g;
        g.shared = groups > 1;
        g.m = rows; g.n = P; g.k = d; g.a = xr; g.lda = d; fa::set_b(g, L.wple_gate); g.c = gur; g.ldc = P;
        g.epi = fa::Epi::Generic; g.act = FA_ACT_GELU; g.mul = ple + r0 * NL * P + (int64_t)l * P;
        g.ldm = (int64_t)NL * P;
        // (split: x's terms, which the residual step above left in xn)
        if ((rc = product(g, xnr, L.wple_gate, L.s_x, L.s_ple, FA_K_GEMM_PLE, 2.0 * rows * P * d, st))) return rc;
      }
      {
        fa::GemmArgs g;
        g.shared = groups > 1;
        g.m = rows; g.n = d; g.k = P; g.a = gur; g.lda = P; fa::set_b(g, L.wple_proj); g.c = or_; g.ldc = d;
        g.ksplit = ks_ple; g.c_split = M * d;
        if ((rc = product(g, g.a, L.wple_proj, L.s_ple, 0.f, FA_K_GEMM_PLE, 2.0 * rows * d * P, st))) return rc;
      }
      fa::Probe pr(m, FA_K_RESIDUAL_NORM, 0, fa::resnorm_bytes(rows, d, ks_ple, g_next));
      if ((rc = fa::launch_residual_norm(ctx, or_, xr, xnr, rows, d, L.g_ple_post, g_next, eps, st, o2_pl, L.scalar,
                                         ks_ple - 1, M * d, s_next)))
        return rc;
      pr.done();
    }
    return FA_OK;
  };
  if (groups == 1) {
    for (int l = 0; l < n_run; l++)
      if ((rc = run_layer(l, 0, B, items_d, group_items_t[0], items_d + 3 * n_items_t, group_items_v[0], s)))
        return rc;
  } else {
    // groups 1.. run on their own streams once the embeddings (and plan) are in
    FA_HIP_CHECK(ctx, hipEventRecord(m->ev_fork, s));
    for (int g = 1; g < groups; g++) FA_HIP_CHECK(ctx, hipStreamWaitEvent(m->mb_stream[g], m->ev_fork, 0));
    rc = FA_OK;
    for (int l = 0; l < n_run && !rc; l++) {
      int64_t it0 = 0, iv0 = n_items_t;  // the group's first tile item, first fp32 item
      for (int g = 0; g < groups && !rc; g++) {
        rc = run_layer(l, gb[g], gb[g + 1], items_d + 3 * it0, group_items_t[g], items_d + 3 * iv0, group_items_v[g],
                       g ? m->mb_stream[g] : s);
        it0 += group_items_t[g];
        iv0 += group_items_v[g];
      }
    }
    // joined also after an error: later calls reuse the workspace on s
    for (int g = 1; g < groups; g++) {
      FA_HIP_CHECK(ctx, hipEventRecord(m->ev_join[g], m->mb_stream[g]));
      FA_HIP_CHECK(ctx, hipStreamWaitEvent(s, m->ev_join[g], 0));
    }
    if (rc) return rc;
  }
  if (hidden) {
    // after the last layer xn holds the final RMSNorm of x (embed.go:237)
    const float* src = final_states ? xn : x;
    FA_HIP_CHECK(ctx, hipMemcpyAsync(hidden, src, (size_t)M * d * 4, hipMemcpyDeviceToDevice, s));
    return FA_OK;
  }
  {
    fa::Probe pr(m, FA_K_POOL_L2, 0, (double)M * d * 4.0 + (double)B * d * 4.0);
    if ((rc = fa::launch_pool(ctx, xn, cu_d, B, d, pooled, s))) return rc;
    pr.done();
  }
  const float* cur = pooled;
  int cur_w = d;
  float* bufs[2] = {hbuf0, hbuf1};
  int nb = 0;
  if (v2) {  // the embedding projection, applied to the pooled vector (embed.go:408-414)
    fa::GemmArgs g;
    g.m = B; g.n = m->E; g.k = d; g.a = pooled; g.lda = d; fa::set_b(g, m->wemb_proj); g.c = bufs[0]; g.ldc = m->E;
    fa::Probe pr(m, FA_K_GEMM_HEAD, 2.0 * B * m->E * d, 0);
    if ((rc = fa::launch_gemm(ctx, g, s))) return rc;
    pr.done();
    cur = bufs[0];
    cur_w = m->E;
    nb = 1;
  }
  // the last dense product splits K (its few rows give few tiles: 3072 -> 768
  // for one pooled row is 12 of them) and the L2 norm adds the partials,
  // unless a Tanh follows it (model.go:296-301, embed.go:415-418: applied in
  // the product's epilogue, so on the whole sum) or K splits are off
  int head_parts = 1;
  for (int i = 0; i < c.n_dense; i++) {
    fa::GemmArgs g;
    g.m = B; g.n = m->dense_out[i]; g.k = cur_w; g.a = cur; g.lda = cur_w; fa::set_b(g, m->dense[i]);
    g.c = bufs[(i + nb) & 1]; g.ldc = m->dense_out[i];
    if (m->dense_act[i] == FA_ACT_TANH) {
      g.epi = fa::Epi::Generic;
      g.act = FA_ACT_TANH;
    } else if (i + 1 == c.n_dense && ksplit > 1) {
      for (int ks : {4, 2})
        if (cur_w % (32 * ks) == 0 && (int64_t)ks * m->dense_out[i] <= maxw) {
          head_parts = ks;
          break;
        }
      g.ksplit = head_parts; g.c_split = (int64_t)B * m->dense_out[i];
    }
    fa::Probe pr(m, FA_K_GEMM_HEAD, 2.0 * B * m->dense_out[i] * cur_w, 0);
    if ((rc = fa::launch_gemm(ctx, g, s))) return rc;
    pr.done();
    cur = bufs[(i + nb) & 1];
    cur_w = m->dense_out[i];
  }
  {
    fa::Probe pr(m, FA_K_POOL_L2, 0, (double)B * dim * 8.0);
    if ((rc = fa::launch_l2norm(ctx, cur, B, cur_w, dim, d_out, s, head_parts,
                                (int64_t)B * cur_w)))
      return rc;
    pr.done();
  }
  return FA_OK;
}

}  // namespace
}  // namespace fa

extern "C" {

int fa_gemma_embed_ids_dev(fa_model* m, const int32_t* d_ids, const int32_t* lengths, int32_t B, int32_t T,
                           int32_t dim, float* d_out) {
  return fa::forward(m, d_ids, lengths, B, T, dim, d_out, 0, nullptr);
}

int fa_gemma_encode_ids_dev(fa_model* m, const int32_t* d_ids, const int32_t* lengths, int32_t B, int32_t T,
                            int32_t n_layers, float* d_hidden) {
  return fa::forward(m, d_ids, lengths, B, T, 0, nullptr, n_layers < 0 ? -1 : n_layers, d_hidden);
}

int fa_gemma_encode_ids(fa_model* m, const int32_t* ids, const int32_t* lengths, int32_t B, int32_t T,
                        int32_t n_layers, float* hidden) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  fa_ctx* ctx = m->ctx;
  if (B < 0 || T < 0) return set_error(ctx, FA_ERR_ARG, "gemma: negative batch shape [%d x %d]", B, T);
  if (B == 0) return FA_OK;
  if (!ids || !lengths || !hidden) return set_error(ctx, FA_ERR_ARG, "gemma: NULL buffer");
  int rc;
  if ((rc = fa::check_ids(m, ids, lengths, B, T))) return rc;
  int64_t M = 0;
  for (int b = 0; b < B; b++) M += lengths[b];
  const int d = m->cfg.hidden_size;
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "gemma");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  if ((rc = m->ids_dev.ensure(ctx, (size_t)B * T * 4))) return rc;
  if ((rc = m->out_dev.ensure(ctx, (size_t)M * d * 4))) return rc;
  char* io;
  const size_t ib = (size_t)B * T * 4, ob = (size_t)M * d * 4;
  if ((rc = fa::io_staging(m, ib + ob, &io))) return rc;
  std::memcpy(io, ids, ib);
  FA_HIP_CHECK(ctx, hipMemcpyAsync(m->ids_dev.ptr, io, ib, hipMemcpyHostToDevice, ctx->stream));
  if ((rc = fa_gemma_encode_ids_dev(m, m->ids_dev.as<int32_t>(), lengths, B, T, n_layers, m->out_dev.as<float>())))
    return rc;
  FA_HIP_CHECK(ctx, hipMemcpyAsync(io + ib, m->out_dev.ptr, ob, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  std::memcpy(hidden, io + ib, ob);
  return FA_OK;
}

int fa_gemma_embed_ids(fa_model* m, const int32_t* ids, const int32_t* lengths, int32_t B, int32_t T, int32_t dim,
                       float* out) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  fa_ctx* ctx = m->ctx;
  if (B < 0 || T < 0) return set_error(ctx, FA_ERR_ARG, "gemma: negative batch shape [%d x %d]", B, T);
  if (B == 0) return FA_OK;
  if (!ids || !lengths || !out) return set_error(ctx, FA_ERR_ARG, "gemma: NULL buffer");
  const fa_gemma_config& c = m->cfg;
  const int full = c.n_dense > 0 ? m->dense_out.back() : (m->variant == 2 ? m->E : c.hidden_size);
  const int dd = dim <= 0 ? full : dim;
  int rc;
  if ((rc = fa::check_ids(m, ids, lengths, B, T))) return rc;
  if (dd > full) return set_error(ctx, FA_ERR_ARG, "gemma: Dim(%d) outside 1..%d", dim, full);
  {
    const int rc_ = fa::refuse_capture(ctx, ctx->stream, "gemma");
    if (rc_) return rc_;
  }
  FA_HIP_CHECK(ctx, hipSetDevice(ctx->device));
  if ((rc = m->ids_dev.ensure(ctx, (size_t)B * T * 4))) return rc;
  if ((rc = m->out_dev.ensure(ctx, (size_t)B * dd * 4))) return rc;
  char* io;
  const size_t ib = (size_t)B * T * 4, ob = (size_t)B * dd * 4;
  if ((rc = fa::io_staging(m, ib + ob, &io))) return rc;
  std::memcpy(io, ids, ib);
  FA_HIP_CHECK(ctx, hipMemcpyAsync(m->ids_dev.ptr, io, ib, hipMemcpyHostToDevice, ctx->stream));
  if ((rc = fa_gemma_embed_ids_dev(m, m->ids_dev.as<int32_t>(), lengths, B, T, dd, m->out_dev.as<float>()))) return rc;
  FA_HIP_CHECK(ctx, hipMemcpyAsync(io + ib, m->out_dev.ptr, ob, hipMemcpyDeviceToHost, ctx->stream));
  FA_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  std::memcpy(out, io + ib, ob);
  return FA_OK;
}

int fa_gemma_set_profiling(fa_model* m, int enabled) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  m->profiling = enabled != 0;
  return FA_OK;
}

int fa_gemma_kernel_stats(fa_model* m, int kind, int64_t* launches, double* ms, double* flops, double* bytes) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  if (kind < 0 || kind >= FA_K_COUNT) return set_error(m->ctx, FA_ERR_ARG, "gemma: kernel kind %d", kind);
  int rc = fa::collect_stats(m);
  if (rc) return rc;
  const fa::KernelStat& s = m->stats[kind];
  if (launches) *launches = s.launches;
  if (ms) *ms = s.ms;
  if (flops) *flops = s.flops;
  if (bytes) *bytes = s.bytes;
  return FA_OK;
}

int fa_gemma_reset_stats(fa_model* m) {
  if (!m) return set_error(nullptr, FA_ERR_ARG, "gemma: NULL model");
  int rc = fa::collect_stats(m);
  for (auto& s : m->stats) s = fa::KernelStat{};
  return rc;
}

}  // extern "C"
