// Decoder layer forward with the grafted MLP (reference forward_layer,
// src/layer_forward_impl.inc:15-290): the attention block is frozen base
// code there (ATen); here every step runs on this library's kernels.
//
//   xn   = rms_norm(x, ln_in)                       glt_rmsnorm_fwd
//   q,k,v = xn . W_{q,k,v}^T                         one MFMA launch, 3 problems
//   RoPE(q, k)                                       glt_rope_fwd
//   a    = causal GQA SDPA(q, k, v)                  glt_attention_fwd
//   x   += a . W_o^T                                 MFMA, residual epilogue
//   x_ffn = rms_norm(x, ln_post)                     glt_rmsnorm_fwd
//   x   += grafted_mlp(x_ffn)                        glt_mlp_fwd (GLT_MLP_RESIDUAL)
#include <algorithm>
#include <cmath>
#include <vector>

#include "gemm.hpp"
#include "layout.hpp"

namespace glt {

namespace {

constexpr size_t kAlign = 256;
size_t up(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

struct Dims {
  int64_t M, D, nq, nk;  // tokens, hidden, q width, k/v width
};
Dims dims(const glt_layer_desc* d) {
  return {(int64_t)d->B * d->T, d->mlp.D, (int64_t)d->n_q_heads * d->head_dim,
          (int64_t)d->n_kv_heads * d->head_dim};
}

// prepared: W_q, W_k, W_v (K = D) and W_o (K = q width), each shuffled
struct Prep {
  size_t q, k, v, o, total;
};
Prep prep_layout(const glt_layer_desc* d) {
  const Dims m = dims(d);
  Prep p{};
  p.q = 0;
  p.k = up(p.q + shuf_elems(m.nq, m.D) * 2);
  p.v = up(p.k + shuf_elems(m.nk, m.D) * 2);
  p.o = up(p.v + shuf_elems(m.nk, m.D) * 2);
  p.total = up(p.o + shuf_elems(m.D, m.nq) * 2);
  return p;
}

// workspace: xn, q, k, v, attention output, RMSNorm mean squares, and the
// MLP's inter when the caller does not keep it
struct Ws {
  size_t xn, q, k, v, a, var_in, var_post, inter, vt, total;
};
Ws ws_layout(const glt_layer_desc* d) {
  const Dims m = dims(d);
  const int64_t N = d->mlp.N;
  Ws w{};
  w.xn = 0;
  w.q = up(w.xn + m.M * m.D * 2);
  w.k = up(w.q + m.M * m.nq * 2);
  w.v = up(w.k + m.M * m.nk * 2);
  w.a = up(w.v + m.M * m.nk * 2);
  w.var_in = up(w.a + m.M * m.nq * 2);
  w.var_post = up(w.var_in + m.M * 4);
  w.inter = up(w.var_post + m.M * 4);
  w.vt = up(w.inter + m.M * N * 2);
  w.total = up(w.vt + glt_attention_workspace_size(d->B, d->T, d->n_kv_heads, d->head_dim));
  return w;
}

glt_status check_layer(const glt_layer_desc* d, const glt_layer_weights* w, const char* who) {
  GLT_CHECK(d && w, GLT_ERR_INVALID_ARG, "%s: null descriptor/weights", who);
  GLT_CHECK(d->B >= 0 && d->T >= 0 && d->n_q_heads > 0 && d->n_kv_heads > 0 &&
                d->n_q_heads % d->n_kv_heads == 0,
            GLT_ERR_SHAPE, "%s: B=%d T=%d heads %d/%d", who, d->B, d->T, d->n_q_heads, d->n_kv_heads);
  GLT_CHECK(d->head_dim == 128, GLT_ERR_UNSUPPORTED, "%s: head_dim %d (only 128)", who, d->head_dim);
  GLT_CHECK(d->mlp.dtype == GLT_DTYPE_BF16, GLT_ERR_DTYPE, "%s: the decoder layer runs in bf16", who);
  GLT_CHECK((int64_t)d->mlp.M == (int64_t)d->B * d->T, GLT_ERR_SHAPE, "%s: mlp.M=%d != B*T=%lld", who, d->mlp.M,
            (long long)d->B * d->T);
  GLT_CHECK(w->q_proj && w->k_proj && w->v_proj && w->o_proj && w->ln_in && w->ln_post, GLT_ERR_INVALID_ARG,
            "%s: null projection / norm weight", who);
  return GLT_OK;
}

GSeg seg(const void* A, int64_t lda, int K, int N, const void* B, int64_t ldb) {
  GSeg s{};
  s.A = A; s.lda = lda; s.a_ks = 1; s.a_col = 0; s.K = K; s.n_lo = 0; s.n_hi = N;
  s.B0 = B; s.ldb0 = ldb; s.b0_row0 = 0; s.b_ks = 1;
  return s;
}
GProb prob(int64_t M, int64_t N, int mode, void* out) {
  GProb p{};
  p.M = (int)M; p.N = (int)N; p.mode = mode; p.out_f32 = 0; p.alpha = 1.f; p.beta = 0.f;
  p.out0 = out; p.ldo = N;
  return p;
}

// Runs out_j = A . W_j^T for the listed problems, on the MFMA kernel with
// the prepared (shuffled) weights when the shapes allow it, else on the
// strided kernel with the row-major weights.
struct Proj {
  const void* w;        // row-major [N, K]
  const uint16_t* shuf; // prepared
  int64_t N;
  void* out;
};
glt_status project(const void* A, int64_t M, int64_t K, const Proj* ps, int n, int mode, const char* label,
                   hipStream_t st) {
  auto mfma_plan = [&](int64_t r0, int64_t rows, GemmPlan& plan) {
    plan.label = label;
    plan.a_kind = LD_BF16;
    plan.b_kind = LD_SHUF;
    for (int j = 0; j < n; ++j) {
      plan.add_problem(prob(rows, ps[j].N, mode, static_cast<char*>(ps[j].out) + r0 * ps[j].N * 2));
      plan.add_seg(seg(static_cast<const char*>(A) + r0 * K * 2, K, (int)K, (int)ps[j].N, ps[j].shuf, shuf_k(K)));
    }
  };
  {
    // on the MFMA kernel, in row blocks when the output passes 31-bit
    // offsets (run_gemm splits it)
    GemmPlan plan;
    mfma_plan(0, M, plan);
    GemmPlan probe;
    mfma_plan(0, std::min<int64_t>(M, 256), probe);
    if (gemm_mfma_eligible(plan) || gemm_mfma_eligible(probe)) return run_gemm(plan, st);
  }
  GemmPlan gen;
  gen.label = label;
  gen.a_kind = gen.b_kind = LD_BF16;
  for (int j = 0; j < n; ++j) {
    gen.add_problem(prob(M, ps[j].N, mode, ps[j].out));
    gen.add_seg(seg(A, K, (int)K, (int)ps[j].N, ps[j].w, K));
  }
  return run_gemm(gen, st, false);
}

}  // namespace

}  // namespace glt

using namespace glt;

extern "C" {

size_t glt_attn_prepared_size(const glt_layer_desc* d) { return d ? prep_layout(d).total : 0; }

glt_status glt_attn_prepare(const glt_layer_desc* d, const glt_layer_weights* w, void* prepared, void* stream) {
  glt_status s = check_layer(d, w, "glt_attn_prepare");
  if (s != GLT_OK) return s;
  GLT_CHECK(prepared && reinterpret_cast<uintptr_t>(prepared) % kAlign == 0, GLT_ERR_ALIGNMENT,
            "glt_attn_prepare: prepared must be %zu-byte aligned", kAlign);
  const Dims m = dims(d);
  const Prep p = prep_layout(d);
  uint16_t* base = static_cast<uint16_t*>(prepared);
  hipStream_t st = as_stream(stream);
  struct Job { const void* src; int64_t rows, K; size_t off; };
  const Job jobs[4] = {{w->q_proj, m.nq, m.D, p.q}, {w->k_proj, m.nk, m.D, p.k}, {w->v_proj, m.nk, m.D, p.v},
                       {w->o_proj, m.D, m.nq, p.o}};
  for (const Job& j : jobs) {
    s = shuffle_b(j.src, GLT_DTYPE_BF16, j.K, false, (int)j.rows, (int)j.K, base + j.off / 2, st);
    if (s != GLT_OK) return s;
  }
  return GLT_OK;
}

size_t glt_layer_fwd_workspace_size(const glt_layer_desc* d) { return d ? ws_layout(d).total : 0; }

glt_status glt_layer_fwd(const glt_layer_desc* d, const glt_layer_weights* w, void* x, void* x_ffn, float* ffn_var,
                         void* gate_pre, void* up_pre, void* inter, void* workspace, size_t workspace_bytes,
                         void* stream) {
  glt_status s = check_layer(d, w, "glt_layer_fwd");
  if (s != GLT_OK) return s;
  const Dims m = dims(d);
  if (m.M == 0) return GLT_OK;
  const Ws L = ws_layout(d);
  GLT_CHECK(x && x_ffn && w->prepared, GLT_ERR_INVALID_ARG, "glt_layer_fwd: null x/x_ffn/prepared");
  GLT_CHECK(workspace && workspace_bytes >= L.total && reinterpret_cast<uintptr_t>(workspace) % kAlign == 0,
            GLT_ERR_WORKSPACE, "glt_layer_fwd: needs %zu workspace bytes, %zu-byte aligned", L.total, kAlign);
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  uint16_t* xn = reinterpret_cast<uint16_t*>(ws + L.xn);
  uint16_t* q = reinterpret_cast<uint16_t*>(ws + L.q);
  uint16_t* k = reinterpret_cast<uint16_t*>(ws + L.k);
  uint16_t* v = reinterpret_cast<uint16_t*>(ws + L.v);
  uint16_t* a = reinterpret_cast<uint16_t*>(ws + L.a);
  float* var_in = reinterpret_cast<float*>(ws + L.var_in);
  float* var_post = ffn_var ? ffn_var : reinterpret_cast<float*>(ws + L.var_post);
  const Prep P = prep_layout(d);
  const uint16_t* pb = static_cast<const uint16_t*>(w->prepared);

  // attention block (reference :29-55)
  s = glt_rmsnorm_fwd(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w->ln_in), xn, var_in,
                      (int32_t)m.M, (int32_t)m.D, d->rms_eps, stream);
  if (s != GLT_OK) return s;
  const Proj qkv[3] = {{w->q_proj, pb + P.q / 2, m.nq, q}, {w->k_proj, pb + P.k / 2, m.nk, k},
                       {w->v_proj, pb + P.v / 2, m.nk, v}};
  if ((s = project(xn, m.M, m.D, qkv, 3, EPI_STORE, "qkv", st)) != GLT_OK) return s;
  if (d->rope_theta > 0.f) {
    s = glt_rope_fwd(q, d->n_q_heads, k, d->n_kv_heads, d->B, d->T, d->head_dim, d->rope_theta, 0, stream);
    if (s != GLT_OK) return s;
  }
  s = glt_attention_fwd(q, k, v, a, d->B, d->T, d->n_q_heads, d->n_kv_heads, d->head_dim,
                        1.0f / std::sqrt((float)d->head_dim), 1, ws + L.vt, L.total - L.vt, stream);
  if (s != GLT_OK) return s;
  const Proj o = {w->o_proj, pb + P.o / 2, m.D, x};
  if ((s = project(a, m.M, m.nq, &o, 1, EPI_RESID, "o_proj", st)) != GLT_OK) return s;

  // grafted MLP block (reference :57-290)
  s = glt_rmsnorm_fwd(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w->ln_post),
                      static_cast<uint16_t*>(x_ffn), var_post, (int32_t)m.M, (int32_t)m.D, d->rms_eps, stream);
  if (s != GLT_OK) return s;
  glt_mlp_desc md = d->mlp;
  md.flags |= GLT_MLP_RESIDUAL;
  return glt_mlp_fwd(&md, &w->mlp, x_ffn, x, gate_pre, up_pre, inter ? inter : ws + L.inter, stream);
}

}  // extern "C"

// ===================================================================== model
// forward_model (reference grafting.hip:224-271) and the shadow-eval
// statistics of its logits (grafting.hip:504-547).
namespace glt {
namespace {

// out[t] = table[ids[t]], 16 bytes per lane when rows allow it
__global__ void __launch_bounds__(256) embedding_kernel(const int32_t* ids, const uint16_t* table, int V, int D,
                                                        uint16_t* out, bool vec) {
  const int64_t t = blockIdx.x;
  const int id = ids[t];
  const bool ok = id >= 0 && id < V;
  const uint16_t* src = table + (int64_t)(ok ? id : 0) * D;
  uint16_t* dst = out + t * D;
  if (vec) {
    for (int c = threadIdx.x; c < D / 8; c += 256) {
      u32x4 v = reinterpret_cast<const u32x4*>(src)[c];
      if (!ok) v = u32x4{0u, 0u, 0u, 0u};
      reinterpret_cast<u32x4*>(dst)[c] = v;
    }
  } else {
    for (int c = threadIdx.x; c < D; c += 256) dst[c] = ok ? src[c] : (uint16_t)0;
  }
}

// Per-row eval terms: f64 sum / sum of squares of the f32 logits, for rows
// t < T-1 the f32 cross-entropy max + log(sum exp(x - max)) - x_label
// against ids[b, t+1], and (rows hash form only) an FNV-1a hash of the row.
struct EvalRow {
  double sum, sumsq;
  uint64_t hash;
  float nll;
  int32_t scored;
};
// the reference's offset basis (grafting.hip:505): the published FNV-1a basis
// 14695981039346656037 with its last digit missing; the hash is defined by it
constexpr uint64_t kFnvBasis = 1469598103934665603ULL;
constexpr uint64_t kFnvPrime = 1099511628211ULL;  // 2^40 + 0x1B3

// Row-hash form: every row is cut into kEvalChunks chunks of
// ceil(V / kEvalChunks) logits (the last ones shorter or empty), which
// defines that hash; one thread walks one chunk in order.
constexpr int kEvalChunks = 16;

__device__ __forceinline__ void chunk_range(int V, int c, int& v0, int& v1) {
  const int L = (V + kEvalChunks - 1) / kEvalChunks;
  v0 = min(V, c * L);
  v1 = min(V, v0 + L);
}

// The reference hash's passes cut every row into 2^shift chunks of
// ceil(V / 2^shift) logits rounded up to a multiple of 8 (the last chunks
// shorter or empty); any cut gives the same hash. One thread walks one chunk,
// so the cut sets the threads: about kHashThreads of them, four wavefronts per
// SIMD (16 chunks per row whatever the rows left half the SIMDs idle at 2048
// rows: 1.29 ms for the two nibble passes, 0.31 this way, half of that from the
// eight runs instead of sixteen), between 16 chunks per row and 1024. The power of
// two costs up to 40 % just past a step (V = 32000: 2048 rows 118 us, 2049 154, 3000
// 188, 4096 255; 16 chunks per row with sixteen runs 420, 421, 419, 435).
constexpr int64_t kHashThreads = 262144;
__host__ __device__ inline int hash_shift(int64_t rows) {
  int sh = 4;
  while (sh < 10 && (rows << (sh + 1)) <= kHashThreads) ++sh;
  return sh;
}

__device__ __forceinline__ void hash_chunk_range(int V, int shift, int c, int& v0, int& v1) {
  const int L = (((V + (1 << shift) - 1) >> shift) + 7) & ~7;
  v0 = min((int64_t)V, (int64_t)c * L);
  v1 = min(V, v0 + L);
}

// Walks the bf16 logits x[v0, v1) in order, f(bits) for one and f2(word) for
// two (the first in the low half): eight 16-byte loads in flight per thread,
// single elements up to the first 16-byte boundary (rows of odd V start off
// it) and after the last whole piece.
template <typename F, typename F2>
__device__ __forceinline__ void walk_chunk(const uint16_t* x, int v0, int v1, F&& f, F2&& f2) {
  int v = v0;
  for (; v < v1 && (reinterpret_cast<uintptr_t>(x + v) & 15) != 0; ++v) f((uint32_t)x[v]);
  for (; v + 64 <= v1; v += 64) {
    u32x4 q[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = *reinterpret_cast<const u32x4*>(x + v + 8 * i);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) f2(q[i][e]);
  }
  for (; v + 8 <= v1; v += 8) {
    const u32x4 q = *reinterpret_cast<const u32x4*>(x + v);
#pragma unroll
    for (int e = 0; e < 4; ++e) f2(q[e]);
  }
  for (; v < v1; ++v) f((uint32_t)x[v]);
}
template <typename F>
__device__ __forceinline__ void walk_chunk(const uint16_t* x, int v0, int v1, F&& f) {
  walk_chunk(x, v0, v1, f, [&](uint32_t w) {
    f(w & 0xFFFFu);
    f(w >> 16);
  });
}

// Row-hash form: one workgroup per 16 rows, 16 threads per row: thread c of
// a row takes chunk c and accumulates its f64 sum and sum of squares, its
// maximum and the FNV-1a hash of the chunk's f32 bytes from the basis. The
// row's threads then share their maxima through LDS, sum exp(x - max) over
// their chunks, and thread 0 of the row adds the parts in chunk order and
// hashes the chunk hashes' little-endian bytes in order.
__global__ void __launch_bounds__(256) eval_rows_kernel(const uint16_t* logits, int64_t ld, const int32_t* ids, int B,
                                                        int T, int V, EvalRow* rows) {
  __shared__ float s_max[16][kEvalChunks], s_se[16][kEvalChunks];
  __shared__ double s_sum[16][kEvalChunks], s_sq[16][kEvalChunks];
  __shared__ uint64_t s_h[16][kEvalChunks];
  const int lr = threadIdx.x >> 4, c = threadIdx.x & (kEvalChunks - 1);
  const int64_t r = (int64_t)blockIdx.x * 16 + lr;
  const bool valid = r < (int64_t)B * T;
  int v0, v1;
  chunk_range(V, c, v0, v1);
  const uint16_t* x = logits + (valid ? r : 0) * ld;
  double s = 0.0, s2 = 0.0;
  float mx = -INFINITY;
  uint64_t h = kFnvBasis;
  if (valid)
    walk_chunk(x, v0, v1, [&](uint32_t h16) {
      const uint32_t bits = h16 << 16;
      const float f = __uint_as_float(bits);
      s += f;
      s2 += (double)f * f;
      mx = fmaxf(mx, f);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        h ^= (bits >> (8 * k)) & 0xFFu;
        h *= kFnvPrime;
      }
    });
  s_max[lr][c] = mx;
  __syncthreads();
  float rmx = -INFINITY;
#pragma unroll
  for (int k = 0; k < kEvalChunks; ++k) rmx = fmaxf(rmx, s_max[lr][k]);
  const int b = valid ? (int)(r / T) : 0, t = valid ? (int)(r - (int64_t)b * T) : 0;
  const bool scored = valid && t < T - 1;
  float se = 0.f;
  if (scored) walk_chunk(x, v0, v1, [&](uint32_t h16) { se += expf(__uint_as_float(h16 << 16) - rmx); });
  s_se[lr][c] = se;
  s_sum[lr][c] = s;
  s_sq[lr][c] = s2;
  s_h[lr][c] = h;
  __syncthreads();
  if (!valid || c != 0) return;
  EvalRow o{0.0, 0.0, kFnvBasis, 0.f, 0};
  float tse = 0.f;
  for (int k = 0; k < kEvalChunks; ++k) {
    o.sum += s_sum[lr][k];
    o.sumsq += s_sq[lr][k];
    tse += s_se[lr][k];
    const uint64_t hk = s_h[lr][k];
    for (int j = 0; j < 8; ++j) {
      o.hash ^= (hk >> (8 * j)) & 0xFFu;
      o.hash *= kFnvPrime;
    }
  }
  if (scored) {
    const int label = ids[(int64_t)b * T + t + 1];
    const float xl = (label >= 0 && label < V) ? __uint_as_float((uint32_t)x[label] << 16) : NAN;
    o.nll = (rmx + logf(tse)) - xl;
    o.scored = 1;
  }
  rows[r] = o;
}

// (max, sum of exp(x - max)) pairs: the sum rescaled to the larger maximum
__device__ __forceinline__ void lse_merge(float& m, float& se, float m2, float se2) {
  const float M = fmaxf(m, m2);
  se = se * __expf(m - M) + se2 * __expf(m2 - M);
  m = M;
}

// Row statistics without the row hash (the reference hash runs in its own
// passes): one workgroup per row reads it once with coalesced 16-byte loads.
// Each thread keeps a running maximum m and the sum of exp(x - m), rescaled
// when m grows (once per 8 logits at most), and f64 sums of x and x^2; the
// threads' parts are merged by a butterfly in each wavefront and the four
// wavefront results in order.
__global__ void __launch_bounds__(256) eval_row_stats_kernel(const uint16_t* logits, int64_t ld, const int32_t* ids,
                                                             int T, int V, EvalRow* rows) {
  __shared__ float s_m[4], s_se[4];
  __shared__ double s_s[4], s_q[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t r = blockIdx.x;
  const uint16_t* x = logits + r * ld;
  double s = 0.0, s2 = 0.0;
  // The running maximum starts at the lowest finite value, so exp(-inf - m) is
  // 0 and the first chunk's rescale of the zero sum needs no test. Each chunk
  // rescales the sum to the new maximum (a factor of 1 when it did not grow),
  // branch-free; exp(x - m) is exp2((x - m) log2(e)): x log2(e) - m log2(e) in one
  // fma, as fast (the pass waits for memory), is off by the rounding of m log2(e),
  // which past m = 1e9 is more than exp2's range.
  constexpr float kLog2e = 1.4426950408889634f;
  float m = -3.4028235e38f, se = 0.f;
  auto add8 = [&](const u32x4& q) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = __uint_as_float(q[e] << 16);
      f[2 * e + 1] = __uint_as_float(q[e] & 0xFFFF0000u);
    }
    float lm = f[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) lm = fmaxf(lm, f[e]);
    const float mn = fmaxf(m, lm);
    se *= __builtin_amdgcn_exp2f((m - mn) * kLog2e);
    m = mn;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      se += __builtin_amdgcn_exp2f((f[e] - mn) * kLog2e);
      // squared in f64 like the reference (static_cast<double>(f) * f): the
      // f32 square of a large or tiny logit overflows or underflows; the
      // product of two f32 values is exact in f64, so one fma is the
      // reference's multiply and add
      const double d = (double)f[e];
      s += d;
      s2 = __builtin_fma(d, d, s2);
    }
  };
  auto add1 = [&](int v) {
    const float f = __uint_as_float((uint32_t)x[v] << 16);
    if (f > m) {
      se *= __expf(m - f);
      m = f;
    }
    se += __expf(f - m);
    const double d = (double)f;
    s += d;
    s2 = __builtin_fma(d, d, s2);
  };
  // whole 16-byte pieces from the first boundary of the row; the elements
  // before it (a row of odd V starts off it) and after the last piece one each
  const int head = min(V, (int)((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / 2);
  const u32x4* xc = reinterpret_cast<const u32x4*>(x + head);
  const int nc = (V - head) >> 3, tail = head + 8 * nc;
  int c = tid;
  for (; c + 768 < nc; c += 1024) {
    u32x4 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = __builtin_nontemporal_load(xc + c + 256 * u);
#pragma unroll
    for (int u = 0; u < 4; ++u) add8(q[u]);
  }
  for (; c < nc; c += 256) add8(__builtin_nontemporal_load(xc + c));
  if (tid < head) add1(tid);
  if (tid < V - tail) add1(tail + tid);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lse_merge(m, se, __shfl_xor(m, o, 64), __shfl_xor(se, o, 64));
    s += __shfl_xor(s, o, 64);
    s2 += __shfl_xor(s2, o, 64);
  }
  if (lane == 0) {
    s_m[tid >> 6] = m;
    s_se[tid >> 6] = se;
    s_s[tid >> 6] = s;
    s_q[tid >> 6] = s2;
  }
  __syncthreads();
  if (tid != 0) return;
  EvalRow o{s_s[0], s_q[0], kFnvBasis, 0.f, 0};
  float rmx = s_m[0], tse = s_se[0];
  for (int k = 1; k < 4; ++k) {
    o.sum += s_s[k];
    o.sumsq += s_q[k];
    lse_merge(rmx, tse, s_m[k], s_se[k]);
  }
  const int t = (int)(r % T);
  if (t < T - 1) {
    const int label = ids[r + 1];
    const float xl = (label >= 0 && label < V) ? __uint_as_float((uint32_t)x[label] << 16) : NAN;
    o.nll = (rmx + logf(tse)) - xl;
    o.scored = 1;
  }
  rows[r] = o;
}

// ------------------------------------------------ the reference's logits hash
// The reference hashes every f32 logit's four little-endian bytes in (b, t, v)
// order with one FNV-1a chain, h = (h ^ byte) * P mod 2^64 (grafting.hip:536-546),
// continued across its eval batches. That chain is computed here exactly, in
// parallel over the chunks of all rows (chunk k = part k % 2^shift of row
// k >> shift), in three passes:
//  * P is odd, so the low byte of h evolves on its own:
//    s' = ((s ^ byte) * P) mod 256. Bit j of s' depends only on bits 0..j of
//    s, so the low nibble is a 16-state chain; and it depends on bit j itself
//    only by XOR, so starting states that differ in the nibble's top bit end
//    differing in exactly that bit: eight runs give the map of 16 states
//    (Map8). Pass 1 runs every chunk from the eight low nibbles 0..7; the maps
//    compose in order from the start hash's nibble to every chunk's starting
//    low nibble.
//  * Pass 2 does the same for the high nibble of the low byte, each chunk's
//    eight runs starting from its known low nibble.
//  * With the low byte s of h known at every step, h ^ byte = h + ((s ^ byte)
//    - s), so a chunk maps h to h * P^(4 n) + B (n logits). Pass 3 runs every
//    chunk once from h = its starting low byte s, giving B = h_end - s P^(4n);
//    the (P^(4n), B) pairs compose in order, h <- h A + B.
// A bf16 logit widens to f32 bits w << 16: its bytes are 0, 0, lo, hi.
//
// Each pass's workgroup (256 consecutive chunks) also composes its maps, and
// the next pass's forms its chunks' starting states from them, so that between
// two passes only one small launch runs over the workgroups. With a factor P^2
// carried along a logit is t ^= lo, t *= P, t ^= hi, t *= P^3. Pass 1 needs
// four bits of each run: a byte per run, four runs per register, P = 3 and P^3
// = 11 mod 16 as shift-adds, 12 instructions per logit (two runs per register
// and 24-bit multiplies, 18 instructions: 166 against 133 us for 2048 rows of
// 128256). Pass 2 needs all eight: two runs per register as 8-bit fields 16
// bits apart, one 24-bit multiply for both, 18 instructions (167 us, 124 of it
// their issue; a packed 16-bit multiply needs no masks and took 12 us more in
// each pass). Reading 525 MB takes 81 us of each pass at least. Fetching the
// chunks' lines eight lanes to a line through LDS, or the next 128 bytes while
// the last are walked, changed the three passes by less than 3 %.
constexpr uint32_t kP8 = (uint32_t)(kFnvPrime & 0xFF);
constexpr uint64_t kP2 = kFnvPrime * kFnvPrime, kP3 = kP2 * kFnvPrime;
constexpr uint64_t inverse64(uint64_t a) {  // of an odd a, mod 2^64 (Newton, doubling the correct bits)
  uint64_t x = a;                           // right in 3 bits
  for (int i = 0; i < 6; ++i) x *= 2 - a * x;
  return x;
}
constexpr uint64_t kP2Inv = inverse64(kP2);
static_assert(kP2Inv * kP2 == 1, "inverse of P^2 mod 2^64");

// Map of 16 nibbles f with f(s ^ 8) = f(s) ^ 8: nibble i of the word is f(i),
// i < 8.
typedef uint32_t Map8;
constexpr Map8 kMapIdentity = 0x76543210u;
__device__ __forceinline__ uint32_t map_apply(Map8 f, uint32_t s) { return ((f >> (4 * (s & 7))) & 15u) ^ (s & 8u); }
__device__ __forceinline__ Map8 map_then(Map8 f, Map8 g) {  // first f, then g
  Map8 h = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) h |= map_apply(g, (f >> (4 * i)) & 15u) << (4 * i);
  return h;
}
// The composition of the maps of threads 0 .. t-1 (in that order) of the 256
// threads; *total that of all.
__device__ __forceinline__ Map8 scan_maps(Map8 f, Map8* lds, Map8* total) {
  const int t = threadIdx.x;
  lds[t] = f;
  __syncthreads();
  for (int w = 1; w < 256; w *= 2) {
    const Map8 g = t >= w ? lds[t - w] : kMapIdentity;
    __syncthreads();
    f = map_then(g, f);
    lds[t] = f;
    __syncthreads();
  }
  const Map8 before = t ? lds[t - 1] : kMapIdentity;
  *total = lds[255];
  __syncthreads();
  return before;
}

// Pass 1 (HIGH false) and 2 (HIGH true) over 256 chunks: maps[k] of chunk k
// and agg[block] of the workgroup's chunks in order. Pass 2 first forms its
// chunks' starting low nibbles from pass 1's maps (lo_maps) and the
// workgroup's (lo_start), and writes them to start[k].
template <bool HIGH>
__global__ void __launch_bounds__(256) hash_nibble_kernel(const uint16_t* logits, int64_t ld, int64_t chunks, int shift,
                                                          int V, const Map8* __restrict__ lo_maps,
                                                          const uint8_t* __restrict__ lo_start,
                                                          uint8_t* __restrict__ start, Map8* __restrict__ maps,
                                                          Map8* __restrict__ agg) {
  __shared__ Map8 lds[256];
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool in = k < chunks;
  Map8 total;
  uint32_t base = 0;
  if (HIGH) {
    const Map8 before = scan_maps(in ? lo_maps[k] : kMapIdentity, lds, &total);
    base = map_apply(before, lo_start[blockIdx.x]);
    if (in) start[k] = (uint8_t)base;
  }
  Map8 f = kMapIdentity;
  if (in) {
    int v0, v1;
    hash_chunk_range(V, shift, (int)(k & ((1 << shift) - 1)), v0, v1);
    const uint16_t* row = logits + (k >> shift) * ld;
    f = 0;
    if constexpr (!HIGH) {
      // byte b of st[j]: run 4 j + b, its low nibble times P^2 (the byte's
      // high nibble is left over); P = 3 and P^3 = 11 mod 16
      constexpr uint32_t kFields = 0x0F0F0F0Fu;
      static_assert((kFnvPrime & 15) == 3 && (kP3 & 15) == 11, "the shifts below");
      uint32_t st[2] = {0, 0};
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) st[i >> 2] |= (i * (uint32_t)(kP2 & 15) & 15u) << (8 * (i & 3));
      auto logit = [&](uint32_t lo, uint32_t hi) {  // each byte in all four
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          uint32_t t = (st[j] ^ lo) & kFields;
          t += t << 1;               // 3 t <= 45
          t = (t ^ hi) & kFields;
          uint32_t t3 = t + (t << 1);
          asm("" : "+v"(t3));        // two shift-adds, not one 32-bit multiply at a quarter of their rate
          st[j] = (t << 3) + t3;     // 11 t <= 165
        }
      };
      walk_chunk(
          row, v0, v1,
          [&](uint32_t w) {
            logit(__builtin_amdgcn_perm(0u, w, 0x00000000u), __builtin_amdgcn_perm(0u, w, 0x01010101u));
          },
          [&](uint32_t w) {
            logit(__builtin_amdgcn_perm(0u, w, 0x00000000u), __builtin_amdgcn_perm(0u, w, 0x01010101u));
            logit(__builtin_amdgcn_perm(0u, w, 0x02020202u), __builtin_amdgcn_perm(0u, w, 0x03030303u));
          });
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        f |= (((st[i >> 2] >> (8 * (i & 3))) * (uint32_t)(kP2Inv & 15)) & 15u) << (4 * i);
    } else {
      // fields 0 and 16 of st[j]: runs 2 j and 2 j + 1 (times P^2; the bits
      // above each field's 8 are left over)
      constexpr uint32_t kFields = 0x00FF00FFu;
      uint32_t st[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a = base | (2 * j) << 4, b = base | (2 * j + 1) << 4;
        st[j] = (a | b << 16) * (uint32_t)(kP2 & 0xFF);
      }
      auto logit = [&](uint32_t lo, uint32_t hi) {  // each byte in both fields
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          st[j] = ((st[j] ^ lo) & kFields) * kP8;
          st[j] = ((st[j] ^ hi) & kFields) * (uint32_t)(kP3 & 0xFF);
        }
      };
      walk_chunk(
          row, v0, v1,
          [&](uint32_t w) {
            logit(__builtin_amdgcn_perm(0u, w, 0x0C000C00u), __builtin_amdgcn_perm(0u, w, 0x0C010C01u));
          },
          [&](uint32_t w) {
            logit(__builtin_amdgcn_perm(0u, w, 0x0C000C00u), __builtin_amdgcn_perm(0u, w, 0x0C010C01u));
            logit(__builtin_amdgcn_perm(0u, w, 0x0C020C02u), __builtin_amdgcn_perm(0u, w, 0x0C030C03u));
          });
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t s2 = ((st[j] & kFields) * (uint32_t)(kP2Inv & 0xFF)) >> 4;
        f |= ((s2 & 15u) | ((s2 >> 16) & 15u) << 4) << (8 * j);
      }
    }
    maps[k] = f;
  }
  scan_maps(f, lds, &total);
  if (threadIdx.x == 0) agg[blockIdx.x] = total;
}

// Starting nibble of every workgroup's first chunk from the start hash's
// nibble, in order.
__global__ void __launch_bounds__(256) hash_starts_kernel(const Map8* __restrict__ agg, int64_t nblocks, uint32_t start,
                                                          uint8_t* __restrict__ bstart) {
  __shared__ Map8 lds[256];
  const int t = threadIdx.x;
  const int64_t q = (nblocks + 255) / 256;
  const int64_t b0 = min(nblocks, t * q), b1 = min(nblocks, b0 + q);
  Map8 f = kMapIdentity, total;
  for (int64_t b = b0; b < b1; ++b) f = map_then(f, agg[b]);
  uint32_t s = map_apply(scan_maps(f, lds, &total), start);
  for (int64_t b = b0; b < b1; ++b) {
    bstart[b] = (uint8_t)s;
    s = map_apply(agg[b], s);
  }
}

// h * P mod 2^64 with P = 2^40 + 0x1B3.
__device__ __forceinline__ uint64_t fnv_mul(uint64_t h) { return (h << 40) + h * 0x1B3ull; }

struct Affine {
  uint64_t a, b;  // h -> h * a + b
};
// first x, then y
__device__ __forceinline__ Affine affine_then(Affine x, Affine y) { return Affine{x.a * y.a, x.b * y.a + y.b}; }

// Pass 3: each chunk run once from h = its starting low byte, reduced to one
// affine map per workgroup of 256 chunks (order-preserving tree).
__global__ void __launch_bounds__(256) hash_affine_kernel(const uint16_t* logits, int64_t ld, int64_t chunks, int shift,
                                                          int V, const uint8_t* __restrict__ start_lo,
                                                          const Map8* __restrict__ hi_maps,
                                                          const uint8_t* __restrict__ hi_start,
                                                          Affine* __restrict__ out) {
  __shared__ uint64_t sa[256], sb[256];
  __shared__ Map8 lds[256];
  const int t = threadIdx.x;
  const int64_t k = (int64_t)blockIdx.x * 256 + t;
  Map8 total;
  const Map8 before = scan_maps(k < chunks ? hi_maps[k] : kMapIdentity, lds, &total);
  Affine f{1, 0};
  if (k < chunks) {
    int v0, v1;
    hash_chunk_range(V, shift, (int)(k & ((1 << shift) - 1)), v0, v1);
    const uint64_t s0 = start_lo[k] | map_apply(before, hi_start[blockIdx.x]) << 4;
    // h with a factor P^2 carried along, as in the other passes: two 64-bit
    // multiplications per logit instead of four
    uint64_t h = s0 * kP2;
    walk_chunk(logits + (k >> shift) * ld, v0, v1, [&](uint32_t w) {
      h = fnv_mul(h ^ (w & 0xFFu));
      h = (h ^ (w >> 8)) * kP3;
    });
    h *= kP2Inv;
    // P^(4 n) by squaring
    uint64_t a = 1, p4 = fnv_mul(fnv_mul(fnv_mul(kFnvPrime)));
    for (uint32_t n = (uint32_t)(v1 - v0); n; n >>= 1, p4 *= p4)
      if (n & 1) a *= p4;
    f = Affine{a, h - s0 * a};
  }
  sa[t] = f.a;
  sb[t] = f.b;
  __syncthreads();
  for (int w = 1; w < 256; w *= 2) {
    if ((t & (2 * w - 1)) == 0) {
      const Affine r = affine_then(Affine{sa[t], sb[t]}, Affine{sa[t + w], sb[t + w]});
      sa[t] = r.a;
      sb[t] = r.b;
    }
    __syncthreads();
  }
  if (t == 0) out[blockIdx.x] = Affine{sa[0], sb[0]};
}

// The whole batch from its rows and (exact hash) its workgroups' affine maps:
// each thread takes a run of consecutive ones, the runs join in order.
struct EvalTotal {
  double nll, sum, sumsq;
  int64_t count;
  Affine hash;
};
__global__ void __launch_bounds__(256) eval_total_kernel(const EvalRow* __restrict__ rows, int64_t R,
                                                         const Affine* __restrict__ aff, int64_t naff,
                                                         EvalTotal* __restrict__ out) {
  __shared__ EvalTotal s[256];
  const int t = threadIdx.x;
  EvalTotal v{0.0, 0.0, 0.0, 0, {1, 0}};
  const int64_t qr = (R + 255) / 256, qa = (naff + 255) / 256;
  for (int64_t r = t * qr; r < min(R, (t + 1) * qr); ++r) {
    v.sum += rows[r].sum;
    v.sumsq += rows[r].sumsq;
    if (rows[r].scored) {
      v.nll += rows[r].nll;
      ++v.count;
    }
  }
  for (int64_t a = t * qa; a < min(naff, (t + 1) * qa); ++a) v.hash = affine_then(v.hash, aff[a]);
  s[t] = v;
  __syncthreads();
  for (int w = 1; w < 256; w *= 2) {
    if ((t & (2 * w - 1)) == 0) {
      const EvalTotal o = s[t + w];
      s[t].nll += o.nll;
      s[t].sum += o.sum;
      s[t].sumsq += o.sumsq;
      s[t].count += o.count;
      s[t].hash = affine_then(s[t].hash, o.hash);
    }
    __syncthreads();
  }
  if (t == 0) *out = s[0];
}

struct ModelWs {
  size_t x, x_ffn, var, layer, total;
};
ModelWs model_ws(const glt_model* m) {
  const glt_layer_desc& d0 = m->descs[0];
  const int64_t M = (int64_t)d0.B * d0.T, D = d0.mlp.D;
  ModelWs w{};
  w.x = 0;
  w.x_ffn = up(w.x + M * D * 2);
  w.var = up(w.x_ffn + M * D * 2);
  w.layer = up(w.var + M * 4);
  size_t lw = 0;
  for (int l = 0; l < m->num_layers; ++l) lw = std::max(lw, glt_layer_fwd_workspace_size(&m->descs[l]));
  w.total = up(w.layer + lw);
  return w;
}

}  // namespace
}  // namespace glt

extern "C" {

glt_status glt_embedding(const int32_t* ids, int64_t n, const uint16_t* table, int32_t V, int32_t D, uint16_t* out,
                         void* stream) {
  GLT_CHECK(n >= 0 && V > 0 && D > 0, GLT_ERR_SHAPE, "glt_embedding: n=%lld V=%d D=%d", (long long)n, V, D);
  if (n == 0) return GLT_OK;
  GLT_CHECK(ids && table && out, GLT_ERR_INVALID_ARG, "glt_embedding: null pointer");
  const bool vec = D % 8 == 0 && (reinterpret_cast<uintptr_t>(table) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  GLT_LAUNCH("embedding", embedding_kernel, dim3((unsigned)n), dim3(256), 0, as_stream(stream), ids, table, V, D, out,
             vec);
  GLT_LAUNCH_CHECK("embedding");
  return GLT_OK;
}

// prepared LM head: [V rows, K = D] (forward), then 256-byte aligned the
// transpose [D rows, K = V] (backward), both in the fragment layout
size_t lm_head_t_offset(int32_t V, int32_t D) { return up((size_t)shuf_elems(V, D) * 2); }

size_t glt_lm_head_prepared_size(int32_t V, int32_t D) {
  return (V > 0 && D > 0) ? lm_head_t_offset(V, D) + (size_t)shuf_elems(D, V) * 2 : 0;
}

glt_status glt_lm_head_prepare(const uint16_t* lm_head, int32_t V, int32_t D, void* prepared, void* stream) {
  GLT_CHECK(V > 0 && D > 0, GLT_ERR_SHAPE, "glt_lm_head_prepare: V=%d D=%d", V, D);
  GLT_CHECK(lm_head && prepared && reinterpret_cast<uintptr_t>(prepared) % kAlign == 0, GLT_ERR_ALIGNMENT,
            "glt_lm_head_prepare: null pointer or prepared not %zu-byte aligned", kAlign);
  hipStream_t st = as_stream(stream);
  uint16_t* p = static_cast<uint16_t*>(prepared);
  glt_status s = shuffle_b(lm_head, GLT_DTYPE_BF16, D, false, V, D, p, st);
  if (s != GLT_OK) return s;
  return shuffle_b(lm_head, GLT_DTYPE_BF16, D, true, D, V, p + lm_head_t_offset(V, D) / 2, st);
}

glt_status glt_lm_head_bwd(const uint16_t* grad, int32_t M, int32_t V, const uint16_t* lm_head, const void* prepared,
                           int32_t D, float* dx, void* stream) {
  GLT_CHECK(M >= 0 && D > 0 && V > 0, GLT_ERR_SHAPE, "glt_lm_head_bwd: M=%d D=%d V=%d", M, D, V);
  if (M == 0) return GLT_OK;
  GLT_CHECK(grad && lm_head && prepared && dx, GLT_ERR_INVALID_ARG, "glt_lm_head_bwd: null pointer");
  // dx[m, d] = sum_v grad[m, v] lm_head[v, d]: B(n = d, k = v) = lm_head^T
  const uint16_t* pt = static_cast<const uint16_t*>(prepared) + lm_head_t_offset(V, D) / 2;
  GemmPlan plan;
  plan.label = "lm_head_bwd";
  plan.a_kind = LD_BF16;
  plan.b_kind = LD_SHUF;
  GProb pr = prob(M, D, EPI_STORE, dx);
  pr.out_f32 = 1;
  plan.add_problem(pr);
  plan.add_seg(seg(grad, V, V, D, pt, shuf_k(V)));
  hipStream_t st = as_stream(stream);
  if (gemm_mfma_eligible(plan)) return run_gemm(plan, st);
  GemmPlan gen;
  gen.label = "lm_head_bwd";
  gen.a_kind = gen.b_kind = LD_BF16;
  gen.add_problem(pr);
  GSeg g = seg(grad, V, V, D, lm_head, 1);
  g.b_ks = D;  // B(n = d, k = v) = lm_head[v * D + d]
  gen.add_seg(g);
  return run_gemm(gen, st, false);
}

glt_status glt_lm_head_fwd(const uint16_t* x, int32_t M, int32_t D, const uint16_t* lm_head, const void* prepared,
                           int32_t V, uint16_t* logits, void* stream) {
  GLT_CHECK(M >= 0 && D > 0 && V > 0, GLT_ERR_SHAPE, "glt_lm_head_fwd: M=%d D=%d V=%d", M, D, V);
  if (M == 0) return GLT_OK;
  GLT_CHECK(x && lm_head && prepared && logits, GLT_ERR_INVALID_ARG, "glt_lm_head_fwd: null pointer");
  const Proj p = {lm_head, static_cast<const uint16_t*>(prepared), V, logits};
  return project(x, M, D, &p, 1, EPI_STORE, "lm_head", as_stream(stream));
}

size_t glt_model_fwd_workspace_size(const glt_model* m) {
  return (m && m->num_layers > 0 && m->descs) ? model_ws(m).total : 0;
}

glt_status glt_model_fwd(const glt_model* m, const int32_t* ids, uint16_t* logits, void* workspace,
                         size_t workspace_bytes, void* stream) {
  GLT_CHECK(m && m->num_layers > 0 && m->descs && m->layers && m->embed && m->final_norm && m->lm_head &&
                m->lm_head_prepared && m->V > 0,
            GLT_ERR_INVALID_ARG, "glt_model_fwd: incomplete model");
  const glt_layer_desc& d0 = m->descs[0];
  for (int l = 1; l < m->num_layers; ++l) {
    const glt_layer_desc& d = m->descs[l];
    GLT_CHECK(d.B == d0.B && d.T == d0.T && d.mlp.D == d0.mlp.D && d.n_q_heads == d0.n_q_heads &&
                  d.n_kv_heads == d0.n_kv_heads && d.head_dim == d0.head_dim,
              GLT_ERR_SHAPE, "glt_model_fwd: layer %d's shape differs from layer 0's", l);
  }
  const int64_t M = (int64_t)d0.B * d0.T;
  const int D = d0.mlp.D;
  if (M == 0) return GLT_OK;
  GLT_CHECK(ids && logits, GLT_ERR_INVALID_ARG, "glt_model_fwd: null ids/logits");
  const ModelWs W = model_ws(m);
  GLT_CHECK(workspace && workspace_bytes >= W.total && reinterpret_cast<uintptr_t>(workspace) % kAlign == 0,
            GLT_ERR_WORKSPACE, "glt_model_fwd: needs %zu workspace bytes, %zu-byte aligned", W.total, kAlign);
  char* ws = static_cast<char*>(workspace);
  uint16_t* x = reinterpret_cast<uint16_t*>(ws + W.x);
  uint16_t* x_ffn = reinterpret_cast<uint16_t*>(ws + W.x_ffn);
  float* var = reinterpret_cast<float*>(ws + W.var);
  glt_status s = glt_embedding(ids, M, m->embed, m->V, D, x, stream);
  if (s != GLT_OK) return s;
  for (int l = 0; l < m->num_layers; ++l) {
    glt_layer_desc d = m->descs[l];
    d.mlp.flags = m->use_explicit_graft ? (d.mlp.flags | GLT_MLP_EXPLICIT) : (d.mlp.flags & ~GLT_MLP_EXPLICIT);
    s = glt_layer_fwd(&d, &m->layers[l], x, x_ffn, var, nullptr, nullptr, nullptr, ws + W.layer,
                      W.total - W.layer, stream);
    if (s != GLT_OK) return s;
  }
  // final norm (into x_ffn) and the LM head
  s = glt_rmsnorm_fwd(x, m->final_norm, x_ffn, var, (int32_t)M, D, d0.rms_eps, stream);
  if (s != GLT_OK) return s;
  return glt_lm_head_fwd(x_ffn, (int32_t)M, D, m->lm_head, m->lm_head_prepared, m->V, logits, stream);
}

}  // extern "C"

namespace glt {
namespace {
struct EvalWs {
  size_t rows, maps_lo, maps_hi, start, agg, bstart_lo, bstart_hi, aff, sums, total;
  int64_t chunks, blocks;
  int shift;
};
// The chunks of R rows fall where hash_shift steps down (2048 rows have 262144,
// 2049 rows 131136), so the buffers are laid out for a bound on them that never
// falls as rows grow: a workspace of the largest batch holds every shorter one.
int64_t hash_chunks_bound(int64_t R) { return std::min(R << 10, std::max(R << 4, kHashThreads)); }
EvalWs eval_ws(int64_t R) {
  EvalWs w{};
  w.shift = hash_shift(R);
  w.chunks = R << w.shift;
  w.blocks = cdiv(w.chunks, 256);
  const int64_t chunks = hash_chunks_bound(R), blocks = cdiv(chunks, 256);
  w.rows = 0;
  w.maps_lo = up(w.rows + R * sizeof(EvalRow));
  w.maps_hi = up(w.maps_lo + chunks * sizeof(Map8));
  w.start = up(w.maps_hi + chunks * sizeof(Map8));
  w.agg = up(w.start + chunks);
  w.bstart_lo = up(w.agg + blocks * sizeof(Map8));
  w.bstart_hi = up(w.bstart_lo + blocks);
  w.aff = up(w.bstart_hi + blocks);
  w.sums = up(w.aff + blocks * sizeof(Affine));
  w.total = up(w.sums + sizeof(EvalTotal));
  return w;
}

}  // namespace
}  // namespace glt

extern "C" {

size_t glt_eval_stats_workspace_size(int32_t B, int32_t T) {
  return (B > 0 && T > 0) ? eval_ws((int64_t)B * T).total : 256;
}

glt_status glt_eval_stats(const uint16_t* logits, int64_t ld, const int32_t* ids, int32_t B, int32_t T, int32_t V,
                          int32_t hash_mode, uint64_t hash_in, glt_eval_result* out, void* workspace,
                          size_t workspace_bytes, void* stream) {
  GLT_CHECK(out && B >= 0 && T >= 0 && V > 0 && ld >= V, GLT_ERR_SHAPE, "glt_eval_stats: B=%d T=%d V=%d", B, T, V);
  GLT_CHECK(hash_mode == GLT_EVAL_HASH_REFERENCE || hash_mode == GLT_EVAL_HASH_ROWS, GLT_ERR_INVALID_ARG,
            "glt_eval_stats: hash_mode %d", hash_mode);
  *out = glt_eval_result{0.0, 0, 0.0, 0.0, hash_in};
  const int64_t R = (int64_t)B * T;
  if (R == 0) return GLT_OK;
  GLT_CHECK(logits && ids, GLT_ERR_INVALID_ARG, "glt_eval_stats: null logits/ids");
  GLT_CHECK(workspace && workspace_bytes >= glt_eval_stats_workspace_size(B, T) &&
                reinterpret_cast<uintptr_t>(workspace) % kAlign == 0,
            GLT_ERR_WORKSPACE, "glt_eval_stats: needs %zu workspace bytes, %zu-byte aligned",
            glt_eval_stats_workspace_size(B, T), kAlign);
  const bool exact = hash_mode == GLT_EVAL_HASH_REFERENCE;
  const EvalWs w = eval_ws(R);
  GLT_CHECK(w.blocks < INT32_MAX, GLT_ERR_SHAPE, "glt_eval_stats: %lld rows", (long long)R);
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  EvalRow* rows = reinterpret_cast<EvalRow*>(ws + w.rows);
  if (exact)
    GLT_LAUNCH("eval_rows", eval_row_stats_kernel, dim3((unsigned)R), dim3(256), 0, st, logits, ld, ids, T, V, rows);
  else
    GLT_LAUNCH("eval_rows", eval_rows_kernel, dim3((unsigned)((R + 15) / 16)), dim3(256), 0, st, logits, ld,
               ids, B, T, V, rows);
  GLT_LAUNCH_CHECK("eval_rows");
  Affine* aff = reinterpret_cast<Affine*>(ws + w.aff);
  if (exact) {
    Map8* maps_lo = reinterpret_cast<Map8*>(ws + w.maps_lo);
    Map8* maps_hi = reinterpret_cast<Map8*>(ws + w.maps_hi);
    Map8* agg = reinterpret_cast<Map8*>(ws + w.agg);
    uint8_t* start = reinterpret_cast<uint8_t*>(ws + w.start);
    uint8_t* b_lo = reinterpret_cast<uint8_t*>(ws + w.bstart_lo);
    uint8_t* b_hi = reinterpret_cast<uint8_t*>(ws + w.bstart_hi);
    const dim3 grid((unsigned)w.blocks);
    GLT_LAUNCH("eval_hash_nibble", hash_nibble_kernel<false>, grid, dim3(256), 0, st, logits, ld, w.chunks, w.shift, V,
               (const Map8*)nullptr, (const uint8_t*)nullptr, (uint8_t*)nullptr, maps_lo, agg);
    GLT_LAUNCH_CHECK("hash_nibble");
    GLT_LAUNCH("eval_hash_scan", hash_starts_kernel, dim3(1), dim3(256), 0, st, agg, w.blocks, (uint32_t)(hash_in & 15),
               b_lo);
    GLT_LAUNCH_CHECK("hash_starts");
    GLT_LAUNCH("eval_hash_nibble", hash_nibble_kernel<true>, grid, dim3(256), 0, st, logits, ld, w.chunks, w.shift, V,
               maps_lo, b_lo, start, maps_hi, agg);
    GLT_LAUNCH_CHECK("hash_nibble");
    GLT_LAUNCH("eval_hash_scan", hash_starts_kernel, dim3(1), dim3(256), 0, st, agg, w.blocks,
               (uint32_t)((hash_in >> 4) & 15), b_hi);
    GLT_LAUNCH_CHECK("hash_starts");
    GLT_LAUNCH("eval_hash_affine", hash_affine_kernel, grid, dim3(256), 0, st, logits, ld, w.chunks, w.shift, V, start,
               maps_hi, b_hi, aff);
    GLT_LAUNCH_CHECK("hash_affine");
  }
  if (exact) {
    EvalTotal* sums = reinterpret_cast<EvalTotal*>(ws + w.sums);
    GLT_LAUNCH("eval_total", eval_total_kernel, dim3(1), dim3(256), 0, st, rows, R, aff, w.blocks, sums);
    GLT_LAUNCH_CHECK("eval_total");
    EvalTotal h;
    GLT_CHECK(hipMemcpyAsync(&h, sums, sizeof h, hipMemcpyDeviceToHost, st) == hipSuccess &&
                  hipStreamSynchronize(st) == hipSuccess,
              GLT_ERR_HIP, "glt_eval_stats: copy of the results failed");
    *out = glt_eval_result{h.nll, h.count, h.sum, h.sumsq, hash_in * h.hash.a + h.hash.b};
    return GLT_OK;
  }
  // the rows form chains the row hashes byte by byte, on the host
  std::vector<EvalRow> h((size_t)R);
  GLT_CHECK(hipMemcpyAsync(h.data(), rows, (size_t)R * sizeof(EvalRow), hipMemcpyDeviceToHost, st) == hipSuccess &&
                hipStreamSynchronize(st) == hipSuccess,
            GLT_ERR_HIP, "glt_eval_stats: copy of the results failed");
  uint64_t hash = hash_in;
  for (const EvalRow& r : h) {
    out->logits_sum += r.sum;
    out->logits_sumsq += r.sumsq;
    if (r.scored) {
      out->total_nll += r.nll;
      ++out->count;
    }
    for (int k = 0; k < 8; ++k) {
      hash ^= (r.hash >> (8 * k)) & 0xFFu;
      hash *= kFnvPrime;
    }
  }
  out->logits_hash = hash;
  return GLT_OK;
}

}  // extern "C"
