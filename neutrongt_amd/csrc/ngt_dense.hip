// Dense full-window attention (all pairs), forward and backward.
//
// Reference: CoreAttention.full_attention
//   NeutronGT/models/graphormer_dist_node_level.py:42-65
//   S = (q * sqrt(d)) k^T      (the reference multiplies by sqrt(d))
//   P = softmax(S, -1);  out = P v;  node_score[j] = sum_i mean_h |S[h,i,j]|
// The backward is what autograd derives: dV = P^T G, dP = G V^T,
// dS = P (dP - rowsum(dP P)) = P (dP - D) with D_i = G_i . out_i,
// dQ = sqrt(d) dS K, dK = sqrt(d) dS^T Q.
// With dropout (training mode, reference att_dropout on P): out = (P o M) v
// with M = keep / (1 - p); dV = (P o M)^T G, dP = (G V^T) o M, and D_i = G_i .
// out_i still equals rowsum(dP o P).  The mask is regenerated from
// (seed, head, query, key) in every kernel (DropoutMask).
//
// The kernels are in ngt_dense_fx.hip (fp32, and bf16 at d = 64: fp32 weights
// on the matrix cores) and ngt_dense_mfma.hip (bf16, d <= 32: bf16 weights);
// this file holds the entry points, their workspace layouts and the two small
// kernels both share.
#include "ngt_common.h"

#include <math.h>
#include <stdlib.h>

#include <type_traits>
#include <utility>

namespace ngt {

// Matrix-core kernels (ngt_dense_mfma.hip).
bool mfma_dense_supported(int d);
MfSplit mfma_fwd_split(int n_q, int n_k, int H, bool node_scores);
MfSplit mfma_dq_split(int n_q, int n_k, int H);
int mfma_fused_blocks(int n_q, int n_k, int H, int d);
int mfma_dense_fwd(int d, const void* q, const void* k, const void* v, int n_q, int n_k, int H,
                   float scale, const DropoutMask* dm, void* out, float* out32, float* lse,
                   float* part, MfSplit sp, float* part_ml, float* part_acc, hipStream_t st);
int mfma_dense_bwd(int d, const void* q, const void* k, const void* v, const void* g,
                   const void* out, const float* out32, const float* lse, float* dsum, int n_q,
                   int n_k, int H, float scale, const DropoutMask* dm, void* gq, void* gk, void* gv,
                   MfSplit sq, float* part_dq, int fused_blocks, hipStream_t st);
// fp32 (and bf16, d = 64) matrix-core kernels (ngt_dense_fx.hip).
MfSplit fx_fwd_split(int n_q, int n_k, int H, int d, bool node_scores);
MfSplit fx_score_split(int n_q, MfSplit keys);
MfSplit fx_dq_split(int n_q, int n_k, int H, int d);
size_t fx_fwd_image_bytes(int dtype, int n_q, int n_k, int H, int d);
size_t fx_bwd_image_bytes(int dtype, int n_q, int n_k, int H, int d);
int fx_dense_fwd(int dtype, int d, const void* q, const void* k, const void* v, int n_q, int n_k,
                 int H, float scale, const DropoutMask* dm, void* out, float* out32, float* lse,
                 float* part, MfSplit sp, MfSplit scores, float* part_ml, float* part_acc,
                 char* images, hipStream_t st);
int fx_dense_bwd(int dtype, int d, const void* q, const void* k, const void* v, const void* go,
                 const void* out, const float* out32, const float* lse, float* dsum, int n_q,
                 int n_k, int H, float scale, const DropoutMask* dm, void* gq, void* gk, void* gv,
                 MfSplit sq, float* part_dq, char* images, hipStream_t st);

namespace {

constexpr int kBlock = 256;

// The key splits' softmax states of one (query, head) per thread, in split
// order: M = max M_s, l = sum l_s e^(M_s - M), out = sum acc_s e^(M_s - M) / l.
template <typename T, int DH>
__global__ __launch_bounds__(kBlock) void k_dense_combine(
    const float* __restrict__ part_ml, const float* __restrict__ part_acc, int32_t n_split,
    int32_t n_q, int32_t H, T* __restrict__ out, float* __restrict__ out32,
    float* __restrict__ lse) {
  const int64_t n = int64_t(n_q) * H;
  for (int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; t < n;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t qi = t / H, h = t % H;
    float M = -INFINITY;
    for (int s = 0; s < n_split; ++s) M = fmaxf(M, part_ml[2 * ((s * H + h) * n_q + qi)]);
    float l = 0.f, acc[DH];
#pragma unroll
    for (int c = 0; c < DH; ++c) acc[c] = 0.f;
    for (int s = 0; s < n_split; ++s) {
      const int64_t r = (s * H + h) * n_q + qi;
      const float a = __expf(part_ml[2 * r] - M);
      l = fmaf(a, part_ml[2 * r + 1], l);
      float pa[DH];
      load_row<float, DH>(part_acc + (s * n_q + qi) * H * DH + h * DH, pa);
#pragma unroll
      for (int c = 0; c < DH; ++c) acc[c] = fmaf(a, pa[c], acc[c]);
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < DH; ++c) acc[c] *= inv;
    store_row<T, DH>(out + t * DH, acc);
    if (out32) store_f32<DH>(out32 + t * DH, acc);
    lse[h * n_q + qi] = M + __logf(l);
  }
}

// node_score[j] = sum over rows of ns_part[:, j] / H.  A block of 1024
// threads takes 64 keys (lane = key) and splits the rows over its 16 waves
// (wave w: rows w, w + 16, ...); the waves' sums are added in wave order, or with
// PAIRS, where the rows are many (query splits), by halves: 8,000 queries in 32
// splits, 4 heads of 32, 6.6e-8 -> 4.0e-8 of float64.
// One thread per key down all rows (2,000 at 16,000 nodes, 8 heads) left the
// loads' latency exposed: 466 us for 128 MB.
constexpr int kScoreThreads = 1024;
constexpr int kScoreWaves = kScoreThreads / kWave;
template <bool PAIRS>
__global__ __launch_bounds__(kScoreThreads) void k_dense_scores(
    const float* __restrict__ part, int32_t rows, int32_t n_k, int32_t H, float* __restrict__ ns) {
  __shared__ float red[kScoreWaves][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x >> 6;
  const int64_t j = int64_t(blockIdx.x) * kWave + lane;
  float s = 0.f;
  if (j < n_k) {
#pragma unroll 8
    for (int r = w; r < rows; r += kScoreWaves) s += part[int64_t(r) * n_k + j];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w == 0 && j < n_k) {
    float t[kScoreWaves];
#pragma unroll
    for (int u = 0; u < kScoreWaves; ++u) t[u] = red[u][lane];
    if (PAIRS) {
#pragma unroll
      for (int n = kScoreWaves / 2; n > 0; n /= 2)
#pragma unroll
        for (int u = 0; u < n; ++u) t[u] += t[u + n];
    } else {
#pragma unroll
      for (int u = 1; u < kScoreWaves; ++u) t[0] += t[u];
    }
    ns[j] = t[0] / float(H);
  }
}

// ------------------------------------------------------------------ host side
inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

size_t bwd_ws(int32_t n_q, int32_t H) { return align256(size_t(n_q) * H * 4); }

int check_args(const char* fn, int dtype, int n_q, int n_k, int H, int d) {
  if (dtype != NGT_F32 && dtype != NGT_BF16)
    return set_error(NGT_ERR_ARG, "%s: unknown dtype %d", fn, dtype);
  if (n_q < 0 || n_k < 0 || H < 1 || H > 65535)
    return set_error(NGT_ERR_ARG, "%s: bad sizes n_q=%d n_k=%d H=%d", fn, n_q, n_k, H);
  if (d != 8 && d != 16 && d != 24 && d != 32 && d != 64)
    return set_error(NGT_ERR_UNSUPPORTED, "%s: head_dim=%d (supported 8,16,24,32,64)", fn, d);
  return NGT_OK;
}

// bf16 with d <= 32 runs on ngt_dense_mfma.hip, everything else on
// ngt_dense_fx.hip.
bool use_bf16(int dtype, int d) { return dtype == NGT_BF16 && mfma_dense_supported(d); }

// Forward workspace: [node-score partials, per query split H * n_k][split
// states (m, l) and unnormalised outputs (with a key split)][the operands'
// pieces (ngt_dense_fx.hip)].
struct FwdLayout {
  size_t ml, acc, images, total;
  MfSplit sp, scores;  // of the keys; of the node scores' queries
};
FwdLayout fwd_layout(int dtype, int32_t n_q, int32_t n_k, int32_t H, int32_t d, bool node_scores) {
  FwdLayout L{};
  const bool b16 = use_bf16(dtype, d);
  L.sp = b16 ? mfma_fwd_split(n_q, n_k, H, node_scores) : fx_fwd_split(n_q, n_k, H, d, node_scores);
  L.scores = b16 ? MfSplit{1, n_q} : fx_score_split(n_q, L.sp);
  size_t off = node_scores ? align256(size_t(L.scores.n_split) * H * n_k * 4) : 0;
  if (L.sp.n_split > 1) {
    L.ml = off;
    off += align256(size_t(L.sp.n_split) * n_q * H * 8);
    L.acc = off;
    off += align256(size_t(L.sp.n_split) * n_q * H * d * 4);
  }
  L.images = off;
  if (!b16) off += fx_fwd_image_bytes(dtype, n_q, n_k, H, d);
  L.total = off;
  return L;
}

// Backward workspace: D_i [n_q, H] fp32, the key splits' partial dQ (two
// passes) or the key blocks' partial dQ (single pass), the operands' pieces.
struct BwdLayout {
  size_t part_dq, images, total;
  MfSplit sq;
  int fused;
};
BwdLayout bwd_layout(int dtype, int32_t n_q, int32_t n_k, int32_t H, int32_t d) {
  BwdLayout L{};
  const bool b16 = use_bf16(dtype, d);
  size_t off = bwd_ws(n_q, H);
  L.part_dq = off;
  L.sq = MfSplit{1, 1};
  if (n_q > 0) {
    L.fused = b16 ? mfma_fused_blocks(n_q, n_k, H, d) : 0;
    L.sq = b16 ? mfma_dq_split(n_q, n_k, H) : fx_dq_split(n_q, n_k, H, d);
    const int parts = L.fused > 0 ? L.fused : (L.sq.n_split > 1 ? L.sq.n_split : 0);
    if (parts > 0) off += align256(size_t(parts) * n_q * H * d * 4);
  }
  L.images = off;
  if (!b16) off += fx_bwd_image_bytes(dtype, n_q, n_k, H, d);
  L.total = off;
  return L;
}

template <typename T>
int launch_combine(int d, const float* part_ml, const float* part_acc, int n_split, int n_q, int H,
                   void* out, float* out32, float* lse, hipStream_t st) {
  KernelTimer timer_("dense_combine", st);
  int64_t blocks = (int64_t(n_q) * H + kBlock - 1) / kBlock;
  if (blocks > 65536) blocks = 65536;
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(int(blocks)), dim3(kBlock), 0, st, part_ml, part_acc, n_split,
                       n_q, H, static_cast<T*>(out), out32, lse);
  };
  switch (d) {
    case 8: run(k_dense_combine<T, 8>); break;
    case 16: run(k_dense_combine<T, 16>); break;
    case 24: run(k_dense_combine<T, 24>); break;
    case 32: run(k_dense_combine<T, 32>); break;
    default: run(k_dense_combine<T, 64>); break;
  }
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

__global__ void k_fill_zero(float* __restrict__ p, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

}  // namespace
}  // namespace ngt

using namespace ngt;

extern "C" int ngt_dense_workspace_bytes(int dtype, int32_t n_q, int32_t n_k, int32_t n_heads,
                                         int32_t head_dim, int32_t node_scores,
                                         size_t* fwd_bytes, size_t* bwd_bytes) {
  const int rc = check_args("ngt_dense_workspace_bytes", dtype, n_q, n_k, n_heads, head_dim);
  if (rc != NGT_OK) return rc;
  if (fwd_bytes) *fwd_bytes = n_q > 0 ? fwd_layout(dtype, n_q, n_k, n_heads, head_dim, node_scores != 0).total : 0;
  if (bwd_bytes) *bwd_bytes = bwd_layout(dtype, n_q, n_k, n_heads, head_dim).total;
  return NGT_OK;
}

extern "C" int ngt_dense_fwd(int dtype, const void* q, const void* k, const void* v, int32_t n_q,
                             int32_t n_k, int32_t n_heads, int32_t head_dim, float scale,
                             float dropout_p, uint64_t seed, const uint64_t* seed_dev,
                             void* out, float* out_f32, float* lse, float* node_score,
                             void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_args("ngt_dense_fwd", dtype, n_q, n_k, n_heads, head_dim);
  if (rc != NGT_OK) return rc;
  if (!(scale > 0.f)) return set_error(NGT_ERR_ARG, "ngt_dense_fwd: scale must be > 0");
  DropoutMask dmv{};
  bool drop = false;
  NGT_CHECK_OK(make_dropout("ngt_dense_fwd", dropout_p, seed, seed_dev, n_q, n_k, &dmv, &drop));
  const DropoutMask* dm = drop ? &dmv : nullptr;
  if (n_q > 0 && (!q || !out || !lse)) return set_error(NGT_ERR_ARG, "ngt_dense_fwd: null q/out/lse");
  if (n_k > 0 && (!k || !v)) return set_error(NGT_ERR_ARG, "ngt_dense_fwd: null k/v");
  FwdLayout L{};
  if (n_q > 0) {
    L = fwd_layout(dtype, n_q, n_k, n_heads, head_dim, node_score != nullptr);
    if (L.total && (!workspace || workspace_bytes < L.total))
      return set_error(NGT_ERR_WORKSPACE, "ngt_dense_fwd: workspace %zu < %zu", workspace_bytes,
                       L.total);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (node_score && n_q == 0 && n_k > 0) {  // no queries: every column score is 0
    hipLaunchKernelGGL(k_fill_zero, dim3(unsigned((n_k + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       st, node_score, int64_t(n_k));
    NGT_HIP_CHECK(hipGetLastError());
  }
  if (n_q == 0) return NGT_OK;
  char* ws = static_cast<char*>(workspace);
  float* part = node_score ? reinterpret_cast<float*>(ws) : nullptr;
  float* part_ml = L.sp.n_split > 1 ? reinterpret_cast<float*>(ws + L.ml) : nullptr;
  float* part_acc = L.sp.n_split > 1 ? reinterpret_cast<float*>(ws + L.acc) : nullptr;
  if (use_bf16(dtype, head_dim))
    rc = mfma_dense_fwd(head_dim, q, k, v, n_q, n_k, n_heads, scale, dm, out, out_f32, lse, part,
                        L.sp, part_ml, part_acc, st);
  else
    rc = fx_dense_fwd(dtype, head_dim, q, k, v, n_q, n_k, n_heads, scale, dm, out, out_f32, lse,
                      part, L.sp, L.scores, part_ml, part_acc, ws + L.images, st);
  if (rc != NGT_OK) return rc;
  if (L.sp.n_split > 1)
    NGT_CHECK_OK((dtype == NGT_F32 ? launch_combine<float> : launch_combine<bf16_t>)(
        head_dim, part_ml, part_acc, L.sp.n_split, n_q, n_heads, out, out_f32, lse, st));
  if (!node_score || n_k == 0) return NGT_OK;
  KernelTimer timer_("dense_scores", st);
  hipLaunchKernelGGL(L.scores.n_split > 1 ? k_dense_scores<true> : k_dense_scores<false>,
                     dim3((n_k + kWave - 1) / kWave), dim3(kScoreThreads), 0, st, part,
                     L.scores.n_split * n_heads, n_k, n_heads, node_score);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

extern "C" int ngt_dense_bwd(int dtype, const void* q, const void* k, const void* v,
                             const void* out, const float* out_f32, const void* grad_out,
                             const float* lse, int32_t n_q,
                             int32_t n_k, int32_t n_heads, int32_t head_dim, float scale,
                             float dropout_p, uint64_t seed, const uint64_t* seed_dev,
                             void* grad_q, void* grad_k, void* grad_v, void* workspace,
                             size_t workspace_bytes, void* stream) {
  int rc = check_args("ngt_dense_bwd", dtype, n_q, n_k, n_heads, head_dim);
  if (rc != NGT_OK) return rc;
  if (!(scale > 0.f)) return set_error(NGT_ERR_ARG, "ngt_dense_bwd: scale must be > 0");
  DropoutMask dmv{};
  bool drop = false;
  NGT_CHECK_OK(make_dropout("ngt_dense_bwd", dropout_p, seed, seed_dev, n_q, n_k, &dmv, &drop));
  const DropoutMask* dm = drop ? &dmv : nullptr;
  if (n_q > 0 && (!q || (!out && !out_f32) || !grad_out || !lse || !grad_q))
    return set_error(NGT_ERR_ARG, "ngt_dense_bwd: null query-side pointer");
  if (n_k > 0 && (!k || !v || !grad_k || !grad_v))
    return set_error(NGT_ERR_ARG, "ngt_dense_bwd: null key-side pointer");
  const BwdLayout L = bwd_layout(dtype, n_q, n_k, n_heads, head_dim);
  if (L.total > 0 && (!workspace || workspace_bytes < L.total))
    return set_error(NGT_ERR_WORKSPACE, "ngt_dense_bwd: workspace %zu < %zu", workspace_bytes,
                     L.total);
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  float* dsum = reinterpret_cast<float*>(ws);  // written by the dQ pass
  float* part_dq = L.sq.n_split > 1 || L.fused > 0 ? reinterpret_cast<float*>(ws + L.part_dq)
                                                   : nullptr;
  if (use_bf16(dtype, head_dim))
    return mfma_dense_bwd(head_dim, q, k, v, grad_out, out, out_f32, lse, dsum, n_q, n_k, n_heads,
                          scale, dm, grad_q, grad_k, grad_v, L.sq, part_dq, L.fused, st);
  return fx_dense_bwd(dtype, head_dim, q, k, v, grad_out, out, out_f32, lse, dsum, n_q, n_k,
                      n_heads, scale, dm, grad_q, grad_k, grad_v, L.sq, part_dq, ws + L.images, st);
}
