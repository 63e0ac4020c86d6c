// Weight and bias gradient of a bf16 linear layer in one pass over its rows:
//   dw[o][i] = sum over rows k of dy[k][o] x[k][i],   db[o] = sum of dy[k][o],
// both fp32.  Part of the backward of the encoder's nn.Linear layers
// (MultiHeadAttention projections and FFN, NeutronGT/models/
// graphormer_dist_node_level.py:130-206) under bf16 autocast.
//
// Bound: the matrix cores for wide layers, launch and memory latency for
// narrow ones.  The contraction runs over the rows, so both operands have to be
// turned: a thread loads 8 rows x 8 columns (16 bytes a row), pairs the rows
// with v_perm and writes each column's 8 rows as one 16-byte LDS unit, which is
// what an MFMA lane reads.  Rows are split over blocks (the outputs are few and
// the rows many); a second kernel adds the splits' partials in split order.
//
// With bias, against a batched library GEMM over row chunks, its chunk sum, a
// GEMM for the rows left over and a column sum (6 launches, now 2): 10,584 x 64
// x 64 30.1 -> 7.6 us, 16,000 x 384 x 128 47.9 -> 18.4, 10,007 x 768 x 768 65.3
// -> 31.7 (375 TFLOP/s), 10,007 x 2,304 x 768 92.0 -> 72.8.  Errors against
// float64 are the library's or smaller.
#include "ngt_common.h"

namespace ngt {
namespace {

constexpr int kBlock = 256;
using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using f32x16 = __attribute__((ext_vector_type(16))) float;

struct WgradArgs {
  const uint16_t *x, *dy;  // [n_rows, n_in], [n_rows, n_out]
  int64_t n_rows;
  int32_t n_out, n_in;
  int32_t tiles_m, tiles_n, splits;
  int64_t rows_per_split;  // a multiple of the stage
  float* part;             // [splits][n_out][n_in]
  float* part_b;           // [splits * tiles_n][n_out], or null
};

// Rows of a stage: T = 64 or 128 columns of both operands fill 32 KB.
constexpr int stage_rows(int t) { return 8192 / t; }

// Byte offset of the unit (8 rows from 8 u) of column c.  The xor spreads both
// the writes (a wave's 16 threads write one column each, 8 columns apart) and
// the reads (8 adjacent columns, one unit) over all banks.
template <int T>
__device__ __forceinline__ int unit_at(int c, int u) {
  return c * (2 * stage_rows(T)) + 16 * (u ^ ((c ^ (c >> 3)) & 7));
}

// 8 rows x 8 columns, rows as loaded: w[r][c / 2]
struct Patch {
  uint32_t w[8][4];
};

// Any row pitch and alignment of 2 bytes: the hardware's unaligned loads take
// 16 bytes a row (32,768 x 47 x 768 in two-byte loads 64.7 us, in these 43.4).
struct __attribute__((packed, aligned(2))) Row16 {
  uint64_t lo, hi;
};

__device__ __forceinline__ void load_patch(Patch& p, const uint16_t* __restrict__ m, int64_t row,
                                           int64_t row_end, int32_t n, int32_t col) {
  if (n >= 8) {
    // the last columns of a row: the 8 that end with it, moved down
    const int32_t back = col + 8 > n ? col + 8 - n : 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      Row16 v{0u, 0u};
      if (row + r < row_end && back < 8)
        v = *reinterpret_cast<const Row16*>(m + (row + r) * n + col - back);
      uint64_t lo = v.lo, hi = v.hi;
      if (back) {
        const int sh = 16 * (back & 3);
        if (back >= 4) lo = hi, hi = 0u;
        if (sh) lo = lo >> sh | hi << (64 - sh), hi >>= sh;
      }
      p.w[r][0] = uint32_t(lo), p.w[r][1] = uint32_t(lo >> 32);
      p.w[r][2] = uint32_t(hi), p.w[r][3] = uint32_t(hi >> 32);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        uint32_t lo = 0u, hi = 0u;
        if (row + r < row_end) {
          const uint16_t* q = m + (row + r) * n + col + 2 * c;
          if (col + 2 * c < n) lo = q[0];
          if (col + 2 * c + 1 < n) hi = q[1];
        }
        p.w[r][c] = lo | hi << 16;
      }
  }
}

// Column j's 8 rows, packed in row order.
__device__ __forceinline__ uint4 column_of(const Patch& p, int j) {
  const uint32_t sel = j & 1 ? 0x07060302u : 0x05040100u;
  const int c = j >> 1;
  return make_uint4(__builtin_amdgcn_perm(p.w[1][c], p.w[0][c], sel),
                    __builtin_amdgcn_perm(p.w[3][c], p.w[2][c], sel),
                    __builtin_amdgcn_perm(p.w[5][c], p.w[4][c], sel),
                    __builtin_amdgcn_perm(p.w[7][c], p.w[6][c], sel));
}

// One block: a T x T tile of dw over one split's rows, 4 waves of (T / 2)^2.
// T = 128 reads its LDS half as often per product; T = 64 leaves less padding
// where a layer is narrow.  Blocks are numbered so that each XCD (block number
// mod 8) gets a contiguous run of (split, tile): the tiles of a split share
// its rows in one L2.
template <int T>
__global__ __launch_bounds__(kBlock) void k_wgrad(const WgradArgs a) {
  constexpr int KB = stage_rows(T);   // rows per stage
  constexpr int PC = T / 8;           // patches per 8 rows
  constexpr int F = T / 64;           // 32 x 32 tiles per wave and direction
  constexpr int OPB = T * KB * 2;     // bytes of one operand's stage
  __shared__ __attribute__((aligned(16))) char lds[2][2 * OPB];
  const int tid = threadIdx.x;
  const int total = a.tiles_m * a.tiles_n * a.splits;
  const int per = (total + 7) / 8;
  const int id = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (int(blockIdx.x / 8) >= per || id >= total) return;  // block-uniform
  const int tiles = a.tiles_m * a.tiles_n;
  const int split = id / tiles, tile = id % tiles;
  const int tm = tile / a.tiles_n, tn = tile % a.tiles_n;
  const int64_t r0 = int64_t(split) * a.rows_per_split;
  const int64_t r1 = r0 + a.rows_per_split < a.n_rows ? r0 + a.rows_per_split : a.n_rows;

  // threads 0 .. 127 carry dy (A), the others x (B)
  const bool is_b = tid >= kBlock / 2;
  const int t2 = tid & (kBlock / 2 - 1);
  const int pc = t2 % PC, pu = t2 / PC;  // 8-column group, unit of 8 rows
  const uint16_t* src = is_b ? a.x : a.dy;
  const int32_t n_src = is_b ? a.n_in : a.n_out;
  const int32_t col = (is_b ? tn : tm) * T + 8 * pc;
  const bool sums = a.part_b && !is_b;

  const int wave = tid >> 6, lane = tid & 63;
  const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
  const int l32 = lane & 31, half = lane >> 5;
  f32x16 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  float bsum[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bsum[j] = 0.f;

  Patch p;
  load_patch(p, src, r0 + 8 * pu, r1, n_src, col);
  int buf = 0, turn = tn;  // the bias sums of a stage fall to one of the row of tiles
  for (int64_t r = r0; r < r1; r += KB) {
    char* base = lds[buf] + (is_b ? OPB : 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint4 w = column_of(p, j);
      *reinterpret_cast<uint4*>(base + unit_at<T>(8 * pc + j, pu)) = w;
    }
    if (sums && turn == 0) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          bsum[2 * c] += __uint_as_float(p.w[k][c] << 16);
          bsum[2 * c + 1] += __uint_as_float(p.w[k][c] & 0xffff0000u);
        }
    }
    turn = turn == 0 ? a.tiles_n - 1 : turn - 1;
    // one barrier a stage: the buffer written next was read before the last one
    __syncthreads();
    if (r + KB < r1) load_patch(p, src, r + KB + 8 * pu, r1, n_src, col);
    const char* la = lds[buf];
    const char* lb = lds[buf] + OPB;
#pragma unroll
    for (int k = 0; k < KB / 16; ++k) {
      bf16x8 fa[F], fb[F];
#pragma unroll
      for (int i = 0; i < F; ++i) {
        fa[i] = *reinterpret_cast<const bf16x8*>(la + unit_at<T>(wm + 32 * i + l32, 2 * k + half));
        fb[i] = *reinterpret_cast<const bf16x8*>(lb + unit_at<T>(wn + 32 * i + l32, 2 * k + half));
      }
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    buf ^= 1;
  }

  float* out = a.part + int64_t(split) * a.n_out * a.n_in;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int32_t c = tn * T + wn + 32 * j + l32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int32_t o = tm * T + wm + 32 * i + 8 * (e / 4) + 4 * half + e % 4;
        if (o < a.n_out && c < a.n_in) out[int64_t(o) * a.n_in + c] = acc[i][j][e];
      }
    }
  if (a.part_b) {
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds[0]);  // [KB / 8][T]
    if (!is_b)
#pragma unroll
      for (int j = 0; j < 8; ++j) red[pu * T + 8 * pc + j] = bsum[j];
    __syncthreads();
    if (tid < T && tm * T + tid < a.n_out) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < KB / 8; ++u) s += red[u * T + tid];
      a.part_b[(int64_t(split) * a.tiles_n + tn) * a.n_out + tm * T + tid] = s;
    }
  }
}

// out[i] = sum over c of in[c * n + i] for dw (blocks below blocks_w) and db.
// A block owns 64 outputs; 16 lanes each add the parts c = lane mod 16 in
// order, then the lane sums are added in lane order.
constexpr int kRedLanes = 16, kRedCols = 64;
template <bool VEC>
__global__ __launch_bounds__(kBlock) void k_wgrad_sum(const float* __restrict__ part,
                                                      int32_t n_parts, int64_t n,
                                                      float* __restrict__ dw, int32_t blocks_w,
                                                      const float* __restrict__ part_b,
                                                      int32_t n_parts_b, int32_t n_out,
                                                      float* __restrict__ db) {
  __shared__ float4 red[kRedLanes][kRedCols / 4];
  const bool bias = int(blockIdx.x) >= blocks_w;  // block-uniform
  const float* in = bias ? part_b : part;
  float* out = bias ? db : dw;
  const int32_t parts = bias ? n_parts_b : n_parts;
  const int64_t len = bias ? n_out : n;
  const int q = threadIdx.x % (kRedCols / 4), lane = threadIdx.x / (kRedCols / 4);
  const int64_t i = int64_t(bias ? blockIdx.x - blocks_w : blockIdx.x) * kRedCols + 4 * q;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (VEC) {
    if (i < len) {
#pragma unroll 4
      for (int32_t c = lane; c < parts; c += kRedLanes) {
        const float4 v = *reinterpret_cast<const float4*>(in + c * len + i);
        s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
      }
    }
  } else {
#pragma unroll 4
    for (int32_t c = lane; c < parts; c += kRedLanes) {
      const float* v = in + c * len + i;
      if (i < len) s.x += v[0];
      if (i + 1 < len) s.y += v[1];
      if (i + 2 < len) s.z += v[2];
      if (i + 3 < len) s.w += v[3];
    }
  }
  red[lane][q] = s;
  __syncthreads();
  if (threadIdx.x >= kRedCols) return;
  const int64_t o = i - 4 * q + threadIdx.x;
  if (o >= len) return;
  const float* f = reinterpret_cast<const float*>(red) + threadIdx.x;
  float t = 0.f;
#pragma unroll
  for (int l = 0; l < kRedLanes; ++l) t += f[l * kRedCols];
  out[o] = t;
}

// Splits of the rows.  Two blocks fit a CU's LDS, so 512 fill the chip in one
// round (10,007 x 768 x 768: 37 / 31 / 41 us at 256 / 512 / 1,024 blocks).  More
// splits than that where one would sum more than 2,560 rows in a chain (the
// error against float64 grows with it: 1.2e-7 at 64 rows, 3.1e-7 at 2,560).
// Fewer where a split would be a stage or two, for then its partial costs more
// to write and add than its products (1,000 x 768 x 768: 21.0 / 18.3 us at 2 / 4
// stages, 16,000 x 128 x 128: 16.9 / 13.9 / 15.0 at 1 / 2 / 4); narrow layers,
// whose partials are small, gain from every split (10,584 x 64 x 64: 7.6 / 9.3
// at 1 / 2).
constexpr int kBlocks = 512;
constexpr int64_t kMaxChain = 2560;
inline int64_t min_stages(bool wide, int64_t tiles) { return !wide ? 1 : tiles < 32 ? 2 : 4; }

// A launch holds fewer than 2^32 threads.
constexpr int64_t kMaxGrid = (int64_t(1) << 32) / kBlock - 8;

struct Plan {
  bool wide;
  int32_t tiles_m, tiles_n, splits;
  int64_t rows_per_split;
};

int make_plan(const char* fn, int64_t n_rows, int32_t n_out, int32_t n_in, Plan* p) {
  if (n_rows < 0 || n_out < 1 || n_in < 1)
    return set_error(NGT_ERR_ARG, "%s: bad sizes n_rows=%lld n_out=%d n_in=%d", fn,
                     static_cast<long long>(n_rows), n_out, n_in);
  p->wide = n_out > 64 && n_in > 64;
  const int t = p->wide ? 128 : 64;
  p->tiles_m = (n_out + t - 1) / t;
  p->tiles_n = (n_in + t - 1) / t;
  const int64_t tiles = int64_t(p->tiles_m) * p->tiles_n;
  const int64_t sums = (int64_t(n_out) * n_in + kRedCols - 1) / kRedCols + n_out / kRedCols + 1;
  if (tiles > (1 << 20) || n_rows > (int64_t(1) << 31) || sums > kMaxGrid)
    return set_error(NGT_ERR_UNSUPPORTED, "%s: %lld rows, %d x %d outputs exceed the grid", fn,
                     static_cast<long long>(n_rows), n_out, n_in);
  const int64_t kb = stage_rows(t);
  const int64_t stages = (n_rows + kb - 1) / kb;
  int64_t splits = kBlocks / tiles;
  if (splits > stages / min_stages(p->wide, tiles)) splits = stages / min_stages(p->wide, tiles);
  if (splits < (n_rows + kMaxChain - 1) / kMaxChain) splits = (n_rows + kMaxChain - 1) / kMaxChain;
  if (splits < 1) splits = 1;
  const int64_t per = (stages + splits - 1) / splits;
  p->rows_per_split = per * kb;
  if (per > 0 && (stages + per - 1) / per * tiles > kMaxGrid)
    return set_error(NGT_ERR_UNSUPPORTED, "%s: %lld rows, %d x %d outputs exceed the grid", fn,
                     static_cast<long long>(n_rows), n_out, n_in);
  p->splits = per > 0 ? static_cast<int32_t>((stages + per - 1) / per) : 0;
  return NGT_OK;
}

inline size_t align16(size_t b) { return (b + 15) & ~size_t(15); }
inline size_t part_bytes(const Plan& p, int32_t n_out, int32_t n_in) {
  return align16(size_t(p.splits) * n_out * n_in * 4);
}
inline size_t part_b_bytes(const Plan& p, int32_t n_out) {
  return align16(size_t(p.splits) * p.tiles_n * n_out * 4);
}

}  // namespace
}  // namespace ngt

using namespace ngt;

extern "C" int ngt_wgrad_workspace_bytes(int64_t n_rows, int32_t n_out, int32_t n_in,
                                         size_t* bytes) {
  Plan p;
  NGT_CHECK_OK(make_plan("ngt_wgrad_workspace_bytes", n_rows, n_out, n_in, &p));
  if (!bytes) return set_error(NGT_ERR_ARG, "ngt_wgrad_workspace_bytes: null bytes");
  *bytes = part_bytes(p, n_out, n_in) + part_b_bytes(p, n_out);
  return NGT_OK;
}

// Where k_wgrad beats the library's GEMMs over row chunks, chunk sum and column
// sum (us with the bias, this / library, rows x n_out x n_in).
// Products: the library's large tiles win once a second round of blocks is under
// way, which the 2,560-row chains ask for: 30,000 x 768 x 768 62 / 87, 32,768 67 / 66,
// 40,000 109 / 85; 896 x 1,024 outputs at 20,000 rows 66 / 92; 65,536 x 512 x 512
// 61 / 68, 100,000 112 / 105.  Between 1 and 2 M outputs its tiles divide the
// chip badly and the line is further out: 2,304 x 768 at 10,007 rows 75 / 93,
// 12,000 111 / 109, 16,000 111 / 125, 20,000 133 / 136, 24,000 165 / 145; 1,536 x
// 768 at 20,000 114 / 119, 32,768 138 / 134; 1,024 x 1,024 at 24,000 106 / 124,
// 32,768 127 / 97.  3,072 x 768 at 7,600 82 / 88, 10,000 119 / 86; above, the
// library's tiles fill it: 3,072 x 1,024 at 5,700 rows 98 / 69, 2,304 x 2,304
// at 3,000 96 / 63.
// Few rows: the partials cost more than the products: 896 x 1,024 at 1,000 rows
// 23 / 21, 1,024 x 1,024 24 / 21 and at 2,000 28 / 29, 768 x 768 at 500 16 / 16.
// Narrow on one side, wide on the other, and many rows: a tile's unused columns
// cost as much as used ones while the rows come from memory: 47 x 768 at 32,768
// rows 44 / 67, 131,072 155 / 138; 48 x 2,048 at 32,768 58 / 36; 48 x 256 at
// 524,288 172 / 222.  Fuller tiles keep longer: 64 x 768 at 131,072 57 / 116, 64 x
// 2,048 152 / 124; 100 x 768 99 / 147, 100 x 1,024 161 / 138.
// Over 166 shapes of 8 to 2,600 columns the choice costs more than 10 % against
// the library in one (2,308 x 191 at 35,131 rows, 260 / 195).
extern "C" int ngt_wgrad_pays(int64_t n_rows, int64_t n_out, int64_t n_in) {
  if (n_rows < 0 || n_out < 1 || n_in < 1 || n_out > 65536 || n_in > 65536 ||
      n_rows > (int64_t(1) << 31))
    return 0;
  const int64_t outputs = n_out * n_in;
  const int64_t narrow = n_out < n_in ? n_out : n_in, wide = n_out < n_in ? n_in : n_out;
  const int64_t most = outputs >= 1000000 && outputs < 2000000 ? 32000000000 : 18000000000;
  if (outputs > 2500000 || n_rows > most / outputs) return 0;
  if (n_rows < 2000 && outputs > 750000) return 0;
  const int64_t span = narrow < 64 ? 60000000 : narrow == 64 ? 150000000 : 120000000;
  if ((narrow <= 64 || (narrow < 256 && narrow % 64)) && wide > 256 && n_rows * wide > span)
    return 0;
  return 1;
}

extern "C" int ngt_wgrad_bf16(const void* x, const void* dy, int64_t n_rows, int32_t n_out,
                              int32_t n_in, float* dw, float* db, void* workspace,
                              size_t workspace_bytes, void* stream) {
  Plan p;
  NGT_CHECK_OK(make_plan("ngt_wgrad_bf16", n_rows, n_out, n_in, &p));
  if (!dw || (n_rows > 0 && (!x || !dy)))
    return set_error(NGT_ERR_ARG, "ngt_wgrad_bf16: null x, dy or dw");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy)) & 1)
    return set_error(NGT_ERR_ARG, "ngt_wgrad_bf16: x and dy must be 2-byte aligned");
  const size_t need = part_bytes(p, n_out, n_in) + part_b_bytes(p, n_out);
  if (need && (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15)))
    return set_error(NGT_ERR_WORKSPACE, "ngt_wgrad_bf16: workspace %zu < %zu or not 16-byte aligned",
                     workspace_bytes, need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(workspace);
  float* part_b = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                           part_bytes(p, n_out, n_in));
  KernelTimer timer_("wgrad", st);
  if (p.splits > 0) {
    WgradArgs a;
    a.x = static_cast<const uint16_t*>(x);
    a.dy = static_cast<const uint16_t*>(dy);
    a.n_rows = n_rows;
    a.n_out = n_out;
    a.n_in = n_in;
    a.tiles_m = p.tiles_m;
    a.tiles_n = p.tiles_n;
    a.splits = p.splits;
    a.rows_per_split = p.rows_per_split;
    a.part = part;
    a.part_b = db ? part_b : nullptr;
    const int total = p.tiles_m * p.tiles_n * p.splits;
    const dim3 grid(static_cast<unsigned>((total + 7) / 8 * 8));
    if (p.wide)
      hipLaunchKernelGGL(k_wgrad<128>, grid, dim3(kBlock), 0, st, a);
    else
      hipLaunchKernelGGL(k_wgrad<64>, grid, dim3(kBlock), 0, st, a);
    NGT_HIP_CHECK(hipGetLastError());
  }
  // no rows: no parts are added and zeros are written
  const int64_t n = int64_t(n_out) * n_in;
  const int64_t blocks_w = (n + kRedCols - 1) / kRedCols;
  const int64_t blocks_b = db ? (n_out + kRedCols - 1) / kRedCols : 0;
  const bool vec = n % 4 == 0 && n_out % 4 == 0;
  const dim3 grid(static_cast<unsigned>(blocks_w + blocks_b));
  if (vec)
    hipLaunchKernelGGL(k_wgrad_sum<true>, grid, dim3(kBlock), 0, st, part, p.splits, n, dw,
                       static_cast<int32_t>(blocks_w), part_b, p.splits * p.tiles_n, n_out, db);
  else
    hipLaunchKernelGGL(k_wgrad_sum<false>, grid, dim3(kBlock), 0, st, part, p.splits, n, dw,
                       static_cast<int32_t>(blocks_w), part_b, p.splits * p.tiles_n, n_out, db);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}
