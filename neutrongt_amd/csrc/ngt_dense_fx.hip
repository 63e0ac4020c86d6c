// Dense full-window attention on the matrix cores with fp32 weights: fp32
// inputs, head_dim d in {8, 16, 24, 32, 64}, and bf16 inputs at d = 64 (P and
// dS keep their 24 bits; the bf16 operands are one piece each).
//
// Products.  An fp32 value is the sum of three bf16 pieces h + m + l (each the
// round-to-nearest of what is left, so the last remainder is zero or below
// 2^-24 of the value).  A product of two such values is hh + (hm + mh) +
// (mm + hl + lh) up to 2^-24.  v_mfma_f32_16x16x32_bf16 multiplies pieces
// exactly, cuts the 8 products of a lane group to 24 bits of the largest, adds
// them and the accumulator with 7 bits to spare and rounds to nearest, lane
// group 0 first and 3 last (probed on gfx950), so a contraction whose largest
// products come last loses less than an fp32 FMA chain.
// At d = 8 a 32 x 32 tile of S takes 128 cycles of bf16 MFMAs where fp32 ones
// take 256, and they leave the vector ALU to the exponentials: the fp32 MFMAs
// do not overlap with vector instructions here (dK/dV at 16,000 nodes, 8
// heads, d = 8: 1,536 MFMA cycles and 800 of vector work per tile ran 2,330
// cycles).  What bounds the kernels is the vector work per score (dK/dV: 320
// vector instructions per tile): the exponential, the split of P (and dS) into
// pieces and, with dropout, the hash.
// Measured (us per launch, forward with node scores / dK/dV / dQ; the earlier
// one-row-per-lane vector kernels -> these): 16,000 nodes, 8 heads, d = 8
// 1,720 / 2,490 / 1,680 -> 1,080 / 1,545 / 970, with dropout 0.5 2,150 /
// 2,810 / 1,980 -> 1,420 / 2,100 / 1,370; all-fp32 MFMAs 1,390 / 1,900 /
// 1,300.  5,000 nodes, 8 heads, d = 64: 8,400 in all -> 650 / 1,210 / 555; the
// same in bf16 (one piece per operand) 1,570 / 5,870 / 2,970 -> 275 / 630 / 290.
//
// A preparation kernel (k_fx_prep) writes the pieces of q * scale, k, v and dO
// once per call, each matrix in the images that the pass reads:
//   row image: per row 3 pieces x d / 8 blocks of 8 columns (16 bytes each),
//     read as A and B operands of S and dP;
//   transposed image: per 32 rows, one line per (piece, column) with the 32
//     rows in the order a lane needs them, read as A operands of the products
//     over rows.
// Lane layouts (g = lane / 16, l = lane % 16; checked on gfx950):
//   A (16 x 32): lane holds A[l][8 g + j], B (32 x 16): B[8 g + j][l], j < 8;
//   D (16 x 16): lane holds D[4 g + i][l], i < 4.
// A contraction's index order is free as long as A and B share it: two score
// tiles (32 streamed rows) give lane (l, g) the rows 4 g + i of both, and those
// 8 values, split, are the B operand of the next product as they stand.
//
// The lanes' side (queries in the forward and dQ pass, keys in the dK/dV
// pass) is the tiles' column, so per-row state (running maximum, sum, lse, D)
// sits in one register per lane; the other side is staged in LDS with line
// lengths that are odd multiples of 16 bytes (16 lanes on 16 bank groups).
// Outputs come out transposed, 4 consecutive columns of a lane's row.
//
// Pieces of an infinity or a NaN would turn products with zero pieces into
// NaN, and below 2^-110 the third piece of an fp32 value is a bf16 subnormal
// that no longer holds all its bits (below 2^-126 the second).  So a head whose
// inputs hold such a value or one past 2^125, and a backward pass whose dO or v
// is so small that dS would be there, runs the same kernels' other body, with
// v_mfma_f32_16x16x4_f32: plain fp32 FMA chains.
#include "ngt_common.h"

#include <math.h>
#include <stdlib.h>

#include <algorithm>

namespace ngt {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Ids as register reads: this file is built with the IEEE mode bit off, and
// the device library's functions behind threadIdx / blockIdx are not inlined
// across that difference (each use would be a call).
__device__ __forceinline__ int tid_x() { return static_cast<int>(__builtin_amdgcn_workitem_id_x()); }
__device__ __forceinline__ int wg_x() { return static_cast<int>(__builtin_amdgcn_workgroup_id_x()); }
__device__ __forceinline__ int wg_y() { return static_cast<int>(__builtin_amdgcn_workgroup_id_y()); }
__device__ __forceinline__ int wg_z() { return static_cast<int>(__builtin_amdgcn_workgroup_id_z()); }

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kT = 16;     // MFMA tile edge
constexpr int kStep = 32;  // streamed rows per step of a wave (two tiles)
constexpr int kPadRows = 64;  // the images' rows come in multiples of this
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kRun = 16;  // stages whose sums meet before they join a total
constexpr float kRebase = 5.5f;  // forward: P entries stay below e^5.5 (fp32 sums)
constexpr float kHuge = 4.2535296e37f;   // 2^125: values past it take the fp32 MFMAs,
constexpr float kTiny = 7.7037198e-34f;  // 2^-110: and values below it (but zero)
constexpr float kFaint = 9.0949470e-13f; // 2^-40: see backward_plain

// Rows (queries or keys) a block owns with G tiles per wave.
constexpr int block_rows(int G) { return kWaves * kT * G; }
constexpr int out_tiles(int dh) { return (dh + 15) / 16; }
// np: pieces per operand, 3 for fp32 inputs and 1 for bf16 ones.
// Row image: bytes per row (np pieces x blocks of 8 columns, d = 24 padded to
// 4 blocks, the line length an odd multiple of 16).
constexpr int col_blocks(int dh) { return dh == 24 ? 4 : dh / 8; }
constexpr int row_bytes(int dh, int np) {
  const int units = np * col_blocks(dh);
  return 16 * (units % 2 ? units : units + 1);
}
// Transposed image: lines per 32 rows, one per (piece, column) in whole
// 16-line tiles; at d = 8 the first tile holds pieces h and m, the second l.
constexpr int t_lines(int dh, int np) { return dh == 8 ? 32 : np * 16 * out_tiles(dh); }
constexpr int kTLine = 80;  // 32 bf16 and 16 bytes of padding
constexpr int t_bytes(int dh, int np) { return t_lines(dh, np) * kTLine; }
template <typename T>
constexpr int pieces() {
  return sizeof(T) == 4 ? 3 : 1;
}
__host__ __device__ inline int padded(int n) { return (n + kPadRows - 1) / kPadRows * kPadRows; }

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ float exp_nat(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

// x combined over the four 16-lane rows of the wave (the lanes of one column).
__device__ __forceinline__ float sum_halves(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float sum_rows(float x) {
  x = sum_halves(x);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float max_rows(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// The dropout word of lane ^ 1 (DPP quad_perm 1,0,3,2).
__device__ __forceinline__ uint32_t swap_pair(uint32_t x) {
  return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0xB1, 0xF, 0xF, true));
}

// Two floats' next pieces, packed; x0, x1 become the remainders (exact).
// NEAREST: pieces rounded to nearest (the operands, once per call), so that
// the products left out are signed and below 2^-24.  Else the leading 16 bits
// (P and dS, per score): a mask and a subtraction at the vector ALU's double
// rate (2.5 cycles each; conversions and shifts take 4.4).  Either way three
// pieces hold all 24 bits.
template <bool NEAREST>
__device__ __forceinline__ uint32_t peel2(float& x0, float& x1) {
  if constexpr (NEAREST) {
    const uint32_t w = pack2_bf16(x0, x1);
    x0 -= __uint_as_float(w << 16);
    x1 -= __uint_as_float(w & 0xffff0000u);
    return w;
  } else {
    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    x0 -= __uint_as_float(u0 & 0xffff0000u);
    x1 -= __uint_as_float(u1 & 0xffff0000u);
    return __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // the two upper halves
  }
}
struct Split {
  bf16x8 h, m, l;
};
template <bool NEAREST>
__device__ __forceinline__ Split split8(float (&x)[8]) {
  uint32_t w[3][4];
#pragma unroll
  for (int n = 0; n < 3; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) w[n][j] = peel2<NEAREST>(x[2 * j], x[2 * j + 1]);
  return {__builtin_bit_cast(bf16x8, make_uint4(w[0][0], w[0][1], w[0][2], w[0][3])),
          __builtin_bit_cast(bf16x8, make_uint4(w[1][0], w[1][1], w[1][2], w[1][3])),
          __builtin_bit_cast(bf16x8, make_uint4(w[2][0], w[2][1], w[2][2], w[2][3]))};
}

// Dropout: 1 / (1 - p) rides in the staged V (forward) and dO (backward), so a
// score only keeps or clears its value.  bits: the 16-bit draw in the upper
// half (the lower half is the other key's and cannot change the comparison
// with thr << 16).
__device__ __forceinline__ bool kept(uint32_t bits, uint32_t thr16) { return bits >= thr16; }

// One operand matrix [n, H, d]: its fp32 rows and, per head, the images.
struct Mat {
  const void* x;        // [n, H, d] of the element type
  const char* row_img;  // [H][padded(n)][row_bytes]
  const char* t_img;    // [H][padded(n) / 32][t_bytes]
  const uint32_t* flag; // [H][padded(n) / 32]: what the step's values are (k...Value)
  int32_t n;
  float scale;          // of x (in the images of fp32 inputs already)
};

// The low N bits of x, each set where some thread of the block has it; a barrier.
template <int N>
__device__ __forceinline__ uint32_t or_over_block(uint32_t x, uint32_t (&waves)[kWaves]) {
  uint32_t w = 0u;
#pragma unroll
  for (int i = 0; i < N; ++i) w |= __ballot(x >> i & 1u) ? 1u << i : 0u;
  waves[tid_x() >> 6] = w;  // one value, whichever lane writes last
  __syncthreads();
  w = waves[0];
#pragma unroll
  for (int i = 1; i < kWaves; ++i) w |= waves[i];
  return w;
}

// -------------------------------------------------------------- preparation
constexpr uint32_t kSpecialValue = 1u;  // some value has no three pieces
constexpr uint32_t kNonzeroValue = 2u, kPlainValue = 4u;  // some value is not 0, not below 2^-40
struct PrepJob {
  const void* x;
  char *row_img, *t_img;  // null: not wanted
  uint32_t* flag;
  int32_t n;
  float scale;
};
struct PrepJobs {
  PrepJob j[4];
};

// Block (step of 32 rows, head, matrix): both images of the step's rows and
// the flag word.  Rows past n are zero.  bf16 inputs are their own single
// piece and stay unscaled.
template <typename T, int DH>
__global__ __launch_bounds__(kBlock) void k_fx_prep(const PrepJobs jobs, int32_t H) {
  const PrepJob job = jobs.j[wg_z()];
  const int step = wg_x(), h = wg_y();
  const int n_pad = padded(job.n);
  if (step * kStep >= n_pad) return;
  __shared__ float xs[kStep][DH + 1];
  constexpr int NP = pieces<T>();
  uint32_t mark = 0u;
  for (int e = tid_x(); e < kStep * DH; e += kBlock) {
    const int r = e / DH, c = e - r * DH;
    const int64_t row = int64_t(step) * kStep + r;
    float v = 0.f;
    if (row < job.n) v = elem<T>::load(static_cast<const T*>(job.x) + (row * H + h) * DH + c);
    if constexpr (NP == 3) v *= job.scale;
    xs[r][c] = v;
    // (compares on the bits: this file does not honour NaNs)
    const uint32_t u = __float_as_uint(v) & 0x7fffffffu;
    if (u > __float_as_uint(kHuge) || (NP == 3 && u != 0u && u < __float_as_uint(kTiny)))
      mark |= kSpecialValue;
    if (u != 0u) mark |= kNonzeroValue;
    if (u >= __float_as_uint(kFaint)) mark |= kPlainValue;
  }
  __shared__ uint32_t waves[kWaves];
  const uint32_t word = or_over_block<3>(mark, waves);
  if (tid_x() == 0) job.flag[int64_t(h) * (n_pad / kStep) + step] = word;
  constexpr int NB = col_blocks(DH);
  for (int e = tid_x(); job.row_img && e < kStep * NB; e += kBlock) {
    const int r = e / NB, cb = e - r * NB;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = 8 * cb + j < DH ? xs[r][(8 * cb + j) % DH] : 0.f;
    const Split sp = split8<true>(x);
    char* p = job.row_img + (int64_t(h) * n_pad + step * kStep + r) * row_bytes(DH, NP) + 16 * cb;
    *reinterpret_cast<bf16x8*>(p) = sp.h;
    if constexpr (NP == 3) {
      *reinterpret_cast<bf16x8*>(p + 16 * NB) = sp.m;
      *reinterpret_cast<bf16x8*>(p + 32 * NB) = sp.l;
    }
  }
  if (!job.t_img) return;
  constexpr int PL = DH == 8 ? 8 : 16 * out_tiles(DH);  // lines per piece
  char* t = job.t_img + (int64_t(h) * (n_pad / kStep) + step) * t_bytes(DH, NP);
  for (int e = tid_x(); e < 4 * PL; e += kBlock) {
    const int c = e / 4, gg = e - 4 * c;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      x[j] = c < DH ? xs[kT * (j / 4) + 4 * gg + j % 4][c < DH ? c : 0] : 0.f;
    const Split sp = split8<true>(x);
    char* p = t + c * kTLine + 16 * gg;
    *reinterpret_cast<bf16x8*>(p) = sp.h;
    if constexpr (NP == 3) {
      *reinterpret_cast<bf16x8*>(p + PL * kTLine) = sp.m;
      *reinterpret_cast<bf16x8*>(p + 2 * PL * kTLine) = sp.l;
    }
    if constexpr (DH == 8)  // the last 8 lines of the second tile
      *reinterpret_cast<uint4*>(p + 3 * PL * kTLine) = make_uint4(0u, 0u, 0u, 0u);
  }
}

// This thread's share of the marks of head h of a matrix.
__device__ __forceinline__ uint32_t marks(const Mat& m, int h) {
  const int steps = padded(m.n) / kStep;
  uint32_t w = 0u;
  for (int t = tid_x(); t < steps; t += kBlock) w |= m.flag[int64_t(h) * steps + t];
  return w;
}
// Whether head h of these matrices takes the fp32 body (the same answer in every
// thread of the block).  Without images (few_scores) all do.
__device__ __forceinline__ bool forward_plain(const Mat& q, const Mat& k, const Mat& v, int h,
                                              uint32_t (&waves)[kWaves]) {
  if (!q.flag) return true;
  return or_over_block<1>(marks(q, h) | marks(k, h) | marks(v, h), waves) != 0u;
}
// The same for the backward, whose dS = p (dO . v - D) is split into pieces too:
// with dO or v below 2^-40 everywhere (zeros alone do no harm) it could lie below
// 2^-110 where it counts.  With one value of each past that, the largest dS lies
// past 2^-80 p and what the pieces drop is below 2^-133.
__device__ __forceinline__ bool backward_plain(const Mat& q, const Mat& k, const Mat& v,
                                               const Mat& g, int h, uint32_t (&waves)[kWaves]) {
  if (!q.flag) return true;
  const uint32_t mg = marks(g, h), mv = marks(v, h);
  const uint32_t special = (marks(q, h) | marks(k, h) | mg | mv) & kSpecialValue;
  const uint32_t w = or_over_block<5>(special | (mg & 6u) | (mv & 6u) << 2, waves);
  const bool faint_g = (w & kNonzeroValue) && !(w & kPlainValue);
  const bool faint_v = (w & kNonzeroValue << 2) && !(w & kPlainValue << 2);
  return (w & kSpecialValue) || faint_g || faint_v;
}

// ------------------------------------------------------- fp32 MFMA products
// A lane's d / 4 elements of row p, columns (d / 4) g ..
template <int DH, typename T>
__device__ __forceinline__ void load_quarter(const T* p, float (&x)[DH / 4]) {
  constexpr int KC = DH / 4;
  if constexpr (sizeof(T) == 2) {
    load_row<T, KC>(p, x);
  } else if constexpr (KC % 4 == 0) {
#pragma unroll
    for (int j = 0; j < KC; j += 4) {
      const float4 w = *reinterpret_cast<const float4*>(p + j);
      x[j] = w.x, x[j + 1] = w.y, x[j + 2] = w.z, x[j + 3] = w.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < KC; j += 2) {
      const float2 w = *reinterpret_cast<const float2*>(p + j);
      x[j] = w.x, x[j + 1] = w.y;
    }
  }
}

// Rows are staged as they are, LD floats apart, and serve both kinds of
// product (an A operand of the products over rows is a column of 4 rows).  At
// d = 8 and 24 the last tile's columns past d read the floats that follow and
// end in registers that nothing stores.
template <typename T, int DH, int G>
struct Fp32Ops {
  static constexpr bool SCALED = true;  // operands carry their Mat's scale
  static constexpr int SB = DH > 32 ? 32 : 64;
  static constexpr int LD = DH + 4;
  static constexpr int MT = out_tiles(DH);
  struct Rows {
    float x[G][DH / 4];
  };
  static __device__ __forceinline__ void load_rows(Rows& r, int u, const Mat& m, int64_t row, int h,
                                                   int H, int g) {
#pragma unroll
    for (int j = 0; j < DH / 4; ++j) r.x[u][j] = 0.f;
    if (row < m.n)
      load_quarter<DH>(static_cast<const T*>(m.x) + (row * H + h) * DH + (DH / 4) * g, r.x[u]);
#pragma unroll
    for (int j = 0; j < DH / 4; ++j) r.x[u][j] *= m.scale;
  }
  template <bool ROW, bool COL>
  struct Staged {
    static constexpr int BYTES = (SB * LD + 16) * 4;
    static constexpr int VPR = DH / 4;
    static constexpr int NV = (SB * VPR + kBlock - 1) / kBlock;
    float* lds;
    float4 w[NV];
    __device__ __forceinline__ void load(const Mat& m, int row0, int h, int H) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = tid_x() + i * kBlock;
        const int r = e / VPR, c = e - r * VPR;
        const bool ok = e < SB * VPR && row0 + r < m.n;  // else read the first piece, use zeros
        const T* p = static_cast<const T*>(m.x) + (int64_t(row0 + (ok ? r : 0)) * H + h) * DH +
                     4 * (ok ? c : 0);
        float4 x;
        if constexpr (sizeof(T) == 4) {
          x = *reinterpret_cast<const float4*>(p);
        } else {
          const uint2 b = *reinterpret_cast<const uint2*>(p);
          x = make_float4(__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xffff0000u),
                          __uint_as_float(b.y << 16), __uint_as_float(b.y & 0xffff0000u));
        }
        w[i] = ok ? x : make_float4(0.f, 0.f, 0.f, 0.f);
        w[i] = make_float4(w[i].x * m.scale, w[i].y * m.scale, w[i].z * m.scale, w[i].w * m.scale);
      }
    }
    __device__ __forceinline__ void store() const {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = tid_x() + i * kBlock;
        const int r = e / VPR, c = e - r * VPR;
        if (e < SB * VPR) *reinterpret_cast<float4*>(lds + r * LD + 4 * c) = w[i];
      }
    }
    // X[t][u] = M R[u]^T for the 16-row tiles t at LDS row r0; chains of two
    // MFMAs meet in a tree
    __device__ __forceinline__ void products(int r0, int g, int l16, const Rows& rows,
                                             f32x4 (&x)[2][G]) const {
      constexpr int NCH = DH / 8;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float a[DH / 4];
        load_quarter<DH>(lds + (r0 + kT * t + l16) * LD + (DH / 4) * g, a);
#pragma unroll
        for (int u = 0; u < G; ++u) {
          f32x4 c[NCH];
#pragma unroll
          for (int n = 0; n < NCH; ++n)
            c[n] = mfma4(a[2 * n + 1], rows.x[u][2 * n + 1],
                         mfma4(a[2 * n], rows.x[u][2 * n], zero4()));
#pragma unroll
          for (int v = 1; v < NCH; v *= 2)
#pragma unroll
            for (int n = 0; n + v < NCH; n += 2 * v) c[n] += c[n + v];
          x[t][u] = c[0];
        }
      }
    }
    // acc[u] (columns x lanes, transposed) += M^T X[u] over 32 rows
    __device__ __forceinline__ void accumulate(int r0, int g, int l16, const f32x4 (&x)[2][G],
                                               f32x4 (&acc)[G][MT]) const {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const float a = lds[(r0 + kT * t + 4 * g + i) * LD + kT * m + l16];
#pragma unroll
            for (int u = 0; u < G; ++u) acc[u][m] = mfma4(a, x[t][u][i], acc[u][m]);
          }
    }
  };
  static __device__ __forceinline__ void finish(f32x4 (&)[G][MT]) {}
};

// ------------------------------------------------------ bf16-piece products
// S and dP contract the columns of two rows' pieces.  A lane's operand is 16
// bytes of a row image, its 16-byte unit chosen by (operand number, g): the
// MFMAs of a tile pair A and B operands so that, over the four g, every piece
// product down to 2^-16 is there once; the smallest come first, and the leading
// products h h in the last lane groups of the last MFMA: all others meet in sums
// 2^-8 of theirs, and S is rounded once at its own size (d = 8; with the h h in
// the first group three more times: S off by up to 1.9 against 1.1 times 2^-24
// sum |q k|, and at d = 16 2.2 against 1.2).
// The dK/dV pass has the two matrices the other way round, and its S has to
// round as the forward's did: exp(S - lse) with another last bit of S is off by
// as much as S is large (at d = 16, 8 heads, 406 nodes dV's error was 3.2e-6,
// with the forward's S 1.2e-6).  The last group is the same from both sides.
// With one piece per operand (d = 64) they are the row's two halves.
template <int DH, int NP>
struct Pairs {
  static_assert(DH == 64, "one piece per operand: d = 64 only");
  static constexpr int NA = 2, NB = 2, N = 2;
  static constexpr __host__ __device__ int a_of(int n) { return n; }
  static constexpr __host__ __device__ int b_of(int n) { return n; }
  static __device__ __forceinline__ int unit(bool, int k, int g) { return 16 * (4 * k + g); }
};
template <int DH>
struct Pairs<DH, 3> {
  static constexpr int NA = DH <= 16 ? 2 : DH == 64 ? 6 : 3;  // A operands
  static constexpr int NB = DH == 8 ? 2 : DH == 64 ? 6 : 3;   // B operands
  static constexpr int N = DH == 8 ? 2 : DH == 16 ? 3 : DH == 64 ? 12 : 6;
  // the N MFMAs, smallest products first
  static constexpr __host__ __device__ int a_of(int n) {
    if constexpr (DH == 8) return 1 - n;
    else if constexpr (DH == 16) return n == 0;  // [h l] x [l h], [m h] x [h m], [m h] x [m h]
    else {
      constexpr int a[6] = {2, 0, 1, 1, 0, 0};
      return DH == 64 ? 2 * a[n / 2] + n % 2 : a[n];
    }
  }
  static constexpr __host__ __device__ int b_of(int n) {
    if constexpr (DH == 8) return 1 - n;
    else if constexpr (DH == 16) return n == 0 ? 1 : n == 1 ? 2 : 0;
    else {
      constexpr int b[6] = {0, 2, 1, 0, 1, 0};
      return DH == 64 ? 2 * b[n / 2] + n % 2 : b[n];
    }
  }
  // byte offset of operand k of a lane's row
  static __device__ __forceinline__ int unit(bool b, int k, int g) {
    constexpr int CB = col_blocks(DH);
    if constexpr (DH == 8) {
      // [h l h m] x [l h m h] first, [l m m h] x [m l m h] last
      const uint32_t units = k == 0 ? (b ? 0x0121u : 0x0112u) : (b ? 0x0102u : 0x1020u);
      return 16 * int(units >> (4 * g) & 15u);
    } else if constexpr (DH == 16) {
      const int hi = g >> 1;  // the second two lane groups
      const int piece = b ? (k == 0 ? !hi : k == 1 ? 2 * !hi : hi)  // mh / lh / hm
                          : (k == 0 ? !hi : 2 * hi);                // mh / hl
      return 16 * (piece * CB + (g & 1));
    } else if constexpr (DH == 64) {
      return 16 * ((k / 2) * CB + 4 * (k % 2) + g);
    } else {
      return 16 * (k * CB + g);
    }
  }
};

template <typename T, int DH, int G>
struct PieceOps {
  static constexpr int NP = pieces<T>();
  static constexpr bool SCALED = NP == 3;
  static constexpr int SB = DH <= 16 || NP == 1 ? 64 : 32;
  static constexpr int MT = out_tiles(DH);
  using P = Pairs<DH, NP>;
  struct Rows {
    bf16x8 x[G][P::NB];
  };
  static __device__ __forceinline__ void load_rows(Rows& r, int u, const Mat& m, int64_t row, int h,
                                                   int H, int g) {
    const int n_pad = padded(m.n);
    const char* p = m.row_img + (int64_t(h) * n_pad + row) * row_bytes(DH, NP);
#pragma unroll
    for (int k = 0; k < P::NB; ++k) {
      uint4 w = make_uint4(0u, 0u, 0u, 0u);
      if (row < n_pad) w = *reinterpret_cast<const uint4*>(p + P::unit(true, k, g));
      r.x[u][k] = __builtin_bit_cast(bf16x8, w);
    }
  }
  template <bool ROW, bool COL>
  struct Staged {
    static constexpr int RB = ROW ? SB * row_bytes(DH, NP) : 0;
    static constexpr int TB = COL ? SB / kStep * t_bytes(DH, NP) : 0;
    static constexpr int BYTES = RB + TB;
    static constexpr int NR = (RB / 16 + kBlock - 1) / kBlock, NT = (TB / 16 + kBlock - 1) / kBlock;
    static constexpr int NV = NR + NT;
    char* lds;
    uint4 w[NV];
    __device__ __forceinline__ void load(const Mat& m, int row0, int h, int H) {
      const int n_pad = padded(m.n);
      const char* r = m.row_img + (int64_t(h) * n_pad + row0) * row_bytes(DH, NP);
      const char* t = m.t_img + (int64_t(h) * (n_pad / kStep) + row0 / kStep) * t_bytes(DH, NP);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int e = 16 * (tid_x() + i * kBlock);
        w[i] = *reinterpret_cast<const uint4*>(r + min(e, RB - 16));
      }
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int e = 16 * (tid_x() + i * kBlock);
        w[NR + i] = *reinterpret_cast<const uint4*>(t + min(e, TB - 16));
      }
    }
    __device__ __forceinline__ void store() const {
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int e = 16 * (tid_x() + i * kBlock);
        if (e < RB) *reinterpret_cast<uint4*>(lds + e) = w[i];
      }
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int e = 16 * (tid_x() + i * kBlock);
        if (e < TB) *reinterpret_cast<uint4*>(lds + RB + e) = w[NR + i];
      }
    }
    __device__ __forceinline__ void products(int r0, int g, int l16, const Rows& rows,
                                             f32x4 (&x)[2][G]) const {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const char* p = lds + (r0 + kT * t + l16) * row_bytes(DH, NP);
        bf16x8 a[P::NA];
#pragma unroll
        for (int k = 0; k < P::NA; ++k)
          a[k] = *reinterpret_cast<const bf16x8*>(p + P::unit(false, k, g));
#pragma unroll
        for (int u = 0; u < G; ++u) {
          x[t][u] = zero4();
#pragma unroll
          for (int n = 0; n < P::N; ++n)
            x[t][u] = mfma32(a[P::a_of(n)], rows.x[u][P::b_of(n)], x[t][u]);
        }
      }
    }
    __device__ __forceinline__ void accumulate(int r0, int g, int l16, const f32x4 (&x)[2][G],
                                               f32x4 (&acc)[G][MT]) const {
      const char* p = lds + RB + (r0 / kStep) * t_bytes(DH, NP) + l16 * kTLine + 16 * g;
      auto line = [&](int tile) {
        return *reinterpret_cast<const bf16x8*>(p + tile * kT * kTLine);
      };
      Split sp[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[j / 4][u][j % 4];
        sp[u] = split8<false>(v);
      }
      if constexpr (DH == 8) {  // rows 0-7: h (then l), rows 8-15: m of M
        const bf16x8 hm = line(0), l = line(1);
#pragma unroll
        for (int u = 0; u < G; ++u) {
          acc[u][0] = mfma32(l, sp[u].h, acc[u][0]);
          acc[u][0] = mfma32(hm, sp[u].l, acc[u][0]);
          acc[u][0] = mfma32(hm, sp[u].m, acc[u][0]);
          acc[u][0] = mfma32(hm, sp[u].h, acc[u][0]);
        }
      } else if constexpr (NP == 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const bf16x8 ah = line(m);
#pragma unroll
          for (int u = 0; u < G; ++u) {
            acc[u][m] = mfma32(ah, sp[u].l, acc[u][m]);
            acc[u][m] = mfma32(ah, sp[u].m, acc[u][m]);
            acc[u][m] = mfma32(ah, sp[u].h, acc[u][m]);
          }
        }
      } else {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const bf16x8 ah = line(m), am = line(MT + m), al = line(2 * MT + m);
#pragma unroll
          for (int u = 0; u < G; ++u) {
            acc[u][m] = mfma32(al, sp[u].h, acc[u][m]);
            acc[u][m] = mfma32(ah, sp[u].l, acc[u][m]);
            acc[u][m] = mfma32(am, sp[u].m, acc[u][m]);
            acc[u][m] = mfma32(am, sp[u].h, acc[u][m]);
            acc[u][m] = mfma32(ah, sp[u].m, acc[u][m]);
            acc[u][m] = mfma32(ah, sp[u].h, acc[u][m]);
          }
        }
      }
    }
  };
  // d = 8: a column's two piece rows meet (lanes g and g + 2)
  static __device__ __forceinline__ void finish(f32x4 (&acc)[G][MT]) {
    if constexpr (DH == 8) {
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][0][i] = sum_halves(acc[u][0][i]);
    }
  }
};

// A stage's sums (at most 64 rows) start from zero and are added to the total
// at its end: one accumulator over 16,000 rows had moved the outputs by 6e-6,
// three times the error of the two levels' sum.
template <int G, int MT>
__device__ __forceinline__ void zero_acc(f32x4 (&x)[G][MT]) {
#pragma unroll
  for (int u = 0; u < G; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t) x[u][t] = zero4();
}
template <int G, int MT>
__device__ __forceinline__ void add_acc(const f32x4 (&x)[G][MT], f32x4 (&acc)[G][MT]) {
#pragma unroll
  for (int u = 0; u < G; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[u][t] += x[u][t];
}
// Multiplies both tiles of a step by f (the scale that unscaled operands leave out).
template <int G>
__device__ __forceinline__ void times(f32x4 (&x)[2][G], float f) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < G; ++u) x[t][u] *= f;
}
template <int DH, int G, typename T>
__device__ __forceinline__ void store_acc(T* __restrict__ row, int u, int g, float f,
                                          const f32x4 (&acc)[G][out_tiles(DH)]) {
#pragma unroll
  for (int m = 0; m < out_tiles(DH); ++m)
    if (kT * m + 4 * g < DH) {
      const float4 w = make_float4(acc[u][m][0] * f, acc[u][m][1] * f, acc[u][m][2] * f,
                                   acc[u][m][3] * f);
      if constexpr (sizeof(T) == 4)
        *reinterpret_cast<float4*>(row + kT * m + 4 * g) = w;
      else
        *reinterpret_cast<uint2*>(row + kT * m + 4 * g) =
            make_uint2(pack2_bf16(w.x, w.y), pack2_bf16(w.z, w.w));
    }
}

// LDS of a kernel whose two bodies share one buffer.
constexpr int max_of(int a, int b) { return a > b ? a : b; }

// ------------------------------------------------------------------ forward
struct FwdArgs {
  Mat q, k, v;
  int32_t H;
  DropoutMask dm;
  uint32_t thr16;
  float drop_scale;
  void* out;
  float *out32, *lse;
  int32_t split_keys;
  float *part_ml, *part_acc;
  int32_t n_split, fwd_bx, score_bx, score_splits;
  int32_t grid_x;      // blocks are numbered y * grid_x + x
  int32_t score_rows;  // queries per split of the column scores
  float* part;         // [split][H][n_k]
};

// One block: block_rows(G) queries of head h, keys of split z.  S^T = K Q^T
// (rows = keys), online softmax per lane's query, O^T += V^T P^T.  The base m
// moves only when some score exceeds it by more than kRebase, so after the
// first step a wave rarely rescales; the column maximum over the lanes that
// share a query is taken only then.
//
// At d = 8, where S is exact enough for the sums to show, a third level: the
// stages of a run (1,024 keys) are added to each other and then to totals in
// LDS, each lane's own, which cost no registers.  250 stages added one by one at
// 16,000 keys had moved out, and through D = dO . out dQ: 8 heads, x 5.9e-7 ->
// 3.9e-7 and dQ 2.2e-6 -> 1.3e-6 against float64 (vector kernels 7.5e-7 and
// 2.0e-6); the forward with dropout 1,408 -> 1,449 us.  With the totals in
// registers it took 134 of them for 111 and the whole pass 50 us more; as a
// struct's members passed by reference 1,480 us.
constexpr bool run_totals(int dh) { return dh == 8; }
template <int DH, int G>
constexpr int totals_bytes() {
  return run_totals(DH) ? G * kBlock * 20 : 0;
}
template <class Ops, typename T, int DH, int G, bool DROP>
__device__ __forceinline__ void fwd_body(const FwdArgs& a, int bx, int h, int z, char* lds) {
  constexpr int SB = Ops::SB, MT = out_tiles(DH);
  const int lane = tid_x() & (kWave - 1);
  const int wave = tid_x() >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int n_q = a.q.n, H = a.H;
  DropoutMask dm = a.dm;
  if constexpr (DROP) dm = drop_for_head(dm, h);
  int qi[G];
  typename Ops::Rows qf;
  float m[G], l[G], thr[G];
  f32x4 acc[G][MT];
  zero_acc(acc);
#pragma unroll
  for (int u = 0; u < G; ++u) {
    qi[u] = bx * block_rows(G) + (wave * G + u) * kT + l16;
    Ops::load_rows(qf, u, a.q, qi[u], h, H, g);
    m[u] = thr[u] = -INFINITY;
    l[u] = 0.f;
  }
  const int k_begin = z * a.split_keys;
  const int k_end = min(a.k.n, k_begin + a.split_keys);
  typename Ops::template Staged<true, false> sk;
  typename Ops::template Staged<false, true> sv;
  sk.lds = reinterpret_cast<decltype(sk.lds)>(lds);
  sv.lds = reinterpret_cast<decltype(sv.lds)>(lds + sk.BYTES);
  if (k_begin < k_end) {
    sk.load(a.k, k_begin, h, H);
    sv.load(a.v, k_begin, h, H);
  }
  // this lane's slots of the totals, kBlock apart, and their base
  f32x4* const tot = reinterpret_cast<f32x4*>(lds + sk.BYTES + sv.BYTES) + tid_x();
  float* const tot_l =
      reinterpret_cast<float*>(lds + sk.BYTES + sv.BYTES + G * kBlock * 16) + tid_x();
  float m_tot[G];
  auto add_totals = [&](bool any) {  // acc, l += the totals
#pragma unroll
    for (int u = 0; u < G; ++u)
      if (any) {
        const float f = m_tot[u] == -INFINITY ? 0.f : exp_nat(m_tot[u] - m[u]);
        acc[u][0] += tot[u * kBlock] * f;
        l[u] += tot_l[u * kBlock] * f;
      }
  };
  int run = 0;  // stages since the totals were last written
  bool any = false;
  for (int kb = k_begin; kb < k_end; kb += SB) {
    __syncthreads();
    sk.store();
    sv.store();
    __syncthreads();
    if (kb + SB < k_end) {
      sk.load(a.k, kb + SB, h, H);
      sv.load(a.v, kb + SB, h, H);
    }
    f32x4 stage[G][MT];  // this stage's share of acc and l
    float lst[G];
    zero_acc(stage);
#pragma unroll
    for (int u = 0; u < G; ++u) lst[u] = 0.f;
    for (int r0 = 0; r0 < SB && kb + r0 < k_end; r0 += kStep) {
      f32x4 s[2][G];  // S^T tiles: rows = keys kb + r0 + 16 t + 4 g + i
      sk.products(r0, g, l16, qf, s);
      if constexpr (!Ops::SCALED) times(s, a.q.scale);
      if (kb + r0 + kStep > k_end) {  // keys past the end drop out
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb + r0 + kT * t + 4 * g + i >= k_end)
#pragma unroll
              for (int u = 0; u < G; ++u) s[t][u][i] = -INFINITY;
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[t][u][i]);
        if (__any(mx > thr[u])) {
          const float m_new = fmaxf(m[u], max_rows(mx));
          const float alpha = m[u] == -INFINITY ? 0.f : exp_nat(m[u] - m_new);
          l[u] *= alpha;
          lst[u] *= alpha;
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            acc[u][t] *= alpha;
            stage[u][t] *= alpha;
          }
          m[u] = m_new;
          thr[u] = m_new + kRebase;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const uint32_t key = uint32_t(kb + r0 + kT * t + 4 * g);
          uint32_t w[2] = {0u, 0u};  // keys +0, +1 and +2, +3
          if constexpr (DROP) {
            w[0] = drop_word(dm, uint32_t(qi[u]), key);
            w[1] = drop_word(dm, uint32_t(qi[u]), key + 2);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = exp_nat(s[t][u][i] - m[u]);
            lst[u] += p;  // the softmax normaliser uses every key
            if constexpr (DROP) {
              const uint32_t bits = i & 1 ? w[i / 2] : w[i / 2] << 16;
              s[t][u][i] = kept(bits, a.thr16) ? p : 0.f;
            } else {
              s[t][u][i] = p;
            }
          }
        }
      }
      sv.accumulate(r0, g, l16, s, stage);
    }
    add_acc(stage, acc);
#pragma unroll
    for (int u = 0; u < G; ++u) l[u] += lst[u];
    if (run_totals(DH) && ++run == kRun && kb + SB < k_end) {
      add_totals(any);
#pragma unroll
      for (int u = 0; u < G; ++u) {
        tot[u * kBlock] = acc[u][0];
        tot_l[u * kBlock] = l[u];
        m_tot[u] = m[u];
        l[u] = 0.f;
      }
      zero_acc(acc);
      run = 0;
      any = true;
    }
  }
  if constexpr (run_totals(DH)) add_totals(any);
  Ops::finish(acc);
  const float ds = DROP && !Ops::SCALED ? a.drop_scale : 1.f;
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const float lsum = sum_rows(l[u]);
    if (qi[u] >= n_q) continue;
    const int64_t row = int64_t(qi[u]) * H + h;
    if (a.part_ml) {  // this split's softmax state, merged in split order later
      store_acc<DH, G>(a.part_acc + (int64_t(z) * n_q * H + row) * DH, u, g, ds, acc);
      if (g == 0) {
        const int64_t r = (int64_t(z) * H + h) * n_q + qi[u];
        a.part_ml[2 * r] = m[u];
        a.part_ml[2 * r + 1] = lsum;
      }
      continue;
    }
    const float inv = a.k.n > 0 ? ds / lsum : 0.f;
    store_acc<DH, G>(static_cast<T*>(a.out) + row * DH, u, g, inv, acc);
    if (a.out32) store_acc<DH, G>(a.out32 + row * DH, u, g, inv, acc);
    if (g == 0)
      a.lse[int64_t(h) * n_q + qi[u]] =
          a.k.n > 0 ? m[u] + __builtin_amdgcn_logf(lsum) * kLn2 : -INFINITY;
  }
}

// Column scores part[z][h][j] = sum |S[h, i, j]| over the queries of split z:
// rows = queries (staged), lanes = keys.  A long column is summed in three levels:
// the stages of a run of kRun are added to each other before they join the total
// (8,000 queries, 4 heads of 32: 7.3e-8 -> 4.7e-8 of float64).
template <class Ops, int DH, int G>
__device__ __forceinline__ void scores_body(const FwdArgs& a, int bx, int h, int z, char* lds) {
  constexpr int SB = Ops::SB;
  const int lane = tid_x() & (kWave - 1);
  const int wave = tid_x() >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int q_begin = z * a.score_rows;
  const int q_end = min(a.q.n, q_begin + a.score_rows);
  int kj[G];
  typename Ops::Rows kf;
  float sum[G], runs[G];
#pragma unroll
  for (int u = 0; u < G; ++u) {
    kj[u] = bx * block_rows(G) + (wave * G + u) * kT + l16;
    sum[u] = runs[u] = 0.f;
    Ops::load_rows(kf, u, a.k, kj[u], h, a.H, g);
  }
  typename Ops::template Staged<true, false> sq;
  sq.lds = reinterpret_cast<decltype(sq.lds)>(lds);
  sq.load(a.q, q_begin, h, a.H);
  int run = kRun;
  for (int qb = q_begin; qb < q_end; qb += SB) {
    __syncthreads();
    sq.store();
    __syncthreads();
    if (qb + SB < q_end) sq.load(a.q, qb + SB, h, a.H);
    float st[G];
#pragma unroll
    for (int u = 0; u < G; ++u) st[u] = 0.f;
    for (int r0 = 0; r0 < SB && qb + r0 < q_end; r0 += kStep) {  // rows past n_q are zero
      f32x4 s[2][G];
      sq.products(r0, g, l16, kf, s);
      if constexpr (!Ops::SCALED) times(s, a.q.scale);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < G; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) st[u] += fabsf(s[t][u][i]);
    }
#pragma unroll
    for (int u = 0; u < G; ++u) runs[u] += st[u];
    if (--run == 0 || qb + SB >= q_end) {
      run = kRun;
#pragma unroll
      for (int u = 0; u < G; ++u) {
        sum[u] += runs[u];
        runs[u] = 0.f;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const float t = sum_rows(sum[u]);
    if (g == 0 && kj[u] < a.k.n) a.part[(int64_t(z) * a.H + h) * a.k.n + kj[u]] = t;
  }
}

template <class Ops, int DH, int G>
constexpr int fwd_lds() {
  return Ops::template Staged<true, false>::BYTES + Ops::template Staged<false, true>::BYTES +
         totals_bytes<DH, G>();
}

// The forward and the column scores in one launch: first the forward blocks (block
// of queries, head, key split), then the score blocks (block of keys, head, query
// split), which fill the CUs that the forward's last round leaves idle.
template <typename T, int DH, int G, bool DROP>
__global__ __launch_bounds__(kBlock) void k_fx_fwd(const FwdArgs a) {
  using F = Fp32Ops<T, DH, G>;
  using P = PieceOps<T, DH, G>;
  __shared__ __align__(16) char lds[max_of(fwd_lds<F, DH, G>(), fwd_lds<P, DH, G>())];
  __shared__ uint32_t waves[kWaves];
  int64_t id = int64_t(wg_y()) * a.grid_x + wg_x();
  const int64_t fwd_blocks = int64_t(a.fwd_bx) * a.H * a.n_split;
  const bool scores = id >= fwd_blocks;
  if (scores) id -= fwd_blocks;
  // block-uniform, before any barrier
  if (scores && id >= int64_t(a.score_bx) * a.H * a.score_splits) return;
  const uint32_t nx = scores ? a.score_bx : a.fwd_bx;
  const uint32_t rest = uint32_t(id) / nx, bx = uint32_t(id) % nx;
  const int h = rest % a.H, z = rest / a.H;
  const bool plain = forward_plain(a.q, a.k, a.v, h, waves);
  if (scores) {
    if (plain)
      scores_body<F, DH, G>(a, bx, h, z, lds);
    else
      scores_body<P, DH, G>(a, bx, h, z, lds);
  } else if (plain) {
    fwd_body<F, T, DH, G, DROP>(a, bx, h, z, lds);
  } else {
    fwd_body<P, T, DH, G, DROP>(a, bx, h, z, lds);
  }
}

// ----------------------------------------------------------------- backward
struct BwdArgs {
  Mat q, k, v, g;
  int32_t H;
  DropoutMask dm;
  uint32_t thr16;
  float drop_scale;
  const void* out;     // of the element type
  const float* out32;  // the forward's fp32 copy, or null
  const float* lse;
  float* dsum;
  float scale;
  void *grad_q, *grad_k, *grad_v;
  int32_t split_keys;
  float* part_dq;
  int32_t n_split, kv_bx, comb_bx;
};

// Query-major: dQ^T += K^T dS^T over the keys of split z, S and dP recomputed
// as in the forward.  D = dO . out per query is formed here and stored (split
// 0) for the dK/dV pass.
template <class Ops, typename T, int DH, int G, bool DROP>
__device__ __forceinline__ void bwd_q_body(const BwdArgs& a, int bx, int h, int z, char* lds) {
  constexpr int SB = Ops::SB, MT = out_tiles(DH);
  const int lane = tid_x() & (kWave - 1);
  const int wave = tid_x() >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int n_q = a.q.n, H = a.H;
  DropoutMask dm = a.dm;
  if constexpr (DROP) dm = drop_for_head(dm, h);
  int qi[G];
  typename Ops::Rows qf, gf;
  float L[G], D[G];
  f32x4 acc[G][MT];
  zero_acc(acc);
#pragma unroll
  for (int u = 0; u < G; ++u) {
    qi[u] = bx * block_rows(G) + (wave * G + u) * kT + l16;
    const bool ok = qi[u] < n_q;
    Ops::load_rows(qf, u, a.q, qi[u], h, H, g);
    Ops::load_rows(gf, u, a.g, qi[u], h, H, g);
    float d = 0.f;
    if (ok) {
      const int64_t o = (int64_t(qi[u]) * H + h) * DH + (DH / 4) * g;
      float gq[DH / 4], oq[DH / 4];
      load_quarter<DH>(static_cast<const T*>(a.g.x) + o, gq);
      if (a.out32)
        load_quarter<DH>(a.out32 + o, oq);
      else
        load_quarter<DH>(static_cast<const T*>(a.out) + o, oq);
#pragma unroll
      for (int j = 0; j < DH / 4; ++j) d = fmaf(gq[j], oq[j], d);
    }
    D[u] = sum_rows(d);
    L[u] = ok ? a.lse[int64_t(h) * n_q + qi[u]] : INFINITY;
    if (ok && z == 0 && g == 0) a.dsum[int64_t(h) * n_q + qi[u]] = D[u];
  }
  const int k_begin = z * a.split_keys;
  const int k_end = min(a.k.n, k_begin + a.split_keys);
  typename Ops::template Staged<true, true> sk;
  typename Ops::template Staged<true, false> sv;
  sk.lds = reinterpret_cast<decltype(sk.lds)>(lds);
  sv.lds = reinterpret_cast<decltype(sv.lds)>(lds + sk.BYTES);
  if (k_begin < k_end) {
    sk.load(a.k, k_begin, h, H);
    sv.load(a.v, k_begin, h, H);
  }
  for (int kb = k_begin; kb < k_end; kb += SB) {
    __syncthreads();
    sk.store();
    sv.store();
    __syncthreads();
    if (kb + SB < k_end) {
      sk.load(a.k, kb + SB, h, H);
      sv.load(a.v, kb + SB, h, H);
    }
    f32x4 stage[G][MT];
    zero_acc(stage);
    for (int r0 = 0; r0 < SB && kb + r0 < k_end; r0 += kStep) {
      f32x4 s[2][G], dp[2][G];
      sk.products(r0, g, l16, qf, s);
      sv.products(r0, g, l16, gf, dp);
      if constexpr (!Ops::SCALED) times(s, a.q.scale);
      if constexpr (!Ops::SCALED && DROP) times(dp, a.drop_scale);
      if (kb + r0 + kStep > k_end) {  // keys past the end: p = 0
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb + r0 + kT * t + 4 * g + i >= k_end)
#pragma unroll
              for (int u = 0; u < G; ++u) s[t][u][i] = -INFINITY;
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const uint32_t key = uint32_t(kb + r0 + kT * t + 4 * g);
          uint32_t w[2] = {0u, 0u};
          if constexpr (DROP) {
            w[0] = drop_word(dm, uint32_t(qi[u]), key);
            w[1] = drop_word(dm, uint32_t(qi[u]), key + 2);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = exp_nat(s[t][u][i] - L[u]);
            float x = dp[t][u][i];
            if constexpr (DROP) {
              const uint32_t bits = i & 1 ? w[i / 2] : w[i / 2] << 16;
              x = kept(bits, a.thr16) ? x : 0.f;
            }
            s[t][u][i] = p * (x - D[u]);
          }
        }
      sk.accumulate(r0, g, l16, s, stage);
    }
    add_acc(stage, acc);
  }
  Ops::finish(acc);
#pragma unroll
  for (int u = 0; u < G; ++u) {
    if (qi[u] >= n_q) continue;
    const int64_t row = int64_t(qi[u]) * H + h;
    if (a.part_dq)
      store_acc<DH, G>(a.part_dq + (int64_t(z) * n_q * H + row) * DH, u, g, 1.f, acc);
    else
      store_acc<DH, G>(static_cast<T*>(a.grad_q) + row * DH, u, g, a.scale, acc);
  }
}

template <class Ops>
constexpr int bwd_q_lds() {
  return Ops::template Staged<true, true>::BYTES + Ops::template Staged<true, false>::BYTES;
}

template <typename T, int DH, int G, bool DROP>
__global__ __launch_bounds__(kBlock) void k_fx_bwd_q(const BwdArgs a) {
  using F = Fp32Ops<T, DH, G>;
  using P = PieceOps<T, DH, G>;
  __shared__ __align__(16) char lds[max_of(bwd_q_lds<F>(), bwd_q_lds<P>())];
  __shared__ uint32_t waves[kWaves];
  const int bx = wg_x(), h = wg_y(), z = wg_z();
  if (backward_plain(a.q, a.k, a.v, a.g, h, waves))
    bwd_q_body<F, T, DH, G, DROP>(a, bx, h, z, lds);
  else
    bwd_q_body<P, T, DH, G, DROP>(a, bx, h, z, lds);
}

// grad_q = scale * sum of the key splits' partial dQ, added in split order.
template <typename T>
__device__ __forceinline__ void dq_combine(const BwdArgs& a, int64_t n, int64_t b, int64_t nb) {
  for (int64_t t = b * kBlock + tid_x(); t < n; t += nb * kBlock) {
    float x = a.part_dq[t];
    for (int s = 1; s < a.n_split; ++s) x += a.part_dq[int64_t(s) * n + t];
    elem<T>::store(static_cast<T*>(a.grad_q) + t, x * a.scale);
  }
}

// Key-major: dV^T += dO^T P and dK^T += (Q scale)^T dS, rows = queries
// (staged, Q already scaled), lanes = keys.
template <class Ops, typename T, int DH, int G, bool DROP>
__device__ __forceinline__ void bwd_kv_body(const BwdArgs& a, int bx, int h, char* lds, float* ls,
                                            float* ds) {
  constexpr int SB = Ops::SB, MT = out_tiles(DH);
  const int lane = tid_x() & (kWave - 1);
  const int wave = tid_x() >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int n_q = a.q.n, H = a.H;
  DropoutMask dm = a.dm;
  if constexpr (DROP) dm = drop_for_head(dm, h);
  int kj[G];
  typename Ops::Rows kf, vf;
  f32x4 dk[G][MT], dv[G][MT];
  zero_acc(dk);
  zero_acc(dv);
#pragma unroll
  for (int u = 0; u < G; ++u) {
    kj[u] = bx * block_rows(G) + (wave * G + u) * kT + l16;
    Ops::load_rows(kf, u, a.k, kj[u], h, H, g);
    Ops::load_rows(vf, u, a.v, kj[u], h, H, g);
  }
  typename Ops::template Staged<true, true> sq, sg;
  sq.lds = reinterpret_cast<decltype(sq.lds)>(lds);
  sg.lds = reinterpret_cast<decltype(sg.lds)>(lds + sq.BYTES);
  float pl = 0.f, pd = 0.f;
  auto prefetch = [&](int qb) {
    sq.load(a.q, qb, h, H);
    sg.load(a.g, qb, h, H);
    if (tid_x() < SB) {
      const bool ok = qb + tid_x() < n_q;  // padded rows: p = exp(-inf) = 0, dO = D = 0
      pl = ok ? a.lse[int64_t(h) * n_q + qb + tid_x()] : INFINITY;
      pd = ok ? a.dsum[int64_t(h) * n_q + qb + tid_x()] : 0.f;
    }
  };
  const int shift = lane & 1 ? 0 : 16;  // this lane's key's half of a word (kj is odd where l16 is)
  if (n_q > 0) prefetch(0);
  for (int qb = 0; qb < n_q; qb += SB) {
    __syncthreads();
    sq.store();
    sg.store();
    if (tid_x() < SB) {
      ls[tid_x()] = pl;
      ds[tid_x()] = pd;
    }
    __syncthreads();
    if (qb + SB < n_q) prefetch(qb + SB);
    f32x4 sdk[G][MT], sdv[G][MT];
    zero_acc(sdk);
    zero_acc(sdv);
    for (int r0 = 0; r0 < SB && qb + r0 < n_q; r0 += kStep) {
      f32x4 s[2][G], dp[2][G];
      sq.products(r0, g, l16, kf, s);
      sg.products(r0, g, l16, vf, dp);
      if constexpr (!Ops::SCALED) times(s, a.q.scale);
      if constexpr (!Ops::SCALED && DROP) times(dp, a.drop_scale);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int r = r0 + kT * t + 4 * g;  // queries qb + r .. + 3
        const f32x4 L = *reinterpret_cast<const f32x4*>(ls + r);
        const f32x4 D = *reinterpret_cast<const f32x4*>(ds + r);
#pragma unroll
        for (int u = 0; u < G; ++u) {
          // the lanes of a key pair need the same four words (one per query):
          // the even lane hashes the first two, the odd one the others
          uint32_t w[4] = {0u, 0u, 0u, 0u};
          if constexpr (DROP) {
            const bool odd = (lane & 1) != 0;
            const uint32_t qr = uint32_t(qb + r) + (odd ? 2u : 0u);
            const uint32_t wa = drop_word(dm, qr, uint32_t(kj[u]));
            const uint32_t wb = drop_word(dm, qr + 1, uint32_t(kj[u]));
            const uint32_t wc = swap_pair(wa), wd = swap_pair(wb);
            w[0] = odd ? wc : wa, w[1] = odd ? wd : wb, w[2] = odd ? wa : wc, w[3] = odd ? wb : wd;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = exp_nat(s[t][u][i] - L[i]);
            if constexpr (DROP) {
              const bool keep = kept(w[i] << shift, a.thr16);
              dp[t][u][i] = p * ((keep ? dp[t][u][i] : 0.f) - D[i]);
              s[t][u][i] = keep ? p : 0.f;
            } else {
              dp[t][u][i] = p * (dp[t][u][i] - D[i]);
              s[t][u][i] = p;
            }
          }
        }
      }
      sg.accumulate(r0, g, l16, s, sdv);
      sq.accumulate(r0, g, l16, dp, sdk);
    }
    add_acc(sdk, dk);
    add_acc(sdv, dv);
  }
  Ops::finish(dk);
  Ops::finish(dv);
#pragma unroll
  for (int u = 0; u < G; ++u) {
    if (kj[u] >= a.k.n) continue;
    const int64_t o = (int64_t(kj[u]) * H + h) * DH;
    store_acc<DH, G>(static_cast<T*>(a.grad_k) + o, u, g, Ops::SCALED ? 1.f : a.scale, dk);
    store_acc<DH, G>(static_cast<T*>(a.grad_v) + o, u, g,
                     Ops::SCALED || !DROP ? 1.f : a.drop_scale, dv);
  }
}

template <class Ops>
constexpr int bwd_kv_lds() {
  return 2 * Ops::template Staged<true, true>::BYTES;
}

// Blocks at grid x >= kv_bx add the dQ splits' partials instead of taking
// keys (that merge needs no launch of its own).
template <typename T, int DH, int G, bool DROP>
__global__ __launch_bounds__(kBlock) void k_fx_bwd_kv(const BwdArgs a) {
  using F = Fp32Ops<T, DH, G>;
  using P = PieceOps<T, DH, G>;
  __shared__ __align__(16) char lds[max_of(bwd_kv_lds<F>(), bwd_kv_lds<P>())];
  __shared__ uint32_t waves[kWaves];
  __shared__ __align__(16) float ls[64];
  __shared__ __align__(16) float ds[64];
  const int bx = wg_x(), h = wg_y();
  if (bx >= a.kv_bx) {  // block-uniform
    dq_combine<T>(a, int64_t(a.q.n) * a.H * DH, int64_t(bx - a.kv_bx) * a.H + h,
               int64_t(a.comb_bx) * a.H);
    return;
  }
  if (backward_plain(a.q, a.k, a.v, a.g, h, waves))
    bwd_kv_body<F, T, DH, G, DROP>(a, bx, h, lds, ls, ds);
  else
    bwd_kv_body<P, T, DH, G, DROP>(a, bx, h, lds, ls, ds);
}

// ------------------------------------------------------------------ host side
inline int blocks_of(int n, int rows) { return (n + rows - 1) / rows; }
inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// 16-row tiles per wave: 2 (each staged operand feeds two MFMAs) where the
// grid still gives the 1,024 SIMDs two waves each, else 1; 1 at d = 64, whose
// accumulators and operands of two tiles would leave one wave per SIMD.
// NGT_DENSE_F32_TILES overrides the choice below d = 64.
int tiles_per_wave(int n, int H, int d) {
  if (d == 64) return 1;
  if (const char* e = getenv("NGT_DENSE_F32_TILES")) return atoi(e) == 1 ? 1 : 2;
  return int64_t(blocks_of(n, block_rows(2))) * H * kWaves >= 2048 ? 2 : 1;
}

MfSplit split_keys_for(int n_q, int n_k, int H, int d, int target_waves, int64_t shared_waves,
                       const char* env) {
  const int rows = block_rows(tiles_per_wave(n_q, H, d));
  const int64_t base = int64_t(blocks_of(n_q, rows)) * H * kWaves;
  const int64_t room = std::max<int64_t>(target_waves - shared_waves, 0);
  int want = base > 0 ? int((room + base / 2) / base) : 1;
  if (const char* e = getenv(env)) want = atoi(e);
  // more than 8 only where those would not give 1,024 waves (few queries: 4 heads
  // of 32, one query, 16,000 keys, forward 73 -> 22 us)
  const int most = base > 0 ? int(std::min<int64_t>(std::max<int64_t>(1024 / base, 8), 32)) : 8;
  want = std::max(1, std::min({want, most, std::max(1, n_k / 256)}));
  if (want <= 1 || n_k <= 0) return {1, std::max(n_k, 1)};
  int keys = (n_k + want - 1) / want;
  keys = (keys + kPadRows - 1) / kPadRows * kPadRows;
  return {(n_k + keys - 1) / keys, keys};
}

size_t row_image_bytes(int n, int H, int d, int np) {
  return align256(size_t(padded(n)) * H * row_bytes(d, np));
}
size_t t_image_bytes(int n, int H, int d, int np) {
  return align256(size_t(padded(n) / kStep) * H * t_bytes(d, np));
}
size_t flag_bytes(int n, int H) { return align256(size_t(padded(n) / kStep) * H * 4); }

// Assigns one matrix's images in the workspace and adds its preparation job.
struct Images {
  char* ws;
  int H, d, np;
  PrepJobs jobs{};
  int n_jobs = 0, max_rows = 0;
  bool none = false;  // no images: the fp32 bodies read the matrices themselves
  Mat add(const void* x, int n, float scale, bool want_row, bool want_t) {
    if (none) return Mat{x, nullptr, nullptr, nullptr, n, scale};
    PrepJob& j = jobs.j[n_jobs++];
    j.x = x;
    j.row_img = j.t_img = nullptr;
    if (want_row) {
      j.row_img = ws;
      ws += row_image_bytes(n, H, d, np);
    }
    if (want_t) {
      j.t_img = ws;
      ws += t_image_bytes(n, H, d, np);
    }
    j.flag = reinterpret_cast<uint32_t*>(ws);
    ws += flag_bytes(n, H);
    j.n = n;
    j.scale = scale;
    max_rows = std::max(max_rows, padded(n));
    return Mat{x, j.row_img, j.t_img, j.flag, n, scale};
  }
};

template <typename T, int DH>
int run_prep(const Images& im, hipStream_t st) {
  if (im.max_rows == 0) return NGT_OK;
  KernelTimer timer_("dense_prep", st);
  hipLaunchKernelGGL((k_fx_prep<T, DH>), dim3(im.max_rows / kStep, im.H, im.n_jobs), dim3(kBlock), 0,
                     st, im.jobs, im.H);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

template <typename T, int DH, int G>
int fx_fwd(FwdArgs a, const DropoutMask* dm, hipStream_t st) {
  a.fwd_bx = blocks_of(a.q.n, block_rows(G));
  a.score_bx = a.part && a.k.n > 0 ? blocks_of(a.k.n, block_rows(G)) : 0;
  a.score_splits = a.score_bx > 0 ? blocks_of(a.q.n, a.score_rows) : 0;
  const int64_t blocks = (int64_t(a.fwd_bx) * a.n_split + int64_t(a.score_bx) * a.score_splits) * a.H;
  if (blocks > INT32_MAX)
    return set_error(NGT_ERR_UNSUPPORTED, "dense: %d x %d x %d scores exceed the grid", a.q.n, a.k.n,
                     a.H);
  a.grid_x = int(std::min<int64_t>(blocks, 1 << 20));
  const dim3 grid(a.grid_x, unsigned((blocks + a.grid_x - 1) / a.grid_x));
  KernelTimer timer_("dense_fwd", st);
  if (dm)
    hipLaunchKernelGGL((k_fx_fwd<T, DH, G, true>), grid, dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL((k_fx_fwd<T, DH, G, false>), grid, dim3(kBlock), 0, st, a);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

template <typename T, int DH, int G>
int fx_bwd_q(const BwdArgs& a, const DropoutMask* dm, hipStream_t st) {
  KernelTimer timer_("dense_bwd_q", st);
  const dim3 grid(blocks_of(a.q.n, block_rows(G)), a.H, a.n_split);
  if (dm)
    hipLaunchKernelGGL((k_fx_bwd_q<T, DH, G, true>), grid, dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL((k_fx_bwd_q<T, DH, G, false>), grid, dim3(kBlock), 0, st, a);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

template <typename T, int DH, int G>
int fx_bwd_kv(BwdArgs a, const DropoutMask* dm, hipStream_t st) {
  KernelTimer timer_("dense_bwd_kv", st);
  a.kv_bx = blocks_of(a.k.n, block_rows(G));
  // merge blocks per head: about 4 elements per thread
  const int64_t n_dq = int64_t(a.q.n) * a.H * DH;
  const int64_t per = int64_t(4) * kBlock * a.H;
  a.comb_bx = a.part_dq ? int((n_dq + per - 1) / per) : 0;
  const dim3 grid(a.kv_bx + a.comb_bx, a.H);
  if (dm)
    hipLaunchKernelGGL((k_fx_bwd_kv<T, DH, G, true>), grid, dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL((k_fx_bwd_kv<T, DH, G, false>), grid, dim3(kBlock), 0, st, a);
  NGT_HIP_CHECK(hipGetLastError());
  return NGT_OK;
}

template <typename T, int DH>
int fx_forward(FwdArgs a, const Images& im, const DropoutMask* dm, hipStream_t st) {
  NGT_CHECK_OK((run_prep<T, DH>(im, st)));
  if constexpr (DH == 64) return fx_fwd<T, DH, 1>(a, dm, st);
  else
    return tiles_per_wave(a.q.n, a.H, DH) == 2 ? fx_fwd<T, DH, 2>(a, dm, st) : fx_fwd<T, DH, 1>(a, dm, st);
}

template <typename T, int DH>
int fx_backward(const BwdArgs& a, const Images& im, const DropoutMask* dm, hipStream_t st) {
  NGT_CHECK_OK((run_prep<T, DH>(im, st)));
  if constexpr (DH == 64) {
    if (a.q.n > 0) NGT_CHECK_OK((fx_bwd_q<T, DH, 1>(a, dm, st)));
    return a.k.n > 0 ? fx_bwd_kv<T, DH, 1>(a, dm, st) : NGT_OK;
  } else {
    if (a.q.n > 0)
      NGT_CHECK_OK((tiles_per_wave(a.q.n, a.H, DH) == 2 ? fx_bwd_q<T, DH, 2>(a, dm, st)
                                                        : fx_bwd_q<T, DH, 1>(a, dm, st)));
    if (a.k.n > 0)
      return tiles_per_wave(a.k.n, a.H, DH) == 2 ? fx_bwd_kv<T, DH, 2>(a, dm, st)
                                                 : fx_bwd_kv<T, DH, 1>(a, dm, st);
    return NGT_OK;
  }
}

}  // namespace

MfSplit fx_fwd_split(int n_q, int n_k, int H, int d, bool node_scores) {
  const int rows = block_rows(tiles_per_wave(n_k, H, d));
  // the score blocks' waves weigh as their rows do against the forward's
  const double weight = node_scores && n_k > 0 ? double(std::min(n_q, n_k)) / n_k : 0.0;
  const int64_t score_waves = int64_t(weight * blocks_of(n_k, rows) * H * kWaves);
  return split_keys_for(n_q, n_k, H, d, 6144, score_waves, "NGT_DENSE_F32_FWD_SPLIT");
}
// Queries per block of the column scores: about the rows that a forward block
// streams, so that neither outlasts the other, and at least 256.  With all
// queries in one block a forward over few keys waited for it (us, vector kernels /
// one block / so): 8 heads of 8, 30,000 queries, 64 keys 40 / 394 / 28; 16,000 and
// 1,000 143 / 260 / 103; 2,500 and 2,500 67 / 79 / 66.  (On a 3-d grid padded with
// 220,000 blocks that exit at once the first took 67.)
MfSplit fx_score_split(int n_q, MfSplit keys) {
  const int rows = std::max(256, keys.split_keys);
  const int want = std::min(std::max(blocks_of(n_q, rows), 1), 1024);
  const int per = blocks_of(blocks_of(n_q, want), kPadRows) * kPadRows;
  return {std::max(blocks_of(n_q, per), 1), std::max(per, kPadRows)};
}
MfSplit fx_dq_split(int n_q, int n_k, int H, int d) {
  return split_keys_for(n_q, n_k, H, d, 6144, 0, "NGT_DENSE_F32_DQ_SPLIT");
}

// Few scores: the fp32 bodies alone, on the matrices as they are.  Their MFMAs
// take 8 times the cycles, but up to here the two preparation launches and the
// pieces' splits cost more.  Forward and backward in us, pieces / fp32 (in brackets
// with dropout): 8 heads of 8, 406 nodes 61 / 36, 2^25 scores (2,048 nodes) 191 /
// 143 (205 / 170); 8 of 16, 2^25 205 / 187 (220 / 220), 2^26 336 / 346; 32 of 24,
// 2^25 285 / 234, 2^27 976 / 1,102; 8 of 32, 2^25 305 / 272 (341 / 355), 4 of 32
// 394 / 415 (398 / 451); 8 of 64, 2^22 179 / 172 (180 / 180), 2^23 232 / 241.  At
// d = 8 and 24 the times cross one power later (2^26 272 / 225 and 463 / 404), but
// the pieces are the more exact there (8 heads of 8, 2,500 nodes: x 3.1e-7 against
// 5.2e-7), so the line stays at 2^25.
// Up to 128 rows on one side an image's row is read by a block or two, and the
// preparation of the other side's is most of the work: 32 heads of 24, 23,170
// queries, 128 keys, forward 256 / 189 (forward and backward 2,209 / 1,568); 128
// queries, 23,170 keys 405 / 187 (1,177 / 659); 8 of 8, 92,681 and 128 135 / 99; at
// 256 173 / 174 and 101 / 89.
// NGT_DENSE_F32_TILES asks for the pieces.
bool few_scores(int dtype, int n_q, int n_k, int H, int d) {
  return dtype == NGT_F32 && !getenv("NGT_DENSE_F32_TILES") &&
         (std::min(n_q, n_k) <= 128 ||
          int64_t(n_q) * n_k <= (int64_t(1) << (d == 64 ? 22 : 25)) / std::max(H, 1));
}

// Bytes of the images and flags that the two directions keep in the workspace.
size_t fx_fwd_image_bytes(int dtype, int n_q, int n_k, int H, int d) {
  if (few_scores(dtype, n_q, n_k, H, d)) return 0;
  const int np = dtype == NGT_F32 ? 3 : 1;
  return row_image_bytes(n_q, H, d, np) + flag_bytes(n_q, H) + row_image_bytes(n_k, H, d, np) +
         t_image_bytes(n_k, H, d, np) + 2 * flag_bytes(n_k, H);
}
size_t fx_bwd_image_bytes(int dtype, int n_q, int n_k, int H, int d) {
  if (few_scores(dtype, n_q, n_k, H, d)) return 0;
  const int np = dtype == NGT_F32 ? 3 : 1;
  return 2 * (row_image_bytes(n_q, H, d, np) + t_image_bytes(n_q, H, d, np) + flag_bytes(n_q, H)) +
         2 * (row_image_bytes(n_k, H, d, np) + flag_bytes(n_k, H)) + t_image_bytes(n_k, H, d, np);
}

// (threshold << 16, scale) of a mask for kept(); a threshold of 2^16 (nothing
// kept) becomes "all kept" with scale 0, as p = 1 is.
static void drop_terms(const DropoutMask* dm, uint32_t* thr16, float* scale) {
  const bool none = dm && dm->thr > 0xffffu;
  *thr16 = dm && !none ? dm->thr << 16 : 0u;
  *scale = !dm ? 1.f : none ? 0.f : dm->scale;
}

int fx_dense_fwd(int dtype, int d, const void* q, const void* k, const void* v, int n_q, int n_k,
                 int H, float scale, const DropoutMask* dm, void* out, float* out32, float* lse,
                 float* part, MfSplit sp, MfSplit scores, float* part_ml, float* part_acc,
                 char* images, hipStream_t st) {
  Images im{images, H, d, dtype == NGT_F32 ? 3 : 1};
  im.none = few_scores(dtype, n_q, n_k, H, d);
  FwdArgs a{};
  drop_terms(dm, &a.thr16, &a.drop_scale);
  a.q = im.add(q, n_q, scale, true, false);
  a.k = im.add(k, n_k, 1.f, true, false);
  a.v = im.add(v, n_k, a.drop_scale, false, true);
  a.H = H;
  if (dm) a.dm = *dm;
  a.out = out, a.out32 = out32, a.lse = lse;
  a.split_keys = sp.split_keys;
  a.n_split = sp.n_split;
  a.score_rows = scores.split_keys;
  if (sp.n_split > 1) a.part_ml = part_ml, a.part_acc = part_acc;
  a.part = part;
  if (dtype == NGT_BF16 && d == 64) return fx_forward<bf16_t, 64>(a, im, dm, st);
  if (dtype == NGT_F32) switch (d) {
      case 8: return fx_forward<float, 8>(a, im, dm, st);
      case 16: return fx_forward<float, 16>(a, im, dm, st);
      case 24: return fx_forward<float, 24>(a, im, dm, st);
      case 32: return fx_forward<float, 32>(a, im, dm, st);
      case 64: return fx_forward<float, 64>(a, im, dm, st);
      default: break;
    }
  return set_error(NGT_ERR_UNSUPPORTED, "dense: head_dim %d", d);
}

int fx_dense_bwd(int dtype, int d, const void* q, const void* k, const void* v, const void* go,
                 const void* out, const float* out32, const float* lse, float* dsum, int n_q,
                 int n_k, int H, float scale, const DropoutMask* dm, void* gq, void* gk, void* gv,
                 MfSplit sq, float* part_dq, char* images, hipStream_t st) {
  Images im{images, H, d, dtype == NGT_F32 ? 3 : 1};
  im.none = few_scores(dtype, n_q, n_k, H, d);
  BwdArgs a{};
  drop_terms(dm, &a.thr16, &a.drop_scale);
  a.q = im.add(q, n_q, scale, true, true);
  a.g = im.add(go, n_q, a.drop_scale, true, true);
  a.k = im.add(k, n_k, 1.f, true, true);
  a.v = im.add(v, n_k, 1.f, true, false);
  a.H = H;
  if (dm) a.dm = *dm;
  a.out = out, a.out32 = out32, a.lse = lse, a.dsum = dsum, a.scale = scale;
  a.grad_q = gq, a.grad_k = gk, a.grad_v = gv;
  a.split_keys = sq.split_keys;
  a.n_split = sq.n_split;
  a.part_dq = n_q > 0 && sq.n_split > 1 ? part_dq : nullptr;
  if (dtype == NGT_BF16 && d == 64) return fx_backward<bf16_t, 64>(a, im, dm, st);
  if (dtype == NGT_F32) switch (d) {
      case 8: return fx_backward<float, 8>(a, im, dm, st);
      case 16: return fx_backward<float, 16>(a, im, dm, st);
      case 24: return fx_backward<float, 24>(a, im, dm, st);
      case 32: return fx_backward<float, 32>(a, im, dm, st);
      case 64: return fx_backward<float, 64>(a, im, dm, st);
      default: break;
    }
  return set_error(NGT_ERR_UNSUPPORTED, "dense: head_dim %d", d);
}

}  // namespace ngt
