// Window adjacency construction: COO edge_index -> query-major CSR,
// key-major (transposed) CSR, the position map between them and the
// degree-binned work lists the attention kernels are scheduled from:
//   rows with more than `chunk` edges -> chunks of `chunk` edges (listed first),
//   rows with small < degree <= chunk -> one work item per row, longest first,
//   rows with degree <= small         -> packed list, longest first; the
//                                        kernels give each such row one edge
//                                        slot (several rows per wave);
// and, when asked for, the rows longest first (the tiled kernels' order): all
// query rows, and the key rows j < min(n_q, n_k) (the window's own nodes).
//
// The reference keeps the window mask as a COO edge_index
// (NeutronGT/core/node_level_pipeline/window_state.py:122-140) and consumes it
// with gathers and torch_scatter adds
// (NeutronGT/models/graphormer_dist_node_level.py:75-97).  Here the ordering is
// made canonical: query-major rows are sorted by (dst, src, edge id) and
// key-major rows by (src, dst, edge id), so the CSR is a pure function of the
// edge list (bit-exact, independent of launch shapes).  Stable sorts make both
// orders: by (dst, src), which leaves the edges in (dst, src, edge id) order,
// then those by src, which gives (src, dst, edge id) and, with query-major
// positions as the values, the map between the two.  Keys are 32 bits; the first
// sort is one of combined keys where both endpoints fit 32 bits (up to 65,535
// rows a side) and else two, by src and by dst: the digit passes are as many,
// but one sort spares a histogram, its scan, the gather of dst between the two
// and the one of src after them (16,384 of 200,000 nodes: the window's whole
// preparation 434 -> 420 us).  Combined 64-bit keys of each order took five
// passes of 12 bytes.  The sorts are rocPRIM's radix sort;
// its default switches to a merge sort below 1 M entries, 23 launches for the
// 0.67 M edges of a 16,384-node window against 5 or 6 (one window's build
// there is bound by launches, not bytes), so sort_edges keeps radix passes
// down to 16 K entries.
#include "ngt_common.h"

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

namespace ngt {
namespace {

constexpr int kBlock = 256;

struct Count3 {
  int32_t split_items;  // chunks of rows longer than `chunk`
  int32_t plain_items;  // rows that fit one item
  int32_t split_rows;
};

struct Count3Plus {
  __host__ __device__ Count3 operator()(const Count3& a, const Count3& b) const {
    return Count3{a.split_items + b.split_items, a.plain_items + b.plain_items,
                  a.split_rows + b.split_rows};
  }
};

inline unsigned bits_for(uint64_t v) {
  unsigned b = 0;
  while (b < 64 && (v >> b) != 0) ++b;
  return b == 0 ? 1 : b;
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Tiles of 16,384 keys (the library's choice) leave most of the chip idle below
// a million edges; tiles of 4,096 fill it but look back over four times as many
// predecessors.  One sort by a 15-bit endpoint with either: 30,000 keys 59 / 30
// us, 230,000 63 / 37, 671,744 67 / 50, 1,800,000 77 / 80, 3,600,000 89 / 124.
constexpr int64_t kSmallTiles = 1200000;
using LargeTiles = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, 16 * 1024>;
using SmallTiles = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<256, 8>,
                                        rocprim::kernel_config<1024, 4>, 8,
                                        rocprim::block_radix_rank_algorithm::match>,
    16 * 1024>;

template <class Config>
hipError_t sort_with(void* temp, size_t& bytes, uint32_t* key_in, uint32_t* key_out,
                     int32_t* val_in, int32_t* val_out, int64_t n, unsigned bits, hipStream_t st) {
  return rocprim::radix_sort_pairs<Config>(temp, bytes, key_in, key_out, val_in, val_out,
                                           size_t(n), 0u, bits, st);
}

// Radix passes clear their counters with memsets, which replays of a captured
// graph do not repeat reliably: under capture every sort is a merge sort, kernels
// only.  (The library's default takes radix passes above a million entries, and
// the row sort below holds both sides' rows.)  That costs a captured build, eager
// against replay: 0.67 M edges of 16,384 nodes 242 / 391 us, 1.8 M of 32,768 387 /
// 612, 3.6 M of 65,000 551 / 791.
using KernelsOnly = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                               rocprim::default_config, (size_t(1) << 32)>;
bool capturing(hipStream_t st) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  return st && hipStreamIsCapturing(st, &s) == hipSuccess && s != hipStreamCaptureStatusNone;
}

int sort_edges(void* temp, size_t bytes, uint32_t* key_in, uint32_t* key_out, int32_t* val_in,
               int32_t* val_out, int64_t n, unsigned bits, hipStream_t st) {
  if (capturing(st))
    NGT_HIP_CHECK(sort_with<KernelsOnly>(temp, bytes, key_in, key_out, val_in, val_out, n, bits,
                                         st));
  else if (n <= kSmallTiles)
    NGT_HIP_CHECK(sort_with<SmallTiles>(temp, bytes, key_in, key_out, val_in, val_out, n, bits, st));
  else
    NGT_HIP_CHECK(sort_with<LargeTiles>(temp, bytes, key_in, key_out, val_in, val_out, n, bits, st));
  return NGT_OK;
}

int sort_edges_bytes(int64_t n, size_t* bytes) {
  size_t a = 0, b = 0;
  uint32_t* k = nullptr;
  int32_t* v = nullptr;
  NGT_HIP_CHECK(sort_with<KernelsOnly>(nullptr, a, k, k, v, v, n, 32u, nullptr));
  if (n <= kSmallTiles)
    NGT_HIP_CHECK(sort_with<SmallTiles>(nullptr, b, k, k, v, v, n, 32u, nullptr));
  else
    NGT_HIP_CHECK(sort_with<LargeTiles>(nullptr, b, k, k, v, v, n, 32u, nullptr));
  *bytes = a > b ? a : b;
  return NGT_OK;
}

// Rows by degree: the library's default, but for capture.
int sort_rows(void* temp, size_t bytes, uint32_t* key_in, uint32_t* key_out, int32_t* val_in,
              int32_t* val_out, int64_t n, hipStream_t st) {
  if (capturing(st))
    NGT_HIP_CHECK(sort_with<KernelsOnly>(temp, bytes, key_in, key_out, val_in, val_out, n, 32u, st));
  else
    NGT_HIP_CHECK(sort_with<rocprim::default_config>(temp, bytes, key_in, key_out, val_in, val_out,
                                                     n, 32u, st));
  return NGT_OK;
}

int sort_rows_bytes(int64_t n, size_t* bytes) {
  size_t a = 0, b = 0;
  uint32_t* k = nullptr;
  int32_t* v = nullptr;
  NGT_HIP_CHECK(sort_with<KernelsOnly>(nullptr, a, k, k, v, v, n, 32u, nullptr));
  NGT_HIP_CHECK(sort_with<rocprim::default_config>(nullptr, b, k, k, v, v, n, 32u, nullptr));
  *bytes = a > b ? a : b;
  return NGT_OK;
}

// 32-bit endpoints, or with dst32 null both in one key, dst << src_bits | src;
// edges outside the window become {n_k, n_q}, which sorts behind every row in
// both orders.
__global__ void k_endpoints(const int64_t* __restrict__ src, const int64_t* __restrict__ dst,
                            int64_t E, int32_t n_q, int32_t n_k, unsigned src_bits,
                            uint32_t* __restrict__ src32, uint32_t* __restrict__ dst32,
                            int32_t* __restrict__ eid, int32_t* __restrict__ info) {
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < E;
       e += int64_t(gridDim.x) * blockDim.x) {
    const int64_t s = src[e];
    const int64_t d = dst[e];
    const bool ok = s >= 0 && s < n_k && d >= 0 && d < n_q;
    const uint32_t s32 = ok ? uint32_t(s) : uint32_t(n_k);
    const uint32_t d32 = ok ? uint32_t(d) : uint32_t(n_q);
    src32[e] = dst32 ? s32 : d32 << src_bits | s32;
    if (dst32) dst32[e] = d32;
    if (!ok) atomicAdd(info + NGT_INFO_BAD_EDGES, 1);
    eid[e] = static_cast<int32_t>(e);
  }
}

__global__ void k_gather_u32(const uint32_t* __restrict__ x, const int32_t* __restrict__ at,
                             int64_t E, uint32_t* __restrict__ out) {
  for (int64_t p = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; p < E;
       p += int64_t(gridDim.x) * blockDim.x)
    out[p] = x[at[p]];
}

// rowptr[r] = first position p of the sorted rows with rows[p] >= r (the rows
// are the keys' bits from `shift` on); edges outside the window (row n_rows)
// sit past rowptr[n_rows].
__device__ __forceinline__ void fill_rowptr(const uint32_t* __restrict__ rows, unsigned shift,
                                            int64_t E, int64_t p, int32_t n_rows,
                                            int32_t* __restrict__ rowptr) {
  const int64_t r_cur = p < E ? int64_t(rows[p] >> shift) : int64_t(n_rows);
  const int64_t r_prev = p > 0 ? int64_t(rows[p - 1] >> shift) : -1;
  for (int64_t r = r_prev + 1; r <= r_cur; ++r) rowptr[r] = static_cast<int32_t>(p);
}

// Query-major rows: row pointers and columns; the columns are also the last
// sort's keys (n_k for an edge outside the window) and the positions its values.
// src_bits: the keys hold src in as many low bits (0: src32 does).
__global__ void k_rows_q(const uint32_t* __restrict__ dst_sorted, const int32_t* __restrict__ perm,
                         const uint32_t* __restrict__ src32, unsigned src_bits, int64_t E,
                         int32_t n_q, int32_t n_k,
                         int32_t* __restrict__ rowptr, int32_t* __restrict__ col,
                         uint32_t* __restrict__ key, int32_t* __restrict__ pos) {
  for (int64_t p = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; p <= E;
       p += int64_t(gridDim.x) * blockDim.x) {
    if (p < E) {
      const uint32_t s =
          src_bits ? dst_sorted[p] & ((1u << src_bits) - 1u) : src32[perm[p]];
      col[p] = s < uint32_t(n_k) ? static_cast<int32_t>(s) : 0;
      key[p] = s;
      pos[p] = static_cast<int32_t>(p);
    }
    fill_rowptr(dst_sorted, src_bits, E, p, n_q, rowptr);
  }
}

// Key-major rows: row pointers, columns, edge ids, and q2t.
__global__ void k_rows_k(const uint32_t* __restrict__ src_sorted, const int32_t* __restrict__ qpos,
                         const int32_t* __restrict__ perm, const uint32_t* __restrict__ dst_sorted,
                         unsigned src_bits, int64_t E, int32_t n_q, int32_t n_k,
                         int32_t* __restrict__ t_rowptr,
                         int32_t* __restrict__ t_col, int32_t* __restrict__ t_perm,
                         int32_t* __restrict__ q2t) {
  for (int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; t <= E;
       t += int64_t(gridDim.x) * blockDim.x) {
    if (t < E) {
      const int32_t p = qpos[t];
      const uint32_t d = dst_sorted[p] >> src_bits;
      t_col[t] = d < uint32_t(n_q) ? static_cast<int32_t>(d) : 0;
      t_perm[t] = perm[p];
      q2t[p] = static_cast<int32_t>(t);
    }
    fill_rowptr(src_sorted, 0u, E, t, n_k, t_rowptr);
  }
}

__device__ __forceinline__ Count3 row_counts(int32_t deg, int32_t chunk) {
  if (deg > chunk) return Count3{(deg + chunk - 1) / chunk, 0, 1};
  return Count3{0, 1, 0};
}

// One order's rows and the lists made for them.  Both orders go through the
// same launches, the query rows first: row r of a side is entry base + r.
struct Side {
  const int32_t* rowptr;
  int32_t n_rows, chunk, small;
  int64_t base;
  int4 *items, *splits;
  int32_t *packed, *order;  // order: every row, longest first (null: not here)
  int32_t info_base, packed_slot, small_slot, max_deg_slot;
};
struct Sides {
  Side s[2];
};
constexpr uint32_t kKeySide = 0x80000000u;  // of a degree: sorts behind the query rows

__device__ __forceinline__ Count3 operator-(const Count3& a, const Count3& b) {
  return Count3{int32_t(uint32_t(a.split_items) - uint32_t(b.split_items)),
                int32_t(uint32_t(a.plain_items) - uint32_t(b.plain_items)),
                int32_t(uint32_t(a.split_rows) - uint32_t(b.split_rows))};
}

// Per row: chunk counts for the scan, and (degree, row) pairs for the sort.
// grid.y = side, as in the two kernels below.
__global__ void k_count(const Sides sides, Count3* __restrict__ cnt,
                        uint32_t* __restrict__ deg_key, int32_t* __restrict__ row_val,
                        int32_t* __restrict__ info) {
  const Side s = sides.s[blockIdx.y];
  const uint32_t flag = blockIdx.y ? kKeySide : 0u;
  int32_t local_max = 0;
  for (int64_t r = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; r < s.n_rows;
       r += int64_t(gridDim.x) * blockDim.x) {
    const int32_t deg = s.rowptr[r + 1] - s.rowptr[r];
    cnt[s.base + r] = row_counts(deg, s.chunk);
    deg_key[s.base + r] = static_cast<uint32_t>(deg) | flag;
    row_val[s.base + r] = static_cast<int32_t>(r);
    local_max = max(local_max, deg);
  }
  if (local_max > 0) atomicMax(info + s.max_deg_slot, local_max);
}

// Chunks of the rows longer than `chunk` (row order) and the split table.
__global__ void k_emit_split(const Sides sides, const Count3* __restrict__ scan) {
  const Side s = sides.s[blockIdx.y];
  for (int64_t r = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; r < s.n_rows;
       r += int64_t(gridDim.x) * blockDim.x) {
    const int32_t beg = s.rowptr[r];
    const int32_t end = s.rowptr[r + 1];
    if (end - beg <= s.chunk) continue;
    const Count3 pre = scan[s.base + r] - scan[s.base];
    const int32_t n = (end - beg + s.chunk - 1) / s.chunk;
    for (int32_t c = 0; c < n; ++c) {
      const int32_t b = beg + c * s.chunk;
      const int32_t slot = pre.split_items + c;
      s.items[slot] = make_int4(static_cast<int32_t>(r), b, min(end, b + s.chunk), slot);
    }
    s.splits[pre.split_rows] = make_int4(static_cast<int32_t>(r), pre.split_items, n, 0);
  }
}

// First index in sorted[0, n) whose value exceeds x.
__device__ __forceinline__ int32_t upper_bound_u32(const uint32_t* __restrict__ sorted, int32_t n,
                                                   uint32_t x) {
  int32_t lo = 0, hi = n;
  while (lo < hi) {
    const int32_t mid = (lo + hi) >> 1;
    if (sorted[mid] <= x) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Packing threshold read from the degrees (small = NGT_SMALL_FROM_DEGREES):
// the first step that packs at least kPackSharePct % of the rows.
constexpr int32_t kPackSteps[4] = {8, 16, 24, 32};
constexpr int64_t kPackSharePct = 78;

__device__ __forceinline__ int32_t packing_threshold(const uint32_t* __restrict__ sdeg,
                                                     int32_t n_rows, int32_t chunk,
                                                     uint32_t flag) {
  int32_t t = 0;
  for (int i = 0; i < 4; ++i) {
    t = min(kPackSteps[i], chunk - 1);
    const int32_t packed = upper_bound_u32(sdeg, n_rows, static_cast<uint32_t>(t) | flag);
    if (int64_t(packed) * 100 >= int64_t(n_rows) * kPackSharePct) break;
  }
  return t;
}

// From the rows sorted by ascending degree: the packed small rows and the
// single-item medium rows, both longest first.  info gets the totals and the
// packing threshold used.
__global__ void k_emit_sorted(const Sides sides, const uint32_t* __restrict__ sorted_deg,
                              const int32_t* __restrict__ sorted_row,
                              const Count3* __restrict__ scan, int32_t* __restrict__ info) {
  const Side s = sides.s[blockIdx.y];
  const uint32_t flag = blockIdx.y ? kKeySide : 0u;
  const uint32_t* sdeg = sorted_deg + s.base;
  const int32_t* srow = sorted_row + s.base;
  const int32_t small =
      s.small < 0 ? packing_threshold(sdeg, s.n_rows, s.chunk, flag) : s.small;
  const int32_t n_small = upper_bound_u32(sdeg, s.n_rows, static_cast<uint32_t>(small) | flag);
  const int32_t n_le_chunk =
      upper_bound_u32(sdeg, s.n_rows, static_cast<uint32_t>(s.chunk) | flag);
  const int32_t n_medium = n_le_chunk - n_small;
  Count3 tot{0, 0, 0};
  if (s.n_rows > 0) {
    const Count3 last = scan[s.base + s.n_rows - 1] - scan[s.base];
    const Count3 own = row_counts(s.rowptr[s.n_rows] - s.rowptr[s.n_rows - 1], s.chunk);
    tot = Count3{last.split_items + own.split_items, last.plain_items + own.plain_items,
                 last.split_rows + own.split_rows};
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    info[s.info_base + 0] = tot.split_items + n_medium;  // work items
    info[s.info_base + 1] = tot.split_items;             // partial slots
    info[s.info_base + 2] = tot.split_rows;              // split rows
    info[s.packed_slot] = n_small;                       // packed rows
    info[s.small_slot] = small;                          // their threshold
  }
  for (int64_t p = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; p < s.n_rows;
       p += int64_t(gridDim.x) * blockDim.x) {
    const int32_t r = srow[p];
    if (p < n_small)
      s.packed[n_small - 1 - p] = r;
    else if (p < n_le_chunk)
      s.items[tot.split_items + (n_le_chunk - 1 - p)] =
          make_int4(r, s.rowptr[r], s.rowptr[r + 1], -1);
    if (s.order) s.order[s.n_rows - 1 - p] = r;
  }
}

// order[n - 1 - p] = srow[p]: rows sorted by ascending degree, reversed.
__global__ void k_emit_order(const int32_t* __restrict__ srow, int32_t n,
                             int32_t* __restrict__ order) {
  for (int32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
    order[n - 1 - p] = srow[p];
}

__global__ void k_ends(const uint32_t* __restrict__ dst_sorted, unsigned src_bits,
                       const uint32_t* __restrict__ src_sorted, const int32_t* __restrict__ rowptr,
                       int32_t n_q, int32_t* __restrict__ info) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int32_t nv = rowptr[n_q];  // valid edges (dropped ones sort last)
    info[NGT_INFO_DST_END] = nv > 0 ? int32_t(dst_sorted[nv - 1] >> src_bits) + 1 : 0;
    info[NGT_INFO_SRC_END] = nv > 0 ? int32_t(src_sorted[nv - 1]) + 1 : 0;
  }
}

__global__ void k_zero(int32_t* p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

inline int grid_for(int64_t n) {
  int64_t g = (n + kBlock - 1) / kBlock;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return static_cast<int>(g);
}

struct CsrLayout {
  size_t src32, dst32, key_a, key_b, key_c, val_a, val_b, cnt, cnt_scan, deg_a, deg_b, row_a,
      row_b, deg_c, row_c, temp, total;
  size_t temp_bytes;
};

int csr_layout(int64_t E, int32_t n_q, int32_t n_k, CsrLayout* L) {
  const int64_t n_rows = int64_t(n_q) + n_k;  // both orders' rows
  size_t sort_bytes = 0, scan_bytes = 0;
  const size_t n = static_cast<size_t>(E > 0 ? E : 1);
  NGT_CHECK_OK(sort_edges_bytes(static_cast<int64_t>(n), &sort_bytes));
  NGT_HIP_CHECK(rocprim::exclusive_scan(nullptr, scan_bytes, (Count3*)nullptr, (Count3*)nullptr,
                                        Count3{0, 0, 0}, size_t(n_rows > 0 ? n_rows : 1),
                                        Count3Plus(), hipStream_t(0)));
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  L->src32 = take(n * 4);
  L->dst32 = take(n * 4);
  L->key_a = take(n * 4);
  L->key_b = take(n * 4);
  L->key_c = take(n * 4);
  L->val_a = take(n * 4);
  L->val_b = take(n * 4);
  L->cnt = take(size_t(n_rows + 1) * sizeof(Count3));
  L->cnt_scan = take(size_t(n_rows + 1) * sizeof(Count3));
  L->deg_a = take(size_t(n_rows + 1) * 4);
  L->deg_b = take(size_t(n_rows + 1) * 4);
  L->row_a = take(size_t(n_rows + 1) * 4);
  L->row_b = take(size_t(n_rows + 1) * 4);
  L->deg_c = take(size_t(n_rows + 1) * 4);
  L->row_c = take(size_t(n_rows + 1) * 4);
  size_t deg_sort_bytes = 0;
  NGT_CHECK_OK(sort_rows_bytes(n_rows > 0 ? n_rows : 1, &deg_sort_bytes));
  L->temp_bytes = sort_bytes > scan_bytes ? sort_bytes : scan_bytes;
  if (deg_sort_bytes > L->temp_bytes) L->temp_bytes = deg_sort_bytes;
  L->temp = take(L->temp_bytes);
  L->total = off;
  return NGT_OK;
}

// Both orders' work lists (q.base = 0, k.base = the query rows).  order_lead
// (optional): the first n_lead key rows, longest first.
int build_worklists(const Sides& sides, int32_t* order_lead, int32_t n_lead, int32_t* info,
                    char* ws, const CsrLayout& L, hipStream_t st) {
  Count3* cnt = reinterpret_cast<Count3*>(ws + L.cnt);
  Count3* scan = reinterpret_cast<Count3*>(ws + L.cnt_scan);
  uint32_t* deg_a = reinterpret_cast<uint32_t*>(ws + L.deg_a);
  uint32_t* deg_b = reinterpret_cast<uint32_t*>(ws + L.deg_b);
  int32_t* row_a = reinterpret_cast<int32_t*>(ws + L.row_a);
  int32_t* row_b = reinterpret_cast<int32_t*>(ws + L.row_b);
  const Side &q = sides.s[0], &k = sides.s[1];
  const int64_t rows = int64_t(q.n_rows) + k.n_rows;
  const dim3 grid(grid_for(q.n_rows > k.n_rows ? q.n_rows : k.n_rows), 2);
  if (rows > 0) {
    hipLaunchKernelGGL(k_count, grid, dim3(kBlock), 0, st, sides, cnt, deg_a, row_a, info);
    NGT_HIP_CHECK(hipGetLastError());
    size_t temp_bytes = L.temp_bytes;
    NGT_HIP_CHECK(rocprim::exclusive_scan(ws + L.temp, temp_bytes, cnt, scan, Count3{0, 0, 0},
                                          size_t(rows), Count3Plus(), st));
    hipLaunchKernelGGL(k_emit_split, grid, dim3(kBlock), 0, st, sides, scan);
    NGT_HIP_CHECK(hipGetLastError());
    NGT_CHECK_OK(sort_rows(ws + L.temp, L.temp_bytes, deg_a, deg_b, row_a, row_b, rows, st));
  }
  hipLaunchKernelGGL(k_emit_sorted, grid, dim3(kBlock), 0, st, sides, deg_b, row_b, scan, info);
  NGT_HIP_CHECK(hipGetLastError());
  if (order_lead && n_lead > 0) {
    // the leading rows alone: their (degree, row) are the first key entries
    uint32_t* deg_c = reinterpret_cast<uint32_t*>(ws + L.deg_c);
    int32_t* row_c = reinterpret_cast<int32_t*>(ws + L.row_c);
    NGT_CHECK_OK(sort_rows(ws + L.temp, L.temp_bytes, deg_a + k.base, deg_c, row_a + k.base, row_c,
                           n_lead, st));
    hipLaunchKernelGGL(k_emit_order, dim3(grid_for(n_lead)), dim3(kBlock), 0, st, row_c, n_lead,
                       order_lead);
    NGT_HIP_CHECK(hipGetLastError());
  }
  return NGT_OK;
}

}  // namespace
}  // namespace ngt

using namespace ngt;

extern "C" int ngt_csr_sizes(int64_t n_edges, int32_t n_q, int32_t n_k, int32_t chunk_q,
                             int32_t chunk_k, int32_t* max_items_q, int32_t* max_splits_q,
                             int32_t* max_items_k, int32_t* max_splits_k) {
  if (n_edges < 0 || n_q < 0 || n_k < 0 || chunk_q <= 0 || chunk_k <= 0)
    return set_error(NGT_ERR_ARG, "ngt_csr_sizes: negative size or non-positive chunk");
  if (n_edges >= (int64_t(1) << 31) - 1)
    return set_error(NGT_ERR_UNSUPPORTED, "ngt_csr_sizes: %lld edges exceed int32 indexing",
                     (long long)n_edges);
  const int64_t cq = (n_edges + chunk_q - 1) / chunk_q;
  const int64_t ck = (n_edges + chunk_k - 1) / chunk_k;
  const int64_t iq = int64_t(n_q) + 2 * cq + 1;
  const int64_t ik = int64_t(n_k) + 2 * ck + 1;
  if (iq >= (int64_t(1) << 31) || ik >= (int64_t(1) << 31))
    return set_error(NGT_ERR_UNSUPPORTED, "ngt_csr_sizes: work list exceeds int32");
  if (max_items_q) *max_items_q = int32_t(iq);
  if (max_items_k) *max_items_k = int32_t(ik);
  if (max_splits_q) *max_splits_q = int32_t((cq < n_q ? cq : n_q) + 1);
  if (max_splits_k) *max_splits_k = int32_t((ck < n_k ? ck : n_k) + 1);
  return NGT_OK;
}

extern "C" int ngt_csr_workspace_bytes(int64_t n_edges, int32_t n_q, int32_t n_k, size_t* bytes) {
  if (!bytes) return set_error(NGT_ERR_ARG, "ngt_csr_workspace_bytes: null output");
  CsrLayout L;
  const int rc = csr_layout(n_edges, n_q, n_k, &L);
  if (rc != NGT_OK) return rc;
  *bytes = L.total;
  return NGT_OK;
}

extern "C" int ngt_csr_build(const int64_t* edge_index, ngt_window_csr* csr, void* workspace,
                             size_t workspace_bytes, void* stream) {
  if (!csr) return set_error(NGT_ERR_ARG, "ngt_csr_build: null csr");
  const int64_t E = csr->n_edges;
  const int32_t n_q = csr->n_q, n_k = csr->n_k;
  if (E < 0 || n_q < 0 || n_k < 0 || csr->chunk_q <= 0 || csr->chunk_k <= 0 ||
      csr->small_q < NGT_SMALL_FROM_DEGREES || csr->small_k < NGT_SMALL_FROM_DEGREES ||
      csr->small_q >= csr->chunk_q || csr->small_k >= csr->chunk_k)
    return set_error(NGT_ERR_ARG,
                     "ngt_csr_build: bad sizes (need 0 <= small < chunk, or small = "
                     "NGT_SMALL_FROM_DEGREES)");
  if (E > 0 && (!edge_index || n_q == 0 || n_k == 0))
    return set_error(NGT_ERR_ARG, "ngt_csr_build: edges given for an empty window");
  if (!csr->rowptr || !csr->t_rowptr || !csr->info || !csr->items_q || !csr->items_k ||
      !csr->splits_q || !csr->splits_k || (n_q > 0 && !csr->packed_q) ||
      (n_k > 0 && !csr->packed_k) || (E > 0 && (!csr->col || !csr->perm || !csr->t_col ||
                                                     !csr->t_perm || !csr->q2t)))
    return set_error(NGT_ERR_ARG, "ngt_csr_build: null output array");
  int32_t miq, msq, mik, msk;
  int rc = ngt_csr_sizes(E, n_q, n_k, csr->chunk_q, csr->chunk_k, &miq, &msq, &mik, &msk);
  if (rc != NGT_OK) return rc;
  if (csr->max_items_q < miq || csr->max_items_k < mik || csr->max_splits_q < msq ||
      csr->max_splits_k < msk)
    return set_error(NGT_ERR_ARG, "ngt_csr_build: work-list arrays smaller than ngt_csr_sizes");
  CsrLayout L;
  rc = csr_layout(E, n_q, n_k, &L);
  if (rc != NGT_OK) return rc;
  if (!workspace || workspace_bytes < L.total)
    return set_error(NGT_ERR_WORKSPACE, "ngt_csr_build: workspace %zu < %zu bytes",
                     workspace_bytes, L.total);

  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  uint32_t* src32 = reinterpret_cast<uint32_t*>(ws + L.src32);
  uint32_t* dst32 = reinterpret_cast<uint32_t*>(ws + L.dst32);
  uint32_t* key_a = reinterpret_cast<uint32_t*>(ws + L.key_a);
  uint32_t* key_b = reinterpret_cast<uint32_t*>(ws + L.key_b);
  uint32_t* key_c = reinterpret_cast<uint32_t*>(ws + L.key_c);
  int32_t* val_a = reinterpret_cast<int32_t*>(ws + L.val_a);
  int32_t* val_b = reinterpret_cast<int32_t*>(ws + L.val_b);

  hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, st, csr->info, NGT_INFO_LEN);
  NGT_HIP_CHECK(hipGetLastError());
  auto sort = [&](uint32_t* key_in, uint32_t* key_out, int32_t* val_in, int32_t* val_out,
                  unsigned bits) -> int {
    return sort_edges(ws + L.temp, L.temp_bytes, key_in, key_out, val_in, val_out, E, bits, st);
  };
  const unsigned bits_q = bits_for(uint64_t(n_q)), bits_k = bits_for(uint64_t(n_k));  // 0 .. n
  const unsigned src_bits = bits_q + bits_k <= 32u ? bits_k : 0u;  // one combined key
  if (E > 0) {
    hipLaunchKernelGGL(k_endpoints, dim3(grid_for(E)), dim3(kBlock), 0, st, edge_index,
                       edge_index + E, E, n_q, n_k, src_bits, src32, src_bits ? nullptr : dst32,
                       val_a, csr->info);
    NGT_HIP_CHECK(hipGetLastError());
    // key_b: dst (above the src_bits of src), query-major
    if (src_bits) {
      NGT_CHECK_OK(sort(src32, key_b, val_a, csr->perm, bits_q + bits_k));
    } else {
      NGT_CHECK_OK(sort(src32, key_a, val_a, val_b, bits_k));  // val_b: edge ids by src
      hipLaunchKernelGGL(k_gather_u32, dim3(grid_for(E)), dim3(kBlock), 0, st, dst32, val_b, E,
                         key_a);
      NGT_HIP_CHECK(hipGetLastError());
      NGT_CHECK_OK(sort(key_a, key_b, val_b, csr->perm, bits_q));
    }
  }
  hipLaunchKernelGGL(k_rows_q, dim3(grid_for(E + 1)), dim3(kBlock), 0, st, key_b, csr->perm, src32,
                     src_bits, E, n_q, n_k, csr->rowptr, csr->col, key_a, val_a);
  NGT_HIP_CHECK(hipGetLastError());
  if (E > 0) NGT_CHECK_OK(sort(key_a, key_c, val_a, val_b, bits_k));  // key_c: src, key-major
  hipLaunchKernelGGL(k_rows_k, dim3(grid_for(E + 1)), dim3(kBlock), 0, st, key_c, val_b, csr->perm,
                     key_b, src_bits, E, n_q, n_k, csr->t_rowptr, csr->t_col, csr->t_perm, csr->q2t);
  NGT_HIP_CHECK(hipGetLastError());
  if (E > 0) {
    hipLaunchKernelGGL(k_ends, dim3(1), dim3(64), 0, st, key_b, src_bits, key_c, csr->rowptr,
                       n_q, csr->info);
    NGT_HIP_CHECK(hipGetLastError());
  }
  const int32_t n_own = n_q < n_k ? n_q : n_k;  // the window's own key rows
  const bool all_keys = n_own == n_k;
  const Sides sides{{
      {csr->rowptr, n_q, csr->chunk_q, csr->small_q, 0, reinterpret_cast<int4*>(csr->items_q),
       reinterpret_cast<int4*>(csr->splits_q), csr->packed_q, csr->order_q, NGT_INFO_ITEMS_Q,
       NGT_INFO_PACKED_Q, NGT_INFO_SMALL_Q, NGT_INFO_MAX_DEG_Q},
      {csr->t_rowptr, n_k, csr->chunk_k, csr->small_k, n_q, reinterpret_cast<int4*>(csr->items_k),
       reinterpret_cast<int4*>(csr->splits_k), csr->packed_k, all_keys ? csr->order_k : nullptr,
       NGT_INFO_ITEMS_K, NGT_INFO_PACKED_K, NGT_INFO_SMALL_K, NGT_INFO_MAX_DEG_K}}};
  return build_worklists(sides, all_keys ? nullptr : csr->order_k, n_own, csr->info, ws, L, st);
}
