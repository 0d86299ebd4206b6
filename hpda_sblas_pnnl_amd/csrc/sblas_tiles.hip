// sblas_tiles.hip -- tile kernels whose work per launch block is fixed in
// advance whatever the row lengths: merge-path CSR (the reference's kernel
// 2, cusparseDcsrmv_mp at src/dspmv_mgpu_v1.cu:267 / src/dspmv_mgpu_v2.cu:457)
// and the COO segmented reduction that consumes row-sorted COO directly (the
// reference converts COO to CSR first, src/dspmv_mgpu_baseline_coo.cu:146-165,
// src/dspmv_mgpu_v1_numa_coo.cu:460-476).
//
// Both write y directly for rows that lie inside one tile and leave, per tile,
// the partial of a row that began in an earlier tile (head) and of a row that
// continues into the next tile (tail).  k_tile_fixup then adds those partials
// in tile order, so every row's sum has a fixed order: no atomics on y.
#include <climits>
#include <mutex>
#include <string>

#include "internal.hpp"
#include "rows_device.hpp"
#include "span_device.hpp"

namespace sblas {
namespace {

__device__ __forceinline__ double tload_val(const double *p, int j) {
  return __builtin_nontemporal_load(p + j);
}
__device__ __forceinline__ double tload_val(const float *p, int j) {
  return static_cast<double>(__builtin_nontemporal_load(p + j));
}
__device__ __forceinline__ double tload_val(const uint16_t *p, int j) {
  const uint32_t h = __builtin_nontemporal_load(p + j);
  return static_cast<double>(__uint_as_float(h << 16));
}

__device__ __forceinline__ double axpby(double alpha, double s, double beta, double yv) {
  return (beta == 0.0) ? alpha * s : alpha * s + beta * yv;
}

// Tile this workgroup takes, -1 for none: each XCD takes a contiguous eighth of
// the tiles (the grid is a multiple of 8), so neighbouring rows meet in one L2
// (banded, 400,009 rows of 140, merge path: 415 us with tiles dealt to the
// XCDs in turn).
__device__ __forceinline__ int tile_of_block(int tiles) { return rows::logical_block(tiles, 1); }

// Products of elements [j0, j0 + ne) into LDS in span order, consecutive
// threads on consecutive elements: every load of values and columns, then the
// x gathers, then the products, each step called once the loads that do not
// depend on it are issued.  Threads past the tile re-read its last element, so
// no load sits under a divergent branch.
template <typename VT>
struct Elements {
  double v[kTileItems];
  int c[kTileItems];
  double xv[kTileItems];
  __device__ __forceinline__ void load(int j0, int ne, const int *__restrict__ col,
                                       const VT *__restrict__ val) {
#pragma unroll
    for (int k = 0; k < kTileItems; k++) {
      const int e = j0 + min(static_cast<int>(threadIdx.x) + k * kTileBlock, ne - 1);
      v[k] = tload_val(val, e);
      c[k] = __builtin_nontemporal_load(col + e);
    }
  }
  __device__ __forceinline__ void gather(const double *__restrict__ x) {
#pragma unroll
    for (int k = 0; k < kTileItems; k++) xv[k] = x[c[k]];
  }
  __device__ __forceinline__ void stage(span::Shared<kTileItems> &sh) {
#pragma unroll
    for (int k = 0; k < kTileItems; k++)
      sh.prod[span::pos<kTileItems>(threadIdx.x + k * kTileBlock)] = v[k] * xv[k];
  }
};

// ---------------------------------------------------------------------------
// merge path (Merrill & Garland, SC'16): the m row ends and nnz elements are
// merged into one list of m + nnz items; tile b owns items [b*T, (b+1)*T).
// A row belongs to the tile holding its row-end item.
//
// The tiles' first rows depend on the row pointers alone: they are found once
// per plan (by the allocation-free form once per call) by one wave a tile that
// probes 64 places a step, and a product starts from one load where it used to
// start from a binary search of up to 22 dependent ones.  Row ends are kept as
// 16-bit offsets in LDS and rows summed by spans (span_device.hpp): 22.8 KB a
// workgroup, seven a CU, where products, sums and a search took 33 KB and four.
// What is left is the x gathers (one L2 request an element).  us before ->
// now, FP64: power law 1,000,003 rows 212 -> 168 (x misses L2), R-MAT scale 20
// 205 -> 99, banded 100,000 rows of 140 90 -> 52, power law 20,000 rows 13.9 ->
// 10.1.
// ---------------------------------------------------------------------------

// carry[b].row0 = number of row ends among the first b*T merge items.  The
// predicate "row end p comes before diagonal d" holds for a prefix of the
// rows; each step keeps the 64th of the range where it stops holding.
__global__ void k_merge_rows(int m, int nnz, int tiles, const int *__restrict__ rp,
                             TileCarry *__restrict__ carry) {
  const int b = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (b >= tiles) return;  // uniform per wave
  const int lane = threadIdx.x & 63;
  const int64_t d = static_cast<int64_t>(b) * kTileSize;
  int lo = static_cast<int>(max<int64_t>(0, d - nnz));
  int hi = static_cast<int>(min<int64_t>(d, m));
  while (lo < hi) {
    const int step = (hi - lo - 1) / 64 + 1;
    const int64_t p = lo + static_cast<int64_t>(lane) * step;
    const bool before = p < hi && static_cast<int64_t>(rp[p + 1]) <= d - p - 1;
    const int c = __popcll(__ballot(before));
    if (c == 0) {
      hi = lo;
    } else {
      hi = static_cast<int>(min<int64_t>(hi, lo + static_cast<int64_t>(c) * step));
      lo += (c - 1) * step + 1;
    }
  }
  if (lane == 0) carry[b].row0 = lo;
}

template <typename VT, bool BETA>
__global__ __launch_bounds__(kTileBlock) void k_csr_merge_path(
    int m, int nnz, int tiles, const int *__restrict__ rp, const int *__restrict__ col,
    const VT *__restrict__ val, const double *__restrict__ x, double *__restrict__ y,
    double alpha, double beta, TileCarry *__restrict__ carry) {
  constexpr int B = kTileBlock, T = kTileSize;
  __shared__ span::Shared<kTileItems> sh;
  __shared__ uint16_t rend[T + 1];  // end of each row in the tile, from its first element
  const int b = tile_of_block(tiles);
  if (b < 0) return;
  const int t = threadIdx.x;
  const int64_t total = static_cast<int64_t>(m) + nnz;
  const int64_t d0 = static_cast<int64_t>(b) * T, d1 = min<int64_t>(d0 + T, total);
  const int i0 = carry[b].row0, i1 = b + 1 < tiles ? carry[b + 1].row0 : m;
  const int j0 = static_cast<int>(d0 - i0), j1 = static_cast<int>(d1 - i1);
  const int ne = j1 - j0;
  // rows [i0, i1) end in this tile; row i1 (if any) may have elements in it
  const int nrows = i1 - i0 + (i1 < m ? 1 : 0);
  span::clear_ends(sh);
  Elements<VT> el;
  if (ne > 0) el.load(j0, ne, col, val);
  // the thread's first row ahead of the gathers (most tiles have fewer rows
  // than threads)
  const int ic = i0 + min(t, max(nrows - 1, 0));
  const int rs0 = rp[ic], re0 = nrows > 0 ? rp[ic + 1] : 0;
  const bool started_before = i0 < m && rp[i0] < j0;
  double y0 = 0.0;
  if (BETA && t < i1 - i0) y0 = y[i0 + t];
  __syncthreads();
  if (ne > 0) el.gather(x);
  auto put_row = [&](int i, int rs, int re) {
    const int e = min(re, j1) - j0, s = max(rs, j0) - j0;
    rend[i] = static_cast<uint16_t>(e);
    if (e > s) span::mark_end(sh, e - 1);
  };
  if (t < nrows) put_row(t, rs0, re0);
  for (int i = t + B; i < nrows; i += B) put_row(i, rp[i0 + i], rp[i0 + i + 1]);
  if (ne > 0) el.stage(sh);
  __syncthreads();
  span::row_sums(sh);

  auto sum = [&](int i) {
    const int e = rend[i], s = i > 0 ? rend[i - 1] : 0;
    return e > s ? sh.prod[span::pos<kTileItems>(e - 1)] : 0.0;
  };
  for (int i = t; i < i1 - i0; i += B) {
    if (i == 0 && started_before) continue;  // completed by the fix-up
    const double s = sum(i);
    const double old = BETA ? (i == t ? y0 : y[i0 + i]) : 0.0;
    y[i0 + i] = BETA ? alpha * s + beta * old : alpha * s;
  }
  if (t == 0) {
    // i0 == i1: no row ends here, the tile lies inside row i0 or begins it
    const bool inside = i0 == i1 && started_before;
    const bool head = started_before;
    const bool tail = !inside && i1 < m && rend[i1 - i0] > (i1 > i0 ? rend[i1 - i0 - 1] : 0);
    TileCarry &cy = carry[b];
    cy.spanning = inside ? 1 : 0;
    cy.head = head ? sum(0) : 0.0;
    cy.head_row = head ? i0 : -1;
    cy.tail = tail ? sum(i1 - i0) : 0.0;
    cy.tail_row = tail ? i1 : -1;
  }
}

// ---------------------------------------------------------------------------
// COO segmented reduction: tile b owns elements [b*T, (b+1)*T) of the
// row-sorted arrays.  An element whose successor has another row id (or that
// ends the tile) closes a segment; spans of elements are summed between those
// marks, so the cost follows the number of elements, not the span of row ids.
// Each thread holds its elements' row ids and their successors', so the marks
// are one ballot per 64 elements and the ids take no LDS.  (us before -> now:
// power law 1,000,003 rows 226 -> 180, R-MAT scale 20 210 -> 122, banded 100,000
// rows of 140 107 -> 67.)  Rows with no element are written (beta*y) by the segment just before them, or by the tile
// whose first element follows them; rows after the last element by the last
// tile.
// ---------------------------------------------------------------------------

// y = beta*y for the rows [a, b) without elements; a run of more than eight
// is left to the whole wave.  Every lane of the wave calls it.
template <bool BETA>
__device__ __forceinline__ void empty_rows(int a, int b, double *__restrict__ y, double alpha,
                                           double beta) {
  const bool many = b - a > 8;
  if (!many)
    for (int q = a; q < b; q++) y[q] = axpby(alpha, 0.0, beta, BETA ? y[q] : 0.0);
  uint64_t mask = __ballot(many);
  while (mask) {
    const int l = __ffsll(static_cast<unsigned long long>(mask)) - 1;
    mask &= mask - 1;
    const int qa = __shfl(a, l, 64), qb = __shfl(b, l, 64);
    for (int q = qa + (static_cast<int>(threadIdx.x) & 63); q < qb; q += 64)
      y[q] = axpby(alpha, 0.0, beta, BETA ? y[q] : 0.0);
  }
}

template <typename VT, bool BETA>
__global__ __launch_bounds__(kTileBlock) void k_coo_tiles(
    int m, int nnz, int tiles, const int *__restrict__ ri, const int *__restrict__ ci,
    const VT *__restrict__ val, const double *__restrict__ x, double *__restrict__ y,
    double alpha, double beta, TileCarry *__restrict__ carry) {
  constexpr int B = kTileBlock, T = kTileSize;
  __shared__ span::Shared<kTileItems> sh;
  const int b = tile_of_block(tiles);
  if (b < 0) return;
  const int t = threadIdx.x;
  const int j0 = b * T;
  const int j1 = min(j0 + T, nnz);
  const int ne = j1 - j0;
  Elements<VT> el;
  el.load(j0, ne, ci, val);
  // row ids of the thread's elements and of their successors: the next lane's,
  // for a wave's last lane one scalar load
  int r[kTileItems], next[kTileItems], after[kTileItems];
  const int wave_end = (__builtin_amdgcn_readfirstlane(t >> 6) + 1) * 64;
#pragma unroll
  for (int k = 0; k < kTileItems; k++) {
    r[k] = __builtin_nontemporal_load(ri + j0 + min(t + k * B, ne - 1));
    after[k] = ri[j0 + min(wave_end + k * B, ne - 1)];
  }
  const int r_first = ri[j0], r_last = ri[j1 - 1];
  const int r_before = j0 > 0 ? ri[j0 - 1] : -1;
  const bool head = r_before == r_first;
  const bool tail = j1 < nnz && ri[j1] == r_last;
#pragma unroll
  for (int k = 0; k < kTileItems; k++) {
    const int e = t + k * B;
    const int down = __shfl_down(r[k], 1, 64);
    next[k] = (t & 63) == 63 ? after[k] : down;
    const uint64_t m64 = __ballot(e == ne - 1 || (e < ne && r[k] != next[k]));
    if ((t & 63) == 0) {
      sh.ends[e >> 5] = static_cast<uint32_t>(m64);
      sh.ends[(e >> 5) + 1] = static_cast<uint32_t>(m64 >> 32);
    }
  }
  el.gather(x);
  el.stage(sh);
  __syncthreads();
  span::row_sums(sh);

  // rows without elements before this tile's first row (and after the last
  // element for the last tile)
  for (int q = r_before + 1 + t; q < r_first; q += B)
    y[q] = axpby(alpha, 0.0, beta, BETA ? y[q] : 0.0);
  if (b == tiles - 1)
    for (int q = r_last + 1 + t; q < m; q += B)
      y[q] = axpby(alpha, 0.0, beta, BETA ? y[q] : 0.0);
  // y of the thread's segments all at once, ahead of the stores
  double old[BETA ? kTileItems : 1];
  if constexpr (BETA) {
#pragma unroll
    for (int k = 0; k < kTileItems; k++) {
      const int e = t + k * B;
      old[k] = e == ne - 1 || (e < ne && r[k] != next[k]) ? y[r[k]] : 0.0;
    }
  }
#pragma unroll
  for (int k = 0; k < kTileItems; k++) {
    const int e = t + k * B;
    const bool last = e == ne - 1, end = last || (e < ne && r[k] != next[k]);
    if (end) {
      const double s = sh.prod[span::pos<kTileItems>(e)];
      if (r[k] == r_first && head) {
        carry[b].head = s;
      } else if (last && tail) {
        carry[b].tail = s;
      } else {
        y[r[k]] = axpby(alpha, s, beta, BETA ? old[BETA ? k : 0] : 0.0);
      }
    }
    const bool gap = end && !last;  // rows up to the next segment's
    empty_rows<BETA>(gap ? r[k] + 1 : 0, gap ? next[k] : 0, y, alpha, beta);
  }
  if (t == 0) {
    const bool spanning = r_first == r_last && head && tail;
    carry[b].spanning = spanning ? 1 : 0;
    carry[b].head_row = head ? r_first : -1;
    carry[b].tail_row = tail && !(r_first == r_last && head) ? r_last : -1;
  }
}

// Rows cut by tile edges (span::close_cut_row), one thread per tile.
__global__ void k_tile_fixup(int tiles, const TileCarry *__restrict__ carry,
                             double *__restrict__ y, double alpha, double beta) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < tiles) span::close_cut_row(b, tiles, carry, y, alpha, beta);
}

// Host-side dispatch helpers ---------------------------------------------------

template <typename VT>
int mp_launch(int m, int64_t nnz, int tiles, const int *rp, const int *col, const VT *val,
              const double *x, double *y, double alpha, double beta, TileCarry *carry,
              hipStream_t s) {
  const dim3 grid((tiles + 7) / 8 * 8), block(kTileBlock);
  if (beta != 0.0)
    hipLaunchKernelGGL((k_csr_merge_path<VT, true>), grid, block, 0, s, m, static_cast<int>(nnz),
                       tiles, rp, col, val, x, y, alpha, beta, carry);
  else
    hipLaunchKernelGGL((k_csr_merge_path<VT, false>), grid, block, 0, s, m, static_cast<int>(nnz),
                       tiles, rp, col, val, x, y, alpha, beta, carry);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT>
int coo_launch(int m, int64_t nnz, int tiles, const int *ri, const int *ci, const VT *val,
               const double *x, double *y, double alpha, double beta, TileCarry *carry,
               hipStream_t s) {
  const dim3 grid((tiles + 7) / 8 * 8), block(kTileBlock);
  if (beta != 0.0)
    hipLaunchKernelGGL((k_coo_tiles<VT, true>), grid, block, 0, s, m, static_cast<int>(nnz), tiles,
                       ri, ci, val, x, y, alpha, beta, carry);
  else
    hipLaunchKernelGGL((k_coo_tiles<VT, false>), grid, block, 0, s, m, static_cast<int>(nnz),
                       tiles, ri, ci, val, x, y, alpha, beta, carry);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

}  // namespace

int launch_merge_rows(int m, int64_t nnz, int tiles, const int *rp, TileCarry *carry,
                      hipStream_t s) {
  if (tiles <= 0) return SBLAS_OK;
  hipLaunchKernelGGL(k_merge_rows, dim3((tiles + 3) / 4), dim3(256), 0, s, m,
                     static_cast<int>(nnz), tiles, rp, carry);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

int launch_csr_merge_path(int val_type, int m, int64_t nnz, int tiles, const int *rp,
                          const int *col, const void *val, const double *x, double *y,
                          double alpha, double beta, TileCarry *carry, hipStream_t s) {
  if (tiles <= 0) return SBLAS_OK;
  switch (val_type) {
    case SBLAS_VAL_F64:
      return mp_launch(m, nnz, tiles, rp, col, static_cast<const double *>(val), x, y, alpha, beta,
                       carry, s);
    case SBLAS_VAL_F32:
      return mp_launch(m, nnz, tiles, rp, col, static_cast<const float *>(val), x, y, alpha, beta,
                       carry, s);
    case SBLAS_VAL_BF16:
      return mp_launch(m, nnz, tiles, rp, col, static_cast<const uint16_t *>(val), x, y, alpha,
                       beta, carry, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

int launch_coo_tiles(int val_type, int m, int64_t nnz, int tiles, const int *row_idx,
                     const int *col_idx, const void *val, const double *x, double *y,
                     double alpha, double beta, TileCarry *carry, hipStream_t s) {
  if (tiles <= 0) return SBLAS_OK;
  switch (val_type) {
    case SBLAS_VAL_F64:
      return coo_launch(m, nnz, tiles, row_idx, col_idx, static_cast<const double *>(val), x, y,
                        alpha, beta, carry, s);
    case SBLAS_VAL_F32:
      return coo_launch(m, nnz, tiles, row_idx, col_idx, static_cast<const float *>(val), x, y,
                        alpha, beta, carry, s);
    case SBLAS_VAL_BF16:
      return coo_launch(m, nnz, tiles, row_idx, col_idx, static_cast<const uint16_t *>(val), x, y,
                        alpha, beta, carry, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

int launch_tile_fixup(int tiles, const TileCarry *carry, double *y, double alpha, double beta,
                      hipStream_t s) {
  if (tiles <= 0) return SBLAS_OK;
  hipLaunchKernelGGL(k_tile_fixup, dim3((tiles + 255) / 256), dim3(256), 0, s, tiles, carry, y,
                     alpha, beta);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

}  // namespace sblas

// ---------------------------------------------------------------------------
// Merge-path SpMV that allocates nothing: the tiles' first rows (k_merge_rows,
// which a plan runs once), then the same two launches as a kernel-2 plan
// (k_csr_merge_path, k_tile_fixup), with the per-tile carries in a file-scope
// device array instead of a plan's workspace.  Every tile writes its carry on
// every call before the fix-up reads it, so nothing needs clearing between
// calls.  One array per GPU, shared by every call on that
// GPU: calls that overlap on one GPU race.
// ---------------------------------------------------------------------------
namespace sblas {
namespace {

constexpr int kNoAllocTiles = 262144;  // 8 MiB of carries: m + nnz <= 2^29 merge items
constexpr int kNoAllocDevices = 64;

static __device__ __align__(256) TileCarry scratch[kNoAllocTiles];

// Device address of `scratch` on each GPU, looked up once per device with
// that device current (each GPU holds its own copy of the array).
struct ScratchAddress {
  std::once_flag once;
  TileCarry *ptr = nullptr;
  hipError_t status = hipSuccess;
};
ScratchAddress g_scratch[kNoAllocDevices];

int scratch_for_current_device(TileCarry **out) {
  int dev = -1;
  SBLAS_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kNoAllocDevices) {
    set_error(SBLAS_ERR_UNSUPPORTED, "spmv noalloc: device index beyond the scratch table");
    return SBLAS_ERR_UNSUPPORTED;
  }
  ScratchAddress &a = g_scratch[dev];
  std::call_once(a.once, [&a] {
    void *p = nullptr;
    a.status = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    a.ptr = static_cast<TileCarry *>(p);
  });
  if (a.status != hipSuccess || !a.ptr) {
    set_error(SBLAS_ERR_HIP, std::string("spmv noalloc: hipGetSymbolAddress(scratch): ") +
                                 hipGetErrorString(a.status));
    return SBLAS_ERR_HIP;
  }
  *out = a.ptr;
  return SBLAS_OK;
}

}  // namespace
}  // namespace sblas

extern "C" int sblas_spmv_csr_noalloc(int m, int n, int64_t nnz, const int *d_row_ptr,
                                      const int *d_col, const void *d_val, int val_type,
                                      double alpha, const double *d_x, double beta, double *d_y,
                                      void *stream) {
  using namespace sblas;
  clear_error();
  if (m < 0 || n < 0 || nnz < 0 || nnz > INT_MAX - 4096 || (m > 0 && (!d_row_ptr || !d_y)) ||
      (nnz > 0 && (!d_col || !d_val || !d_x)) || val_type < SBLAS_VAL_F64 ||
      val_type > SBLAS_VAL_BF16) {
    set_error(SBLAS_ERR_ARGS, "spmv noalloc: invalid sizes, pointers or value type");
    return SBLAS_ERR_ARGS;
  }
  if (m == 0) return SBLAS_OK;
  const int64_t items = static_cast<int64_t>(m) + nnz;
  const int64_t tiles = (items + kTileSize - 1) / kTileSize;
  if (tiles > kNoAllocTiles) {
    set_error(SBLAS_ERR_ARGS, "spmv noalloc: m + nnz exceeds 2^29 (the scratch holds 262144 "
                              "tile carries of 2048 merge items)");
    return SBLAS_ERR_ARGS;
  }
  TileCarry *carry = nullptr;
  int st = scratch_for_current_device(&carry);
  if (st != SBLAS_OK) return st;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  st = launch_merge_rows(m, nnz, static_cast<int>(tiles), d_row_ptr, carry, s);
  if (st != SBLAS_OK) return st;
  st = launch_csr_merge_path(val_type, m, nnz, static_cast<int>(tiles), d_row_ptr, d_col, d_val,
                             d_x, d_y, alpha, beta, carry, s);
  if (st != SBLAS_OK) return st;
  return launch_tile_fixup(static_cast<int>(tiles), carry, d_y, alpha, beta, s);
}
