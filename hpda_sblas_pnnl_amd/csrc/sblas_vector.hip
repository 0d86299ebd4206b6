// sblas_vector.hip -- vector-CSR SpMV / SpMM for gfx950, the split-row merge
// and small helpers.
//
// Replaces the reference's kernel 1 (cusparseDcsrmv, call sites
// src/dspmv_mgpu_v1.cu:261, src/dspmv_mgpu_baseline.cu:125,
// src/dspmv_mgpu_v1_numa.cu:696) and its host merges
// (src/dspmv_mgpu_v1.cu:304-319, src/dspmv_mgpu_v2.cu:486-544).
//
// Design: a 64-lane wave is cut into sub-waves of SUBW lanes, one row per
// sub-wave at a time; SUBW follows the mean row length.  A launch block owns a
// contiguous run of rows of one chunk (rows_per_block), so consecutive blocks
// touch neighbouring parts of x; with xcd_remap the logical block order is
// re-dealt so that each XCD (blocks are dealt round-robin over the 8 XCDs)
// owns a contiguous 1/8 of the rows and keeps its own x window in its L2.
// Matrix values and column indices are streamed with non-temporal loads so
// they do not evict x from L2 / MALL.  Products and sums are FP64 for every
// stored value type.
#include "internal.hpp"
#include "rows_device.hpp"
#include "span_device.hpp"

namespace sblas {
namespace {

__device__ __forceinline__ double load_val(const double *p, int j) {
  return __builtin_nontemporal_load(p + j);
}
__device__ __forceinline__ double load_val(const float *p, int j) {
  return static_cast<double>(__builtin_nontemporal_load(p + j));
}
__device__ __forceinline__ double load_val(const uint16_t *p, int j) {
  const uint32_t h = __builtin_nontemporal_load(p + j);
  return static_cast<double>(__uint_as_float(h << 16));
}
__device__ __forceinline__ int load_col(const int *p, int j) {
  return __builtin_nontemporal_load(p + j);
}

// Sum over the SUBW lanes of each aligned sub-wave (xor butterfly).
template <int SUBW>
__device__ __forceinline__ double subwave_sum(double v) {
#pragma unroll
  for (int off = SUBW / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, SUBW);
  return v;
}

using rows::logical_block;

__device__ __forceinline__ int chunk_of_block(const DevChunk *chunks, int nchunks, int b) {
  int lo = 0, hi = nchunks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (chunks[mid].blk_begin <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <typename VT, int SUBW, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_csr_vector(
    const DevChunk *__restrict__ chunks, int nchunks, int rows_per_block, int total_blocks,
    int xcd_remap, const int *__restrict__ rp, const int *__restrict__ col,
    const VT *__restrict__ val, const double *__restrict__ x, double *__restrict__ y,
    double alpha, double beta, double *__restrict__ partials) {
  const int b = logical_block(total_blocks, xcd_remap);
  if (b < 0) return;
  const int c = nchunks > 1 ? chunk_of_block(chunks, nchunks, b) : 0;
  const DevChunk ch = chunks[c];
  constexpr int SUBS = BLOCK / SUBW;
  const int sub = threadIdx.x / SUBW;
  const int lane = threadIdx.x % SUBW;
  const int row0 = ch.row_begin + (b - ch.blk_begin) * rows_per_block;
  const int row1 = min(row0 + rows_per_block, ch.row_end);
  for (int r = row0 + sub; r < row1; r += SUBS) {
    const int rs = rp[r], re = rp[r + 1];
    const int s = max(rs, ch.lo), e = min(re, ch.hi);
    double sum = 0.0;
    int j = s + lane;
    // two independent accumulators keep two loads in flight per lane
    double sum2 = 0.0;
    for (; j + SUBW < e; j += 2 * SUBW) {
      const double v0 = load_val(val, j);
      const int c0 = load_col(col, j);
      const double v1 = load_val(val, j + SUBW);
      const int c1 = load_col(col, j + SUBW);
      sum += v0 * x[c0];
      sum2 += v1 * x[c1];
    }
    if (j < e) sum += load_val(val, j) * x[load_col(col, j)];
    sum = subwave_sum<SUBW>(sum + sum2);
    if (lane == 0) {
      if (rs < ch.lo || re > ch.hi) {
        partials[2 * c + (r == ch.row_begin ? 0 : 1)] = sum;
      } else {
        y[r] = (beta == 0.0) ? alpha * sum : alpha * sum + beta * y[r];
      }
    }
  }
}

// k right-hand sides, X row-major (n x K), Y row-major (m x K).  Lane l of a
// sub-wave handles vector l % K and every (SUBW/K)-th element of the row, so
// K neighbouring lanes read one contiguous K*8-byte row of X.
template <typename VT, int SUBW, int K, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_csr_vector_mrhs(
    const DevChunk *__restrict__ chunks, int nchunks, int rows_per_block, int total_blocks,
    int xcd_remap, const int *__restrict__ rp, const int *__restrict__ col,
    const VT *__restrict__ val, const double *__restrict__ X, double *__restrict__ Y,
    double alpha, double beta, double *__restrict__ partials) {
  static_assert(SUBW >= K, "sub-wave narrower than K");
  const int b = logical_block(total_blocks, xcd_remap);
  if (b < 0) return;
  const int c = nchunks > 1 ? chunk_of_block(chunks, nchunks, b) : 0;
  const DevChunk ch = chunks[c];
  constexpr int SUBS = BLOCK / SUBW;
  constexpr int STEP = SUBW / K;
  const int sub = threadIdx.x / SUBW;
  const int lane = threadIdx.x % SUBW;
  const int vec = lane % K;
  const int grp = lane / K;
  const int row0 = ch.row_begin + (b - ch.blk_begin) * rows_per_block;
  const int row1 = min(row0 + rows_per_block, ch.row_end);
  for (int r = row0 + sub; r < row1; r += SUBS) {
    const int rs = rp[r], re = rp[r + 1];
    const int s = max(rs, ch.lo), e = min(re, ch.hi);
    double sum = 0.0;
    for (int j = s + grp; j < e; j += STEP) {
      const double v = load_val(val, j);
      const int cc = load_col(col, j);
      sum += v * X[static_cast<int64_t>(cc) * K + vec];
    }
#pragma unroll
    for (int off = SUBW / 2; off >= K; off >>= 1) sum += __shfl_xor(sum, off, SUBW);
    if (grp == 0) {
      if (rs < ch.lo || re > ch.hi) {
        partials[(2 * c + (r == ch.row_begin ? 0 : 1)) * K + vec] = sum;
      } else {
        double *yp = Y + static_cast<int64_t>(r) * K + vec;
        *yp = (beta == 0.0) ? alpha * sum : alpha * sum + beta * (*yp);
      }
    }
  }
}

// Row blocks.  Phase 1 issues every global load the block needs that does not
// depend on another: ITEMS values and columns per thread (consecutive threads
// on consecutive elements, so each load instruction of a wave covers whole
// cache lines), the bounds of the thread's rows and, with beta != 0, their y;
// then the x gathers, whose products go to LDS.  Phase 2 sums the rows by
// spans of elements (span_device.hpp).  Phase 3 writes y, consecutive threads
// on consecutive rows, from bounds that are still in registers.  XT float: x
// gathered from its FP32 copy (narrow values: half the bytes per gather and per
// cached line of x; an FP32 value times an FP32 x is exact in FP64, so x's
// rounding is the only one added).
//
// What bounds it: the x gathers, one L2 request an element (about 2.1e11 a
// second on this GPU), and on small matrices the chain of dependent loads.
// Against the form that gave each row a group of lanes, with the sums in an
// LDS array of their own (28 KB of LDS, 5 workgroups a CU; now 18.7 KB and 8),
// us before -> now, FP64: power law 20,000 rows 8.0 -> 6.9, 200,000 rows 25.5
// -> 22.3; R-MAT 30,000 rows 14.2 -> 10.1, 300,000 rows 38.6 -> 31.5, scale 22
// over column segments 463 -> 442; banded 100,000 rows of 140 56.6 -> 42.7.
template <typename VT, int ITEMS, bool BETA, typename XT>
__global__ __launch_bounds__(span::kBlock) void k_csr_stream(
    const RowBlock *__restrict__ blocks, int nblocks, int xcd_remap,
    const int *__restrict__ rp, const int *__restrict__ col, const VT *__restrict__ val,
    const XT *__restrict__ x, double *__restrict__ y, double alpha, double beta,
    double *__restrict__ partials) {
  constexpr int B = span::kBlock;
  constexpr int RPT = kStreamRowsMax / B;  // rows per thread
  __shared__ span::Shared<ITEMS> sh;
  const int b = logical_block(nblocks, xcd_remap);
  if (b < 0) return;
  const RowBlock rb = blocks[b];
  const int lo = rb.lo, hi = rb.hi;
  const int t = threadIdx.x;
  const int r0 = rb.row_begin, nrows = rb.row_end - rb.row_begin;
  span::clear_ends(sh);

  // phase 1.  Threads past the window re-read its last element (same cache
  // line), so no load sits under a divergent branch.
  double v[ITEMS];
  int c[ITEMS];
  if (hi > lo) {
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const int e = min(lo + t + k * B, hi - 1);
      v[k] = load_val(val, e);
      c[k] = load_col(col, e);
    }
  }
  int rs[RPT], re[RPT];
  double yv[BETA ? RPT : 1];
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    if (k == 0 || k * B < nrows) {
      const int r = r0 + min(t + k * B, nrows - 1);
      rs[k] = rp[r];
      re[k] = rp[r + 1];
      if constexpr (BETA) yv[k] = y[r];
    }
  }
  __syncthreads();
  if (hi > lo) {
    XT xv[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) xv[k] = x[c[k]];
#pragma unroll
    for (int k = 0; k < RPT; k++)
      if (t + k * B < nrows && min(re[k], hi) > max(rs[k], lo))
        span::mark_end(sh, min(re[k], hi) - 1 - lo);
#pragma unroll
    for (int k = 0; k < ITEMS; k++)
      sh.prod[span::pos<ITEMS>(t + k * B)] = v[k] * static_cast<double>(xv[k]);
  }
  __syncthreads();

  // phase 2
  span::row_sums(sh);

  // phase 3: y for whole rows, partials for rows cut by the window
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = t + k * B;
    if (i < nrows) {
      const int e = min(re[k], hi);
      const double s = e > max(rs[k], lo) ? sh.prod[span::pos<ITEMS>(e - 1 - lo)] : 0.0;
      if ((i == 0 || i == nrows - 1) && (rs[k] < lo || re[k] > hi)) {
        partials[2 * b + (i == 0 ? 0 : 1)] = s;
      } else {
        y[r0 + i] = BETA ? alpha * s + beta * yv[BETA ? k : 0] : alpha * s;
      }
    }
  }
}

// Split rows: y[row] = alpha * (partials of the row in chunk order) + beta*y.
__global__ void k_merge(const int *__restrict__ rows, const int *__restrict__ ptr,
                        const int *__restrict__ slots, int groups,
                        const double *__restrict__ partials, int k, double *__restrict__ y,
                        double alpha, double beta) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = t / k, v = t % k;
  if (g >= groups) return;
  double s = 0.0;
  for (int q = ptr[g]; q < ptr[g + 1]; q++) s += partials[slots[q] * k + v];
  double *yp = y + static_cast<int64_t>(rows[g]) * k + v;
  *yp = (beta == 0.0) ? alpha * s : alpha * s + beta * (*yp);
}

// Index validation at plan time: flag[0] = 1 when some a[i] is outside
// [lo, hi) or, with `sorted`, a[i] > a[i+1].  Every offending thread stores
// the same value.
__global__ void k_check_indices(int64_t count, const int *__restrict__ a, int lo, int hi,
                                int sorted, int *__restrict__ flag) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int v = a[i];
  bool bad = v < lo || v >= hi;
  if (sorted && i + 1 < count) bad = bad || v > a[i + 1];
  if (bad) flag[0] = 1;
}

__global__ void k_scale(int64_t count, double beta, double *__restrict__ y) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < count) y[i] = (beta == 0.0) ? 0.0 : beta * y[i];
}

template <typename VT>
int launch_vector_typed(const VectorLaunch &L, const DevChunk *chunks, int nchunks,
                        const int *rp, const int *col, const VT *val, const double *x,
                        double *y, double alpha, double beta, double *partials,
                        hipStream_t s) {
  constexpr int B = 256;
  const dim3 grid(L.grid), block(B);
#define SBLAS_VEC_CASE(W)                                                                 \
  case W:                                                                                 \
    hipLaunchKernelGGL((k_csr_vector<VT, W, B>), grid, block, 0, s, chunks, nchunks,      \
                       L.rows_per_block, L.total_blocks, L.xcd_remap, rp, col, val, x, y, \
                       alpha, beta, partials);                                            \
    break;
  switch (L.subwave) {
    SBLAS_VEC_CASE(2)
    SBLAS_VEC_CASE(4)
    SBLAS_VEC_CASE(8)
    SBLAS_VEC_CASE(16)
    SBLAS_VEC_CASE(32)
    SBLAS_VEC_CASE(64)
    default:
      set_error(SBLAS_ERR_ARGS, "vector kernel: sub-wave must be a power of two in [2,64]");
      return SBLAS_ERR_ARGS;
  }
#undef SBLAS_VEC_CASE
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT, int K>
int launch_mrhs_k(const VectorLaunch &L, const DevChunk *chunks, int nchunks, const int *rp,
                  const int *col, const VT *val, const double *X, double *Y, double alpha,
                  double beta, double *partials, hipStream_t s) {
  constexpr int B = 256;
  const dim3 grid(L.grid), block(B);
  const int w = L.subwave < K ? K : L.subwave;
#define SBLAS_MRHS_CASE(W)                                                                 \
  case W:                                                                                  \
    if constexpr (W >= K)                                                                  \
      hipLaunchKernelGGL((k_csr_vector_mrhs<VT, W, K, B>), grid, block, 0, s, chunks,      \
                         nchunks, L.rows_per_block, L.total_blocks, L.xcd_remap, rp, col,  \
                         val, X, Y, alpha, beta, partials);                                \
    break;
  switch (w) {
    SBLAS_MRHS_CASE(2)
    SBLAS_MRHS_CASE(4)
    SBLAS_MRHS_CASE(8)
    SBLAS_MRHS_CASE(16)
    SBLAS_MRHS_CASE(32)
    SBLAS_MRHS_CASE(64)
    default:
      set_error(SBLAS_ERR_ARGS, "spmm kernel: bad sub-wave");
      return SBLAS_ERR_ARGS;
  }
#undef SBLAS_MRHS_CASE
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT>
int launch_mrhs_typed(int k, const VectorLaunch &L, const DevChunk *chunks, int nchunks,
                      const int *rp, const int *col, const VT *val, const double *X, double *Y,
                      double alpha, double beta, double *partials, hipStream_t s) {
  switch (k) {
    case 1: return launch_mrhs_k<VT, 1>(L, chunks, nchunks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 2: return launch_mrhs_k<VT, 2>(L, chunks, nchunks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 4: return launch_mrhs_k<VT, 4>(L, chunks, nchunks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 8: return launch_mrhs_k<VT, 8>(L, chunks, nchunks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 16: return launch_mrhs_k<VT, 16>(L, chunks, nchunks, rp, col, val, X, Y, alpha, beta, partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "spmm: k must be 1, 2, 4, 8 or 16");
      return SBLAS_ERR_ARGS;
  }
}

template <typename VT, int ITEMS, typename XT>
int launch_stream_items(const StreamLaunch &L, const RowBlock *blocks, const int *rp,
                        const int *col, const VT *val, const XT *x, double *y, double alpha,
                        double beta, double *partials, hipStream_t s) {
  const dim3 grid(L.grid), block(span::kBlock);
  if (beta != 0.0)
    hipLaunchKernelGGL((k_csr_stream<VT, ITEMS, true, XT>), grid, block, 0, s, blocks, L.nblocks,
                       L.xcd_remap, rp, col, val, x, y, alpha, beta, partials);
  else
    hipLaunchKernelGGL((k_csr_stream<VT, ITEMS, false, XT>), grid, block, 0, s, blocks, L.nblocks,
                       L.xcd_remap, rp, col, val, x, y, alpha, beta, partials);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT, typename XT>
int launch_stream_typed(const StreamLaunch &L, const RowBlock *blocks, const int *rp,
                        const int *col, const VT *val, const XT *x, double *y, double alpha,
                        double beta, double *partials, hipStream_t s) {
  switch (L.items) {
    case 8:
      return launch_stream_items<VT, 8>(L, blocks, rp, col, val, x, y, alpha, beta, partials, s);
    case 16:
      return launch_stream_items<VT, 16>(L, blocks, rp, col, val, x, y, alpha, beta, partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "stream kernel: items per thread must be 8 or 16");
      return SBLAS_ERR_ARGS;
  }
}

}  // namespace

int launch_csr_stream(int val_type, const StreamLaunch &L, const RowBlock *blocks,
                      const int *rp, const int *col, const void *val, const double *x,
                      double *y, double alpha, double beta, double *partials, hipStream_t s,
                      const float *x32) {
  if (L.grid <= 0) return SBLAS_OK;
  const float *v32 = static_cast<const float *>(val);
  const uint16_t *v16 = static_cast<const uint16_t *>(val);
  switch (val_type) {
    case SBLAS_VAL_F64:
      return launch_stream_typed(L, blocks, rp, col, static_cast<const double *>(val), x, y,
                                 alpha, beta, partials, s);
    case SBLAS_VAL_F32:
      return x32 ? launch_stream_typed(L, blocks, rp, col, v32, x32, y, alpha, beta, partials, s)
                 : launch_stream_typed(L, blocks, rp, col, v32, x, y, alpha, beta, partials, s);
    case SBLAS_VAL_BF16:
      return x32 ? launch_stream_typed(L, blocks, rp, col, v16, x32, y, alpha, beta, partials, s)
                 : launch_stream_typed(L, blocks, rp, col, v16, x, y, alpha, beta, partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

int launch_csr_vector(int val_type, const VectorLaunch &L, const DevChunk *chunks, int nchunks,
                      const int *rp, const int *col, const void *val, const double *x,
                      double *y, double alpha, double beta, double *partials,
                      hipStream_t s) {
  if (L.grid <= 0) return SBLAS_OK;
  switch (val_type) {
    case SBLAS_VAL_F64:
      return launch_vector_typed(L, chunks, nchunks, rp, col, static_cast<const double *>(val),
                                 x, y, alpha, beta, partials, s);
    case SBLAS_VAL_F32:
      return launch_vector_typed(L, chunks, nchunks, rp, col, static_cast<const float *>(val),
                                 x, y, alpha, beta, partials, s);
    case SBLAS_VAL_BF16:
      return launch_vector_typed(L, chunks, nchunks, rp, col,
                                 static_cast<const uint16_t *>(val), x, y, alpha, beta,
                                 partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

int launch_csr_vector_mrhs(int val_type, int k, const VectorLaunch &L, const DevChunk *chunks,
                           int nchunks, const int *rp, const int *col, const void *val,
                           const double *X, double *Y, double alpha, double beta,
                           double *partials, hipStream_t s) {
  if (L.grid <= 0) return SBLAS_OK;
  switch (val_type) {
    case SBLAS_VAL_F64:
      return launch_mrhs_typed(k, L, chunks, nchunks, rp, col, static_cast<const double *>(val),
                               X, Y, alpha, beta, partials, s);
    case SBLAS_VAL_F32:
      return launch_mrhs_typed(k, L, chunks, nchunks, rp, col, static_cast<const float *>(val),
                               X, Y, alpha, beta, partials, s);
    case SBLAS_VAL_BF16:
      return launch_mrhs_typed(k, L, chunks, nchunks, rp, col,
                               static_cast<const uint16_t *>(val), X, Y, alpha, beta,
                               partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

int launch_merge(const int *rows, const int *ptr, const int *slots, int groups,
                 const double *partials, int k, double *y, double alpha, double beta,
                 hipStream_t s) {
  if (groups <= 0) return SBLAS_OK;
  const int threads = groups * k;
  hipLaunchKernelGGL(k_merge, dim3((threads + 255) / 256), dim3(256), 0, s, rows, ptr, slots,
                     groups, partials, k, y, alpha, beta);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

int check_indices(const int *a, int64_t count, int lo, int hi, bool sorted, hipStream_t s,
                  bool *ok) {
  *ok = true;
  if (count <= 0) return SBLAS_OK;
  int *flag = nullptr;
  SBLAS_HIP_TRY(hipMalloc(&flag, sizeof(int)));
  int h = 0;
  hipError_t e = hipMemcpyAsync(flag, &h, sizeof(int), hipMemcpyHostToDevice, s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_check_indices, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256),
                       0, s, count, a, lo, hi, sorted ? 1 : 0, flag);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(&h, flag, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFree(flag);
  if (e != hipSuccess) {
    set_error(SBLAS_ERR_HIP, std::string("index check: ") + hipGetErrorString(e));
    return SBLAS_ERR_HIP;
  }
  *ok = (h == 0);
  return SBLAS_OK;
}

int launch_scale(int64_t count, double beta, double *y, hipStream_t s) {
  if (count <= 0) return SBLAS_OK;
  hipLaunchKernelGGL(k_scale, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, s,
                     count, beta, y);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

}  // namespace sblas
