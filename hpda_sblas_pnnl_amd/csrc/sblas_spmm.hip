// sblas_spmm.hip -- multi-vector products over row blocks (kernel 1, k = 2, 4,
// 8 or 16 right-hand sides, X and Y row-major) for gfx950.
//
// The reference has no multi-vector form; its counterpart is k calls of
// kernel 1 (cusparseDcsrmv, src/dspmv_mgpu_v1.cu:261).
//
// What bounds it: the gathers of X.  Each element reads one k*8-byte row of X,
// so the kernel wants one L2 request and as few lanes as possible per element,
// and nothing else competing for them.  One workgroup takes one row block (at
// most 256*ITEMS elements, kStreamRowsMax rows):
//
// 1. Columns and values are loaded with consecutive threads on consecutive
//    elements (whole lines, each read once) and staged in LDS; the thread of a
//    row marks the row's last element of the window in a bit mask and leaves
//    the row's number beside it.
// 2. L = K/2 lanes, two vectors (16 bytes) each, form a group; a group owns
//    2^es consecutive elements whatever the row lengths, so every lane issues
//    the same number of gathers (eight in flight per lane) and no lane waits
//    for a longer row.  A row ending inside the span is written by its group;
//    the span's first ended row and what follows its last end are kept.
// 3. A segmented scan over the groups (lane shifts inside a wave, one LDS
//    exchange between the four waves) completes the rows that cross spans, in
//    an order fixed by the block alone.
//
// The form before gave each row k lanes, read its columns and values from
// global memory with the lanes of a wave on eight different rows (three
// requests an element instead of one) and waited for the longest of those
// rows.  Times before -> now, FP64 values unless said (us):
//   R-MAT scale 22, k = 2 / 4 / 8 / 16: 818 / 1175 / 1424 / 2041 ->
//     683 / 949 / 1168 / 1498
//   banded, 400,009 rows of 140, k = 2 / 4 / 8 / 16: 450 / 522 / 673 / 1134 ->
//     260 / 292 / 321 / 411
//   27 a row in a band, 300,000 rows, k = 2 / 8, beta 0.5: 87 / 204 -> 45 / 65
//   power law, 20,000 rows, k = 2 / 8: 16.6 / 42.3 -> 7.2 / 10.3
// On the banded matrix at k = 4 the 56 M gathers are 92 % of the L2 requests
// (61 M) and their rate, 2.1e11 a second, is the bound; on R-MAT at k = 8, 51 M
// of the 82 M requests miss L2 and bring 6 GB (5.3 TB/s) of the 268 MB of X and
// the matrix.
#include "internal.hpp"
#include "rows_device.hpp"

namespace sblas {
namespace {

typedef double dbl2 __attribute__((ext_vector_type(2)));
// rows of X and Y start on any 8-byte boundary
typedef dbl2 dbl2_u __attribute__((aligned(8)));

__device__ __forceinline__ double widen(double v) { return v; }
__device__ __forceinline__ double widen(float v) { return static_cast<double>(v); }
__device__ __forceinline__ double widen(uint16_t v) {
  return static_cast<double>(__uint_as_float(static_cast<uint32_t>(v) << 16));
}

constexpr int kSpmmBlock = kStreamBlock;
constexpr int kSpmmBatch = 8;  // elements of a span between two looks at its row ends

// LDS place of element e of the block: spans of 2^es elements are two apart,
// so the groups of a wave read distinct banks, and pairs stay aligned
__device__ __forceinline__ int span_pos(int e, int es) { return e + 2 * (e >> es); }

// BETA: beta != 0, Y is read (with the gathers of the batch a row ends in, so
// its latency is theirs)
template <typename VT, int K, int ITEMS, bool BETA>
__global__ __launch_bounds__(kSpmmBlock) void k_spmm_blocks(
    const RowBlock *__restrict__ blocks, int nblocks, int xcd_remap, const int *__restrict__ rp,
    const int *__restrict__ col, const VT *__restrict__ val, const double *__restrict__ X,
    double *__restrict__ Y, double alpha, double beta, double *__restrict__ partials) {
  constexpr int B = kSpmmBlock, CAP = B * ITEMS;
  constexpr int L = K / 2, G = B / L, WAVES = B / 64;
  constexpr int U = BETA ? kSpmmBatch / 2 : kSpmmBatch;  // gathers in flight per lane
  __shared__ __attribute__((aligned(16))) VT vsh[CAP + 2 * G];
  __shared__ __attribute__((aligned(16))) int csh[CAP + 2 * G];
  __shared__ uint16_t rowof[CAP];         // at a row's last element: the row's number
  __shared__ uint32_t ends[CAP / 32];     // bit e: element e is its row's last
  __shared__ dbl2 wave_tail[WAVES][L];
  __shared__ int wave_has[WAVES];
  const int b = rows::logical_block(nblocks, xcd_remap);
  if (b < 0) return;
  const RowBlock rb = blocks[b];
  const int lo = rb.lo, cnt = rb.hi - rb.lo;
  const int r0 = rb.row_begin, nrows = rb.row_end - rb.row_begin;
  const int t = threadIdx.x;

  // 1. loads, none under a branch; threads past the window re-read its last
  // element, so the places up to the next multiple of eight hold valid columns
  VT v[ITEMS];
  int c[ITEMS];
  if (cnt > 0) {
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const int e = lo + min(t + k * B, cnt - 1);
      v[k] = __builtin_nontemporal_load(val + e);
      c[k] = __builtin_nontemporal_load(col + e);
    }
  }
  const bool cut_first = rp[r0] < lo, cut_last = rp[r0 + nrows] > rb.hi;
  for (int i = t; i < CAP / 32; i += B) ends[i] = 0;
  __syncthreads();
  // span of each group: the block's elements over all groups, at least a batch
  int es = 3;
  while ((G << es) < cnt) es++;
  if (cnt > 0) {
    const int filled = (cnt + kSpmmBatch - 1) & ~(kSpmmBatch - 1);
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const int e = t + k * B;
      if (e < filled) {
        vsh[span_pos(e, es)] = v[k];
        csh[span_pos(e, es)] = c[k];
      }
    }
  }
  const int lane = t % L;
  // a finished row (two vectors of it): into Y, or the partial slots of the
  // rows that the window cuts
  auto finish = [&](int i, dbl2 s, dbl2 old) {
    if ((i == 0 && cut_first) || (i == nrows - 1 && cut_last)) {
      *reinterpret_cast<dbl2_u *>(partials + static_cast<int64_t>(2 * b + (i == 0 ? 0 : 1)) * K +
                                  2 * lane) = s;
    } else {
      *reinterpret_cast<dbl2_u *>(Y + static_cast<int64_t>(r0 + i) * K + 2 * lane) =
          BETA ? alpha * s + beta * old : alpha * s;
    }
  };
  for (int i = t; i < nrows; i += B) {
    const int s = max(rp[r0 + i], lo) - lo, e = min(rp[r0 + i + 1], rb.hi) - lo;
    if (e > s) {
      rowof[e - 1] = static_cast<uint16_t>(i);
      atomicOr(&ends[(e - 1) >> 5], 1u << ((e - 1) & 31));
    }
  }
  // rows without elements in the window
  for (int i = t / L; i < nrows; i += G) {
    if (min(rp[r0 + i + 1], rb.hi) <= max(rp[r0 + i], lo)) {
      dbl2 old = {0.0, 0.0};
      if (BETA) old = *reinterpret_cast<const dbl2_u *>(Y + static_cast<int64_t>(r0 + i) * K + 2 * lane);
      finish(i, dbl2{0.0, 0.0}, old);
    }
  }
  __syncthreads();

  // 2. the group's span
  const int g = t / L;
  const int span0 = g << es;
  const int span = min(1 << es, cnt - span0);
  const VT *vs = vsh + span_pos(span0, es);
  const int *cs = csh + span_pos(span0, es);
  const double *Xl = X + 2 * lane;
  dbl2 acc = {0.0, 0.0}, head = {0.0, 0.0}, head_old = {0.0, 0.0};
  int head_row = -1;
  for (int s = 0; s < span; s += U) {
    dbl2 xv[U], old[BETA ? U : 1];
    uint32_t m = ends[(span0 + s) >> 5] >> ((span0 + s) & 31);
#pragma unroll
    for (int u = 0; u < U; u++)
      xv[u] = *reinterpret_cast<const dbl2_u *>(Xl + static_cast<int64_t>(cs[s + u]) * K);
    if constexpr (BETA) {
#pragma unroll
      for (int u = 0; u < U; u++)
        if ((m >> u) & 1)
          old[u] = *reinterpret_cast<const dbl2_u *>(
              Y + static_cast<int64_t>(r0 + rowof[span0 + s + u]) * K + 2 * lane);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const double a = widen(vs[s + u]);
      acc.x += a * xv[u].x;
      acc.y += a * xv[u].y;
      if ((m >> u) & 1) {
        const int i = rowof[span0 + s + u];
        if (head_row < 0) {  // may have begun in an earlier span: finished in step 3
          head_row = i;
          head = acc;
          if (BETA) head_old = old[BETA ? u : 0];
        } else {
          finish(i, acc, old[BETA ? u : 0]);
        }
        acc = dbl2{0.0, 0.0};
      }
    }
  }

  // 3. what each group leaves after its last row end, summed over the groups
  // back to the last one with a row end (inclusive), then shifted by a group
  const int wl = t & 63, w = t >> 6;
  dbl2 tail = acc;
  int has = head_row >= 0 ? 1 : 0;
#pragma unroll
  for (int d = L; d < 64; d <<= 1) {
    const double px = __shfl_up(tail.x, d, 64), py = __shfl_up(tail.y, d, 64);
    const int ph = __shfl_up(has, d, 64);
    if (wl >= d && !has) {
      tail.x += px;
      tail.y += py;
      has = ph;
    }
  }
  if (wl >= 64 - L) {
    wave_tail[w][lane] = tail;
    if (lane == 0) wave_has[w] = has;
  }
  dbl2 carry = {__shfl_up(tail.x, L, 64), __shfl_up(tail.y, L, 64)};
  int carry_has = __shfl_up(has, L, 64);
  if (wl < L) {
    carry = dbl2{0.0, 0.0};
    carry_has = 0;
  }
  __syncthreads();
  if (head_row >= 0) {
    if (!carry_has) {
      for (int p = w - 1; p >= 0; p--) {
        carry += wave_tail[p][lane];
        if (wave_has[p]) break;
      }
    }
    finish(head_row, carry + head, head_old);
  }
}

template <typename VT, int K, int ITEMS>
int launch_spmm_k(const StreamLaunch &L, const RowBlock *blocks, const int *rp, const int *col,
                  const VT *val, const double *X, double *Y, double alpha, double beta,
                  double *partials, hipStream_t s) {
  const dim3 grid(L.grid), block(kSpmmBlock);
  if (beta != 0.0)
    hipLaunchKernelGGL((k_spmm_blocks<VT, K, ITEMS, true>), grid, block, 0, s, blocks, L.nblocks,
                       L.xcd_remap, rp, col, val, X, Y, alpha, beta, partials);
  else
    hipLaunchKernelGGL((k_spmm_blocks<VT, K, ITEMS, false>), grid, block, 0, s, blocks, L.nblocks,
                       L.xcd_remap, rp, col, val, X, Y, alpha, beta, partials);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT, int ITEMS>
int launch_spmm_items(int k, const StreamLaunch &L, const RowBlock *blocks, const int *rp,
                      const int *col, const VT *val, const double *X, double *Y, double alpha,
                      double beta, double *partials, hipStream_t s) {
  switch (k) {
    case 2: return launch_spmm_k<VT, 2, ITEMS>(L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 4: return launch_spmm_k<VT, 4, ITEMS>(L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 8: return launch_spmm_k<VT, 8, ITEMS>(L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
    case 16: return launch_spmm_k<VT, 16, ITEMS>(L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "spmm: k must be 1, 2, 4, 8 or 16");
      return SBLAS_ERR_ARGS;
  }
}

template <typename VT>
int launch_spmm_typed(int k, const StreamLaunch &L, const RowBlock *blocks, const int *rp,
                      const int *col, const VT *val, const double *X, double *Y, double alpha,
                      double beta, double *partials, hipStream_t s) {
  if (L.items == 16)
    return launch_spmm_items<VT, 16>(k, L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
  if (L.items == 2)
    return launch_spmm_items<VT, 2>(k, L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
  return launch_spmm_items<VT, 8>(k, L, blocks, rp, col, val, X, Y, alpha, beta, partials, s);
}

}  // namespace

int launch_csr_blocks_mrhs(int val_type, int k, const StreamLaunch &L, const RowBlock *blocks,
                           const int *rp, const int *col, const void *val, const double *X,
                           double *Y, double alpha, double beta, double *partials,
                           hipStream_t s) {
  if (L.grid <= 0) return SBLAS_OK;
  if (L.items != 2 && L.items != 8 && L.items != 16) {
    set_error(SBLAS_ERR_ARGS, "spmm kernel: items per thread must be 2, 8 or 16");
    return SBLAS_ERR_ARGS;
  }
  switch (val_type) {
    case SBLAS_VAL_F64:
      return launch_spmm_typed(k, L, blocks, rp, col, static_cast<const double *>(val), X, Y,
                               alpha, beta, partials, s);
    case SBLAS_VAL_F32:
      return launch_spmm_typed(k, L, blocks, rp, col, static_cast<const float *>(val), X, Y, alpha,
                               beta, partials, s);
    case SBLAS_VAL_BF16:
      return launch_spmm_typed(k, L, blocks, rp, col, static_cast<const uint16_t *>(val), X, Y,
                               alpha, beta, partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

}  // namespace sblas
