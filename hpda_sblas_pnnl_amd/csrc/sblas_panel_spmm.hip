// sblas_panel_spmm.hip -- products of two and four vectors over column panels
// in sorted groups, for gfx950.
//
// On banded matrices the row-block form (sblas_spmm.hip) is bound by the rate
// at which L2 serves one request an element.  Here a workgroup stages the
// vectors' window of a column panel (kPanelCols rows of X: 64 KB at two vectors,
// 128 KB at four) in LDS by whole lines and gathers from there, over the format
// of the single-vector product (sorted_panel_device.hpp): the matrix is streamed
// once, ten bytes an FP64 element, and X crosses L2 once per row panel that
// its columns meet.  One lane owns a row of a 64-row group and keeps its K
// sums in registers for the length of a slice; between slices they live in LDS
// (the order of the rows changes from slice to slice).  Padding meets a row of
// zeros behind the window, so the gathers of a batch need no branch and leave
// together (a branch an element ran them one after another: 308 against 122 us
// below).
//
// 512 threads at two vectors (two workgroups a CU: one stages while the other
// sums) and 1024 at four, where a window leaves room for one workgroup and what
// is left over its floor is the staging nothing hides (512 threads: 186 against
// 166 us; loading a wave's first elements ahead of the window: spills; two
// waves a group in short row panels: 0.85x the time at 256 rows, 1.1x at 1344).
// Products and sums are FP64 for every stored type, also where the
// single-vector product rounds x to FP32.
//
// n = 400009, 140 elements a row in a band of 20000, us (row blocks before):
//   FP64  k = 2   122 (287)   k = 4   166 (309)   floor 114 and 117 at 6 TB/s
//   FP32  k = 2   125 (249)   BF16  k = 2   112 (244)
#include <type_traits>

#include "internal.hpp"
#include "panel_device.hpp"
#include "sorted_panel_device.hpp"

namespace sblas {
namespace {

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef dbl2 dbl2_u __attribute__((aligned(8)));

constexpr size_t kLdsMost = size_t{160} << 10;  // of a workgroup

template <int K>
__host__ __device__ constexpr int spmm_threads() {
  return K == 4 ? 1024 : 512;
}
// LDS in bytes: window, sums, row order (whole rounds of a word a thread),
// group offsets
template <int K>
__host__ __device__ constexpr size_t spmm_lds(int R) {
  return sizeof(double) * K * (kPanelCols + 1 + static_cast<size_t>(R)) +
         sizeof(uint32_t) * ((R / 2 + 63) / 64 * 64 + R / 64 + 1);
}

// ld: doubles from one row of X (Y) to the next; X, Y and slots point at the
// pass's first vector, slots are ks apart
template <typename VT, int K>
__global__ __launch_bounds__(spmm_threads<K>()) void k_panel_spmm(
    int n, int R, int npanels, int xcd_remap, const PanelInfo *__restrict__ info,
    const int *__restrict__ slice_base, const int64_t *__restrict__ slice_off,
    const uint16_t *__restrict__ perm, const uint32_t *__restrict__ goff,
    const VT *__restrict__ pval, const uint16_t *__restrict__ pcol, const double *__restrict__ X,
    int ld, double *__restrict__ Y, double alpha, double beta, double *__restrict__ slots, int ks) {
  constexpr int T = spmm_threads<K>(), W = kPanelCols, H = K / 2;
  constexpr bool PACKED = sorted_panel::kPackedBf16<VT>;
  extern __shared__ __attribute__((aligned(16))) double lds[];
  int p = blockIdx.x;
  if (xcd_remap) {
    const int per = gridDim.x >> 3;
    p = (p & 7) * per + (p >> 3);
  }
  if (p >= npanels) return;  // uniform per workgroup
  const PanelInfo pi = info[p];
  const int G = R >> 6, words = R >> 1;
  double *xs = lds, *sums = lds + (W + 1) * K;
  uint32_t *order = reinterpret_cast<uint32_t *>(sums + static_cast<size_t>(R) * K);
  uint32_t *group = order + (words + 63) / 64 * 64;
  const int t = threadIdx.x, w = t >> 6, l = t & 63, wv = t & ~63;
  const bool x16 = (reinterpret_cast<uintptr_t>(X) & 15) == 0;  // a row is an even number of doubles
  const int s0 = slice_base[p], s1 = slice_base[p + 1];
  // the sums, and the row of X that padding meets; the barrier outside the
  // slices, since a panel of empty rows has none and its sums are read below all
  // the same
  for (int i = t; i < (R + 1) * K; i += T) xs[W * K + i] = 0.0;
  __syncthreads();

  for (int s = s0; s < s1; s++) {
    const int64_t sb = slice_off[s];
    if (slice_off[s + 1] == sb) continue;  // uniform
    // X window (rows past n repeat the last one: their columns never occur),
    // row order and group offsets
    const int c0 = (pi.q_lo + (s - s0)) * W;
    if (x16) {
#pragma unroll 4
      for (int i = 0; i < W * H; i += T) {
        const int q = i + t;
        const int c = min(c0 + q / H, n - 1);
        panel::load16_to_lds(X + static_cast<int64_t>(c) * ld + 2 * (q % H), xs + 2 * (i + wv));
      }
    } else {
      const uint32_t *xw = reinterpret_cast<const uint32_t *>(X);
#pragma unroll 1
      for (int i = 0; i < W * 2 * K; i += T) {
        const int q = i + t;
        const int c = min(c0 + q / (2 * K), n - 1);
        panel::load4_to_lds(xw + static_cast<int64_t>(c) * 2 * ld + q % (2 * K),
                            reinterpret_cast<uint32_t *>(xs) + i + wv);
      }
    }
    const uint32_t *po = reinterpret_cast<const uint32_t *>(perm + static_cast<int64_t>(s) * R);
    for (int i = 0; i + wv < words; i += T)  // uniform per wave
      panel::load4_to_lds(po + min(i + t, words - 1), order + i + wv);
    const uint32_t go = t <= G ? goff[static_cast<int64_t>(s) * (G + 1) + t] : 0u;
    panel::wait_vector_memory();
    if (t <= G) group[t] = go;
    __syncthreads();

    for (int g = w; g < G; g += T / 64) {
      const int gb = __builtin_amdgcn_readfirstlane(static_cast<int>(group[g]));
      const int len =
          __builtin_amdgcn_readfirstlane(static_cast<int>(group[g + 1] - group[g]) >> 6);
      if (len == 0) break;  // groups come longest first
      const int row = reinterpret_cast<const uint16_t *>(order)[64 * g + l];
      dbl2 acc[H];
#pragma unroll
      for (int h = 0; h < H; h++) acc[h] = *reinterpret_cast<dbl2 *>(sums + row * K + 2 * h);
      const VT *vs = pval + sb + gb + l;
      const uint16_t *cs = pcol + sb + gb + l;
      // N elements of the lane's row from element k on
      auto add = [&](int k, auto count) {
        constexpr int N = decltype(count)::value;
        VT v[N];
        uint32_t c[N];
#pragma unroll
        for (int u = 0; u < N; u++) {
          v[u] = __builtin_nontemporal_load(vs + 64 * (k + u));
          if constexpr (!PACKED) c[u] = __builtin_nontemporal_load(cs + 64 * (k + u));
        }
#pragma unroll
        for (int u = 0; u < N; u++) {
          if constexpr (PACKED) c[u] = static_cast<uint32_t>(v[u]) & 0xFFFFu;
          // padding (value 0) meets the row of zeros past the window
          const double a = sorted_panel::widen1(v[u]);
          const dbl2 *x = reinterpret_cast<const dbl2 *>(xs + min(c[u], uint32_t{W}) * K);
#pragma unroll
          for (int h = 0; h < H; h++) acc[h] += a * x[h];
        }
      };
      int k = 0;
      for (; k + 16 <= len; k += 16) add(k, std::integral_constant<int, 16>());
      if (len & 8) add(k, std::integral_constant<int, 8>()), k += 8;
      if (len & 4) add(k, std::integral_constant<int, 4>()), k += 4;
      if (len & 2) add(k, std::integral_constant<int, 2>()), k += 2;
      if (len & 1) add(k, std::integral_constant<int, 1>());
#pragma unroll
      for (int h = 0; h < H; h++) *reinterpret_cast<dbl2 *>(sums + row * K + 2 * h) = acc[h];
    }
    __syncthreads();  // sums written; the window no longer read
  }
  for (int i = t; i < pi.nrow * H; i += T) {
    const int rl = i / H, h = i % H;
    const dbl2 a = *reinterpret_cast<dbl2 *>(sums + rl * K + 2 * h);
    const bool first = rl == 0 && (pi.flags & 1), last = rl == pi.nrow - 1 && (pi.flags & 2);
    if (first || last) {
      *reinterpret_cast<dbl2_u *>(slots + static_cast<int64_t>(2 * p + (first ? 0 : 1)) * ks +
                                  2 * h) = a;
    } else {
      dbl2_u *y = reinterpret_cast<dbl2_u *>(Y + static_cast<int64_t>(pi.row0 + rl) * ld + 2 * h);
      *y = beta == 0.0 ? alpha * a : alpha * a + beta * *y;
    }
  }
}

template <typename VT, int K>
int launch_pass(const PanelFormat &f, const VT *val, int n, int k, int v0, int xcd_remap,
                const double *X, double *Y, double alpha, double beta, hipStream_t s) {
  const size_t lds = spmm_lds<K>(f.rows);
  const void *fn = reinterpret_cast<const void *>(&k_panel_spmm<VT, K>);
  SBLAS_HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(lds)));
  const int grid = xcd_remap ? (f.npanels + 7) / 8 * 8 : f.npanels;
  hipLaunchKernelGGL((k_panel_spmm<VT, K>), dim3(grid), dim3(spmm_threads<K>()), lds, s, n, f.rows,
                     f.npanels, xcd_remap, f.info, f.slice_base, f.slice_off, f.perm, f.goff, val,
                     f.pcol, X + v0, k, Y + v0, alpha, beta, f.partials + v0, k);
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT>
int launch_passes(const PanelFormat &f, const VT *val, int n, int k, int each, int xcd_remap,
                  const double *X, double *Y, double alpha, double beta, hipStream_t s) {
  for (int v0 = 0; v0 < k; v0 += each) {
    const int st = each == 4
                       ? launch_pass<VT, 4>(f, val, n, k, v0, xcd_remap, X, Y, alpha, beta, s)
                       : launch_pass<VT, 2>(f, val, n, k, v0, xcd_remap, X, Y, alpha, beta, s);
    if (st != SBLAS_OK) return st;
  }
  return SBLAS_OK;
}

}  // namespace

// A slice costs a window's staging whatever it holds, so the line lies at the
// elements of a slice.  Two vectors, row blocks / this form, by elements a slice:
// 1.0 at 1600, 1.2-1.5 at 2700-3200, 1.0 at 3700 (7 a row, where row blocks reuse
// lines), 1.5-2.4 from 5600 up.  Four: 0.9-1.1 at 3100, 1.13 at 6000, 1.76 and 1.86
// at 22700 and 10400.  Four as two passes of two, where the sums of a row panel
// leave no room for the wide window: 0.6-0.8 up to 5600, 1.15 and 1.4 at 26400.
// Eight as two passes of four: 0.99 at 10400, 0.96 at 22700.
int panel_spmm_vectors(const PanelFormat &f, int k) {
  if (f.layout != kPanelSorted || f.npanels <= 0) return 0;
  if (k == 2 && spmm_lds<2>(f.rows) <= kLdsMost) return f.avg_slice >= kPanelCols ? 2 : 0;
  if (k == 4 && spmm_lds<4>(f.rows) <= kLdsMost) return f.avg_slice >= 1.25 * kPanelCols ? 4 : 0;
  if (k == 4 && spmm_lds<2>(f.rows) <= kLdsMost) return f.avg_slice >= 4.0 * kPanelCols ? 2 : 0;
  return 0;
}

int launch_panel_spmm(int val_type, const PanelFormat &f, int n, int k, int each, int xcd_remap,
                      const double *X, double *Y, double alpha, double beta, hipStream_t s) {
  switch (val_type) {
    case SBLAS_VAL_F64:
      return launch_passes(f, static_cast<const double *>(f.pval), n, k, each, xcd_remap, X, Y,
                           alpha, beta, s);
    case SBLAS_VAL_F32:
      return launch_passes(f, static_cast<const float *>(f.pval), n, k, each, xcd_remap, X, Y,
                           alpha, beta, s);
    case SBLAS_VAL_BF16:
      return launch_passes(f, f.packed, n, k, each, xcd_remap, X, Y, alpha, beta, s);
    default:
      set_error(SBLAS_ERR_ARGS, "unknown value type");
      return SBLAS_ERR_ARGS;
  }
}

}  // namespace sblas
