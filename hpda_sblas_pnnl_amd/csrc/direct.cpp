// direct.cpp -- one product of a CSR matrix in host memory without a plan: the
// path of the reference's drop-in calls (include/spmv_kernel.h:211-296) for
// matrices that fit a call context.
//
// A plan is made to be kept; a call that uses one once pays for its set-up: a
// stream, some sixteen device allocations and frees, eight small uploads and as
// many waits, and the row pointers sent back to the host that holds them (310 of
// the 460 us of a call on a 20,000-row matrix of 315,000 elements; 4.2 MB of
// transfers are the rest).  Here a call borrows a context that lives with the
// process: one per device, a stream, one device allocation that grows to the
// largest call (at most kContextBytes) and one pinned buffer.  What the kernel
// needs beside the matrix (row blocks and merge lists, or the CSR5-style tile
// words) is built on the host while the elements are on their way and goes up
// in one transfer; indices are checked on the device (an
// out-of-range column is replaced by 0 in the uploaded copy, so the product
// stays in bounds, and its flag comes back before y is touched).  A second
// thread's call that finds the context borrowed takes the plan path.
//
// us a call before -> now (power law): 2,000 rows 261 -> 98; 20,000 rows kernels
// 1 / 2 / 3 455 / 507 / 664 -> 242 / 254 / 278; 200,000 rows (42 MB) 2229 ->
// 1318.  What is left at 20,000 rows are the copies from pageable memory (4.2
// MB, 147 us); sent through the pinned ring they took longer (297 us a call),
// so calls under 8 MB copy straight.
#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "direct.hpp"
#include "host_util.hpp"
#include "plan.hpp"

namespace sblas {
namespace {

constexpr size_t kContextBytes = size_t{64} << 20;  // device memory of a context, at most
constexpr size_t kPinnedBytes = size_t{1} << 20;    // its pinned buffer
constexpr size_t kFlagAt = kPinnedBytes - 64;       // the index flag's place there
constexpr int kMaxDevices = 64;
constexpr int kEvents = 7;

// Contexts live until the process ends: no HIP call runs from a static
// destructor.
struct CallContext {
  std::mutex mu;
  bool failed = false;  // set-up failed once: the plan path from then on
  hipStream_t stream = nullptr;
  hipEvent_t ev[kEvents] = {};
  char *pinned = nullptr;
  char *dev = nullptr;
  size_t dev_bytes = 0;

  bool ready(size_t bytes, size_t pinned_bytes = kPinnedBytes) {
    if (failed) return false;
    if (!stream) {
      failed = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess;
      for (hipEvent_t &e : ev) failed = failed || hipEventCreate(&e) != hipSuccess;
      void *p = nullptr;
      failed = failed || hipHostMalloc(&p, pinned_bytes, hipHostMallocDefault) != hipSuccess;
      pinned = static_cast<char *>(p);
    }
    if (failed) {
      (void)hipGetLastError();  // the plan path's launches must not find it
      return false;
    }
    if (bytes > dev_bytes) {
      if (dev) (void)hipFree(dev);
      dev = nullptr;
      dev_bytes = 0;
      const size_t want = (bytes + (size_t{1} << 20) - 1) >> 20 << 20;
      void *p = nullptr;
      if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      dev = static_cast<char *>(p);
      dev_bytes = want;
    }
    return true;
  }
};
CallContext g_contexts[kMaxDevices];

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch())
      .count();
}

// Places in the context's device memory, 256 bytes apart.
struct Layout {
  size_t used = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (bytes + 255) & ~size_t{255};
    return at;
  }
};

// Host arrays that go up together: each gets a place behind `start`.
struct Pack {
  struct Part {
    const void *src;
    size_t bytes, at;
  };
  Layout &room;
  size_t start;
  std::vector<Part> parts;
  explicit Pack(Layout &l) : room(l), start(l.used) {}
  template <typename T>
  size_t add(const std::vector<T> &v) {
    const size_t bytes = sizeof(T) * v.size();
    parts.push_back(Part{v.data(), bytes, room.take(bytes)});
    return parts.back().at;
  }
};

bool env_set(const char *name) {
  const char *e = std::getenv(name);
  return e && *e;
}

double seconds(hipEvent_t a, hipEvent_t b) {
  float ms = 0.f;
  return hipEventElapsedTime(&ms, a, b) == hipSuccess ? ms / 1000.0 : 0.0;
}

int failed(const char *what) {
  set_error(SBLAS_ERR_HIP, what);
  return SBLAS_ERR_HIP;
}

int run(CallContext &c, int m, int n, int nnz, double alpha, const double *val,
        const int *rp, const int *col, const double *x, double beta, double *y, int kernel,
        int part_mode, spmv_ret &ret, bool &handled) {
  const bool merge_path = kernel == SBLAS_KERNEL_MERGE, csr5 = kernel == SBLAS_KERNEL_CSR5;
  const char *ec = std::getenv("SBLAS_CHUNKS");
  const int C = std::max(1, ec && *ec ? std::atoi(ec) : 1);
  const int cap = kStreamBlock * 8;
  int tiles = static_cast<int>((static_cast<int64_t>(m) + nnz + kTileSize - 1) / kTileSize);
  const int sigma = csr5 ? autotune_sigma(nnz, m) : 0;
  Layout at;
  const size_t o_col = at.take(sizeof(int) * nnz), o_val = at.take(sizeof(double) * nnz);
  const size_t o_rp = at.take(sizeof(int) * (static_cast<size_t>(m) + 1));
  const size_t o_x = at.take(sizeof(double) * n), o_y = at.take(sizeof(double) * m);
  const size_t o_flag = at.take(sizeof(int));
  // an upper bound of what the kernel needs beside them: a row block (16
  // bytes), its partials (16) and lists (at most two rows, slots and pointers,
  // 24) for nnz/2048 + m/kStreamRowsMax blocks beside what chunk edges and long
  // rows add; a carry a tile; or the transposed elements, a flag word a lane,
  // a tile word, a carry a workgroup and the lists of rows
  const size_t most_blocks = 2 * (static_cast<size_t>(nnz) / cap + m / kStreamRowsMax +
                                  2 * static_cast<size_t>(C)) + 64;
  const size_t most_tiles = csr5 ? static_cast<size_t>(nnz) / (64 * sigma) + 1 : 0;
  const size_t more = merge_path ? sizeof(TileCarry) * static_cast<size_t>(tiles)
                      : csr5     ? most_tiles * (64 * sigma * 12 + 256 + 4 + sizeof(TileCarry)) +
                                   sizeof(int) * static_cast<size_t>(m)
                                 : 64 * most_blocks;
  const size_t room = at.used + more + 4096;  // the last: rounding of the places
  if (room > kContextBytes || C > 4096) return SBLAS_OK;
  if (!c.ready(room)) {
    clear_error();
    return SBLAS_OK;
  }
  // spmv_ret: comm_time the copies of the caller's arrays and y; part_time what a
  // plan's creation would do, on the host (host_s, while the arrays are copied) and
  // on the device (its lists uploaded, indices checked, a format laid out)
  double host_s = -now_s();
  for (int r = 0; r < m; r++)
    if (rp[r + 1] < rp[r]) {
      handled = true;
      set_error(SBLAS_ERR_ARGS, "plan: row_ptr must be non-decreasing");
      return SBLAS_ERR_ARGS;
    }
  handled = true;
  hipStream_t s = c.stream;
  char *d = c.dev;
  int *d_col = reinterpret_cast<int *>(d + o_col), *d_rp = reinterpret_cast<int *>(d + o_rp);
  int *d_flag = reinterpret_cast<int *>(d + o_flag);
  double *d_val = reinterpret_cast<double *>(d + o_val);
  double *d_x = reinterpret_cast<double *>(d + o_x), *d_y = reinterpret_cast<double *>(d + o_y);
  // an event costs about 6 us of a call, so neighbouring steps share theirs
  enum { UP_A, UP_B, PREP_A, COMP_A, COMP_B, MERGE_B, DOWN_B };
  // whatever happens below, nothing of this call is left on the stream when
  // the context is handed on
  struct Drain {
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  } drain{s};

  host_s += now_s();
  (void)hipEventRecord(c.ev[UP_A], s);
  {
    StagingLease ring((sizeof(int) + sizeof(double)) * static_cast<size_t>(nnz) +
                      sizeof(double) * (static_cast<size_t>(n) + m));
    int st;
    if ((st = ring.to_device(d_col, col, sizeof(int) * nnz, s)) != SBLAS_OK ||
        (st = ring.to_device(d_val, val, sizeof(double) * nnz, s)) != SBLAS_OK ||
        (st = ring.to_device(d_rp, rp, sizeof(int) * (static_cast<size_t>(m) + 1), s)) !=
            SBLAS_OK ||
        (st = ring.to_device(d_x, x, sizeof(double) * n, s)) != SBLAS_OK)
      return st;
    if (beta != 0.0 && (st = ring.to_device(d_y, y, sizeof(double) * m, s)) != SBLAS_OK) return st;
  }
  (void)hipEventRecord(c.ev[UP_B], s);
  // what the kernel needs beside the matrix, while the transfers run
  host_s -= now_s();
  int *flag_home = reinterpret_cast<int *>(c.pinned + kFlagAt);
  *flag_home = 0;
  StreamLaunch L{};
  Csr5Host c5;
  std::vector<RowBlock> rb;
  std::vector<int> mrows, mptr, mslots;
  Pack pack(at);
  size_t o_rows = 0, o_mrows = 0, o_mptr = 0, o_mslots = 0, o_tile = 0, o_lane = 0, o_nz = 0,
         o_empty = 0;
  if (csr5) {
    csr5_host_format(m, nnz, sigma, rp, c5);
    tiles = c5.tiles;
    o_tile = pack.add(c5.tile_nz);
    o_lane = pack.add(c5.flags);
    o_nz = pack.add(c5.rows_nz);
    o_empty = pack.add(c5.empty);
  } else if (!merge_path) {
    const std::vector<ExecChunk> ex =
        exec_chunks_from_bounds(m, rp, element_bounds(part_mode, m, rp, nnz, C, 1));
    rb = build_row_blocks(ex, rp, cap);
    std::vector<ExecChunk> as_chunks;
    as_chunks.reserve(rb.size());
    for (const RowBlock &b : rb) as_chunks.push_back(ExecChunk{b.lo, b.hi, b.row_begin, b.row_end});
    merge_lists(as_chunks, rp, mrows, mptr, mslots);
    o_rows = pack.add(rb);
    o_mrows = pack.add(mrows);
    o_mptr = pack.add(mptr);
    o_mslots = pack.add(mslots);
    const char *er = std::getenv("SBLAS_XCD_REMAP");
    L.items = 8;
    L.nblocks = static_cast<int>(rb.size());
    L.xcd_remap = !(er && *er) || std::atoi(er) != 0 ? 1 : 0;
    L.grid = L.xcd_remap ? (L.nblocks + 7) / 8 * 8 : L.nblocks;
  }
  const int groups = static_cast<int>(mrows.size());
  const int64_t padded = static_cast<int64_t>(csr5 ? tiles : 0) * 64 * sigma;
  const size_t pack_bytes = at.used - pack.start;
  const size_t o_part = at.take(sizeof(double) * 2 * rb.size());
  const size_t o_carry = at.take(merge_path ? sizeof(TileCarry) * static_cast<size_t>(tiles)
                                 : csr5     ? sizeof(TileCarry) * ((tiles + 3) / 4)
                                            : 0);
  const size_t o_colT = at.take(sizeof(int) * padded), o_valT = at.take(sizeof(double) * padded);
  if (at.used > c.dev_bytes || (!merge_path && !csr5 && rb.empty())) {
    handled = false;  // more than foreseen: the plan path
    return SBLAS_OK;
  }
  std::vector<char> large;
  if (pack_bytes > 0) {
    char *stage = c.pinned;
    if (pack_bytes > kFlagAt) {
      large.resize(pack_bytes);
      stage = large.data();
    }
    for (const Pack::Part &q : pack.parts)
      if (q.bytes) std::memcpy(stage + (q.at - pack.start), q.src, q.bytes);
    host_s += now_s();
    (void)hipEventRecord(c.ev[PREP_A], s);
    if (hipMemcpyAsync(d + pack.start, stage, pack_bytes, hipMemcpyHostToDevice, s) != hipSuccess ||
        (!large.empty() && hipStreamSynchronize(s) != hipSuccess))
      return failed("upload failed");
  } else {
    host_s += now_s();
    (void)hipEventRecord(c.ev[PREP_A], s);
  }
  if (hipMemcpyAsync(d_flag, flag_home, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess)
    return failed("upload failed");
  int st = launch_sanitize_cols(nnz, d_col, n, d_flag, s);
  if (st != SBLAS_OK) return st;

  TileCarry *carry = reinterpret_cast<TileCarry *>(d + o_carry);
  double *partials = reinterpret_cast<double *>(d + o_part);
  auto ints = [&](size_t o) { return reinterpret_cast<int *>(d + o); };
  auto words = [&](size_t o) { return reinterpret_cast<uint32_t *>(d + o); };
  double *d_valT = reinterpret_cast<double *>(d + o_valT);
  if (merge_path)
    st = launch_merge_rows(m, nnz, tiles, d_rp, carry, s);
  else if (csr5)
    st = launch_csr5_transpose(SBLAS_VAL_F64, sigma, padded, nnz, d_col, d_val, ints(o_colT),
                               d_valT, s);
  if (st != SBLAS_OK) return st;
  (void)hipEventRecord(c.ev[COMP_A], s);
  if (merge_path) {
    st = launch_csr_merge_path(SBLAS_VAL_F64, m, nnz, tiles, d_rp, d_col, d_val, d_x, d_y, alpha,
                               beta, carry, s);
  } else if (csr5) {
    st = launch_csr5(SBLAS_VAL_F64, sigma, tiles, nnz, words(o_tile), words(o_lane), ints(o_nz),
                     ints(o_colT), d_valT, d_x, d_y, alpha, beta, carry, s);
  } else {
    st = launch_csr_stream(SBLAS_VAL_F64, L, reinterpret_cast<RowBlock *>(d + o_rows), d_rp, d_col,
                           d_val, d_x, d_y, alpha, beta, partials, s);
  }
  if (st != SBLAS_OK) return st;
  (void)hipEventRecord(c.ev[COMP_B], s);
  const bool merged = merge_path || csr5 || groups > 0;
  if (merged) {
    st = merge_path ? launch_tile_fixup(tiles, carry, d_y, alpha, beta, s)
         : csr5     ? launch_csr5_finish((tiles + 3) / 4, carry, static_cast<int>(c5.empty.size()),
                                         ints(o_empty), alpha, beta, d_y, s)
                    : launch_merge(ints(o_mrows), ints(o_mptr), ints(o_mslots), groups, partials,
                                   1, d_y, alpha, beta, s);
    if (st != SBLAS_OK) return st;
    (void)hipEventRecord(c.ev[MERGE_B], s);
  }
  // y by way of the pinned buffer where it fits, so that one wait serves the
  // flag and y, and y stays untouched when an index was out of range
  const size_t y_bytes = sizeof(double) * static_cast<size_t>(m);
  const bool by_pinned = y_bytes <= kFlagAt;
  if (hipMemcpyAsync(flag_home, d_flag, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
      (by_pinned &&
       hipMemcpyAsync(c.pinned, d_y, y_bytes, hipMemcpyDeviceToHost, s) != hipSuccess))
    return failed("download failed");
  (void)hipEventRecord(c.ev[DOWN_B], s);
  if (hipStreamSynchronize(s) != hipSuccess) return failed("kernel execution failed");
  if (*flag_home != 0) {
    set_error(SBLAS_ERR_ARGS, "plan: a column index is outside [0, n)");
    return SBLAS_ERR_ARGS;
  }
  double y_s = 0.0;
  if (by_pinned) {
    std::memcpy(y, c.pinned, y_bytes);
  } else {
    const double t1 = now_s();
    if (hipMemcpyAsync(y, d_y, y_bytes, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return failed("download failed");
    y_s = now_s() - t1;
  }
  const int done = merged ? MERGE_B : COMP_B;
  ret.part_time = host_s + seconds(c.ev[PREP_A], c.ev[COMP_A]);
  ret.comm_time = seconds(c.ev[UP_A], c.ev[UP_B]) + seconds(c.ev[done], c.ev[DOWN_B]) + y_s;
  ret.comp_time = seconds(c.ev[COMP_A], c.ev[COMP_B]);
  ret.merg_time = merged ? seconds(c.ev[COMP_B], c.ev[MERGE_B]) : 0.0;
  return SBLAS_OK;
}

}  // namespace

int direct_csr(int device, int m, int n, int nnz, double alpha, const double *val, const int *rp,
               const int *col, const double *x, double beta, double *y, int kernel, int part_mode,
               spmv_ret &ret, bool &handled) {
  handled = false;
  if (device < 0 || device >= kMaxDevices || m < 1 || n < 1 || nnz < 1 ||
      kernel < SBLAS_KERNEL_VECTOR || kernel > SBLAS_KERNEL_CSR5 ||
      part_mode == SBLAS_PART_V2 || env_set("SBLAS_VARIANT"))
    return SBLAS_OK;
  CallContext &c = g_contexts[device];
  std::unique_lock<std::mutex> lock(c.mu, std::try_to_lock);
  if (!lock.owns_lock()) return SBLAS_OK;
  try {
    return run(c, m, n, nnz, alpha, val, rp, col, x, beta, y, kernel, part_mode, ret,
               handled);
  } catch (const std::bad_alloc &) {
    handled = true;
    set_error(SBLAS_ERR_ALLOC, "host allocation failed");
    return SBLAS_ERR_ALLOC;
  }
}

}  // namespace sblas

// The HIP error that a call context leaves behind whose pinned buffer cannot be had,
// -1 if it can (not in sblas.h; used by the tests).
extern "C" int sblas_internal_call_context_error(size_t pinned_bytes) {
  sblas::CallContext c;
  const bool ok = c.ready(0, pinned_bytes);
  const int left = static_cast<int>(hipGetLastError());
  for (hipEvent_t e : c.ev)
    if (e) (void)hipEventDestroy(e);
  if (c.stream) (void)hipStreamDestroy(c.stream);
  if (ok) (void)hipHostFree(c.pinned);
  return ok ? -1 : left;
}
