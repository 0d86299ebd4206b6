// span_device.hpp -- row sums of staged products by spans of elements, shared
// by the row-block kernel (sblas_vector.hip) and the merge-path kernel
// (sblas_tiles.hip), and the wave scans under them (also sblas_csr5.hip).
//
// A workgroup of 256 threads holds up to 256*ITEMS products in LDS in element
// order, and a bit mask of the elements that are the last of their row.
// Thread t sums the ITEMS consecutive products of its span; a row that ends
// inside the span and began there is complete, and its sum is left in the
// place of its last product.  What follows a span's last row end is carried by
// a segmented scan (lane moves inside a wave, one exchange through LDS between
// the four waves) to the next span with a row end.  Every thread does the same
// work whatever the row lengths, where one group of lanes per row waits for
// the longest row of its wave and needs a second pass for very long ones; the
// order of every sum is fixed by the row's place in the window alone.
#pragma once

#include "internal.hpp"

namespace sblas {
namespace span {

// Wave-wide scans on DPP lane moves.  Lanes whose source lies outside the
// move (row_shr past a 16-lane row start, rows that a broadcast does not
// reach) read 0, the identity of both scans.
//   row_shr:d   lane l reads l-d inside its row of 16 (d = 1, 2, 4, 8)
//   row_bcast15 rows 1 and 3 read lane 15 of the row before (row mask 0xa)
//   row_bcast31 rows 2 and 3 read lane 31 (row mask 0xc)
//   wave_shr:1  lane l reads l-1
// so after the four in-row steps each lane holds its row prefix, and the two
// broadcasts add the totals of the rows before it.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_mov(double v) {
  return __builtin_amdgcn_update_dpp(0.0, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_mov(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;

// inclusive prefix sum over the 64 lanes
__device__ __forceinline__ int wave_incl_sum(int v) {
  v += dpp_mov<kRowShr1, 0xf>(v);
  v += dpp_mov<kRowShr2, 0xf>(v);
  v += dpp_mov<kRowShr4, 0xf>(v);
  v += dpp_mov<kRowShr8, 0xf>(v);
  v += dpp_mov<kRowBcast15, 0xa>(v);
  v += dpp_mov<kRowBcast31, 0xc>(v);
  return v;
}

// One step of the segmented scan: (v, head) absorbs the moved-in partner
// unless a segment already begins inside this lane's range.
template <int CTRL, int ROWS>
__device__ __forceinline__ void seg_step(double &v, int &head) {
  const double vu = dpp_mov<CTRL, ROWS>(v);
  const int hu = dpp_mov<CTRL, ROWS>(head);
  if (!head) {
    v += vu;
    head = hu;
  }
}

// inclusive segmented sum over the 64 lanes; head = 1 opens a segment.  On
// return head tells whether a segment opens at or before the lane.
__device__ __forceinline__ double wave_seg_sum(double v, int &head) {
  seg_step<kRowShr1, 0xf>(v, head);
  seg_step<kRowShr2, 0xf>(v, head);
  seg_step<kRowShr4, 0xf>(v, head);
  seg_step<kRowShr8, 0xf>(v, head);
  seg_step<kRowBcast15, 0xa>(v, head);
  seg_step<kRowBcast31, 0xc>(v, head);
  return v;
}

constexpr int kBlock = 256;

template <int ITEMS>
struct Shared {
  // element e at e + e/ITEMS: threads' spans start in distinct banks
  double prod[kBlock * ITEMS + kBlock];
  uint32_t ends[kBlock * ITEMS / 32];
  double wave_tail[kBlock / 64];
  int wave_has[kBlock / 64];
};

template <int ITEMS>
__device__ __forceinline__ int pos(int e) {
  return e + e / ITEMS;
}

template <int ITEMS>
__device__ __forceinline__ void clear_ends(Shared<ITEMS> &sh) {
  const int t = threadIdx.x;
  if (t < kBlock * ITEMS / 32) sh.ends[t] = 0;
}

// element e is the last of its row (after a barrier behind clear_ends)
template <int ITEMS>
__device__ __forceinline__ void mark_end(Shared<ITEMS> &sh, int e) {
  atomicOr(&sh.ends[e >> 5], 1u << (e & 31));
}

// Row sums: called with products and marks in place behind a barrier; returns
// behind a barrier with the sum of each row that ends in the window at
// sh.prod[pos(its last element)].  Products past the window may hold anything:
// they follow every row end.
template <int ITEMS>
__device__ __forceinline__ void row_sums(Shared<ITEMS> &sh) {
  static_assert(sizeof(Shared<ITEMS>) % sizeof(double) == 0, "LDS counted in doubles");
  static_assert(ITEMS == 4 || ITEMS == 8 || ITEMS == 16, "spans of whole mask parts");
  const int t = threadIdx.x;
  const uint32_t m = (sh.ends[(t * ITEMS) >> 5] >> ((t * ITEMS) & 31)) & ((1u << ITEMS) - 1u);
  double *span = sh.prod + t * (ITEMS + 1);
  double p[ITEMS];
#pragma unroll
  for (int s = 0; s < ITEMS; s++) p[s] = span[s];
  const int first = __ffs(static_cast<int>(m)) - 1;  // the span's first row end, -1: none
  double acc = 0.0, head = 0.0;
#pragma unroll
  for (int s = 0; s < ITEMS; s++) {
    acc += p[s];
    if ((m >> s) & 1u) {
      if (s == first) head = acc; else span[s] = acc;
      acc = 0.0;
    }
  }
  int has = m != 0 ? 1 : 0;
  const double tail = wave_seg_sum(acc, has);
  const int w = t >> 6, l = t & 63;
  if (l == 63) {
    sh.wave_tail[w] = tail;
    sh.wave_has[w] = has;
  }
  double carry = dpp_mov<kWaveShr1, 0xf>(tail);
  const int carry_has = dpp_mov<kWaveShr1, 0xf>(has);
  __syncthreads();
  if (first >= 0) {
    if (!carry_has) {
      for (int p = w - 1; p >= 0; p--) {
        carry += sh.wave_tail[p];
        if (sh.wave_has[p]) break;
      }
    }
    span[first] = carry + head;
  }
  __syncthreads();
}

// A row cut by tile edges whose last tile before the cut is b: the head
// partials of the following tiles are added in order (through tiles that lie
// wholly inside the row) and y is written once.
__device__ __forceinline__ void close_cut_row(int b, int tiles,
                                              const TileCarry *__restrict__ carry,
                                              double *__restrict__ y, double alpha, double beta) {
  const TileCarry c = carry[b];
  if (c.tail_row < 0 || c.spanning) return;
  const int r = c.tail_row;
  double s = c.tail;
  int n = b + 1;
  while (n < tiles && carry[n].spanning) s += carry[n++].head;
  if (n < tiles && carry[n].head_row == r) s += carry[n].head;
  y[r] = (beta == 0.0) ? alpha * s : alpha * s + beta * y[r];
}

}  // namespace span
}  // namespace sblas
