// Composition of row interchanges, shared by the LU panels and the solves
// (zml lapack/laswp.zig:26-40 applies them one after the other).
#pragma once

#include <cstdint>

namespace zmlhip {

// An interchange of row i with row ip - 1 as compose_swaps takes it. An entry of ipiv
// below 1 names no row (a cleared ipiv): that interchange touches nothing.
__device__ __forceinline__ int2 swap_entry(int i, int32_t ip) {
  return i >= 0 && ip >= 1 ? make_int2(i, ip - 1) : make_int2(-1, -1);
}

// Where the interchanges ev[0], ev[1], .., ev[cnt - 1] (rows x <-> y, in this order,
// each from swap_entry; in LDS, 16-byte aligned, cnt <= NS, entry cnt (-1, -1) when
// cnt is odd) leave every row they touch. 2 NS threads, two per interchange:
// thread 2 s + side stands for "the content of row ev[s].x (side 0) or ev[s].y after
// interchange s", which is what the other row held before: the content after the last
// earlier interchange that touched it, or its own row. Those links, found by a scan
// over the list, are followed (and shortened) in `node` (2 NS words of LDS).
// Returns true in the one thread per touched row that stands for its last
// interchange, with the row in dst and the row whose content ends there in src.
// All threads call it; the list may be overwritten after the caller's next barrier.
//
// Every thread does the same work, about 8 instructions per entry of the list
// (8 us for 256 interchanges with two waves per SIMD), where one lane walking the
// list needs a dependent LDS exchange of 100 ns for each.
template <int NS>
__device__ __forceinline__ bool compose_swaps(const int2* ev, int cnt, int* node, int& dst, int& src) {
  const int t = threadIdx.x, s0 = t >> 1;
  const int w0 = __builtin_amdgcn_readfirstlane(s0 & ~31);   // the wave's first interchange
  const int2 me = s0 < cnt ? ev[s0] : make_int2(-1, -1);
  const bool mine = me.x >= 0;
  // (-2 is in no entry: a thread without an interchange finds no link and is none's)
  const int row = !mine ? -2 : t & 1 ? me.y : me.x, other = !mine ? -2 : t & 1 ? me.x : me.y;
  int link = mine ? ~other : -1;               // < 0: the row itself
  bool later = false;                          // touched again
  // two entries per read (the list ends with an empty one when cnt is odd)
  const int4* const ev2 = reinterpret_cast<const int4*>(ev);
  const int pairs = (cnt + 1) >> 1, b0 = min(w0 >> 1, pairs), b1 = min((w0 >> 1) + 16, pairs);
#pragma unroll 8
  for (int s = 0; s < b0; ++s) {
    const int4 e = ev2[s];
    link = e.x == other ? 4 * s : link;
    link = e.y == other ? 4 * s + 1 : link;
    link = e.z == other ? 4 * s + 2 : link;
    link = e.w == other ? 4 * s + 3 : link;
  }
#pragma unroll 4
  for (int s = b0; s < b1; ++s) {
    const int4 e = ev2[s];
    link = (2 * s < s0) & (e.x == other) ? 4 * s : link;
    link = (2 * s < s0) & (e.y == other) ? 4 * s + 1 : link;
    link = (2 * s + 1 < s0) & (e.z == other) ? 4 * s + 2 : link;
    link = (2 * s + 1 < s0) & (e.w == other) ? 4 * s + 3 : link;
    later |= (2 * s > s0) & ((e.x == row) | (e.y == row));
    later |= (2 * s + 1 > s0) & ((e.z == row) | (e.w == row));
  }
#pragma unroll 8
  for (int s = b1; s < pairs; ++s) {
    const int4 e = ev2[s];
    later |= (e.x == row) | (e.y == row) | (e.z == row) | (e.w == row);
  }
  node[t] = link;
  __syncthreads();
  // (links lead to ever earlier interchanges; an entry read here may already have been
  // moved further along its chain, which is as good)
  volatile int* const nd = node;
  while (link >= 0) {
    link = nd[link];
    nd[t] = link;
  }
  dst = row;
  src = ~link;
  return mine && !later && !((t & 1) && me.x == me.y);
}

}  // namespace zmlhip
