// shp_flow.h - worlds solved by several workgroups: how the workgroups join a
// world and hand words to each other (both solvers).
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "shp_engine.h"

namespace shp {

// Agent-scope accesses of a single word, which other workgroups' wavefronts
// read and write while this one runs.
template <class X>
__device__ __forceinline__ X peek(const X* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class X>
__device__ __forceinline__ void poke(X* p, X v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls before a wait on another workgroup gives up and flags the step
// (SHP_FLAG_STALL).  The waits end by themselves: what one waits for is held by
// a wavefront that has joined the world, so that it runs, and comes earlier in
// the schedule.
constexpr int FLOW_POLLS = 1 << 20;
// seats of a world beyond any grid's
constexpr int FLOW_ANY_SEATS = 1 << 29;

// 16 bytes past the L1 cache (sc1, as agent-scope atomics compile to; there is
// none of 16 bytes): from two addresses, waiting for both, and to one.  A lane
// trusts a word of 8 bytes only by the count that it carries itself.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load_pair(const void* a, const void* b, u32x4& x, u32x4& y) {
  asm volatile(
      "global_load_dwordx4 %0, %2, off sc1\n\t"
      "global_load_dwordx4 %1, %3, off sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(x), "=&v"(y)
      : "v"(a), "v"(b)
      : "memory");
}

// (a wait state before the data's registers may be written)
__device__ __forceinline__ void store_16(void* p, u32x4 x) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(x) : "memory");
}

// The workgroups that share a world wait for each other's results, so each of
// them must be running.  They join by a counter; the first to come closes it
// once all `want` have joined or after a bounded wait (on a GPU busy with
// other streams some may not have started), and those that come later leave.
// Returns the caller's seat and their number in *groups (-1: leave; the seats
// from c.flow_seats on leave too, as if they had come too late).  Seats
// follow each other in space (pairs are in the order of their bodies), so
// when all have come, those of an XCD, to which workgroups go in turn, are
// consecutive: what neighbours exchange stays in its L2.
constexpr int FLOW_JOIN_POLLS = 4096;  // about 0.5 ms
enum { FLOW_CLOSED = 1 << 30 };

constexpr int XCDS = 8;

static __device__ __forceinline__ int flow_join(const Ctx& c, int* seats, int* groups_word, int blk,
                                                int want, int* s_tmp, int* groups) {
  if (threadIdx.x == 0) {
    constexpr int AGENT = __HIP_MEMORY_SCOPE_AGENT;
    int s = __hip_atomic_fetch_add(seats, 1, __ATOMIC_RELAXED, AGENT), g = 0;
    if (s >= c.flow_seats) {  // closed, or one too many
      s = -1;
    } else if (s == 0) {
      for (int n = 0; n < FLOW_JOIN_POLLS && peek(seats) < min(want, c.flow_seats); ++n)
        __builtin_amdgcn_s_sleep(1);
      g = min(__hip_atomic_fetch_or(seats, FLOW_CLOSED, __ATOMIC_RELAXED, AGENT), c.flow_seats);
      poke(groups_word, g);
    } else {  // the first one runs and always writes it
      for (int n = 0; n < c.flow_polls && (g = peek(groups_word)) == 0; ++n)
        __builtin_amdgcn_s_sleep(1);
      if (g == 0) {  // counted in, and now missing
        atomicOr(&c.counters[CNT_FLAGS], SHP_FLAG_STALL);
        s = -1;
      }
    }
    if (g == want) s = blk % XCDS * (want / XCDS) + min(blk % XCDS, want % XCDS) + blk / XCDS;
    s_tmp[0] = s;
    s_tmp[1] = g;
  }
  __syncthreads();
  *groups = s_tmp[1];
  const int seat = s_tmp[0];
  __syncthreads();
  return seat;
}

// Workgroups of world w, of at most `groups`.
__device__ __forceinline__ int flow_want(const Ctx& c, int w, int groups) {
  const int nb = c.body_off[w + 1] - c.body_off[w];
  return min(groups, (nb + FLOW_GROUP_BODIES - 1) / FLOW_GROUP_BODIES);
}

// An FP64 velocity in four words of 8 bytes, 48 bits of it in each beside the
// body's turn.
__device__ __forceinline__ void flow_pack(const double* v, uint32_t turn, u32x4* x) {
  const uint32_t a0 = __double2loint(v[0]), a1 = __double2hiint(v[0]);
  const uint32_t b0 = __double2loint(v[1]), b1 = __double2hiint(v[1]);
  const uint32_t d0 = __double2loint(v[2]), d1 = __double2hiint(v[2]);
  const uint32_t t = turn << 16;
  x[0] = u32x4{a0, (a1 & 0xFFFFu) | t, (a1 >> 16) | (b0 << 16), (b0 >> 16) | t};
  x[1] = u32x4{b1, (d0 & 0xFFFFu) | t, (d0 >> 16) | (d1 << 16), (d1 >> 16) | t};
}

__device__ __forceinline__ void flow_unpack(u32x4 x, u32x4 y, double* v) {
  v[0] = __hiloint2double((x[1] & 0xFFFFu) | (x[2] << 16), x[0]);
  v[1] = __hiloint2double(y[0], (x[2] >> 16) | (x[3] << 16));
  v[2] = __hiloint2double((y[2] >> 16) | (y[3] << 16), (y[1] & 0xFFFFu) | (y[2] << 16));
}

}  // namespace shp
