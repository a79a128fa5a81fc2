// pxh_queue.h -- the work queues of the persistent kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pxh {

// Phase A and B deal out work through kQueues independent queues (queue q
// serves work items q, q + kQueues, ...), so that no single counter takes
// every fetch.
constexpr int kQueues = 16;
constexpr int kQueueStride = 64;  // ints between queue heads (256 B)

// Next work item of this wave's queue, or n when it is empty.  The whole wave
// calls it.  The items are dealt to the kQueues queues in granules of G
// consecutive items, round robin; a queue hands its items out in order.
// Workgroups go to the XCDs round robin, so queue q is served by XCD q % 8
// alone: a granule's items (neighbouring rows of one call, in phase A) share
// that XCD's L2.
//
// One lane adds, in the source: additions of several lanes of a wave are
// several operations, between which another wave's may fall, unless the
// compiler merges them.  Two compiler effects shape the form.  The branch's
// lane number is hidden from it, because it may join a branch on lane 0 with
// another one at the end of the caller's loop, and let lanes 1..63 go round
// that loop by themselves, for ever.  And an addition of 1 in lane 0 and 0
// elsewhere makes it sum the lanes in a loop of 64 rounds and 20 instructions
// for every item (8,192 glyphs on 8,192 x 8,192: the composition 395 us,
// 279 us with one addition).
template <int G = 1>
__device__ __forceinline__ int queue_next(int32_t* heads, int n) {
  const uint32_t q = blockIdx.x % kQueues;
  int lane = (int)(threadIdx.x & 63);
  asm volatile("" : "+v"(lane));
  int old = 0;
  if (lane == 0) old = atomicAdd(heads + q * kQueueStride, 1);
  // the same in every lane: keep it (and what derives from it) scalar
  const uint32_t k = (uint32_t)__builtin_amdgcn_readfirstlane(old);
  // The item is increasing in k, so a queue is empty once one is >= n.  k ends
  // at n / kQueues and an addition per wave: 32 unsigned bits hold the item.
  const uint32_t item = (k / G * kQueues + q) * G + k % G;
  return item < (uint32_t)n ? (int)item : n;
}

}  // namespace pxh
