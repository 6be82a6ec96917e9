// mdk_brick.h -- limits and extents of the brick list (k_brick_list), shared by
// host and device code.
#pragma once
#include <hip/hip_runtime.h>

#define BRICK_THREADS_MAX 512
#define BRICK_CELLS 216
#define BRICK_CAP_MAX 2560  // staged atoms: 40 KB of LDS, below 64 KB with the list kernel's masks
#define BRICK_H_SHIFT 24

// A brick's record: first atom, own atoms, staged atoms.  The pair passes stage
// exactly the atoms that the record counts, so it counts none where the list
// kernel writes no bstage words: for a brick that does not fit (the build is
// flagged), and for one without atoms of its own, whatever the cells around it
// hold (a void, the gap beside a slab).
__host__ __device__ inline int4 brick_extent(int a0, int own, int total, int threads, int cap) {
  const bool listed = own > 0 && own <= threads && total < cap;
  return make_int4(a0, listed ? own : 0, listed ? total : 0, 0);
}
