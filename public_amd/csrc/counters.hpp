// Device cells of the step loops: which forward state an adjoint step reads
// and which checkpoint a subset restores.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

namespace cruna {

// The forward state of the next backward step: the step counter *ntp (set
// by the host before the loop) selects trajectory slot nt (or the only slot
// of a one-slot trajectory), then counts down.  One thread writes.
__global__ void k_adjoint_slot(const double **q0p, int *ntp, const double *traj, long stride,
                               int nslots) {
  if (threadIdx.x != 0) return;
  const int nt = *ntp;
  q0p[0] = traj + (long)(nslots > 1 ? nt - 1 : 0) * stride;
  ntp[0] = nt - 1;
}

// Subset checkpoints inside a recorded period: the subset counter *sp
// (device cell) names the checkpoint to restore; every thread copies its
// share of that state of M = 5 N values into q, one value at a time (grid-stride).
__global__ __launch_bounds__(256) void k_restore_ckpt(double *__restrict__ q, const double *__restrict__ ckpt,
                                                      const int *__restrict__ sp, long M) {
  const int s = *sp;
  const double *src = ckpt + (long)s * M;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < M; i += (long)gridDim.x * 256) q[i] = src[i];
}

// Set an int cell (counter) from the stream, so that a recorded graph can
// reset it without a memset node.
__global__ void k_set_int(int *p, int v, int delta) {
  if (threadIdx.x == 0) p[0] = v == INT_MIN ? p[0] + delta : v;
}

// Point the forward-state cell at a given state.  One thread writes.
__global__ void k_set_state_ptr(const double **q0p, const double *q) {
  if (threadIdx.x == 0) q0p[0] = q;
}

}  // namespace cruna
