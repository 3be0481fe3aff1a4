// gp_xfer.hip — transposition between a caller's device arrays (instance-major
// flattening, the layout of the host set/get calls) and the buckets'
// structure-of-arrays rows, for callers whose state or torques live in HBM.
//
// One launch moves every array of every bucket that a call names: a table
// entry per (bucket, array), entry e owning workgroups [first, first of e + 1).
// What bounds it is the launch, not the bytes: with one launch per bucket and
// array, a batch of 13 buckets took 78 launches of 3.4 us for its state,
// torques, new state and accelerations, and takes 4 now. A workgroup moves
// the rows of 64 lanes, each wave one row at a time: consecutive threads touch
// consecutive lanes of a row, and the flat array's lines, which hold a lane's
// whole row set, are re-read from the compute unit's own L1 instead of by
// workgroups on other XCDs.
#include <hip/hip_runtime.h>

#include "gp_internal.h"

namespace gp {

constexpr int kXferWaves = 4;

__global__ void __launch_bounds__(64 * kXferWaves) flat_xfer_kernel(const XferEntry* __restrict__ t, int n,
                                                                    unsigned block0, double* flat0, double* flat1,
                                                                    int to_soa) {
  const unsigned b = block0 + blockIdx.x;
  int e = 0;  // the last entry whose first workgroup is at most b (uniform)
  for (int hi = n; hi - e > 1;) {
    const int mid = (e + hi) / 2;
    if (t[mid].first <= b) e = mid;
    else hi = mid;
  }
  const XferEntry x = t[e];
  const int64_t l = (int64_t)(b - x.first) * 64 + (threadIdx.x & 63);
  if (l >= x.B) return;
  double* __restrict__ s = x.soa + l;
  double* __restrict__ f = (x.second ? flat1 : flat0) + x.off[l];
  const size_t Bp = x.Bp;
  const int k0 = (int)(threadIdx.x >> 6), rows = x.rows;
  if (to_soa) {
#pragma unroll 4
    for (int k = k0; k < rows; k += kXferWaves) s[k * Bp] = f[k];
  } else {
#pragma unroll 4
    for (int k = k0; k < rows; k += kXferWaves) f[k] = s[k * Bp];
  }
}

int launch_flat_xfer(const XferEntry* d_table, int n, unsigned blocks, double* flat0, double* flat1, int to_soa,
                     void* stream) {
  constexpr unsigned kMost = 1u << 23;  // a launch's threads stay below 2^32
  for (unsigned b = 0; n > 0 && b < blocks; b += kMost) {
    const unsigned g = blocks - b < kMost ? blocks - b : kMost;
    hipLaunchKernelGGL(flat_xfer_kernel, dim3(g), dim3(64 * kXferWaves), 0, (hipStream_t)stream, d_table, n, b, flat0,
                       flat1, to_soa);
    const int err = (int)hipGetLastError();
    if (err) return err;
  }
  return 0;
}

}  // namespace gp
