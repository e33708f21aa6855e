// Workgroup orders: which piece of a launch a workgroup takes, as plain integer functions (a
// host test compiles them by themselves).  Each is a permutation of 0 .. n - 1 for every n:
// a kernel's grid is what its work divides into, not a multiple of 8 XCDs or of the
// batch-groups.
#pragma once

namespace nsa {

// Workgroup id -> logical id such that each XCD (ids dispatched round-robin over 8)
// receives a contiguous range of logical ids.
__host__ __device__ __forceinline__ int xcd_contiguous(int i, int n) {
  const int xcd = i & 7, k = i >> 3;
  const int base = n >> 3, rem = n & 7;
  return (xcd < rem ? xcd * (base + 1) : rem * (base + 1) + (xcd - rem) * base) + k;
}
// Logical id of a workgroup of the selection kernels (ids: batch-group major, timesteps
// ascending).  A timestep's cost grows with the blocks it can select, so with contiguous
// ranges the XCDs that held the early timesteps finished first, and ascending order left
// the longest workgroups for the last, partly filled round.  Late timesteps go first, and the
// XCDs take runs of kXcdRun ids in turn, which keeps neighbouring timesteps on one L2; with
// whole batch-groups to share out (a multiple of 8) each XCD takes a contiguous range, its own
// groups, so that its L2 holds one group's K / V (the dQ kernel of the stored dS has
// ceil(waves / 4) workgroups, not whole ones per group: the ranges then end within a group).
// Forward / dQ in us, before -> after: H64 G4 T2048 dk 192 160 / 163 -> 137 / 140, T8192 634 /
// 657 -> 613 / 624; B2 H16 G4 T4096 dk 64 118 / 215 -> 106 / 128 (runs of 1, 2 and 4 alike; of
// 16 and 64 up to 10 % slower).
constexpr int kXcdRun = 4;
__host__ __device__ __forceinline__ int sel_workgroup(int i, int n, int nbg) {
  if (nbg % 8 == 0) return n - 1 - xcd_contiguous(i, n);
  const int full = n / (8 * kXcdRun) * (8 * kXcdRun);
  if (i < full) {
    const int k = i >> 3;
    return n - 1 - ((k / kXcdRun * 8 + (i & 7)) * kXcdRun + k % kXcdRun);
  }
  return n - 1 - (full + xcd_contiguous(i - full, n - full));
}

}  // namespace nsa
