// Device-side symbolic pipeline: the term sort, the S pattern and the per-slot pair lists of
// the Schur BA path built on the GPU (the host analysis in problem.cpp computes the same
// arrays; both are checked against each other element by element).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "api_internal.hpp"
#include "problem.hpp"

namespace sgpu {

// Stable LSD radix sort of (key, value) pairs of 32-bit unsigned keys by their low key_bits
// bits (8-bit digits; equal keys keep their input order).  keys/vals are sorted in place
// through the two scratch arrays of n elements each.
void radix_sort_pairs(hipStream_t s, DeviceArena& arena, uint32_t* keys, uint32_t* vals,
                      uint32_t* keys_tmp, uint32_t* vals_tmp, int64_t n, int key_bits);

// Exclusive prefix sum of n int64 counts (in place), on the device.
void exclusive_scan_i64(hipStream_t s, DeviceArena& arena, int64_t* data, int64_t n);

// The arrays of the term sort and the analysis that the numeric kernels read, on the device:
// the reprojection terms in sorted order, the point and camera lists over them, the members'
// blocks, and the pairs of S slots (2 per pair).
struct DeviceTerms {
  int32_t *obs_point = nullptr, *obs_pose = nullptr, *obs_intr = nullptr;
  double* obs_uv = nullptr;
  int32_t *pt_ptr = nullptr, *pt_nu = nullptr, *pt_block = nullptr, *pose_block = nullptr;
  int32_t *cam_ptr = nullptr, *cam_nu = nullptr, *cam_obs = nullptr;
  int32_t *cm_point = nullptr, *cm_intr = nullptr;
  double* cm_uv = nullptr;
  int32_t* pairs = nullptr;
};

// analyze() of a problem built with build_host_problem_sorted(.., false), with the term sort
// (stable radix passes over the sort key's arguments, the last argument first), the lists over
// the sorted terms, the S pattern and the pair lists built on the device.  They stay there
// (T, allocated from `arena`): P keeps the caller's order, and S.pt_nu, cam_nu, cam_obs and
// pairs are left empty.
Symbolic analyze_device(const HostProblem& P, hipStream_t s, DeviceArena& arena, DeviceTerms& T);

}  // namespace sgpu
