// Batched Schur LM for many small, independent bundle-adjustment windows.
//
// Every window (one shared pinhole, SE(3) poses with pose 0 constant, marginalized
// points, Huber reprojection terms) has at most kBatchMaxCams cameras, so its reduced
// camera system (n = 6 (cameras - 1) <= 180) lives in LDS as a packed lower triangle, its
// right-hand side as one more row.
// One workgroup runs one complete LM iteration of one window:
//   per point (threads): M_o = A^T A of its observations, H_ll + nu n I, H_ll^-1, s;
//   per camera (16 lanes): the own terms M H^-1 (H - M) of its observations, rhs and
//     gradient, summed in registers;
//   per segment of at most 8 points that two cameras share (threads): the cross terms
//     -M_i H^-1 M_j, lifted by P = [hat(-x) | I] and summed in registers, into S with
//     LDS atomics;
//   dense LDLt of S in LDS (the reference's rule on each 6x6 pivot block), solves;
//   back-substitution, T <- exp(delta) T, merit of the proposal (FP64), and the LM
//   decision with the same rules and check order as the single-problem optimizer.
// One launch advances every unfinished window by one iteration; the host captures a
// sequence of launches in a hipGraph.  Precision T = float computes the Jacobians and
// Schur products in FP32 (S, the factorization, the merit and the decisions stay FP64).
//
// An iteration is bound by the latency of dependent LDS and FP64 steps, its data (0.2 MB a
// window) lies in L2.  Cycles of one iteration of a window of 9 cameras and 5300 observations
// at 512 threads: points 57k, own terms 99k, cross terms 139k (a thread per point that added
// all its terms to S with LDS atomics, 36 a pair at about 40 cycles a wavefront: 621k to
// 668k for the three); factor 71k in panels of 12 columns (258k to 544k with one thread per 6x6
// pivot); solves 18k, back-substitution 33k, merit 27k (57k with a search for the point of
// each observation).  24 windows of 5 to 30 cameras, 20 persistent iterations: 16.0 -> 5.4 ms;
// 1000 such windows, FP32 products, 10 launches: 33.9 -> 12.3 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cstring>
#include <cmath>
#include <numeric>
#include <vector>

#include "api_internal.hpp"
#include "block6.hpp"
#include "eliminate.hpp"
#include "lie.hpp"

namespace sgpu {

constexpr int kBatchMaxCams = 31;
constexpr int kRec = 21;     // doubles of a point's record
constexpr int kSegment = 8;  // most pairs of a segment

// Two camera blocks of a window: its first pair and its first full and partial segment there.
struct BatchSlot {
  int64_t pair, full, part;
};

struct BatchDev {
  int32_t nprob;
  const int32_t* order;      // launch slot -> problem (largest first)
  const int32_t* cam0;       // problem -> first camera (prefix, nprob + 1)
  const int32_t* pt0;        // problem -> first point
  const int32_t* obs0;       // problem -> first observation
  const double* intr;        // 4 per problem
  const double* poses_init;  // 7 per camera
  const double* points_init; // 3 per point
  double* poses[2];
  double* points[2];
  const int32_t* obs_cam;    // camera within the problem, sorted by point
  const double* obs_uv;
  const int32_t* pt_obs;     // global point -> first observation (npt_total + 1)
  const int32_t* obs_pt;     // observation -> point within the problem
  const int32_t* cam_pt;     // observations camera by camera: their point within the problem
  const double* cam_uv;      // and uv
  const int32_t* cam_ptr;    // camera -> its first entry of those (prefix)
  const int4* seg;           // segments of pairs (see segment())
  const int64_t* seg_ptr;    // problem -> first segment (prefix, nprob + 1)
  const int64_t* pair_ptr;   // problem -> its first pair (prefix, nprob + 1)
  const int32_t* pair_pt;    // point within the problem of each pair
  const int32_t* same;       // an observation per pair of observations of a point by one camera
  const int64_t* same_ptr;   // problem -> first entry of same (prefix, nprob + 1)
  const int32_t* pt_nu;      // reduced terms per point
  const int32_t* cam_nu;     // reduced terms per camera
  double* rec;               // kRec per point: x, H_ll^-1 (all 9: its triangles differ by rounding), damped
                             // H_ll upper (00, 01, 02, 11, 12, 22), neg-gradient s
  // per-problem LM state
  int32_t* cur;
  double* nu;
  double* merit;
  double* init_merit;
  int32_t* rejects;
  int32_t* steps;
  int32_t* done;
  int32_t* term;
  // parameters
  int32_t robust;
  double delta;
  double nu0;
  int64_t num_iterations;
  double function_tolerance, gradient_tolerance, parameter_tolerance;
  int64_t max_consecutive_rejects;
  int32_t lds_doubles;  // dynamic LDS per workgroup
  int32_t n_max;        // largest RCS dimension of the batch
};

namespace {

__host__ __device__ __forceinline__ int pk(int r, int c) {  // r >= c
  return int((unsigned(r) * unsigned(r + 1)) >> 1) + c;
}

// n pairs of camera blocks i and j < i from pair `first` of the problem (which may lie past 2^31).
__device__ __forceinline__ int4 segment(int i, int j, int n, int64_t first) {
  return make_int4(i | j << 8 | n << 16, 0, int(uint32_t(first)), int(first >> 32));
}

template <int NT>
__device__ double wg_sum(double v, double* red) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < NT / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

template <int NT>
__device__ double wg_max(double v, double* red) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v = fmax(v, __shfl_xor(v, m, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < NT / 64; ++w) t = fmax(t, red[w]);
  __syncthreads();
  return t;
}

__device__ __forceinline__ double huber_weight(int robust, double delta, double nrm) {
  if (robust != 1) return 1.0;
  if (nrm == 0.0) return 0.0;
  const double a = nrm <= delta ? nrm * nrm : 2.0 * delta * nrm - delta * delta;
  return sqrt(a) / nrm;
}

// camera_from_world R (row-major), t and the camera centre c, per camera, into LDS.
__device__ void cam_cache(const double* pose, double* out) {
  double inv[7], R[9];
  se3_inverse(pose, inv);
  so3_matrix(inv, R);
  for (int k = 0; k < 9; ++k) out[k] = R[k];
  for (int k = 0; k < 3; ++k) out[9 + k] = inv[4 + k];
  for (int k = 0; k < 3; ++k) out[12 + k] = pose[4 + k];
}

// Residual r = uv - K pi(R x + t) (FP64) and the Jacobian A = diag(f) dpi R (2x3, in T).
template <typename T>
__device__ __forceinline__ void obs_eval(const double* cc, const double* K, const double* uv,
                                         const double x[3], double r[2], T A[6]) {
  const double xc0 = cc[0] * x[0] + cc[1] * x[1] + cc[2] * x[2] + cc[9];
  const double xc1 = cc[3] * x[0] + cc[4] * x[1] + cc[5] * x[2] + cc[10];
  const double xc2 = cc[6] * x[0] + cc[7] * x[1] + cc[8] * x[2] + cc[11];
  const double iz = 1.0 / xc2;
  r[0] = uv[0] - (K[0] * xc0 * iz + K[2]);
  r[1] = uv[1] - (K[1] * xc1 * iz + K[3]);
  const T d00 = T(K[0] * iz), d02 = T(-K[0] * xc0 * iz * iz);
  const T d11 = T(K[1] * iz), d12 = T(-K[1] * xc1 * iz * iz);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    A[j] = d00 * T(cc[j]) + d02 * T(cc[6 + j]);
    A[3 + j] = d11 * T(cc[3 + j]) + d12 * T(cc[6 + j]);
  }
}

// The Jacobian's Gram matrix of a point in one camera.
template <typename T>
__device__ __forceinline__ void obs_gram(const double* cc, const double* K, const double x[3], T M[9]) {
  const double uv[2] = {0.0, 0.0};
  double r[2];
  T A[6];
  obs_eval<T>(cc, K, uv, x, r, A);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) M[3 * i + j] = A[i] * A[j] + A[3 + i] * A[3 + j];
}

// v + v of the lane that the DPP control kCtrl selects.
template <int kCtrl>
__device__ __forceinline__ double dpp_add(double v) {
  const int2 b = __builtin_bit_cast(int2, v);
  return v + __builtin_bit_cast(double, make_int2(__builtin_amdgcn_mov_dpp(b.x, kCtrl, 0xf, 0xf, true),
                                                  __builtin_amdgcn_mov_dpp(b.y, kCtrl, 0xf, 0xf, true)));
}

// Sum over each 16 consecutive lanes, in all of them.
__device__ __forceinline__ double row_sum(double v) {
  v = dpp_add<0xb1>(v);     // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4e>(v);     // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x124>(v);    // row_ror:4
  return dpp_add<0x128>(v);  // row_ror:8
}

template <typename T>
__device__ __forceinline__ void gram3(const T A[6], T M[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) M[3 * i + j] = A[i] * A[j] + A[3 + i] * A[3 + j];
}

template <typename T>
__device__ __forceinline__ void mul3(const T* A, const T* B, T* C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[3 * i + j] = A[3 * i] * B[j] + A[3 * i + 1] * B[3 + j] + A[3 * i + 2] * B[6 + j];
}

// u v - w t with the rounding fixed: w t rounded first, u v rounded first, or both.
__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
template <int kRounded, typename T>
__device__ __forceinline__ T cross(T u, T v, T w, T t) {
#pragma clang fp contract(off)
  if constexpr (kRounded == 1) return fma_t(u, v, -(w * t));
  if constexpr (kRounded == 2) return fma_t(-w, t, u * v);
  return u * v - w * t;
}

// B = P^T N P (P = [hat(-x) | I]): f(a, b, B_ab) for its 36 entries. The FP32 products of a
// mixed run are summed in FP64, and their rounding decides how a window goes on whose steps are
// often rejected: ends differed by up to 1e-3 in such windows when only the choice of the fused
// product was left to the compiler, which changes it with the code around. So it is written
// down, for the own term of an observation (kOwn) and the cross terms as each has always been.
template <bool kOwn, typename T, typename F>
__device__ __forceinline__ void lift(const T x[3], const T N[9], F f) {
  T HN[9], NHt[9], HNHt[9];
  HN[0] = cross<1>(x[1], N[6], x[2], N[3]);
  HN[1] = cross<1>(x[1], N[7], x[2], N[4]);
  HN[2] = cross<2>(x[1], N[8], x[2], N[5]);
  HN[3] = cross<2>(x[2], N[0], x[0], N[6]);
  HN[4] = cross<1>(x[2], N[1], x[0], N[7]);
  HN[5] = cross<1>(x[2], N[2], x[0], N[8]);
  HN[6] = cross<1>(x[0], N[3], x[1], N[0]);
  HN[7] = cross<2>(x[0], N[4], x[1], N[1]);
  HN[8] = cross<1>(x[0], N[5], x[1], N[2]);
  NHt[0] = cross<0>(x[1], N[2], x[2], N[1]);
  NHt[1] = cross<2>(x[2], N[0], x[0], N[2]);
  NHt[2] = cross<1>(x[0], N[1], x[1], N[0]);
  NHt[3] = cross<1>(x[1], N[5], x[2], N[4]);
  NHt[4] = cross<kOwn ? 1 : 0>(x[2], N[3], x[0], N[5]);
  NHt[5] = cross<2>(x[0], N[4], x[1], N[3]);
  NHt[6] = cross<2>(x[1], N[8], x[2], N[7]);
  NHt[7] = cross<1>(x[2], N[6], x[0], N[8]);
  NHt[8] = cross<kOwn ? 2 : 0>(x[0], N[7], x[1], N[6]);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    HNHt[3 * i] = cross<1>(x[1], HN[3 * i + 2], x[2], HN[3 * i + 1]);
    HNHt[3 * i + 1] = i == 0 ? cross<2>(x[2], HN[0], x[0], HN[2])
                             : cross<1>(x[2], HN[3 * i], x[0], HN[3 * i + 2]);
    HNHt[3 * i + 2] = cross<1>(x[0], HN[3 * i + 1], x[1], HN[3 * i]);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      f(a, b, HNHt[3 * a + b]);
      f(a, b + 3, HN[3 * a + b]);
      f(a + 3, b, NHt[3 * a + b]);
      f(a + 3, b + 3, N[3 * a + b]);
    }
}

constexpr int kPanel = 12;  // columns factored at a time: two 6x6 pivot blocks
typedef double mfma_d4 __attribute__((ext_vector_type(4)));

// eliminate_columns by the block pivot rule itself, for a panel with a pivot that it zeroes or
// could zero later: p and q as there; false if a pivot is not finite.
__device__ __forceinline__ bool eliminate_general(double (&p)[kPanel], double (&q)[kPanel], int w, double& dv,
                                  double& rv) {
  const int li = threadIdx.x & 15;
  bool ok = true;
  static_for<0, kPanel / 6>([&](auto blk) __attribute__((always_inline)) {
    constexpr int b0 = 6 * blk;
    if (b0 >= w) return;
    double a6[36], L[36], d[6], di[6];
    static_for<0, 6>([&](auto i) __attribute__((always_inline)) {
      static_for<0, i + 1>([&](auto j) __attribute__((always_inline)) {
        a6[6 * i + j] = a6[6 * j + i] = row_value<b0 + i>(p[b0 + j]);
      });
    });
    if (!ldlt6(a6, L, d, di)) {
      ok = false;
      for (int k = 0; k < 36; ++k) L[k] = (k % 7 == 0) ? 1.0 : 0.0;
      for (int k = 0; k < 6; ++k) d[k] = di[k] = 0.0;
    }
    static_for<0, 6>([&](auto i) __attribute__((always_inline)) {
      static_for<0, i>([&](auto t) __attribute__((always_inline)) {
        p[b0 + i] -= p[b0 + t] * L[6 * i + t];
        q[b0 + i] -= q[b0 + t] * L[6 * i + t];
      });
      dv = li == b0 + i ? d[i] : dv;
      rv = li == b0 + i ? di[i] : rv;
    });
    static_for<0, 6>([&](auto t) __attribute__((always_inline)) {
      const double lp = p[b0 + t] * di[t], lq = q[b0 + t] * di[t];
      static_for<b0 + 6, kPanel>([&](auto c) __attribute__((always_inline)) {
        const double u = row_value<c>(p[b0 + t]);
        p[c] -= lp * u;
        q[c] -= lq * u;
      });
    });
    // the pivot rows' own U: L_jj diag(d)
    static_for<0, 6>([&](auto i) __attribute__((always_inline)) {
      static_for<0, i>([&](auto t) __attribute__((always_inline)) {
        p[b0 + t] = li == b0 + i ? L[6 * i + t] * d[t] : p[b0 + t];
      });
    });
  });
  return ok;
}

// LDLt of the n x n system in S (packed lower triangle) with its right-hand side as row n, in
// place: S's columns become U = L D, row n the forward-solved right-hand side times D, rd
// the reciprocal pivots (0 for a zero pivot).
//
// Panels of 12 columns.  Each wavefront repeats the panel's pivot rows and eliminates 64 of
// the rows below in registers (eliminate_columns: no barrier or LDS access between pivots),
// then the trailing update runs on the matrix cores in 16x16 tiles.  The bound is the chain of
// n pivots and the tiles' LDS accesses (17 per lane and tile).
template <int NT>
__device__ __forceinline__ void window_ldlt(double* S, int n, double* rd, int* flags) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int lr = lane & 15, lc = lane >> 4;
  for (int o = 0; o < n; o += kPanel) {
    const int w = min(kPanel, n - o), r0 = o + w;  // rows below: r0..n (n: the right-hand side)
    double p[kPanel], q[kPanel], dv = 1.0, rv = 0.0;
    for (int c0 = r0 + 64 * wv; c0 <= n; c0 += NT) {
      const int r = min(c0 + lane, n), pr = o + min(lr, w - 1);
      auto load = [&] {
#pragma unroll
        for (int c = 0; c < kPanel; ++c) {
          const int cc = o + min(c, w - 1);
          p[c] = S[pk(max(pr, cc), min(pr, cc))];
          q[c] = S[pk(r, cc)];
        }
      };
      load();
      eliminate_columns<kPanel>(p, q, w, dv);
      rv = recip_nr(dv);
      // a pivot that the rule zeroes, or would once a larger one follows it (or not finite)
      double mx[2] = {1.0, 1.0};
      static_for<0, kPanel>([&](auto c) __attribute__((always_inline)) {
        mx[c / 6] = fmax(mx[c / 6], fabs(row_value<c>(dv)));
      });
      const double ad = fabs(dv);
      if (__any(lr < w && !(ad > (lr < 6 ? mx[0] : mx[1]) * 1e-12 && ad < __builtin_inf()))) {
        load();
        if (!eliminate_general(p, q, w, dv, rv)) flags[1] = 1;
      }
      if (c0 + lane <= n)
#pragma unroll
        for (int c = 0; c < kPanel; ++c)
          if (c < w) S[pk(r, o + c)] = q[c];
    }
    __syncthreads();  // every wavefront has read the pivot rows
    if (wv == 0 && lane < w) {
#pragma unroll
      for (int c = 0; c < kPanel; ++c)
        if (c < lane) S[pk(o + lane, o + c)] = p[c];
      rd[o + lane] = rv;
    }
    __syncthreads();
    // S(r, c) -= U(r, :) D^+ U(c, :)^T for r0 <= c <= r <= n, c < n
    const int nt = (n + 1 - r0 + 15) / 16;
    for (int t = wv; t < nt * (nt + 1) / 2; t += NT / 64) {
      int ti = int((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
      ti += (ti + 1) * (ti + 2) / 2 <= t;
      ti -= ti * (ti + 1) / 2 > t;
      const int tj = t - ti * (ti + 1) / 2;
      const int R = r0 + 16 * ti, c = r0 + 16 * tj + lr;
      mfma_d4 acc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = R + lc + 4 * i;
        acc[i] = S[c <= r && r <= n ? pk(r, c) : 0];
      }
      const int ra = min(R + lr, n), rc = min(c, n);
#pragma unroll
      for (int k = 0; k < kPanel; k += 4) {
        const int kk = o + min(k + lc, w - 1);
        const double rk = (k + lc < w ? -1.0 : 0.0) * rd[kk];  // a product, so that the load has no branch
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(rk * S[pk(ra, kk)], S[pk(rc, kk)], acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = R + lc + 4 * i;
        if (c <= r && r <= n && c < n) S[pk(r, c)] = acc[i];
      }
    }
    __syncthreads();
  }
}

// x = L^-T D^+ (row n of S) with the factor of window_ldlt.
template <int NT>
__device__ __forceinline__ void window_backsolve(const double* S, int n, const double* rd, double* x) {
  const int tid = threadIdx.x, lr = tid & 15;
  for (int e = tid; e < n; e += NT) x[e] = S[pk(n, e)] * rd[e];
  __syncthreads();
  for (int o = (n - 1) / kPanel * kPanel; o >= 0; o -= kPanel) {
    const int w = min(kPanel, n - o), me = o + min(lr, w - 1);
    if (tid < 64) {  // the panel's own columns, each 16 lanes alike
      double l[kPanel], v = x[me];
      const double rme = rd[me];
#pragma unroll
      for (int c = 1; c < kPanel; ++c) {  // the masks are products, so that the loads have no branches
        const int row = o + min(c, w - 1);
        l[c] = S[pk(row, min(me, row))] * (c < w && lr < c ? rme : 0.0);
      }
      static_for<0, kPanel - 1>([&](auto i) __attribute__((always_inline)) {
        constexpr int c = kPanel - 1 - i;
        v -= l[c] * row_value<c>(v);
      });
      if (tid < w) x[me] = v;
    }
    __syncthreads();
    for (int r = tid; r < o; r += NT) {
      double s[2] = {0.0, 0.0};
      if (w == kPanel) {
#pragma unroll
        for (int c = 0; c < kPanel; ++c) s[c & 1] += S[pk(o + c, r)] * x[o + c];
      } else {
        for (int c = 0; c < w; ++c) s[0] += S[pk(o + c, r)] * x[o + c];
      }
      x[r] -= (s[0] + s[1]) * rd[r];
    }
    __syncthreads();
  }
}

// The same system by 6x6 pivot blocks, L(:, k) = S(:, k) D_k^+ with D_k = L_6 diag(d) L_6^T
// (stored in the packed diagonal block, strict lower L_6 and diagonal d), and its solution
// into x.  The windows with FP32 Schur products keep this elimination so that they keep their
// results: their S is near singular once nu has fallen, and LM magnifies the rounding of single
// windows by 1e11.  Accuracy does not decide: of 36,000 runs of windows, 10 iterations each, 222 end
// more than 1e-4 from the same window's FP64 run with this order and 222 with the order of
// window_ldlt, 18 more than 0.1% above its cost and 18 below with either (geometric mean of the
// distances 8.9e-7).  Runs before the sums per camera and segment, whose S depended on the order
// of LDS atomics, differ among themselves by up to 5e-4 (norms over 1000 windows, 20 runs of a
// batch); the present ones repeat to 1e-15 and lie among those.  The order of window_ldlt takes
// 9.9 ms for 10 iterations of such a batch instead of 12.3 ms.
__device__ __forceinline__ void d_solve(const double* S, int k, double v[6]) {
  const int o = 6 * k;
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int j = 0; j < i; ++j) v[i] -= S[pk(o + i, o + j)] * v[j];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const double d = S[pk(o + i, o + i)];
    v[i] = d == 0.0 ? 0.0 : v[i] / d;
  }
#pragma unroll
  for (int i = 5; i >= 0; --i)
#pragma unroll
    for (int j = i + 1; j < 6; ++j) v[i] -= S[pk(o + j, o + i)] * v[j];
}

template <int NT>
__device__ __forceinline__ void window_block_solve(double* S, int n, double* W, double* x, int* flags) {
  const int tid = threadIdx.x, nbk = n / 6;
  for (int k = 0; k < nbk; ++k) {
    const int o = 6 * k, m = n - o - 6;
    if (tid == 0) {
      double Dk[36], L6[36], dk[6];
#pragma unroll
      for (int a = 0; a < 6; ++a)
#pragma unroll
        for (int b = 0; b <= a; ++b) Dk[6 * a + b] = Dk[6 * b + a] = S[pk(o + a, o + b)];
      if (!ldlt6(Dk, L6, dk)) {
        flags[1] = 1;
        for (int a = 0; a < 6; ++a) dk[a] = 0.0;
      }
#pragma unroll
      for (int a = 0; a < 6; ++a) {
#pragma unroll
        for (int b = 0; b < a; ++b) S[pk(o + a, o + b)] = L6[6 * a + b];
        S[pk(o + a, o + a)] = dk[a];
      }
    }
    __syncthreads();
    // W = S(:, k) below the diagonal block; L(:, k) = W D_k^+
    for (int r = o + 6 + tid; r < n; r += NT) {
      double v[6];
#pragma unroll
      for (int t = 0; t < 6; ++t) {
        v[t] = S[pk(r, o + t)];
        W[6 * (r - o - 6) + t] = v[t];
      }
      d_solve(S, k, v);
#pragma unroll
      for (int t = 0; t < 6; ++t) S[pk(r, o + t)] = v[t];
    }
    __syncthreads();
    // trailing update S(r, c) -= L(r, k) . W(c, k) for o + 6 <= c <= r, a row's columns over as
    // many threads as there are per row
    const int parts = m > 0 ? NT / m : 0;
    for (int e = tid; e < max(parts, 1) * m; e += NT) {
      const int i = e % m, part = e / m, r = o + 6 + i;
      double l[6];
#pragma unroll
      for (int t = 0; t < 6; ++t) l[t] = S[pk(r, o + t)];
      const int per = (i + 1 + max(parts, 1) - 1) / max(parts, 1);
      const int c1 = min((part + 1) * per, i + 1);
#pragma unroll 4
      for (int j = part * per; j < c1; ++j) {
        const double* w = W + 6 * j;
        S[pk(r, o + 6 + j)] -= l[0] * w[0] + l[1] * w[1] + l[2] * w[2] + l[3] * w[3] + l[4] * w[4] + l[5] * w[5];
      }
    }
    __syncthreads();
  }
  for (int e = tid; e < n; e += NT) x[e] = S[pk(n, e)];
  __syncthreads();
  for (int k = 0; k < nbk; ++k) {
    const int o = 6 * k;
    for (int r = o + 6 + tid; r < n; r += NT) {
      double s = 0.0;
#pragma unroll
      for (int t = 0; t < 6; ++t) s += S[pk(r, o + t)] * x[o + t];
      x[r] -= s;
    }
    __syncthreads();
  }
  for (int k = tid; k < nbk; k += NT) {
    double v[6];
    for (int t = 0; t < 6; ++t) v[t] = x[6 * k + t];
    d_solve(S, k, v);
    for (int t = 0; t < 6; ++t) x[6 * k + t] = v[t];
  }
  __syncthreads();
  for (int k = nbk - 1; k > 0; --k) {
    const int o = 6 * k;
    for (int r = tid; r < o; r += NT) {
      double s = 0.0;
#pragma unroll
      for (int a = 0; a < 6; ++a) s += S[pk(o + a, r)] * x[o + a];
      x[r] -= s;
    }
    __syncthreads();
  }
}

// One LM iteration of unfinished window p by the whole workgroup (lds: the dynamic LDS, red
// and flags (0: singular marginal block, 1: bad pivot) its static scratch).  Thread 0 takes
// the LM decision and writes the window's state; the other threads return before it, so a
// caller that goes on synchronizes first.
template <typename T, int NT>
__device__ __forceinline__ void batch_iteration(const BatchDev& d, int p, double* lds, double* red, int* flags) {
  const int c0 = d.cam0[p], nc = d.cam0[p + 1] - c0;
  const int q0 = d.pt0[p], np = d.pt0[p + 1] - q0;
  const int o0 = d.obs0[p], no = d.obs0[p + 1] - o0;
  const int nbk = nc - 1, n = 6 * nbk;  // camera 0 is constant
  const int cur = d.cur[p], nxt = 1 - cur;
  const double nu = d.nu[p];
  const double* K = d.intr + 4 * p;
  double* S = lds;                    // packed, row n the right-hand side
  double* grad = S + pk(d.n_max + 1, 0);
  double* xs = grad + d.n_max;
  double* rd = xs + d.n_max;          // reciprocal pivots (FP32 Schur products: 6 columns of S)
  double* cams = rd + (std::is_same<T, double>::value ? 1 : 6) * d.n_max;  // 15 per camera
  const int tid = threadIdx.x;
  const double* poses = d.poses[cur] + 7 * int64_t(c0);
  const double* points = d.points[cur] + 3 * int64_t(q0);
  // ---- linearize + Schur -------------------------------------------------------------------
  for (int c = tid; c < nc; c += NT) cam_cache(poses + 7 * c, cams + 15 * c);
  for (int e = tid; e < pk(n + 1, 0); e += NT) S[e] = 0.0;
  if (tid < 4) flags[tid] = 0;
  __syncthreads();
  double gmax = 0.0;
  for (int b = tid; b < np; b += NT) {
    const int gb = q0 + b;
    const double x[3] = {points[3 * b], points[3 * b + 1], points[3 * b + 2]};
    const int ob = d.pt_obs[gb], oe = d.pt_obs[gb + 1];
    double H[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, s[3] = {0, 0, 0};
    for (int o = ob; o < oe; ++o) {
      double r[2];
      T A[6], M[9];
      obs_eval<T>(cams + 15 * d.obs_cam[o], K, d.obs_uv + 2 * int64_t(o), x, r, A);
      const double w = huber_weight(d.robust, d.delta, sqrt(r[0] * r[0] + r[1] * r[1]));
      const double rw0 = d.robust == 1 ? w * r[0] : r[0], rw1 = d.robust == 1 ? w * r[1] : r[1];
      gram3(A, M);
      for (int k = 0; k < 9; ++k) H[k] += double(M[k]);
      for (int k = 0; k < 3; ++k) s[k] += double(A[k]) * rw0 + double(A[3 + k]) * rw1;
    }
    const double damp = nu * double(d.pt_nu[gb]);
    H[0] += damp;
    H[4] += damp;
    H[8] += damp;
    const double a0 = H[4] * H[8] - H[7] * H[5], a1 = H[3] * H[8] - H[6] * H[5], a2 = H[3] * H[7] - H[6] * H[4];
    const double det = H[0] * a0 - H[1] * a1 + H[2] * a2;
    double Hi[9];
    if (det == 0.0 || !isfinite(det)) {
      flags[0] = 1;
      for (int k = 0; k < 9; ++k) Hi[k] = 0.0;
    } else {
      Hi[0] = a0 / det;
      Hi[1] = (H[2] * H[7] - H[8] * H[1]) / det;
      Hi[2] = (H[1] * H[5] - H[4] * H[2]) / det;
      Hi[3] = -a1 / det;
      Hi[4] = (H[0] * H[8] - H[6] * H[2]) / det;
      Hi[5] = (H[2] * H[3] - H[5] * H[0]) / det;
      Hi[6] = a2 / det;
      Hi[7] = (H[1] * H[6] - H[7] * H[0]) / det;
      Hi[8] = (H[0] * H[4] - H[3] * H[1]) / det;
    }
    double* rec = d.rec + kRec * int64_t(gb);
    constexpr int up[6] = {0, 1, 2, 4, 5, 8};
    for (int k = 0; k < 3; ++k) {
      rec[k] = x[k];
      rec[18 + k] = s[k];
      gmax = fmax(gmax, fabs(s[k]));
    }
    for (int k = 0; k < 9; ++k) rec[3 + k] = Hi[k];
    for (int k = 0; k < 6; ++k) rec[12 + k] = H[up[k]];
  }
  __syncthreads();  // the point records are read below
  // own terms, camera by camera: 21 entries of M H^-1 (H - M) lifted, rhs and gradient
  for (int c = 1 + tid / 16; c < nc; c += NT / 16) {
    const int ci = c - 1;
    double own[33];
#pragma unroll
    for (int e = 0; e < 33; ++e) own[e] = 0.0;
    for (int q = d.cam_ptr[c0 + c] + (tid & 15); q < d.cam_ptr[c0 + c + 1]; q += 16) {
      const double* rec = d.rec + kRec * int64_t(q0 + d.cam_pt[q]);
      double h[kRec];
#pragma unroll
      for (int k = 0; k < kRec; ++k) h[k] = rec[k];
      const double x[3] = {h[0], h[1], h[2]};
      double r[2];
      T A[6], M[9], R[9], Z[9], N[9];
      obs_eval<T>(cams + 15 * c, K, d.cam_uv + 2 * int64_t(q), x, r, A);
      const double w = huber_weight(d.robust, d.delta, sqrt(r[0] * r[0] + r[1] * r[1]));
      const double rw0 = d.robust == 1 ? w * r[0] : r[0], rw1 = d.robust == 1 ? w * r[1] : r[1];
      gram3(A, M);
      const T Hi[9] = {T(h[3]), T(h[4]), T(h[5]), T(h[6]), T(h[7]), T(h[8]), T(h[9]), T(h[10]), T(h[11])};
      const double y[3] = {h[3] * h[18] + h[4] * h[19] + h[5] * h[20], h[6] * h[18] + h[7] * h[19] + h[8] * h[20],
                           h[9] * h[18] + h[10] * h[19] + h[11] * h[20]};
      double v[3], t[3];
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        constexpr int at[9] = {12, 13, 14, 13, 15, 16, 14, 16, 17};
        R[k] = T(h[at[k]] - double(M[k]));
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        v[k] = double(A[k]) * rw0 + double(A[3 + k]) * rw1;
        t[k] = double(M[3 * k]) * y[0] + double(M[3 * k + 1]) * y[1] + double(M[3 * k + 2]) * y[2] - v[k];
      }
      // rhs += P^T t = [x cross t; t]; gradient -= P^T v
      own[21] += x[1] * t[2] - x[2] * t[1];
      own[22] += x[2] * t[0] - x[0] * t[2];
      own[23] += x[0] * t[1] - x[1] * t[0];
      own[27] -= x[1] * v[2] - x[2] * v[1];
      own[28] -= x[2] * v[0] - x[0] * v[2];
      own[29] -= x[0] * v[1] - x[1] * v[0];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        own[24 + k] += t[k];
        own[30 + k] -= v[k];
      }
      mul3(M, Hi, Z);
      mul3(Z, R, N);
      const T xt[3] = {T(x[0]), T(x[1]), T(x[2])};
      lift<true>(xt, N, [&](int a, int b2, T val) {
        if (b2 <= a) own[a * (a + 1) / 2 + b2] += double(val);
      });
    }
#pragma unroll
    for (int e = 0; e < 33; ++e) own[e] = row_sum(own[e]);
    // the diagonal block also takes the damping (one per reduced term), and below the terms of
    // a point's repeated observations of one camera: atomic, as those may come first
    if ((tid & 15) == 0) {
#pragma unroll
      for (int a = 0; a < 6; ++a) {
#pragma unroll
        for (int b = 0; b <= a; ++b)
          atomicAdd(&S[pk(6 * ci + a, 6 * ci + b)],
                    own[a * (a + 1) / 2 + b] + (a == b ? nu * double(d.cam_nu[c0 + c]) : 0.0));
        S[pk(n, 6 * ci + a)] = own[21 + a];
        grad[6 * ci + a] = own[27 + a];
      }
    }
  }
  // cross terms: a thread per segment of points shared by two cameras
  const int32_t* pairs = d.pair_pt + d.pair_ptr[p];
  for (int64_t e = d.seg_ptr[p] + tid; e < d.seg_ptr[p + 1]; e += NT) {
    const int4 sg = d.seg[e];
    const int bi = sg.x & 255, bj = sg.x >> 8 & 255;
    double acc[36], ci[12], cj[12];
#pragma unroll
    for (int k = 0; k < 36; ++k) acc[k] = 0.0;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      ci[k] = cams[15 * (bi + 1) + k];
      cj[k] = cams[15 * (bj + 1) + k];
    }
    const int32_t* pt = pairs + (int64_t(sg.w) << 32 | uint32_t(sg.z));
    for (int q = 0; q < sg.x >> 16; ++q) {
      const double* h = d.rec + kRec * int64_t(q0 + pt[q]);
      const double x[3] = {h[0], h[1], h[2]};
      const T xt[3] = {T(x[0]), T(x[1]), T(x[2])};
      const T Hi[9] = {T(h[3]), T(h[4]), T(h[5]), T(h[6]), T(h[7]), T(h[8]), T(h[9]), T(h[10]), T(h[11])};
      T M[9], Z[9], N[9];
      obs_gram<T>(ci, K, x, M);
      mul3(M, Hi, Z);
      obs_gram<T>(cj, K, x, M);
      mul3(Z, M, N);
      lift<false>(xt, N, [&](int a, int b2, T val) { acc[6 * a + b2] -= double(val); });
    }
    double* row = S + pk(6 * bi, 6 * bj);
#pragma unroll
    for (int a = 0; a < 6; ++a)
#pragma unroll
      for (int b2 = 0; b2 < 6; ++b2) atomicAdd(row + (6 * bi * a + a * (a + 1) / 2 + b2), acc[6 * a + b2]);
  }
  // a point's repeated observations of one camera: the pair in both orders, B + B^T
  for (int64_t e = d.same_ptr[p] + tid; e < d.same_ptr[p + 1]; e += NT) {
    const int ci = d.obs_cam[d.same[e]] - 1;
    const double* h = d.rec + kRec * int64_t(q0 + d.obs_pt[d.same[e]]);
    const double x[3] = {h[0], h[1], h[2]};
    const T xt[3] = {T(x[0]), T(x[1]), T(x[2])};
    const T Hi[9] = {T(h[3]), T(h[4]), T(h[5]), T(h[6]), T(h[7]), T(h[8]), T(h[9]), T(h[10]), T(h[11])};
    T M[9], Z[9], N[9];
    obs_gram<T>(cams + 15 * (ci + 1), K, x, M);
    mul3(M, Hi, Z);
    mul3(Z, M, N);
    lift<false>(xt, N, [&](int a, int b2, T val) {
      atomicAdd(&S[pk(6 * ci + max(a, b2), 6 * ci + min(a, b2))], (a == b2 ? -2.0 : -1.0) * double(val));
    });
  }
  __syncthreads();
  for (int e = tid; e < n; e += NT) gmax = fmax(gmax, fabs(grad[e]));
  const double max_grad = wg_max<NT>(gmax, red);
  if constexpr (std::is_same<T, double>::value) {
    window_ldlt<NT>(S, n, rd, flags);
    window_backsolve<NT>(S, n, rd, xs);
  } else {
    window_block_solve<NT>(S, n, rd, xs, flags);
  }
  // ---- back-substitution, update, proposal merit ----------------------------------------------
  double dd = 0.0, dg = 0.0, dmax = 0.0;
  double* pnew = d.points[nxt] + 3 * int64_t(q0);
  for (int b = tid; b < np; b += NT) {
    const int gb = q0 + b;
    double h[kRec];
#pragma unroll
    for (int k = 0; k < kRec; ++k) h[k] = d.rec[kRec * int64_t(gb) + k];
    const double x[3] = {h[0], h[1], h[2]};
    double acc[3] = {h[18], h[19], h[20]};
    for (int o = d.pt_obs[gb]; o < d.pt_obs[gb + 1]; ++o) {
      const int ci = d.obs_cam[o] - 1;
      if (ci < 0) continue;
      T M[9];
      obs_gram<T>(cams + 15 * (ci + 1), K, x, M);
      const double* dx = xs + 6 * ci;
      const double q[3] = {dx[1] * x[2] - dx[2] * x[1] + dx[3], dx[2] * x[0] - dx[0] * x[2] + dx[4],
                           dx[0] * x[1] - dx[1] * x[0] + dx[5]};
      for (int k = 0; k < 3; ++k)
        acc[k] += double(M[3 * k]) * q[0] + double(M[3 * k + 1]) * q[1] + double(M[3 * k + 2]) * q[2];
    }
    const double* Hi = h + 3;
    for (int k = 0; k < 3; ++k) {
      const double dk = Hi[3 * k] * acc[0] + Hi[3 * k + 1] * acc[1] + Hi[3 * k + 2] * acc[2];
      pnew[3 * b + k] = x[k] + dk;
      dd += dk * dk;
      dg += dk * h[18 + k];
      dmax = fmax(dmax, fabs(dk));
    }
  }
  double* tnew = d.poses[nxt] + 7 * int64_t(c0);
  for (int c = tid; c < nc; c += NT) {
    if (c == 0) {
      for (int k = 0; k < 7; ++k) tnew[k] = poses[k];
      continue;
    }
    double t[6], T1[7];
    for (int k = 0; k < 6; ++k) {
      t[k] = xs[6 * (c - 1) + k];
      dd += t[k] * t[k];
      dg += t[k] * grad[6 * (c - 1) + k];
      dmax = fmax(dmax, fabs(t[k]));
    }
    se3_oplus(poses + 7 * c, t, T1);
    for (int k = 0; k < 7; ++k) tnew[7 * c + k] = T1[k];
  }
  __syncthreads();  // proposal poses are read below
  // cameras of the proposal into the cache
  for (int c = tid; c < nc; c += NT) cam_cache(tnew + 7 * c, cams + 15 * c);
  __syncthreads();
  double cost = 0.0;
  for (int o = tid; o < no; o += NT) {
    const int go = o0 + o;
    const double* xp = pnew + 3 * d.obs_pt[go];
    const double x[3] = {xp[0], xp[1], xp[2]};
    double r[2];
    double A[6];
    obs_eval<double>(cams + 15 * d.obs_cam[go], K, d.obs_uv + 2 * int64_t(go), x, r, A);
    const double nrm2 = r[0] * r[0] + r[1] * r[1];
    if (d.robust == 1) {
      const double w = huber_weight(1, d.delta, sqrt(nrm2));
      cost += w * w * nrm2;
    } else {
      cost += nrm2;
    }
  }
  const double new_merit = wg_sum<NT>(cost, red);
  const double dd_s = wg_sum<NT>(dd, red);
  const double dg_s = wg_sum<NT>(dg, red);
  const double max_step = wg_max<NT>(dmax, red);
  if (tid != 0) return;
  // ---- LM decision (step_nlls_inner order, optimizer_step.rs:366-443) -------------------------
  int reason = 0, accepted = 0;
  double nu_next = nu, merit = d.merit[p];
  int rejects = d.rejects[p];
  if (max_grad < d.gradient_tolerance) {
    reason = 3;  // GradientTolerance
  } else if (flags[0] || flags[1]) {
    nu_next = 2.0 * nu;
    if (++rejects >= d.max_consecutive_rejects) reason = 5;
  } else if (max_step < d.parameter_tolerance) {
    if (new_merit < merit) {
      accepted = 1;
      merit = new_merit;
    }
    reason = 4;
  } else {
    const double pred = nu * dd_s + dg_s;
    const double actual = merit - new_merit;
    const double rho = fabs(pred) > DBL_MIN ? actual / pred : (actual > 0 ? 1.0 : 0.0);
    if (rho > 0.0 && new_merit < merit) {
      const double f = 1.0 - pow(2.0 * rho - 1.0, 3.0);
      nu_next = nu * fmax(f, 1.0 / 3.0);
      rejects = 0;
      if ((merit - new_merit) / (fabs(merit) + DBL_MIN) < d.function_tolerance) reason = 2;
      merit = new_merit;
      accepted = 1;
    } else {
      nu_next = 2.0 * nu;
      if (++rejects >= d.max_consecutive_rejects) reason = 5;
    }
  }
  const int steps = d.steps[p] + 1;
  if (steps >= d.num_iterations && reason == 0) reason = 1;
  if (accepted) d.cur[p] = nxt;
  d.nu[p] = nu_next;
  d.merit[p] = merit;
  d.rejects[p] = rejects;
  d.steps[p] = steps;
  if (reason) {
    d.done[p] = 1;
    d.term[p] = reason;
  }
}

// One LM iteration of every unfinished window: one workgroup per window, largest first.
template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_batch_step(BatchDev d) {
  extern __shared__ double lds[];
  __shared__ double red[NT / 64];
  __shared__ int flags[4];
  const int p = d.order[blockIdx.x];
  if (d.done[p]) return;  // uniform per workgroup
  batch_iteration<T, NT>(d, p, lds, red, flags);
}

// Every window's LM run in one launch: each workgroup takes the next window (largest first)
// from a queue counter and runs up to `iterations` LM iterations of it until it terminates,
// then takes the next; the grid is sized to the resident workgroups.  Nothing waits on
// another workgroup, and every loop is bounded (windows, iterations), so the grid always
// drains.  t_start / t_end: the device wall clock when a window was taken and when its run
// ended.
template <typename T, int NT>
__global__ void __launch_bounds__(NT)
    k_batch_persistent(BatchDev d, int32_t iterations, int32_t* __restrict__ queue,
                       unsigned long long* __restrict__ t_start, unsigned long long* __restrict__ t_end) {
  extern __shared__ double lds[];
  __shared__ double red[NT / 64];
  __shared__ int flags[4];
  __shared__ int s_slot, s_done;
  for (;;) {
    if (threadIdx.x == 0) s_slot = atomicAdd(queue, 1);
    __syncthreads();
    const int slot = s_slot;
    if (slot >= d.nprob) return;  // uniform per workgroup
    const int p = d.order[slot];
    if (threadIdx.x == 0) {
      t_start[p] = (unsigned long long)wall_clock64();
      s_done = d.done[p];
    }
    __syncthreads();
    for (int it = 0; it < iterations && !s_done; ++it) {
      // p is uniform, but read from LDS the compiler cannot know it: made a scalar so that
      // the addresses derived from it stay in scalar registers
      batch_iteration<T, NT>(d, __builtin_amdgcn_readfirstlane(p), lds, red, flags);
      __syncthreads();
      if (threadIdx.x == 0) s_done = d.done[p];
      __syncthreads();
    }
    if (threadIdx.x == 0) t_end[p] = (unsigned long long)wall_clock64();
    __syncthreads();
  }
}

// Every window's current variables, side by side.
__global__ void __launch_bounds__(256)
    k_batch_gather(BatchDev d, double* __restrict__ poses, double* __restrict__ points) {
  const int p = blockIdx.x, cur = d.cur[p];
  const int64_t c0 = 7 * int64_t(d.cam0[p]), c1 = 7 * int64_t(d.cam0[p + 1]);
  const int64_t q0 = 3 * int64_t(d.pt0[p]), q1 = 3 * int64_t(d.pt0[p + 1]);
  for (int64_t e = c0 + threadIdx.x; e < c1; e += 256) poses[e] = d.poses[cur][e];
  for (int64_t e = q0 + threadIdx.x; e < q1; e += 256) points[e] = d.points[cur][e];
}

// The lists of a window that follow from its sorted observations, one workgroup per window:
// the point of each observation, the observations camera by camera, and the points that two
// cameras share with their segments.  A wavefront takes a camera and goes through the window's observations 64 at
// a time, in order; an entry's place is the camera's (the pair's) count so far plus the
// entries of lower lanes, so the lists come out as if written one by one.  Built on the host
// they cost 250 ms for 1000 windows of 5300 observations, most of it page faults of 230 MB.
constexpr int kListThreads = 512;
__global__ void __launch_bounds__(kListThreads)
    k_batch_lists(BatchDev d, const BatchSlot* __restrict__ slots, const int64_t* __restrict__ slot_ptr,
                  int32_t* obs_pt, int32_t* __restrict__ cam_pt, double* __restrict__ cam_uv,
                  int32_t* __restrict__ pair_pt, int4* __restrict__ seg) {
  const int p = blockIdx.x, lane = threadIdx.x & 63;
  const int c0 = d.cam0[p], nc = d.cam0[p + 1] - c0, q0 = d.pt0[p], np = d.pt0[p + 1] - q0;
  const int o0 = d.obs0[p], o1 = d.obs0[p + 1];
  for (int b = threadIdx.x; b < np; b += kListThreads)
    for (int o = d.pt_obs[q0 + b]; o < d.pt_obs[q0 + b + 1]; ++o) obs_pt[o] = b;
  __syncthreads();
  const unsigned long long below = (1ull << lane) - 1;
  int32_t* pairs = pair_pt + d.pair_ptr[p];
  const BatchSlot* sl = slots + slot_ptr[p];  // one more than there are slots: the end
  seg += d.seg_ptr[p];
  for (int ci = 1, k = 0; ci < nc - 1; ++ci)
    for (int cj = 0; cj < ci; ++cj, ++k) {
      if (k % (kListThreads / 64) != threadIdx.x >> 6) continue;
      const BatchSlot z = sl[k];
      const int64_t n = sl[k + 1].pair - z.pair, full = n / kSegment;
      for (int64_t t = lane; t < full; t += 64) seg[z.full + t] = segment(ci, cj, kSegment, z.pair + t * kSegment);
      if (lane == 0 && n % kSegment)
        seg[z.part] = segment(ci, cj, int(n % kSegment), z.pair + full * kSegment);
    }
  for (int c = threadIdx.x >> 6; c < nc; c += kListThreads / 64) {
    const int ci = c - 1;
    int q = d.cam_ptr[c0 + c];
    // lane j: where the next pair of blocks ci and j goes
    long long to = lane < ci ? sl[ci * (ci - 1) / 2 + lane].pair : 0;
    for (int z = o0; z < o1; z += 64) {
      const int o = z + lane;
      const bool mine = o < o1 && d.obs_cam[min(o, o1 - 1)] == c;
      const unsigned long long m = __ballot(mine);
      if (m == 0) continue;
      int b = 0, first = 0;
      unsigned with = 0;  // blocks j < ci that see the point, and whether one does twice
      bool twice = false;
      if (mine) {
        const int at = q + __popcll(m & below);
        b = obs_pt[o];
        cam_pt[at] = b;
        cam_uv[2 * int64_t(at)] = d.obs_uv[2 * int64_t(o)];
        cam_uv[2 * int64_t(at) + 1] = d.obs_uv[2 * int64_t(o) + 1];
        first = d.pt_obs[q0 + b];
        for (int j = first; j < o; ++j) {
          const int cj = d.obs_cam[j] - 1;
          if (cj < 0 || cj == ci) continue;
          twice |= (with >> cj & 1) != 0;
          with |= 1u << cj;
        }
      }
      q += __popcll(m);
      const bool counts = __ballot(twice) != 0;
      for (int cj = 0; cj < ci; ++cj) {
        const unsigned long long see = __ballot(with >> cj & 1);
        if (see == 0) continue;
        int n = with >> cj & 1, before = __popcll(see & below), all = __popcll(see);
        if (counts) {  // several pairs of one point: a running sum over the lanes
          if (n) {
            n = 0;
            for (int j = first; j < o; ++j) n += d.obs_cam[j] - 1 == cj;
          }
          int sum = n;
          for (int s = 1; s < 64; s *= 2) {
            const int lower = __shfl_up(sum, s);
            if (lane >= s) sum += lower;
          }
          before = sum - n;
          all = __shfl(sum, 63);
        }
        const long long at = __shfl(to, cj) + before;
        for (int k = 0; k < n; ++k) pairs[at + k] = b;
        if (lane == cj) to += all;
      }
    }
  }
}

__global__ void k_batch_zero_queue(int32_t* queue) {
  if (threadIdx.x == 0) *queue = 0;
}

// State from the initial values and the initial merit.
template <int NT>
__global__ void __launch_bounds__(NT) k_batch_init(BatchDev d) {
  __shared__ double red[NT / 64];
  __shared__ double cams[15 * kBatchMaxCams];
  const int p = blockIdx.x;
  const int c0 = d.cam0[p], nc = d.cam0[p + 1] - c0;
  const int q0 = d.pt0[p], np = d.pt0[p + 1] - q0;
  const int o0 = d.obs0[p], no = d.obs0[p + 1] - o0;
  for (int e = threadIdx.x; e < 7 * nc; e += NT) d.poses[0][7 * int64_t(c0) + e] = d.poses_init[7 * int64_t(c0) + e];
  for (int e = threadIdx.x; e < 3 * np; e += NT) d.points[0][3 * int64_t(q0) + e] = d.points_init[3 * int64_t(q0) + e];
  for (int c = threadIdx.x; c < nc; c += NT) cam_cache(d.poses_init + 7 * int64_t(c0 + c), cams + 15 * c);
  __syncthreads();
  const double* K = d.intr + 4 * p;
  double cost = 0.0;
  for (int o = threadIdx.x; o < no; o += NT) {
    const int go = o0 + o;
    const double* xp = d.points_init + 3 * int64_t(q0 + d.obs_pt[go]);
    const double x[3] = {xp[0], xp[1], xp[2]};
    double r[2], A[6];
    obs_eval<double>(cams + 15 * d.obs_cam[go], K, d.obs_uv + 2 * int64_t(go), x, r, A);
    const double nrm2 = r[0] * r[0] + r[1] * r[1];
    if (d.robust == 1) {
      const double w = huber_weight(1, d.delta, sqrt(nrm2));
      cost += w * w * nrm2;
    } else {
      cost += nrm2;
    }
  }
  const double m = wg_sum<NT>(cost, red);
  if (threadIdx.x == 0) {
    d.cur[p] = 0;
    d.nu[p] = d.nu0;
    d.merit[p] = m;
    d.init_merit[p] = m;
    d.rejects[p] = 0;
    d.steps[p] = 0;
    d.done[p] = d.num_iterations <= 0 ? 1 : 0;
    d.term[p] = d.num_iterations <= 0 ? 1 : 0;
  }
}

}  // namespace
}  // namespace sgpu

using namespace sgpu;

struct sgpu_batch {
  BatchDev d{};
  DeviceArena arena;
  hipStream_t stream = nullptr;
  int precision = 0;
  int threads = 256;           // chosen by the autotuner
  double tune_ms[3] = {0, 0, 0};
  size_t lds_bytes = 0;
  int64_t ncam = 0, npt = 0, nobs = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  int graph_iters = 0;
  // the persistent launch: queue counter, per-window wall-clock stamps, its own graph
  double *out_poses = nullptr, *out_points = nullptr;  // results, gathered
  int32_t* queue = nullptr;
  unsigned long long* t_start = nullptr;
  unsigned long long* t_end = nullptr;
  int persistent_grid = 0;     // resident workgroups of the persistent kernel's size
  int persistent_threads = 256;  // the persistent kernel's workgroup size (its own autotuner)
  double ptune_ms[3] = {0, 0, 0};
  double clock_khz = 0.0;   // device wall-clock rate
  hipGraph_t pgraph = nullptr;
  hipGraphExec_t pgraph_exec = nullptr;
  int pgraph_iters = -1;

  ~sgpu_batch() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (pgraph_exec) (void)hipGraphExecDestroy(pgraph_exec);
    if (pgraph) (void)hipGraphDestroy(pgraph);
    if (stream) (void)hipStreamDestroy(stream);
  }

  void launch_persistent(int iterations) {
    hipLaunchKernelGGL(k_batch_zero_queue, dim3(1), dim3(64), 0, stream, queue);
    const dim3 g(persistent_grid);
    const int nt = persistent_threads;
    if (precision == SGPU_PRECISION_MIXED) {
      if (nt == 128) hipLaunchKernelGGL((k_batch_persistent<float, 128>), g, dim3(128), lds_bytes, stream, d, iterations, queue, t_start, t_end);
      else if (nt == 512) hipLaunchKernelGGL((k_batch_persistent<float, 512>), g, dim3(512), lds_bytes, stream, d, iterations, queue, t_start, t_end);
      else hipLaunchKernelGGL((k_batch_persistent<float, 256>), g, dim3(256), lds_bytes, stream, d, iterations, queue, t_start, t_end);
    } else {
      if (nt == 128) hipLaunchKernelGGL((k_batch_persistent<double, 128>), g, dim3(128), lds_bytes, stream, d, iterations, queue, t_start, t_end);
      else if (nt == 512) hipLaunchKernelGGL((k_batch_persistent<double, 512>), g, dim3(512), lds_bytes, stream, d, iterations, queue, t_start, t_end);
      else hipLaunchKernelGGL((k_batch_persistent<double, 256>), g, dim3(256), lds_bytes, stream, d, iterations, queue, t_start, t_end);
    }
  }

  void launch_init() {
    hipLaunchKernelGGL((k_batch_init<256>), dim3(d.nprob), dim3(256), 0, stream, d);
  }
  void launch_step(int nt) {
    const dim3 g(d.nprob);
    if (precision == SGPU_PRECISION_MIXED) {
      if (nt == 128) hipLaunchKernelGGL((k_batch_step<float, 128>), g, dim3(128), lds_bytes, stream, d);
      else if (nt == 512) hipLaunchKernelGGL((k_batch_step<float, 512>), g, dim3(512), lds_bytes, stream, d);
      else hipLaunchKernelGGL((k_batch_step<float, 256>), g, dim3(256), lds_bytes, stream, d);
    } else {
      if (nt == 128) hipLaunchKernelGGL((k_batch_step<double, 128>), g, dim3(128), lds_bytes, stream, d);
      else if (nt == 512) hipLaunchKernelGGL((k_batch_step<double, 512>), g, dim3(512), lds_bytes, stream, d);
      else hipLaunchKernelGGL((k_batch_step<double, 256>), g, dim3(256), lds_bytes, stream, d);
    }
  }
};

namespace {

// Device arrays in one allocation.  A small batch's creation is bound by the calls: with an
// allocation, a copy and a free for each of its 40 arrays four windows of 2 cameras took 1.06 ms
// (creation and destruction), so 0.75.  Up to kStage bytes of host values go up in one copy, more go
// from where they are (a second pass over them would cost more).
struct DeviceBlock {
  static constexpr size_t kStage = size_t(1) << 20;
  struct Part {
    void* dst;  // where the array's address goes
    const void* src;
    size_t at, bytes;
  };
  std::vector<Part> parts;
  size_t size = 0, filled = 0;  // bytes in all, and up to the end of the last host values
  template <typename T>
  void add(T*& dst, size_t n, const std::remove_const_t<T>* src = nullptr) {
    parts.push_back({&dst, src, size, n * sizeof(T)});
    size = (size + std::max<size_t>(n * sizeof(T), 1) + 255) & ~size_t(255);
    if (src) filled = parts.back().at + parts.back().bytes;
  }
  template <typename T>
  void add(const T*& dst, const std::vector<T>& v) {
    add(dst, v.size(), v.data());
  }
  void commit(DeviceArena& arena) {
    char* base = arena.alloc<char>(size);
    std::vector<char> stage(filled <= kStage ? filled : 0);
    for (const Part& p : parts) {
      void* at = base + p.at;
      std::memcpy(p.dst, &at, sizeof(at));
      if (!p.src || !p.bytes) continue;
      if (!stage.empty()) std::memcpy(stage.data() + p.at, p.src, p.bytes);
      else SGPU_HIP(hipMemcpy(at, p.src, p.bytes, hipMemcpyHostToDevice));
    }
    if (!stage.empty()) SGPU_HIP(hipMemcpy(base, stage.data(), stage.size(), hipMemcpyHostToDevice));
  }
};

template <typename F>
void set_lds(F kernel, size_t bytes) {
  SGPU_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
}
}  // namespace

extern "C" {

sgpu_status sgpu_batch_create(const sgpu_batch_desc* desc, const sgpu_opt_params* params,
                              sgpu_batch** out) {
  return guarded([&] {
    if (!desc || !params || !out) throw Error(SGPU_ERR_INVALID_ARGUMENT, "desc, params and out required");
    *out = nullptr;
    const int64_t P = desc->num_problems;
    if (P <= 0 || P > INT32_MAX / 2 || !desc->cam_ptr || !desc->point_ptr || !desc->obs_ptr ||
        !desc->intrinsics || !desc->poses || !desc->points || !desc->obs_cam || !desc->obs_point ||
        !desc->obs_uv)
      throw Error(SGPU_ERR_INVALID_ARGUMENT, "incomplete batch description");
    if (params->precision != SGPU_PRECISION_F64 && params->precision != SGPU_PRECISION_MIXED)
      throw Error(SGPU_ERR_INVALID_ARGUMENT, "unknown precision");
    if (params->solver != SGPU_SOLVER_SCHUR_BLOCK_SPARSE_LDLT)
      throw Error(SGPU_ERR_UNSUPPORTED, "the batched path solves each window directly");
    const int64_t C = desc->cam_ptr[P], Q = desc->point_ptr[P], O = desc->obs_ptr[P];
    if (desc->cam_ptr[0] != 0 || desc->point_ptr[0] != 0 || desc->obs_ptr[0] != 0 || O > INT32_MAX ||
        Q > INT32_MAX || C > INT32_MAX)
      throw Error(SGPU_ERR_INVALID_ARGUMENT, "bad prefix arrays");
    int n_max = 0;
    std::vector<int32_t> cam0(P + 1), pt0(P + 1), obs0(P + 1), pt_obs(Q + 1), pt_nu(Q, 0), cam_nu(C, 0),
        cam_ptr(C + 1, 0), same;
    std::vector<int64_t> pair_ptr(P + 1, 0), seg_ptr(P + 1, 0), same_ptr(P + 1, 0), slot_ptr(P + 1, 0);
    std::vector<BatchSlot> slots;
    for (int64_t p = 0; p <= P; ++p) {
      cam0[p] = int32_t(desc->cam_ptr[p]);
      pt0[p] = int32_t(desc->point_ptr[p]);
      obs0[p] = int32_t(desc->obs_ptr[p]);
    }
    bool sorted = true;
    for (int64_t p = 0; p < P; ++p) {
      const int64_t nc = cam0[p + 1] - cam0[p], np = pt0[p + 1] - pt0[p], no = obs0[p + 1] - obs0[p];
      if (nc < 2 || nc > kBatchMaxCams || np < 1 || no < 1)
        throw Error(nc > kBatchMaxCams ? SGPU_ERR_UNSUPPORTED : SGPU_ERR_INVALID_ARGUMENT,
                    "each window needs 2.." + std::to_string(kBatchMaxCams) +
                        " cameras, points and observations");
      n_max = std::max<int>(n_max, int(6 * (nc - 1)));
      const int32_t* oc = desc->obs_cam + obs0[p];
      const int32_t* op = desc->obs_point + obs0[p];
      int32_t* first = pt_obs.data() + pt0[p];
      for (int64_t k = 0; k < no; ++k) {
        if (oc[k] < 0 || oc[k] >= nc || op[k] < 0 || op[k] >= np)
          throw Error(SGPU_ERR_INDEX_OUT_OF_RANGE, "observation index out of range");
        ++first[op[k]];
        sorted &= k == 0 || op[k] > op[k - 1] || (op[k] == op[k - 1] && oc[k] >= oc[k - 1]);
      }
    }
    // observations of each window by (point, camera) (CostFn::sort order): two stable counting
    // passes, none if they come that way
    for (int64_t q = 0, at = 0; q <= Q; ++q) {
      const int32_t c = pt_obs[q];
      pt_obs[q] = int32_t(at);
      at += c;
    }
    const int32_t* obs_cam = desc->obs_cam;
    const double* uv = desc->obs_uv;
    std::vector<int32_t> cam_sorted;
    std::vector<double> uv_sorted;
    if (!sorted) {
      cam_sorted.resize(O);
      uv_sorted.resize(2 * O);
      std::vector<int32_t> by_cam, to(pt_obs);
      for (int64_t p = 0; p < P; ++p) {
        const int64_t no = obs0[p + 1] - obs0[p], ob = obs0[p];
        int32_t at[kBatchMaxCams + 1] = {};
        by_cam.resize(no);
        for (int64_t k = 0; k < no; ++k) ++at[desc->obs_cam[ob + k] + 1];
        for (int c = 0; c < kBatchMaxCams; ++c) at[c + 1] += at[c];
        for (int64_t k = 0; k < no; ++k) by_cam[at[desc->obs_cam[ob + k]]++] = int32_t(k);
        for (int64_t k = 0; k < no; ++k) {
          const int64_t o = ob + by_cam[k], q = to[pt0[p] + desc->obs_point[o]]++;
          cam_sorted[q] = desc->obs_cam[o];
          uv_sorted[2 * q] = desc->obs_uv[2 * o];
          uv_sorted[2 * q + 1] = desc->obs_uv[2 * o + 1];
        }
      }
      obs_cam = cam_sorted.data();
      uv = uv_sorted.data();
    }
    for (int64_t p = 0; p < P; ++p) {
      const int64_t nc = cam0[p + 1] - cam0[p], np = pt0[p + 1] - pt0[p];
      // reduced terms (distinct (camera, point) pairs), and how many points each two cameras
      // (other than camera 0) share
      const int64_t nslot = (nc - 1) * (nc - 2) / 2;
      int64_t slot[kBatchMaxCams * kBatchMaxCams / 2 + 1] = {};
      int32_t at[kBatchMaxCams + 1] = {};
      for (int64_t b = 0; b < np; ++b) {
        const int32_t o0 = pt_obs[pt0[p] + b], o1 = pt_obs[pt0[p] + b + 1];
        int32_t last = -1, nu = 0;
        for (int32_t i = o0; i < o1; ++i) {
          const int32_t c = obs_cam[i], ci = c - 1;
          ++at[c + 1];
          if (c != last) ++nu, ++cam_nu[cam0[p] + c];
          last = c;
          if (ci < 0) continue;
          int64_t* row = slot + ci * (ci - 1) / 2 + 1;
          for (int32_t j = o0; j < i; ++j) {
            const int32_t cj = obs_cam[j] - 1;
            if (cj == ci) same.push_back(i);
            else if (cj >= 0) ++row[cj];
          }
        }
        pt_nu[pt0[p] + b] = nu;
      }
      // the observations camera by camera
      for (int64_t c = 0; c < nc; ++c) at[c + 1] += at[c];
      for (int64_t c = 0; c < nc; ++c) cam_ptr[cam0[p] + c + 1] = obs0[p] + at[c + 1];
      // the points that two cameras share, pair by pair, in segments: full ones first, so that
      // the threads of a wavefront run alike
      int64_t nseg = 0, pairs = 0;
      const size_t s0 = slots.size();
      for (int64_t k = 0; k < nslot; ++k) {
        slots.push_back({pairs, nseg, 0});
        pairs += slot[k + 1];
        nseg += slot[k + 1] / kSegment;
      }
      for (int64_t k = 0; k < nslot; ++k)
        if (slot[k + 1] % kSegment) slots[s0 + size_t(k)].part = nseg++;
      slots.push_back({pairs, nseg, 0});
      slot_ptr[p + 1] = int64_t(slots.size());
      pair_ptr[p + 1] = pair_ptr[p] + pairs;
      seg_ptr[p + 1] = seg_ptr[p] + nseg;
      same_ptr[p + 1] = int64_t(same.size());
    }
    const int nt_max = 512;
    const size_t lds_doubles = size_t(pk(n_max + 1, 0)) + (params->precision == SGPU_PRECISION_MIXED ? 8 : 3) * size_t(n_max) + 15 * size_t(kBatchMaxCams);
    const size_t lds_bytes = lds_doubles * 8;
    if (lds_bytes + 8 * (nt_max / 64) + 16 + 8 > 160 * 1024)  // + red, flags, queue slot
      throw Error(SGPU_ERR_UNSUPPORTED, "window too large for the LDS-resident solve");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw Error(SGPU_ERR_NO_DEVICE, "no HIP device");
    if (params->device < 0 || params->device >= ndev) throw Error(SGPU_ERR_NO_DEVICE, "device out of range");
    SGPU_HIP(hipSetDevice(params->device));
    auto* b = new sgpu_batch();
    try {
      b->precision = params->precision;
      b->lds_bytes = lds_bytes;
      b->ncam = C;
      b->npt = Q;
      b->nobs = O;
      SGPU_HIP(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
      // launch order: largest windows first (load balance)
      std::vector<int32_t> order(P);
      std::iota(order.begin(), order.end(), 0);
      std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t c) {
        return obs0[a + 1] - obs0[a] > obs0[c + 1] - obs0[c];
      });
      BatchDev& d = b->d;
      DeviceArena& A = b->arena;
      d.nprob = int32_t(P);
      // every array in one allocation, those with values from the host first
      DeviceBlock B;
      int32_t *obs_pt, *cam_pt, *pair_pt;
      double* cam_uv;
      int4* seg;
      const int64_t* sp;
      B.add(d.order, order);
      B.add(d.cam0, cam0);
      B.add(d.pt0, pt0);
      B.add(d.obs0, obs0);
      B.add(d.intr, size_t(4) * P, desc->intrinsics);
      B.add(d.poses_init, size_t(7) * C, desc->poses);
      B.add(d.points_init, size_t(3) * Q, desc->points);
      B.add(d.obs_cam, size_t(O), obs_cam);
      B.add(d.obs_uv, 2 * size_t(O), uv);
      B.add(d.pt_obs, pt_obs);
      B.add(d.cam_ptr, cam_ptr);
      B.add(d.pair_ptr, pair_ptr);
      B.add(d.seg_ptr, seg_ptr);
      B.add(sp, slot_ptr);
      B.add(d.same, same);
      B.add(d.same_ptr, same_ptr);
      B.add(d.pt_nu, pt_nu);
      B.add(d.cam_nu, cam_nu);
      B.add(obs_pt, size_t(O));
      B.add(cam_pt, size_t(O));
      B.add(cam_uv, 2 * size_t(O));
      B.add(pair_pt, size_t(pair_ptr[P]));
      B.add(seg, size_t(seg_ptr[P]));
      for (int i = 0; i < 2; ++i) {
        B.add(d.poses[i], size_t(7) * C);
        B.add(d.points[i], size_t(3) * Q);
      }
      B.add(d.rec, size_t(kRec) * Q);
      B.add(d.cur, P);
      B.add(d.nu, P);
      B.add(d.merit, P);
      B.add(d.init_merit, P);
      B.add(d.rejects, P);
      B.add(d.steps, P);
      B.add(d.done, P);
      B.add(d.term, P);
      B.add(b->out_poses, size_t(7) * C);
      B.add(b->out_points, size_t(3) * Q);
      B.add(b->queue, 1);
      B.add(b->t_start, P);
      B.add(b->t_end, P);
      B.commit(A);
      d.seg = seg;
      {
        DeviceArena tmp;  // freed once the lists are there
        const BatchSlot* sl = tmp.upload(slots, nullptr);
        hipLaunchKernelGGL(k_batch_lists, dim3(unsigned(P)), dim3(kListThreads), 0, b->stream, d, sl, sp, obs_pt,
                           cam_pt, cam_uv, pair_pt, seg);
        SGPU_HIP(hipGetLastError());
        SGPU_HIP(hipStreamSynchronize(b->stream));
        d.obs_pt = obs_pt;
        d.cam_pt = cam_pt;
        d.cam_uv = cam_uv;
        d.pair_pt = pair_pt;
      }
      d.robust = desc->huber_delta > 0.0 ? 1 : 0;
      d.delta = desc->huber_delta;
      d.nu0 = params->initial_lm_damping;
      d.num_iterations = params->num_iterations;
      d.function_tolerance = params->function_tolerance;
      d.gradient_tolerance = params->gradient_tolerance;
      d.parameter_tolerance = params->parameter_tolerance;
      d.max_consecutive_rejects = params->max_consecutive_rejects;
      d.lds_doubles = int32_t(lds_doubles);
      d.n_max = n_max;
      set_lds(k_batch_step<double, 128>, lds_bytes);
      set_lds(k_batch_step<double, 256>, lds_bytes);
      set_lds(k_batch_step<double, 512>, lds_bytes);
      set_lds(k_batch_step<float, 128>, lds_bytes);
      set_lds(k_batch_step<float, 256>, lds_bytes);
      set_lds(k_batch_step<float, 512>, lds_bytes);
      set_lds(k_batch_persistent<double, 128>, lds_bytes);
      set_lds(k_batch_persistent<double, 256>, lds_bytes);
      set_lds(k_batch_persistent<double, 512>, lds_bytes);
      set_lds(k_batch_persistent<float, 128>, lds_bytes);
      set_lds(k_batch_persistent<float, 256>, lds_bytes);
      set_lds(k_batch_persistent<float, 512>, lds_bytes);
      int khz = 0;
      SGPU_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, params->device));
      if (khz <= 0) throw Error(SGPU_ERR_HIP, "device wall-clock rate unavailable");
      b->clock_khz = double(khz);
      // autotuner: one LM iteration of the whole batch per candidate workgroup size, from
      // the same initial state; the fastest is kept
      hipEvent_t e0, e1;
      SGPU_HIP(hipEventCreate(&e0));
      SGPU_HIP(hipEventCreate(&e1));
      const int cand[3] = {128, 256, 512};
      float best = 1e30f;
      for (int i = 0; i < 3; ++i) {  // first launches of each variant, untimed
        b->launch_init();
        b->launch_step(cand[i]);
      }
      for (int i = 0; i < 3; ++i) {
        b->launch_init();
        SGPU_HIP(hipEventRecord(e0, b->stream));
        b->launch_step(cand[i]);
        SGPU_HIP(hipEventRecord(e1, b->stream));
        SGPU_HIP(hipGetLastError());
        SGPU_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SGPU_HIP(hipEventElapsedTime(&ms, e0, e1));
        b->tune_ms[i] = ms;
        if (ms < best) {
          best = ms;
          b->threads = cand[i];
        }
      }
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      // the persistent kernel keeps more registers live than the per-iteration one, so it
      // has its own choice: for each size, the grid of every resident workgroup and one
      // timed persistent launch of one LM iteration per window; the fastest is kept
      {
        int cus = 0;
        SGPU_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, params->device));
        int grids[3] = {0, 0, 0};
        for (int i = 0; i < 3; ++i) {
          const int nt = cand[i];
          const void* fn = nullptr;
          if (b->precision == SGPU_PRECISION_MIXED)
            fn = nt == 128 ? reinterpret_cast<const void*>(k_batch_persistent<float, 128>)
                 : nt == 512 ? reinterpret_cast<const void*>(k_batch_persistent<float, 512>)
                             : reinterpret_cast<const void*>(k_batch_persistent<float, 256>);
          else
            fn = nt == 128 ? reinterpret_cast<const void*>(k_batch_persistent<double, 128>)
                 : nt == 512 ? reinterpret_cast<const void*>(k_batch_persistent<double, 512>)
                             : reinterpret_cast<const void*>(k_batch_persistent<double, 256>);
          int per_cu = 0;
          SGPU_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, nt, lds_bytes));
          grids[i] = int(std::max<int64_t>(1, std::min<int64_t>(P, int64_t(std::max(per_cu, 1)) * cus)));
        }
        hipEvent_t p0, p1;
        SGPU_HIP(hipEventCreate(&p0));
        SGPU_HIP(hipEventCreate(&p1));
        float pbest = 1e30f;
        for (int rep = 0; rep < 2; ++rep)  // the first pass is untimed
          for (int i = 0; i < 3; ++i) {
            b->persistent_threads = cand[i];
            b->persistent_grid = grids[i];
            b->launch_init();
            SGPU_HIP(hipEventRecord(p0, b->stream));
            b->launch_persistent(1);
            SGPU_HIP(hipEventRecord(p1, b->stream));
            SGPU_HIP(hipGetLastError());
            SGPU_HIP(hipEventSynchronize(p1));
            float ms = 0;
            SGPU_HIP(hipEventElapsedTime(&ms, p0, p1));
            if (rep == 1) b->ptune_ms[i] = ms;
          }
        int pick = 0;
        for (int i = 0; i < 3; ++i)
          if (b->ptune_ms[i] < pbest) {
            pbest = float(b->ptune_ms[i]);
            pick = i;
          }
        b->persistent_threads = cand[pick];
        b->persistent_grid = grids[pick];
        (void)hipEventDestroy(p0);
        (void)hipEventDestroy(p1);
      }
      b->launch_init();
      SGPU_HIP(hipStreamSynchronize(b->stream));
    } catch (...) {
      delete b;
      throw;
    }
    *out = b;
  });
}

sgpu_status sgpu_batch_run(sgpu_batch* b, int32_t iterations, int32_t use_graph, double* seconds) {
  return guarded([&] {
    if (!b || iterations < 0) throw Error(SGPU_ERR_INVALID_ARGUMENT, "bad arguments");
    const auto t0 = std::chrono::steady_clock::now();
    if (use_graph) {
      if (!b->graph_exec || b->graph_iters != iterations) {
        if (b->graph_exec) (void)hipGraphExecDestroy(b->graph_exec);
        if (b->graph) (void)hipGraphDestroy(b->graph);
        b->graph_exec = nullptr;
        b->graph = nullptr;
        SGPU_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        for (int i = 0; i < iterations; ++i) b->launch_step(b->threads);
        SGPU_HIP(hipStreamEndCapture(b->stream, &b->graph));
        SGPU_HIP(hipGraphInstantiate(&b->graph_exec, b->graph, nullptr, nullptr, 0));
        b->graph_iters = iterations;
      }
      SGPU_HIP(hipGraphLaunch(b->graph_exec, b->stream));
    } else {
      for (int i = 0; i < iterations; ++i) b->launch_step(b->threads);
    }
    SGPU_HIP(hipGetLastError());
    SGPU_HIP(hipStreamSynchronize(b->stream));
    if (seconds)
      *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  });
}

sgpu_status sgpu_batch_run_persistent(sgpu_batch* b, int32_t iterations, int32_t use_graph,
                                      double* seconds) {
  return guarded([&] {
    if (!b || iterations < 0) throw Error(SGPU_ERR_INVALID_ARGUMENT, "bad arguments");
    const auto t0 = std::chrono::steady_clock::now();
    if (use_graph) {
      if (!b->pgraph_exec || b->pgraph_iters != iterations) {
        if (b->pgraph_exec) (void)hipGraphExecDestroy(b->pgraph_exec);
        if (b->pgraph) (void)hipGraphDestroy(b->pgraph);
        b->pgraph_exec = nullptr;
        b->pgraph = nullptr;
        SGPU_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        b->launch_persistent(iterations);
        SGPU_HIP(hipStreamEndCapture(b->stream, &b->pgraph));
        SGPU_HIP(hipGraphInstantiate(&b->pgraph_exec, b->pgraph, nullptr, nullptr, 0));
        b->pgraph_iters = iterations;
      }
      SGPU_HIP(hipGraphLaunch(b->pgraph_exec, b->stream));
    } else {
      b->launch_persistent(iterations);
    }
    SGPU_HIP(hipGetLastError());
    SGPU_HIP(hipStreamSynchronize(b->stream));
    if (seconds)
      *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  });
}

sgpu_status sgpu_batch_latencies(const sgpu_batch* b, double* start_ms, double* end_ms) {
  return guarded([&] {
    if (!b || !start_ms || !end_ms) throw Error(SGPU_ERR_INVALID_ARGUMENT, "bad arguments");
    const size_t P = size_t(b->d.nprob);
    std::vector<unsigned long long> ts(P), te(P);
    SGPU_HIP(hipMemcpy(ts.data(), b->t_start, P * 8, hipMemcpyDeviceToHost));
    SGPU_HIP(hipMemcpy(te.data(), b->t_end, P * 8, hipMemcpyDeviceToHost));
    const unsigned long long t0 = *std::min_element(ts.begin(), ts.end());
    for (size_t p = 0; p < P; ++p) {
      start_ms[p] = double(ts[p] - t0) / b->clock_khz;
      end_ms[p] = double(te[p] - t0) / b->clock_khz;
    }
  });
}

sgpu_status sgpu_batch_reset(sgpu_batch* b) {
  return guarded([&] {
    if (!b) throw Error(SGPU_ERR_INVALID_ARGUMENT, "null batch");
    b->launch_init();
    SGPU_HIP(hipStreamSynchronize(b->stream));
  });
}

sgpu_status sgpu_batch_results(sgpu_batch* b, double* poses_out, double* points_out, double* initial_cost,
                               double* final_cost, int32_t* num_steps, int32_t* termination) {
  return guarded([&] {
    if (!b) throw Error(SGPU_ERR_INVALID_ARGUMENT, "null batch");
    const BatchDev& d = b->d;
    const size_t P = size_t(d.nprob);
    if (poses_out || points_out) {
      hipLaunchKernelGGL(k_batch_gather, dim3(d.nprob), dim3(256), 0, b->stream, d, b->out_poses, b->out_points);
      SGPU_HIP(hipGetLastError());
      if (poses_out)
        SGPU_HIP(hipMemcpyAsync(poses_out, b->out_poses, size_t(7) * b->ncam * 8, hipMemcpyDeviceToHost, b->stream));
      if (points_out)
        SGPU_HIP(hipMemcpyAsync(points_out, b->out_points, size_t(3) * b->npt * 8, hipMemcpyDeviceToHost, b->stream));
      SGPU_HIP(hipStreamSynchronize(b->stream));
    }
    if (initial_cost) SGPU_HIP(hipMemcpy(initial_cost, d.init_merit, P * 8, hipMemcpyDeviceToHost));
    if (final_cost) SGPU_HIP(hipMemcpy(final_cost, d.merit, P * 8, hipMemcpyDeviceToHost));
    if (num_steps) SGPU_HIP(hipMemcpy(num_steps, d.steps, P * 4, hipMemcpyDeviceToHost));
    if (termination) SGPU_HIP(hipMemcpy(termination, d.term, P * 4, hipMemcpyDeviceToHost));
  });
}

sgpu_status sgpu_batch_info(const sgpu_batch* b, int32_t* threads, double* tune_ms3, int64_t* lds_bytes,
                            int32_t* persistent_threads, double* persistent_tune_ms3,
                            int32_t* persistent_grid) {
  return guarded([&] {
    if (!b) throw Error(SGPU_ERR_INVALID_ARGUMENT, "null batch");
    if (threads) *threads = b->threads;
    if (persistent_threads) *persistent_threads = b->persistent_threads;
    if (persistent_tune_ms3)
      for (int i = 0; i < 3; ++i) persistent_tune_ms3[i] = b->ptune_ms[i];
    if (persistent_grid) *persistent_grid = b->persistent_grid;
    if (tune_ms3)
      for (int i = 0; i < 3; ++i) tune_ms3[i] = b->tune_ms[i];
    if (lds_bytes) *lds_bytes = int64_t(b->lds_bytes);
  });
}

void sgpu_batch_destroy(sgpu_batch* b) { delete b; }

}  // extern "C"
