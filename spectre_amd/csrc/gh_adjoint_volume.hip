// Volume part of the GH adjoint (the RHS linearised at u) on uniform and ragged
// domains, without a derivative array:
//   gh_adjoint_sums_kernel: one workgroup per (element, half of the symmetric
//     pairs), of large elements per 512 points too: the partial derivatives of u
//     from LDS, reduced on the spot to the ten weighted sums per point that the
//     point-wise adjoint reads;
//   gh_adjoint_point_kernel: one thread per point, the point-wise adjoint (50
//     values into ubar) and the scalars that the adjoint of the derivatives needs;
//   gh_adjoint_sweeps_kernel: one workgroup per (element, pair): the adjoint of
//     the pair's 15 derivatives from gbar, contracted into logical ones in LDS,
//     transposed differentiation sweeps, and the face terms.
//
// 30 doubles per point go through the work array.  The arrangement before wrote
// 150 derivatives and 150 derivative adjoints per point and read both back, and
// its point kernel ran one wave per SIMD through some 600 dependent global
// accesses (193 of the 343 us of 300 x 6^3).  Here the point kernel's fields are
// in LDS, where re-reading them between its phases costs no global latency.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "device_common.hpp"
#include "gh_adjoint.hpp"
#include "kernels.hpp"
#include "rk3.hpp"

namespace sxd {
namespace {

// Work array of an element, blocks of Np doubles at kGhAdjointDoubles times its
// point offset: the two halves' sums (10 each: lapse, shift, q), then lapse,
// shift and inverse spatial metric (10).
constexpr int kSums = 10, kScalars = 20;
static_assert(kScalars + 10 == kGhAdjointDoubles, "work array layout");

struct ElementShape {
  int64_t off, e;
  int n0, n1, n2, np;
};

template <bool RAGGED>
__device__ __forceinline__ ElementShape element_shape(int64_t at, int n0, int n1, int n2,
                                                      const MixedElement* el,
                                                      const int32_t* list) {
  ElementShape s;
  if constexpr (RAGGED) {
    s.e = list[at];
    const MixedElement m = el[s.e];
    s.n0 = m.n[0], s.n1 = m.n[1], s.n2 = m.n[2];
    s.np = m.np;
    s.off = m.off;
  } else {
    s.e = at;
    s.n0 = n0, s.n1 = n1, s.n2 = n2;
    s.np = n0 * n1 * n2;
    s.off = at * s.np;
  }
  return s;
}

// S fields of a pair are staged together (5, or 1 for elements whose five fields
// exceed the LDS), next to each other per point.  Dynamic LDS: S Np doubles,
// then the D matrices.  Grid: (elements and halves, chunks of the element's
// points).
template <bool RAGGED, int S>
__global__ void __launch_bounds__(512)
gh_adjoint_sums_kernel(int n0, int n1, int n2, const MixedElement* __restrict__ el,
                       const int32_t* __restrict__ list, const double* __restrict__ u,
                       const double* __restrict__ gammas, const double* __restrict__ inv_jac,
                       const double* __restrict__ gbar, double* __restrict__ work,
                       const double* __restrict__ dtab) {
  extern __shared__ double s_lds[];
  const int half = blockIdx.x % 2;
  const ElementShape m = element_shape<RAGGED>(blockIdx.x / 2, n0, n1, n2, el, list);
  const int np = m.np;
  const int n[3] = {m.n0, m.n1, m.n2};
  const double* D[3];
  stage_diff_matrices(dtab, n, s_lds + S * np, D);
  const double* ue = u + 50 * m.off;
  const double* ge = gbar + 50 * m.off;
  const double* ije = inv_jac + 9 * m.off;
  const double* ga = gammas + 3 * m.off;
  const int T = blockDim.x;
  for (int base = blockIdx.y * T; base < np; base += gridDim.y * T) {
    const unsigned p = base + threadIdx.x;
    const bool active = p < static_cast<unsigned>(np);
    const int row = p / m.n0, k = row / m.n1;
    const int i = p - row * m.n0, j = row - k * m.n1;
    double a[10], ij[9], gamma1 = 0.0, gamma2 = 0.0;
#pragma unroll
    for (int x = 0; x < 10; ++x) a[x] = 0.0;
    if (active) {
#pragma unroll
      for (int c = 0; c < 9; ++c) ij[c] = (ije + c * np)[p];
      gamma1 = (ga + np)[p];
      gamma2 = (ga + 2 * np)[p];
    }
#pragma unroll 1
    for (int pr = 5 * half; pr < 5 * half + 5; ++pr) {
      const int comp[5] = {pr, 10 + pr, 20 + 3 * pr, 21 + 3 * pr, 22 + 3 * pr};
#pragma unroll
      for (int c0 = 0; c0 < 5; c0 += S) {
        __syncthreads();
        for (unsigned x = threadIdx.x; x < static_cast<unsigned>(np); x += T)
#pragma unroll
          for (int c = 0; c < S; ++c) s_lds[S * x + c] = (ue + comp[c0 + c] * np)[x];
        __syncthreads();
        if (!active) continue;
        double der[S][3];
        auto sums = [&](int d, int nd, const double* w, const double* x, int step) {
#pragma unroll
          for (int c = 0; c < S; ++c) der[c][d] = w[0] * x[c];
#pragma unroll 2
          for (int l = 1; l < nd; ++l) {
            x += step;
            const double a = w[l];
#pragma unroll
            for (int c = 0; c < S; ++c) der[c][d] = fma(a, x[c], der[c][d]);
          }
        };
        sums(0, m.n0, D[0] + i * m.n0, s_lds + S * row * m.n0, S);
        sums(1, m.n1, D[1] + j * m.n1, s_lds + S * (i + m.n0 * m.n1 * k), S * m.n0);
        sums(2, m.n2, D[2] + k * m.n2, s_lds + S * (i + m.n0 * j), S * m.n0 * m.n1);
        double w[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) w[c] = (ge + comp[c] * np)[p];
#pragma unroll
        for (int c = 0; c < S; ++c) {
          const int f = c0 + c;  // field of the pair: g, Pi, Phi_0..2
          double d[3];
#pragma unroll
          for (int x = 0; x < 3; ++x)
            d[x] = fma(ij[ij3(2, x)], der[c][2],
                       fma(ij[ij3(1, x)], der[c][1], ij[ij3(0, x)] * der[c][0]));
          if (f == 0) {
            const double s = gamma1 * gamma2 * w[1] + (1.0 + gamma1) * w[0];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              a[0] = fma(gamma2 * w[2 + x], d[x], a[0]);
              a[1 + x] = fma(s, d[x], a[1 + x]);
            }
          } else if (f == 1) {
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              a[0] = fma(-w[2 + x], d[x], a[0]);
              a[1 + x] = fma(w[1], d[x], a[1 + x]);
            }
          } else {
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              a[1 + x] = fma(w[f], d[x], a[1 + x]);
              a[4 + sym3(x, f - 2)] = fma(w[1], d[x], a[4 + sym3(x, f - 2)]);
            }
          }
        }
      }
    }
    if (!active) continue;
    double* out = work + kGhAdjointDoubles * m.off + kSums * half * np;
#pragma unroll
    for (int x = 0; x < 10; ++x) (out + x * np)[p] = a[x];
  }
}

// One wave per workgroup; LDS: 50 fields of its 64 points (25.6 KB, so that four
// waves, one per SIMD, share a CU).
template <bool RAGGED>
__global__ void __launch_bounds__(64)
gh_adjoint_point_kernel(int64_t total, int np_uniform, const MixedElement* __restrict__ el,
                        const int32_t* __restrict__ point_el, const double* __restrict__ u,
                        const double* __restrict__ gammas, const double* __restrict__ gbar,
                        double* __restrict__ work, double* __restrict__ ubar) {
  __shared__ double s_u[50 * 64];
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  if (gid >= total) return;
  int64_t off;
  int np;
  if constexpr (RAGGED) {
    const MixedElement& m = el[point_el[gid]];
    off = m.off;
    np = m.np;
  } else {
    np = np_uniform;
    off = gid / np * np;
  }
  const int p = static_cast<int>(gid - off);
  const double* up = u + 50 * off + p;
  // a thread reads only its own column of the block: no barrier
#pragma unroll
  for (int c = 0; c < 50; ++c) s_u[64 * c + threadIdx.x] = up[c * np];
  double* w = work + kGhAdjointDoubles * off + p;
  GhDerivativeSums sums;
  sums.lapse = w[0] + w[kSums * np];
#pragma unroll
  for (int x = 0; x < 3; ++x) sums.shift[x] = w[(1 + x) * np] + w[(kSums + 1 + x) * np];
#pragma unroll
  for (int x = 0; x < 6; ++x) sums.q[x] = w[(4 + x) * np] + w[(kSums + 4 + x) * np];
  const double* ga = gammas + 3 * off + p;
  double ub[50];
  GhVjpPoint pt;
  gh_time_derivative_vjp((LdsField)(s_u + threadIdx.x), 64, sums, ga[0], ga[np], ga[2 * np],
                         gbar + 50 * off + p, np, ub, &pt);
  double* out = ubar + 50 * off + p;
#pragma unroll
  for (int c = 0; c < 50; ++c) out[c * np] = ub[c];
  w[kScalars * np] = pt.lapse;
#pragma unroll
  for (int x = 0; x < 3; ++x) w[(kScalars + 1 + x) * np] = pt.shift[x];
#pragma unroll
  for (int x = 0; x < 6; ++x) w[(kScalars + 4 + x) * np] = pt.isp[x];
}

// S fields of the pair at a time (5, or 1 where their 15 Np derivative adjoints
// exceed the LDS).  Dynamic LDS: 3 S Np doubles, then
// the D matrices.  contrib: face terms, [E][6][50][F] (uniform domains) or per
// record as `table` places them.  list_or_first: RAGGED: length of `list`,
// otherwise the launch's first element.
template <bool RAGGED, int S, bool UPDATE>
__global__ void __launch_bounds__(512)
gh_adjoint_sweeps_kernel(int list_or_first, int n0, int n1, int n2,
                         const MixedElement* __restrict__ el, const int32_t* __restrict__ list, const double* __restrict__ gammas,
                         const double* __restrict__ inv_jac, const double* __restrict__ gbar,
                         const double* __restrict__ work, double* __restrict__ ubar,
                         const double* __restrict__ dtab, const double* __restrict__ contrib,
                         int F, const MortarCorrection* __restrict__ table,
                         Rk3AdjointUpdate update) {
  extern __shared__ double s_lds[];
  int64_t at;
  int pr;
  if constexpr (RAGGED) {
    const int x = blockIdx.x % kNumXcds, slot = blockIdx.x / kNumXcds;
    at = slot / 10 * kNumXcds + x;
    pr = slot % 10;
    if (at >= list_or_first) return;
  } else {
    const int64_t item = xcd_local_element(blockIdx.x, gridDim.x);
    at = item / 10;
    pr = static_cast<int>(item - 10 * at);
    at += list_or_first;
  }
  const ElementShape m = element_shape<RAGGED>(at, n0, n1, n2, el, list);
  const int np = m.np;
  const int n[3] = {m.n0, m.n1, m.n2};
  const int comp[5] = {pr, 10 + pr, 20 + 3 * pr, 21 + 3 * pr, 22 + 3 * pr};
  const double* D[3];
  stage_diff_matrices(dtab, n, s_lds + 3 * S * np, D);
  const double* ge = gbar + 50 * m.off;
  const double* ije = inv_jac + 9 * m.off;
  const double* ga = gammas + 3 * m.off;
  const double* we = work + kGhAdjointDoubles * m.off;
  double* ube = ubar + 50 * m.off;
#pragma unroll
  for (int c0 = 0; c0 < 5; c0 += S) {
    if (c0 > 0) __syncthreads();  // the previous field's sweeps have read the LDS
    for (unsigned p = threadIdx.x; p < static_cast<unsigned>(np); p += blockDim.x) {
      double w[5], ij[9];
      GhVjpPoint pt;
#pragma unroll
      for (int c = 0; c < 5; ++c) w[c] = (ge + comp[c] * np)[p];
#pragma unroll
      for (int c = 0; c < 9; ++c) ij[c] = (ije + c * np)[p];
      pt.lapse = (we + kScalars * np)[p];
#pragma unroll
      for (int x = 0; x < 3; ++x) pt.shift[x] = (we + (kScalars + 1 + x) * np)[p];
#pragma unroll
      for (int x = 0; x < 6; ++x) pt.isp[x] = (we + (kScalars + 4 + x) * np)[p];
      const double gamma1 = (ga + np)[p], gamma2 = (ga + 2 * np)[p];
#pragma unroll
      for (int c = 0; c < S; ++c) {
        double d[3];
        gh_pair_dubar(d, c0 + c, pt, gamma1, gamma2, w);
#pragma unroll
        for (int j = 0; j < 3; ++j)
          s_lds[3 * S * p + 3 * c + j] =
              fma(ij[ij3(j, 2)], d[2], fma(ij[ij3(j, 1)], d[1], ij[ij3(j, 0)] * d[0]));
      }
    }
    __syncthreads();
    for (unsigned p = threadIdx.x; p < static_cast<unsigned>(np); p += blockDim.x) {
      const int row = p / m.n0, k = row / m.n1;
      const int i = p - row * m.n0, j = row - k * m.n1;
      double acc[S];
#pragma unroll
      for (int c = 0; c < S; ++c) acc[c] = (ube + comp[c0 + c] * np)[p];
      auto sweep = [&](int d, int nd, const double* w, const double* x, int step) {
#pragma unroll 2
        for (int l = 0; l < nd; ++l) {
          const double a = w[l * nd];
#pragma unroll
          for (int c = 0; c < S; ++c) acc[c] = fma(a, x[3 * c + d], acc[c]);
          x += step;
        }
      };
      sweep(0, m.n0, D[0] + i, s_lds + 3 * S * row * m.n0, 3 * S);
      sweep(1, m.n1, D[1] + j, s_lds + 3 * S * (i + m.n0 * m.n1 * k), 3 * S * m.n0);
      sweep(2, m.n2, D[2] + k, s_lds + 3 * S * (i + m.n0 * j), 3 * S * m.n0 * m.n1);
      if constexpr (!RAGGED) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int at_d = d == 0 ? i : d == 1 ? j : k, nd = d == 0 ? n0 : d == 1 ? n1 : n2;
          if (at_d != 0 && at_d != nd - 1) continue;
          const int f = d == 0 ? j + n1 * k : d == 1 ? i + n0 * k : i + n0 * j;
          const double* from =
              contrib + (m.e * 6 + 2 * d + (at_d == 0 ? 0 : 1)) * 50 * static_cast<int64_t>(F) + f;
#pragma unroll
          for (int c = 0; c < S; ++c) acc[c] += from[static_cast<int64_t>(comp[c0 + c]) * F];
        }
      } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int at_d = d == 0 ? i : d == 1 ? j : k, nd = n[d];
          if (at_d != 0 && at_d != nd - 1) continue;
          const int nf = d == 0 ? m.n1 * m.n2 : d == 1 ? m.n0 * m.n2 : m.n0 * m.n1;
          const int f = d == 0 ? j + m.n1 * k : d == 1 ? i + m.n0 * k : i + m.n0 * j;
          const MortarCorrection lower = table[6 * m.e + 2 * d];
          const MortarCorrection upper = table[6 * m.e + 2 * d + 1];
          const int mortars = at_d == 0 ? lower.count : upper.count;
          const double* from = contrib + 50 * (at_d == 0 ? lower.off : upper.off) + f;
          for (int q = 0; q < mortars; ++q, from += 50 * nf)
#pragma unroll
            for (int c = 0; c < S; ++c) acc[c] += from[comp[c0 + c] * nf];
        }
      }
      if constexpr (UPDATE) {
        double* mu = update.mu + 50 * m.off;
#pragma unroll
        for (int c = 0; c < S; ++c)
          acc[c] = rk3_adjoint_value(update.substep, update.dt, (ge + comp[c0 + c] * np)[p],
                                     acc[c], mu + comp[c0 + c] * np + p);
        if (update.substep == 0) continue;
      }
#pragma unroll
      for (int c = 0; c < S; ++c) (ube + comp[c0 + c] * np)[p] = acc[c];
    }
  }
}

// A thread per point up to 512: two workgroups per element are few, so that more
// waves count for more than fewer stagings (300 x 6^3: 33.8 us with two points
// per thread, 24.9 with one).
int sums_threads(int np) { return std::min(512, (np + 63) / 64 * 64); }

constexpr int kLdsDoubles = 160 * 1024 / 8;

}  // namespace

bool gh_adjoint_supported(const int32_t ext[3]) {
  const int np = ext[0] * ext[1] * ext[2];
  return 3 * np + ext[0] * ext[0] + ext[1] * ext[1] + ext[2] * ext[2] <= kLdsDoubles;
}

namespace {
// One launch of the sums, or of the sweeps, over elements of up to np points
// and d_doubles entries of their D matrices.
template <bool RAGGED>
int launch_sums(int count, int np, int d_doubles, const int32_t ext[3], const MixedElement* el,
                const int32_t* list, const double* u, const double* gammas, const double* inv_jac,
                const double* gbar, double* work, const double* dtab, hipStream_t stream) {
  // ragged elements have at most 193 points on a face, so that five fields fit
  const bool five = RAGGED || 5 * np + d_doubles <= kLdsDoubles;
  const int lds = ((five ? 5 : 1) * np + d_doubles) * 8;
  auto kernel = &gh_adjoint_sums_kernel<RAGGED, 5>;
  if constexpr (!RAGGED)
    if (!five) kernel = &gh_adjoint_sums_kernel<RAGGED, 1>;
  if (!allow_lds(reinterpret_cast<const void*>(kernel), lds)) return SXD_ERR_UNSUPPORTED;
  // Field by field a chunk of the points stages the fields again in any case, so
  // each chunk is a workgroup: with two per element for all of them whole
  // adjoints of 8 x 16^3 took 1361 us, 64 x 16^3 2062, of 8 x 18^3 1438, with the
  // chunks 347, 1200 and 366.
  const int threads = sums_threads(np);
  const int chunks = five ? 1 : (np + threads - 1) / threads;
  // a uniform domain has too few elements for the limit: each has at least an eighth
  // of the threads in points, at 150 doubles a point
  const int limit = RAGGED ? launch_limit(2, threads) : count;
  for (int first = 0; first < count; first += limit) {
    hipLaunchKernelGGL(kernel, dim3(2 * std::min(limit, count - first), chunks), dim3(threads),
                       lds, stream, ext[0], ext[1], ext[2], el, RAGGED ? list + first : nullptr, u,
                       gammas, inv_jac, gbar, work, dtab);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  return SXD_OK;
}

template <bool RAGGED>
int launch_sweeps(int count, int np, int d_doubles, const int32_t ext[3], const MixedElement* el,
                  const int32_t* list, const double* gammas, const double* inv_jac,
                  const double* gbar, const double* work, double* ubar, const double* dtab,
                  const double* contrib, int F, const MortarCorrection* table,
                  hipStream_t stream, const Rk3AdjointUpdate& up) {
  // All five fields also where they leave one workgroup per CU: a field at a time
  // each point's scalars are read and its adjoints formed five times (300 elements
  // of 6^3 .. 10^3 223 -> 149 us, whole adjoint of 256 elements of 10^3 671 -> 618).
  const bool five = 15 * np + d_doubles <= kLdsDoubles;
  const int lds = ((five ? 15 : 3) * np + d_doubles) * 8;
  const bool update = up.substep >= 0;
  const auto kernel = five ? (update ? &gh_adjoint_sweeps_kernel<RAGGED, 5, true>
                                     : &gh_adjoint_sweeps_kernel<RAGGED, 5, false>)
                           : (update ? &gh_adjoint_sweeps_kernel<RAGGED, 1, true>
                                     : &gh_adjoint_sweeps_kernel<RAGGED, 1, false>);
  if (!allow_lds(reinterpret_cast<const void*>(kernel), lds)) return SXD_ERR_UNSUPPORTED;
  const int threads = np > 512 ? 512 : np > 128 ? 256 : 128;
  const int limit = launch_limit(10, threads);
  for (int first = 0; first < count; first += limit) {
    const int n = std::min(limit, count - first);
    const int blocks = RAGGED ? (n + kNumXcds - 1) / kNumXcds * kNumXcds * 10 : 10 * n;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(threads), lds, stream, RAGGED ? n : first,
                       ext[0], ext[1], ext[2], el, RAGGED ? list + first : nullptr, gammas,
                       inv_jac, gbar, work, ubar, dtab, contrib, F, table, up);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  return SXD_OK;
}
}  // namespace

int launch_gh_adjoint_points(int num_elements, const int32_t ext[3], const double* u,
                             const double* gammas, const double* inv_jac, const double* gbar,
                             double* ubar, double* work, hipStream_t stream) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  if (!gh_adjoint_supported(ext)) return SXD_ERR_UNSUPPORTED;
  const int np = ext[0] * ext[1] * ext[2];
  const int d_doubles = ext[0] * ext[0] + ext[1] * ext[1] + ext[2] * ext[2];
  const int rc = launch_sums<false>(num_elements, np, d_doubles, ext, nullptr, nullptr, u, gammas,
                                    inv_jac, gbar, work, dtab, stream);
  if (rc != SXD_OK) return rc;
  const int64_t total = static_cast<int64_t>(num_elements) * np;
  hipLaunchKernelGGL(gh_adjoint_point_kernel<false>,
                     dim3(static_cast<unsigned>((total + 63) / 64)), dim3(64), 0, stream, total,
                     np, nullptr, nullptr, u, gammas, gbar, work, ubar);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

int launch_gh_adjoint_sweeps(int num_elements, const int32_t ext[3], const double* gammas,
                             const double* inv_jac, const double* gbar, const double* work,
                             double* ubar, const double* contrib, int F, hipStream_t stream,
                             const Rk3AdjointUpdate& up) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  const int np = ext[0] * ext[1] * ext[2];
  const int d_doubles = ext[0] * ext[0] + ext[1] * ext[1] + ext[2] * ext[2];
  return launch_sweeps<false>(num_elements, np, d_doubles, ext, nullptr, nullptr, gammas, inv_jac,
                              gbar, work, ubar, dtab, contrib, F, nullptr, stream, up);
}

int launch_ragged_gh_adjoint_points(const std::vector<RaggedClass>& classes, const int32_t* list,
                                    const MixedElement* el, const int32_t* point_el,
                                    int64_t total_points, const double* u, const double* gammas,
                                    const double* inv_jac, const double* gbar, double* ubar,
                                    double* work, hipStream_t stream) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  const int32_t none[3] = {0, 0, 0};
  for (const RaggedClass& c : classes) {
    const int rc = launch_sums<true>(c.count, c.np_max, c.d_doubles, none, el, list + c.begin, u,
                                     gammas, inv_jac, gbar, work, dtab, stream);
    if (rc != SXD_OK) return rc;
  }
  hipLaunchKernelGGL(gh_adjoint_point_kernel<true>,
                     dim3(static_cast<unsigned>((total_points + 63) / 64)), dim3(64), 0, stream,
                     total_points, 0, el, point_el, u, gammas, gbar, work, ubar);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

int launch_ragged_gh_adjoint_sweeps(const std::vector<RaggedClass>& classes, const int32_t* list,
                                    const MixedElement* el, const double* gammas,
                                    const double* inv_jac, const double* gbar,
                                    const double* work, double* ubar,
                                    const MortarCorrection* table, const double* contrib,
                                    hipStream_t stream, const Rk3AdjointUpdate& up) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  const int32_t none[3] = {0, 0, 0};
  for (const RaggedClass& c : classes) {
    const int rc = launch_sweeps<true>(c.count, c.np_max, c.d_doubles, none, el, list + c.begin,
                                       gammas, inv_jac, gbar, work, ubar, dtab, contrib, 0, table,
                                       stream, up);
    if (rc != SXD_OK) return rc;
  }
  return SXD_OK;
}

}  // namespace sxd
