// Adjoint (transpose) of the ScalarWave DG right-hand side and of the RK3
// update, for gradients of functionals of the evolved state.
//
// For fixed gamma2 and inverse Jacobian the ScalarWave RHS u -> dt is linear;
// these kernels apply its exact transpose gbar -> ubar, written by hand from
// the forward operations (the reference has no adjoint):
//  * volume: the transposed point-wise terms give the adjoints of the 15
//    inertial derivatives, the transposed inverse-Jacobian contraction those
//    of the logical derivatives (staged in LDS), and the transposed
//    differentiation sweeps ubar_c(p) += sum_j sum_m D_j(m, idx_j(p)) x_cj(m);
//  * faces (transposed UpwindPenalty + lift): with the constant speeds
//    (0, 1, -1) the correction reduces to bc_Pi = -(v+_ext + v-_int) / 2,
//    bc_Phi = (v-_int n_int - v+_ext n_ext) / 2; its transpose sends
//    s_in = (b.n_int - a) / 2 to the interior point and
//    s_ext = -(a + b.n_ext) / 2 to the exterior point, with (a, b) the lift
//    factor times (gbar_Pi, gbar_Phi) at the interior point.
// Each point gathers the face contributions that land on it (its own faces'
// interior terms and the neighbours' exterior terms) and adds them in the
// order (contributing element, direction), the order in which the oracle
// scatters them, so results equal the oracle bit for bit.  Bound by the latency
// of its phases (512 x 6^3: 13.4 us, 5 us of traffic).  Face terms that were
// sorted first and evaluated in turn, each with loads, square roots and a
// division of its own, were a serial chain of six, and LDS reads of all
// components in flight spilled up to 1 KB per thread: 512 elements of 6^3 14.5,
// of 7^3 29.5 -> 16.3, of 8^3 45.5 -> 23.2, of 10^3 278 -> 58 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include <cstdint>

#include "device_common.hpp"
#include "gh_adjoint.hpp"
#include "kernels.hpp"
#include "rk3.hpp"
#include "sw_point.hpp"

namespace sxd {
namespace {

template <int N, bool UPDATE>
__global__ void __launch_bounds__((N * N * N + 63) / 64 * 64)
sw_rhs_adjoint_kernel(const int32_t* __restrict__ nbr, const double* __restrict__ gbar,
                      const double* __restrict__ gamma2, const double* __restrict__ inv_jac,
                      double* __restrict__ ubar, const double* __restrict__ dtab,
                      Rk3AdjointUpdate update) {
  constexpr int NP = N * N * N;
  // logical-derivative adjoints [c][j][p]; then, a column per point, the face
  // terms' factors [slot] and normals [d][i]
  __shared__ double s_x[15 * NP];
  const int64_t e = xcd_local_element(blockIdx.x, gridDim.x);
  const int t = threadIdx.x;
  const double* g = gbar + e * 5 * NP;
  const double* ij = inv_jac + e * 9 * NP;
  double gp[5], g2 = 0.0;
  const int idx[3] = {t % N, (t / N) % N, t / (N * N)};
  // the neighbours' values of all faces of the point, in flight during the sums
  int64_t nbr_of[3] = {0, 0, 0};
  double ijn[3][3], gn[3][4];
  if (t < NP) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (idx[d] != 0 && idx[d] != N - 1) continue;
      const int64_t en = nbr[6 * e + 2 * d + (idx[d] == 0 ? 0 : 1)];
      const int stride = d == 0 ? 1 : d == 1 ? N : N * N;
      const int q = t + (idx[d] == 0 ? 1 : -1) * (N - 1) * stride;
      nbr_of[d] = en;
#pragma unroll
      for (int i = 0; i < 3; ++i) ijn[d][i] = inv_jac[(en * 9 + ij3(d, i)) * NP + q];
#pragma unroll
      for (int c = 0; c < 4; ++c) gn[d][c] = gbar[(en * 5 + 1 + c) * NP + q];
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) gp[c] = g[c * NP + t];
    g2 = gamma2[e * NP + t];
    double dub[15];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      dub[i] = g2 * gp[2 + i];
      dub[3 + i] = -gp[2 + i];
#pragma unroll
      for (int jj = 0; jj < 3; ++jj) dub[6 + 3 * jj + i] = i == jj ? -gp[1] : 0.0;
    }
    double ijp[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) ijp[c] = ij[c * NP + t];
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        double s = ijp[ij3(j, 0)] * dub[3 * c + 0];
        s = fma(ijp[ij3(j, 1)], dub[3 * c + 1], s);
        s = fma(ijp[ij3(j, 2)], dub[3 * c + 2], s);
        s_x[(3 * c + j) * NP + t] = s;
      }
  }
  __syncthreads();
  const double* D = diff_matrix(dtab, N);
  double ub[5];
  if (t < NP) {
    ub[0] = 0.0;
    ub[1] = 0.0 - gp[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) ub[2 + i] = 0.0 - g2 * gp[2 + i];
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    if (t >= NP) break;
    double acc = ub[c];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int stride = j == 0 ? 1 : j == 1 ? N : N * N;
      const int base = t - idx[j] * stride;
#pragma unroll
      for (int m = 0; m < N; ++m)
        acc = fma(D[m * N + idx[j]], s_x[(3 * c + j) * NP + base + m * stride], acc);
    }
    ub[c] = acc;
    // a component's LDS reads stay behind the sums before: all in flight at
    // once they need more registers than there are
    __builtin_amdgcn_sched_barrier(0);
  }
  // Face terms, added in ascending (element, direction) order of the face they
  // stem from: slot 2 d the interior term of the own face, slot 2 d + 1 the
  // exterior term of the neighbour's.  Their factors are formed together, and
  // the order is a packed list of slots by rank.
  constexpr int64_t kNoFace = INT64_MAX;
  int64_t key[6];
  int terms = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const bool on = idx[d] == 0 || idx[d] == N - 1;
    const int s = idx[d] == 0 ? 0 : 1;
    key[2 * d] = on ? e * 8 + 2 * d + s : kNoFace;
    key[2 * d + 1] = on ? nbr_of[d] * 8 + 2 * d + (1 - s) : kNoFace;
    terms += on ? 2 : 0;
  }
  __syncthreads();  // the sweeps have read the LDS
  if (t >= NP) return;
  double* mine = s_x + t;
  unsigned order = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (idx[d] != 0 && idx[d] != N - 1) continue;
    const int s = idx[d] == 0 ? 0 : 1;
    int rank_in = 0, rank_ex = 0;
#pragma unroll
    for (int x = 0; x < 6; ++x) {
      rank_in += key[x] < key[2 * d];
      rank_ex += key[x] < key[2 * d + 1];
    }
    order |= static_cast<unsigned>(2 * d) << (3 * rank_in) |
             static_cast<unsigned>(2 * d + 1) << (3 * rank_ex);
    // own normal (as interior and as the neighbour's exterior normal), and the
    // neighbour's own
    double n[3], nq[3], mag, magq;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double v = ij[ij3(d, i) * NP + t];
      n[i] = s == 0 ? v * -1.0 : v;
      nq[i] = s == 1 ? ijn[d][i] * -1.0 : ijn[d][i];
    }
    flat_normalize(n, &mag);
    flat_normalize(nq, &magq);
    // s_in = 0.5 (fac b.n - fac a), s_ex = -0.5 (fac a + fac b.n)
    auto half_sum = [&](double fac, const double* b, double sign) {
      const double a = fac * b[0];
      double bn = (fac * b[1]) * n[0];
      bn = fma(fac * b[2], n[1], bn);
      bn = fma(fac * b[3], n[2], bn);
      return sign > 0.0 ? 0.5 * (bn - a) : -0.5 * (a + bn);
    };
    mine[2 * d * NP] = half_sum(lift_factor(N, mag), gp + 1, 1.0);
    mine[(2 * d + 1) * NP] = half_sum(lift_factor(N, magq), gn[d], -1.0);
#pragma unroll
    for (int i = 0; i < 3; ++i) mine[(6 + 3 * d + i) * NP] = n[i];
  }
  for (int x = 0; x < terms; ++x, order >>= 3) {
    const int slot = order & 7, exterior = slot & 1;
    const double f = mine[slot * NP];
    const double* n = mine + (6 + 3 * (slot >> 1)) * NP;
    ub[0] = exterior ? ub[0] - g2 * f : ub[0] + g2 * f;
    ub[1] = exterior ? ub[1] + f : ub[1] - f;
#pragma unroll
    for (int i = 0; i < 3; ++i) ub[2 + i] = ub[2 + i] + n[i * NP] * f;
  }
  if constexpr (UPDATE) {
#pragma unroll
    for (int c = 0; c < 5; ++c)
      ub[c] = rk3_adjoint_value(update.substep, update.dt, gp[c], ub[c],
                                update.mu + (e * 5 + c) * NP + t);
    if (update.substep == 0) return;
  }
#pragma unroll
  for (int c = 0; c < 5; ++c) ubar[(e * 5 + c) * NP + t] = ub[c];
}

template <int N>
int launch_sw_adjoint_n(int num_elements, const int32_t* nbr, const double* gbar,
                        const double* gamma2, const double* inv_jac, double* ubar,
                        const double* dtab, hipStream_t stream, const Rk3AdjointUpdate& up) {
  constexpr int threads = (N * N * N + 63) / 64 * 64;
  hipLaunchKernelGGL((up.substep < 0 ? &sw_rhs_adjoint_kernel<N, false>
                                     : &sw_rhs_adjoint_kernel<N, true>),
                     dim3(num_elements), dim3(threads), 0, stream, nbr, gbar, gamma2, inv_jac,
                     ubar, dtab, up);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

// Transpose of one Rk3HesthavenSsp substep (Rk3HesthavenSsp.cpp:55-81),
// substeps in reverse order.  lam: adjoint of the substep's output; a:
// A^T lam (adjoint RHS); mu: accumulated adjoint of the step's input u.
//   substep 2 (u3 = (u + 2 u2 + 2 dt L(u2)) / 3): lam_out = 2/3 (lam + dt a), mu = lam / 3
//   substep 1 (u2 = (3 u + u1 + dt L(u1)) / 4):   lam_out = (lam + dt a) / 4, mu += 3/4 lam
//   substep 0 (u1 = u + dt L(u)):                 mu += lam + dt a
__global__ void __launch_bounds__(256)
rk3_adjoint_substep_kernel(int substep, int64_t n, double dt, const double* lam,
                           const double* __restrict__ a, double* __restrict__ mu,
                           double* lam_out) {  // lam_out may be lam (element-wise in place)
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double out = rk3_adjoint_value(substep, dt, lam[i], a[i], mu + i);
  if (substep > 0) lam_out[i] = out;
}

// ---------------------------------------------------------------------------
// Generalized harmonic: adjoint of the RHS linearised at the state u (the RHS
// is nonlinear): the point-wise adjoint (gh_adjoint_volume.hip); the face points'
// transposed lifted UpwindPenalty terms of each face they lie on, as interior
// point of their own face and as exterior point of the neighbour's, into a
// per-face work array; then the transposed differentiation sweeps
// (gh_adjoint_volume.hip), which add the face terms.
//
// Faces, one thread per (element, face, face point): the point's face terms
// (its own correction's and the neighbour's, gh_face_pair_vjp) go to its
// slot of contrib [E][6][50][F] (F = largest face), which the transposed
// sweeps add; no two threads write the same value.  Grid: E * 6 * F threads.
__global__ void __launch_bounds__(64)
gh_adjoint_face_kernel(int64_t total, int F, int n0, int n1, int n2,
                       const int32_t* __restrict__ nbr, const double* __restrict__ u,
                       const double* __restrict__ gammas, const double* __restrict__ inv_jac,
                       const double* __restrict__ gbar, double* __restrict__ contrib) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= total) return;
  const int np = n0 * n1 * n2;
  const int n[3] = {n0, n1, n2};
  const int64_t e = gid / (6 * F);
  const int r = static_cast<int>(gid % (6 * F));
  const int dir = r / F, f = r % F;
  const int d = dir >> 1, s = dir & 1;
  const int ad = d == 0 ? 1 : 0, bd = d == 2 ? 1 : 2;
  if (n[d] == 1 || f >= n[ad] * n[bd]) return;
  int pi[3], qi[3];
  pi[ad] = qi[ad] = f % n[ad];
  pi[bd] = qi[bd] = f / n[ad];
  pi[d] = s == 0 ? 0 : n[d] - 1;
  qi[d] = s == 0 ? n[d] - 1 : 0;
  const int p = pi[0] + n0 * (pi[1] + n1 * pi[2]);
  const int q = qi[0] + n0 * (qi[1] + n1 * qi[2]);
  const int64_t en = nbr[6 * e + dir];
  const double* gap = gammas + e * 3 * np + p;
  const double* gaq = gammas + en * 3 * np + q;
  // normal covectors pointing out of each point's own element
  double np_row[3], nq_row[3];
  for (int i = 0; i < 3; ++i) {
    np_row[i] = inv_jac[(e * 9 + ij3(d, i)) * np + p];
    nq_row[i] = inv_jac[(en * 9 + ij3(d, i)) * np + q];
    if (s == 0) np_row[i] = np_row[i] * -1.0;
    if (s == 1) nq_row[i] = nq_row[i] * -1.0;
  }
  double* out = contrib + (e * 6 + dir) * 50 * static_cast<int64_t>(F) + f;
  // this element's face (d, s) at p and the neighbour's face (d, 1 - s) at
  // q: each point is the other's exterior
  gh_face_pair_vjp(u + e * 50 * np + p, gap[np], gap[2 * np], np_row, u + en * 50 * np + q,
                   gaq[np], gaq[2 * np], nq_row, n[d], np, gbar + e * 50 * np + p,
                   gbar + en * 50 * np + q, np, out, F);
}

}  // namespace

bool sw_adjoint_supported(const int32_t ext[3]) {
  return ext[0] == ext[1] && ext[1] == ext[2] && ext[0] >= 2 && ext[0] <= 10;
}

int launch_sw_rhs_adjoint(int num_elements, const int32_t ext[3], const int32_t* nbr,
                          const double* gbar, const double* gamma2, const double* inv_jac,
                          double* ubar, hipStream_t stream, const Rk3AdjointUpdate& up) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  if (!sw_adjoint_supported(ext)) return SXD_ERR_UNSUPPORTED;
  switch (ext[0]) {
#define SXD_ADJ_CASE(n) \
  case n:               \
    return launch_sw_adjoint_n<n>(num_elements, nbr, gbar, gamma2, inv_jac, ubar, dtab, stream, \
                                  up);
    SXD_ADJ_CASE(2)
    SXD_ADJ_CASE(3)
    SXD_ADJ_CASE(4)
    SXD_ADJ_CASE(5)
    SXD_ADJ_CASE(6)
    SXD_ADJ_CASE(7)
    SXD_ADJ_CASE(8)
    SXD_ADJ_CASE(9)
    SXD_ADJ_CASE(10)
#undef SXD_ADJ_CASE
    default: return SXD_ERR_UNSUPPORTED;
  }
}

int gh_adjoint_face_slots(const int32_t ext[3]) {
  return std::max({ext[1] * ext[2], ext[0] * ext[2], ext[0] * ext[1]});
}

int launch_gh_rhs_adjoint(int num_elements, const int32_t ext[3], const int32_t* nbr,
                          const double* u, const double* gammas, const double* inv_jac,
                          const double* gbar, double* ubar, double* work,
                          double* scratch_faces, hipStream_t stream,
                          const Rk3AdjointUpdate& up) {
  if (!gh_adjoint_supported(ext)) return SXD_ERR_UNSUPPORTED;
  const int rc = launch_gh_adjoint_points(num_elements, ext, u, gammas, inv_jac, gbar, ubar,
                                          work, stream);
  if (rc != SXD_OK) return rc;
  const int F = gh_adjoint_face_slots(ext);
  const int64_t faces = static_cast<int64_t>(num_elements) * 6 * F;
  hipLaunchKernelGGL(gh_adjoint_face_kernel, dim3(static_cast<unsigned>((faces + 63) / 64)),
                     dim3(64), 0, stream, faces, F, ext[0], ext[1], ext[2], nbr, u, gammas,
                     inv_jac, gbar, scratch_faces);
  if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  return launch_gh_adjoint_sweeps(num_elements, ext, gammas, inv_jac, gbar, work, ubar,
                                  scratch_faces, F, stream, up);
}

int launch_rk3_adjoint_substep(int substep, int64_t n, double dt, const double* lam,
                               const double* a, double* mu, double* lam_out, hipStream_t stream) {
  if (n == 0) return SXD_OK;
  hipLaunchKernelGGL(rk3_adjoint_substep_kernel, dim3(static_cast<unsigned>((n + 255) / 256)),
                     dim3(256), 0, stream, substep, n, dt, lam, a, mu, lam_out);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

}  // namespace sxd
