// GH right-hand side in two kernels for any extents whose five fields of a
// symmetric pair fit the LDS: uniform domains beyond the fused kernel
// (anisotropic extents, N > 8) and the volume terms of ragged ones.
//
//   gh_state_kernel: one thread per grid point.  What gh_point_pair reads of a
//     point (lapse, shift, inverse spatial metric, normal contractions and
//     the dt Pi partial sums, kGhStateDoubles values) and, on uniform
//     domains, the normals and speeds of the face points.
//   gh_pair_kernel: one workgroup per (element, symmetric pair).  The pair's
//     five fields are staged in LDS once; the derivative sums, the
//     inverse-Jacobian contraction, the pair's algebra and (uniform domains)
//     the lifted corrections of all faces follow, and dt is written once.
//
// The two replace a pipeline that wrote all 150 derivatives of a point to HBM,
// read them back with the point's whole state in one lane, and read and wrote
// dt once per face dimension: 462 doubles per point of volume traffic against
// 235 here, and a register file that held one wave per SIMD.  The pair kernel
// is bound by its LDS reads (15 N per point and pair plus the D rows); the ten
// workgroups of an element run next to each other on one XCD, so the state and
// the inverse Jacobian they share come from its L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_common.hpp"
#include "gh_point.hpp"
#include "kernels.hpp"
#include "rk3.hpp"

namespace sxd {
namespace {

// State of a point, element-local blocks of Np doubles at
// kGhStateDoubles * (point offset of the element).
constexpr int kLapse = 0, kShift = 1, kInvSp = 4, kHalfPhi = 10, kPhiNormal = 13, kPiNormal = 22,
              kPartial = 25;
static_assert(kPartial + 10 == kGhStateDoubles, "state layout");
// Values of a face point: n, nv, lam (4), gamma2, |n|; blocks of the element's
// face points, the six faces in direction order.
constexpr int kGhSideDoubles = 12;

__device__ __forceinline__ int face_index(int n0, int n1, int d, int i, int j, int k) {
  return d == 0 ? j + n1 * k : d == 1 ? i + n0 * k : i + n0 * j;
}

// RAGGED: grid (list length, chunks of 128 points of the largest element).
template <bool RAGGED>
__global__ void __launch_bounds__(128)
gh_state_kernel(int64_t total, int n0, int n1, int n2, const MixedElement* __restrict__ el,
                const int32_t* __restrict__ list, const double* __restrict__ u,
                const double* __restrict__ gammas, const double* __restrict__ inv_jac,
                double* __restrict__ state, double* __restrict__ sides) {
  int64_t off;
  int np, p;
  if constexpr (RAGGED) {
    const MixedElement& m = el[list[blockIdx.x]];
    off = m.off;
    np = m.np;
    p = blockIdx.y * blockDim.x + threadIdx.x;
    if (p >= np) return;
  } else {
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= total) return;
    np = n0 * n1 * n2;
    off = gid / np * np;
    p = static_cast<int>(gid - off);
  }
  const double* ue = u + 50 * off + p;
  const double* ga = gammas + 3 * off + p;
  double up[50];
#pragma unroll
  for (int c = 0; c < 50; ++c) up[c] = ue[c * np];
  const double gamma1 = ga[np], gamma2 = ga[2 * np];
  GhPointState st;
  gh_point_setup(st, up, ga[0], gamma1, gamma2);
  double* o = state + kGhStateDoubles * off + p;
  o[kLapse * np] = st.lapse;
#pragma unroll
  for (int i = 0; i < 3; ++i) o[(kShift + i) * np] = st.shift[i];
#pragma unroll
  for (int i = 0; i < 6; ++i) o[(kInvSp + i) * np] = st.inv_sp[i];
#pragma unroll
  for (int i = 0; i < 3; ++i) o[(kHalfPhi + i) * np] = st.half_phi_two_normals[i];
#pragma unroll
  for (int i = 0; i < 9; ++i) o[(kPhiNormal + i) * np] = st.phi_one_normal[i];
#pragma unroll
  for (int i = 0; i < 3; ++i) o[(kPiNormal + i) * np] = st.pi_one_normal[i];
#pragma unroll
  for (int i = 0; i < 10; ++i) o[(kPartial + i) * np] = st.dt_pi_partial[i];
  if constexpr (!RAGGED) {
    const int i = p % n0, j = (p / n0) % n1, k = p / (n0 * n1);
    const int points = 2 * (n1 * n2 + n0 * n2 + n0 * n1);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int at = d == 0 ? i : d == 1 ? j : k, nd = d == 0 ? n0 : d == 1 ? n1 : n2;
      if (at != 0 && at != nd - 1) continue;
      const int side = at == 0 ? 0 : 1;
      GhFaceSide s;
      double mag;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        s.n[a] = inv_jac[9 * off + ij3(d, a) * np + p];
        if (side == 0) s.n[a] = s.n[a] * -1.0;
      }
      gh_normalize(s.n, s.nv, &mag, st.inv_sp);
      gh_char_speeds(s.lam, gamma1, st.lapse, st.shift, s.n);
      double* so = sides + kGhSideDoubles * (off / np) * points +
                   face_begin(n0, n1, n2, 2 * d + side) + face_index(n0, n1, d, i, j, k);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        so[a * points] = s.n[a];
        so[(3 + a) * points] = s.nv[a];
      }
#pragma unroll
      for (int a = 0; a < 4; ++a) so[(6 + a) * points] = s.lam[a];
      so[10 * points] = gamma2;
      so[11 * points] = mag;
    }
  }
}

// The pair's fields of a point lie next to each other in LDS: a pencil step
// reads them at one address with constant offsets (a block per field costs an
// address each, which made 44 M vector instructions of 512 x 8^3 instead of
// 27 M), and the stride of 5 doubles spreads the lanes over all banks (a
// stride of 6, for 16-byte loads, puts the xi rows of 8 points on two banks:
// 203 against 191 us).
constexpr int kPairStride = 5;

struct PairFields {
  double v[5];
};
__device__ __forceinline__ PairFields pair_fields(const double* at) {
  return {{at[0], at[1], at[2], at[3], at[4]}};
}

// der[c][d] = sum over l of row[l] * field c at x + l step (first term a
// product, then fused multiply-adds).
__device__ __forceinline__ void pair_derivatives(double der[5][3], int d, int n,
                                                 const double* row, const double* x, int step) {
  PairFields f = pair_fields(x);
  double w = row[0];
#pragma unroll
  for (int c = 0; c < 5; ++c) der[c][d] = w * f.v[c];
#pragma unroll 2
  for (int l = 1; l < n; ++l) {
    x += step;
    f = pair_fields(x);
    w = row[l];
#pragma unroll
    for (int c = 0; c < 5; ++c) der[c][d] = fma(w, f.v[c], der[c][d]);
  }
}

// Doubles of dynamic LDS: the pair's fields, (FACES) the five lifted
// corrections of the element's face points, and the D matrices.
__host__ __device__ inline int pair_lds_doubles(int n0, int n1, int n2, bool faces) {
  return kPairStride * n0 * n1 * n2 + (faces ? 10 * (n1 * n2 + n0 * n2 + n0 * n1) : 0) +
         n0 * n0 + n1 * n1 + n2 * n2;
}

// FACES (uniform domains): faces whose neighbour is -1 take the ghost state
// [E][50][Np] as exterior state, as gh_face_pass_kernel does; their
// corrections are added before those of the internal faces.
// list_or_first: RAGGED: length of `list`, otherwise the launch's first element.
// RAGGED: with a table of lifted corrections (launch_ragged_gh_volume) those of
// the faces a point lies on are added, each face's mortars in order.
template <bool RAGGED, bool FACES, bool UPDATE>
__global__ void __launch_bounds__(512)
gh_pair_kernel(int list_or_first, int n0, int n1, int n2, const MixedElement* __restrict__ el,
               const int32_t* __restrict__ list, const int32_t* __restrict__ nbr,
               const double* __restrict__ u, const double* __restrict__ gammas,
               const double* __restrict__ inv_jac, const double* __restrict__ state,
               const double* __restrict__ sides, const double* __restrict__ ghost,
               double* __restrict__ dt, const double* __restrict__ dtab,
               const MortarCorrection* __restrict__ table, const double* __restrict__ corr,
               Rk3Update update) {
  extern __shared__ double s_lds[];
  int64_t e, off;
  int pr;
  if constexpr (RAGGED) {
    // elements in list order over the XCDs in turn, an element's pairs
    // next to each other on its XCD
    const int x = blockIdx.x % kNumXcds, slot = blockIdx.x / kNumXcds;
    const int at = slot / 10 * kNumXcds + x;
    if (at >= list_or_first) return;
    pr = slot % 10;
    e = list[at];
    const MixedElement m = el[e];
    n0 = m.n[0], n1 = m.n[1], n2 = m.n[2];
    off = m.off;
  } else {
    const int64_t item = xcd_local_element(blockIdx.x, gridDim.x);
    e = item / 10;
    pr = static_cast<int>(item - 10 * e);
    e += list_or_first;
    off = e * n0 * n1 * n2;
  }
  const int np = n0 * n1 * n2;
  const int nf0 = n1 * n2, nf1 = n0 * n2, nf2 = n0 * n1;
  const int points = 2 * (nf0 + nf1 + nf2);
  const int comp[5] = {pr, 10 + pr, 20 + 3 * pr, 21 + 3 * pr, 22 + 3 * pr};
  const int n[3] = {n0, n1, n2};
  double* s_u = s_lds;
  double* s_bc = s_u + kPairStride * np;
  const double* D[3];
  stage_diff_matrices(dtab, n, s_bc + (FACES ? 5 * points : 0), D);
  // workgroup-uniform bases, so that loads take a scalar base and a 32-bit
  // offset
  const double* ue = u + 50 * off;
  const double* ije = inv_jac + 9 * off;
  const double* ga = gammas + 3 * off;
  const double* se = state + kGhStateDoubles * off;
  for (unsigned p = threadIdx.x; p < static_cast<unsigned>(np); p += blockDim.x) {
    PairFields f;
#pragma unroll
    for (int c = 0; c < 5; ++c) f.v[c] = (ue + comp[c] * np)[p];
    double* at = s_u + kPairStride * p;
#pragma unroll
    for (int c = 0; c < 5; ++c) at[c] = f.v[c];
  }
  __syncthreads();
  if constexpr (FACES) {
    for (int x = threadIdx.x; x < points; x += blockDim.x) {
      const int d = x < 2 * nf0 ? 0 : x < 2 * (nf0 + nf1) ? 1 : 2;
      const int nf = d == 0 ? nf0 : d == 1 ? nf1 : nf2;
      const int nd = d == 0 ? n0 : d == 1 ? n1 : n2;
      const int first = face_begin(n0, n1, n2, 2 * d);
      const int side = x - first >= nf ? 1 : 0;
      const int f = x - first - side * nf;
      const int na = d == 0 ? n1 : n0;
      const int b = f / na, a = f - b * na;
      // volume index of the point on the lower face, and across the element
      const int low = d == 0 ? n0 * f : d == 1 ? a + n0 * n1 * b : f;
      const int across = (nd - 1) * (d == 0 ? 1 : d == 1 ? n0 : n0 * n1);
      const int p = low + side * across;
      const int64_t en = nbr[6 * e + 2 * d + side];
      const double* si = sides + kGhSideDoubles * e * points;
      const unsigned xi = x;
      GhFaceSide fi, fe;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        fi.n[i] = (si + i * points)[xi];
        fi.nv[i] = (si + (3 + i) * points)[xi];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) fi.lam[i] = (si + (6 + i) * points)[xi];
      fi.gamma2 = (si + 10 * points)[xi];
      const double fac = lift_factor(nd, (si + 11 * points)[xi]);
      const double* un;
      if (en < 0) {
        un = ghost + 50 * off + p;
        double g[10], lapse, shift[3], inv_sp[6];
#pragma unroll
        for (int c = 0; c < 10; ++c) g[c] = un[c * np];
        gh_lapse_shift(&lapse, shift, inv_sp, g);
#pragma unroll
        for (int i = 0; i < 3; ++i) fe.n[i] = fi.n[i] * -1.0;
        gh_ghost_normal(fe.n, fe.nv, inv_sp);
        gh_char_speeds(fe.lam, ga[np + p], lapse, shift, fe.n);
        fe.gamma2 = fi.gamma2;
      } else {
        un = u + 50 * en * np + low + (1 - side) * across;
        const double* so = sides + kGhSideDoubles * en * points + first + (1 - side) * nf + f;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          fe.n[i] = so[i * points];
          fe.nv[i] = so[(3 + i) * points];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) fe.lam[i] = so[(6 + i) * points];
        fe.gamma2 = so[10 * points];
      }
      double phie[3], pki[13], pke[13], bc[5];
#pragma unroll
      for (int i = 0; i < 3; ++i) phie[i] = un[comp[2 + i] * np];
      const PairFields own = pair_fields(s_u + kPairStride * p);
      gh_package_pair(pki, own.v[0], own.v[1], own.v + 2, fi);
      gh_package_pair(pke, un[comp[0] * np], un[comp[1] * np], phie, fe);
      gh_boundary_terms_pair(bc, pki, fi.lam, pke, fe.lam);
#pragma unroll
      for (int c = 0; c < 5; ++c) s_bc[5 * x + c] = bc[c] * fac;
    }
    __syncthreads();
  }
  const unsigned by_n0 = divisor(n0), by_n1 = divisor(n1);
  for (unsigned p = threadIdx.x; p < static_cast<unsigned>(np); p += blockDim.x) {
    const int row = divide(p, by_n0), k = divide(row, by_n1);
    const int i = p - row * n0, j = row - k * n1;
    double der[5][3];
    pair_derivatives(der, 0, n0, D[0] + i * n0, s_u + kPairStride * row * n0, kPairStride);
    pair_derivatives(der, 1, n1, D[1] + j * n1, s_u + kPairStride * (i + nf2 * k),
                     kPairStride * n0);
    pair_derivatives(der, 2, n2, D[2] + k * n2, s_u + kPairStride * (i + n0 * j),
                     kPairStride * nf2);
    double ij[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) ij[c] = (ije + c * np)[p];
    double dg[3], dpi[3], dphi[9];
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        double s = ij[ij3(0, a)] * der[c][0];
        s = fma(ij[ij3(1, a)], der[c][1], s);
        s = fma(ij[ij3(2, a)], der[c][2], s);
        if (c == 0) dg[a] = s;
        else if (c == 1) dpi[a] = s;
        else dphi[a + 3 * (c - 2)] = s;
      }
    // corrections of the point's faces, loaded together with its state: a
    // face's first mortar here, further ones where they are added
    bool on[3] = {false, false, false};
    int mortars[3];
    const double* from[3];
    double first[3][5];
    if constexpr (RAGGED) {
      if (table != nullptr) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int at = d == 0 ? i : d == 1 ? j : k, nd = d == 0 ? n0 : d == 1 ? n1 : n2;
          on[d] = at == 0 || at == nd - 1;
          if (!on[d]) continue;
          const int nf = d == 0 ? nf0 : d == 1 ? nf1 : nf2;
          const MortarCorrection lower = table[6 * e + 2 * d], upper = table[6 * e + 2 * d + 1];
          mortars[d] = at == 0 ? lower.count : upper.count;
          from[d] = corr + 50 * (at == 0 ? lower.off : upper.off) +
                    face_index(n0, n1, d, i, j, k);
#pragma unroll
          for (int c = 0; c < 5; ++c) first[d][c] = from[d][comp[c] * nf];
        }
      }
    }
    const double gamma1 = (ga + np)[p], gamma2 = (ga + 2 * np)[p];
    GhPointState st;
    st.lapse = (se + kLapse * np)[p];
#pragma unroll
    for (int a = 0; a < 3; ++a) st.shift[a] = (se + (kShift + a) * np)[p];
#pragma unroll
    for (int a = 0; a < 6; ++a) st.inv_sp[a] = (se + (kInvSp + a) * np)[p];
#pragma unroll
    for (int a = 0; a < 3; ++a) st.half_phi_two_normals[a] = (se + (kHalfPhi + a) * np)[p];
#pragma unroll
    for (int a = 0; a < 9; ++a) st.phi_one_normal[a] = (se + (kPhiNormal + a) * np)[p];
#pragma unroll
    for (int a = 0; a < 3; ++a) st.pi_one_normal[a] = (se + (kPiNormal + a) * np)[p];
    st.gamma1p1 = 1.0 + gamma1;
    st.gamma12 = gamma1 * gamma2;
    st.gamma2 = gamma2;
    double out[5];
    const PairFields own = pair_fields(s_u + kPairStride * p);
    gh_point_pair(out, st, (se + (kPartial + pr) * np)[p], own.v[1], own.v + 2, dg, dpi, dphi);
    if constexpr (FACES) {
      const int steps = ghost != nullptr ? 6 : 3;
      for (int step = 0; step < steps; ++step) {
        const int d = step % 3;
        const int at = d == 0 ? i : d == 1 ? j : k, nd = d == 0 ? n0 : d == 1 ? n1 : n2;
        if (at != 0 && at != nd - 1) continue;
        const int dir = 2 * d + (at == 0 ? 0 : 1);
        if (steps == 6 && (nbr[6 * e + dir] < 0) != (step < 3)) continue;
        const double* bc =
            s_bc + 5 * (face_begin(n0, n1, n2, dir) + face_index(n0, n1, d, i, j, k));
#pragma unroll
        for (int c = 0; c < 5; ++c) out[c] = out[c] + bc[c];
      }
    }
    if constexpr (RAGGED) {
      if (table != nullptr) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (!on[d]) continue;
          const double* src = from[d];
#pragma unroll
          for (int c = 0; c < 5; ++c) out[c] = out[c] + first[d][c];
          const int nf = d == 0 ? nf0 : d == 1 ? nf1 : nf2;
          for (int q = 1; q < mortars[d]; ++q) {
            src += 50 * nf;
#pragma unroll
            for (int c = 0; c < 5; ++c) out[c] = out[c] + src[comp[c] * nf];
          }
        }
      }
    }
    if constexpr (UPDATE) {
      // the fields are read from the LDS once more: held in registers since the
      // point-wise terms they would cost a wavefront per SIMD
      asm volatile("" ::: "memory");
      const PairFields uk = pair_fields(s_u + kPairStride * p);
      const double h = rk3_step_size(update);
      const double* u0 = update.u0 + 50 * off;
      double first_u[5];
#pragma unroll
      for (int c = 0; c < 5; ++c)
        first_u[c] = update.substep == 0 ? uk.v[c] : (u0 + comp[c] * np)[p];
#pragma unroll
      for (int c = 0; c < 5; ++c)
        out[c] = rk3_value(update.substep, h, first_u[c], uk.v[c], out[c]);
    }
    double* dte = dt + 50 * off;
#pragma unroll
    for (int c = 0; c < 5; ++c) (dte + comp[c] * np)[p] = out[c];
  }
}

// Threads of a workgroup that takes np points in rounds.  Up to 256 points, or
// where the launch has no second workgroup for a CU: one round (2 elements of
// 7x7x6 16.6 us, with 192 threads 19.3).  Up to 768, where several workgroups
// share a CU: 192 or 256, whichever leaves fewer lanes idle in the last round (360
// elements of 7x7x6 with 192 / 256 / 320 / 512 threads 81 / 85 / 101 / 100 us, of
// 8x8x7 115 / 106 / 141 / 125, of 9^3 202 / 191 / 224 / 197).  Beyond: 512, the more
// so where the LDS leaves one workgroup per CU (360 of 10x9x9 283 / 259 / 251 / 228;
// 64 of 14^3 249 / 203 / 182 / 154).  The fewest idle lanes alone can mean 64 threads:
// 526 us on 360 of 10x9x9, 577 on 64 of 14^3.
int pair_threads(int np, int num_elements) {
  if (np > 768) return 512;
  if (np <= 256 || 10 * num_elements <= kNumCus) return std::min(512, (np + 63) / 64 * 64);
  return (np + 191) / 192 * 192 < (np + 255) / 256 * 256 ? 192 : 256;
}

}  // namespace

// Whether the two kernels take less time than the fused one (isotropic N = 3
// .. 8).  The fused kernel fills whole CUs, so its time goes in rounds of kNumCus x
// (workgroups per CU) elements; the pair kernel's workgroups are a tenth of an
// element and its time is a launch's worth plus a time per element.
// Measured in microseconds (periodic; the Dirichlet closure has the same
// crossings), fused / pairs: 8^3 at 128 elements 66 / 51, 200 71 / 76, 300 136 / 112,
// 512 146 / 194; 7^3 at 128 76 / 40, 343 151 / 95, 512 158 / 145, 2048 622 / 581;
// 6^3 at 64 33 / 22, 200 36 / 43, 300 65 / 57, 512 73 / 94; 5^3 at 256 38 / 36,
// 512 44 / 58, 576 73 / 68; 4^3 at 300 35 / 27, 768 40 / 46; 3^3 at 300 25 / 23,
// 768 29 / 35.
bool gh_pairs_faster(int num_elements, const int32_t ext[3]) {
  struct Cost {
    double element, round;  // pairs: 14 + element * elements; fused: round * rounds
    int per_cu;
  };
  static const Cost cost[6] = {{0.028, 26.0, 4}, {0.043, 35.0, 4}, {0.085, 37.0, 2},
                               {0.155, 34.0, 1}, {0.25, 79.0, 1},  {0.366, 71.0, 1}};
  if (ext[0] < 3 || ext[0] > 8 || ext[1] != ext[0] || ext[2] != ext[0]) return false;
  const Cost& c = cost[ext[0] - 3];
  const int per_round = kNumCus * c.per_cu;
  const int rounds = (num_elements + per_round - 1) / per_round;
  return 14.0 + c.element * num_elements < c.round * rounds;
}

size_t gh_pairs_work_doubles(int num_elements, const int32_t ext[3]) {
  const size_t np = static_cast<size_t>(ext[0]) * ext[1] * ext[2];
  return num_elements * (kGhStateDoubles * np +
                         kGhSideDoubles * 2 * (np / ext[0] + np / ext[1] + np / ext[2]));
}

bool gh_pairs_supported(const int32_t ext[3]) {
  return pair_lds_doubles(ext[0], ext[1], ext[2], true) * 8 <= 160 * 1024;
}

int launch_gh_rhs_pairs(int num_elements, const int32_t ext[3], const int32_t* nbr,
                        const double* u, const double* gammas, const double* inv_jac, double* dt,
                        double* work, const double* ghost, hipStream_t stream,
                        const Rk3Update& up) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  const int np = ext[0] * ext[1] * ext[2];
  const int64_t total = static_cast<int64_t>(num_elements) * np;
  const int lds = pair_lds_doubles(ext[0], ext[1], ext[2], true) * 8;
  const auto pair_kernel = up.substep < 0 ? &gh_pair_kernel<false, true, false>
                                          : &gh_pair_kernel<false, true, true>;
  if (!allow_lds(reinterpret_cast<const void*>(pair_kernel), lds)) return SXD_ERR_UNSUPPORTED;
  double* sides = work + kGhStateDoubles * total;
  hipLaunchKernelGGL(gh_state_kernel<false>, dim3(static_cast<unsigned>((total + 127) / 128)),
                     dim3(128), 0, stream, total, ext[0], ext[1], ext[2], nullptr, nullptr, u,
                     gammas, inv_jac, work, sides);
  if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  const int threads = pair_threads(np, num_elements);
  const int limit = launch_limit(10, threads);
  for (int first = 0; first < num_elements; first += limit) {
    hipLaunchKernelGGL(pair_kernel, dim3(10 * std::min(limit, num_elements - first)),
                       dim3(threads), lds, stream, first, ext[0], ext[1], ext[2], nullptr, nullptr,
                       nbr, u, gammas, inv_jac, work, sides, ghost, dt, dtab, nullptr, nullptr,
                       up);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  return SXD_OK;
}

int launch_ragged_gh_state(int count, const int32_t* list, const MixedElement* el, int np_max,
                           const double* u, const double* gammas, double* state,
                           hipStream_t stream) {
  if (count == 0) return SXD_OK;
  if (state == nullptr) return SXD_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(gh_state_kernel<true>, dim3(count, (np_max + 127) / 128), dim3(128), 0,
                     stream, 0, 0, 0, 0, el, list, u, gammas, nullptr, state, nullptr);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

int launch_ragged_gh_volume(const std::vector<RaggedClass>& classes, const int32_t* list,
                            const MixedElement* el, const double* u, const double* gammas,
                            const double* inv_jac, double* dt, const double* state,
                            const MortarCorrection* table, const double* corr,
                            hipStream_t stream, const Rk3Update& up) {
  const double* dtab = device_diff_matrices();
  if (dtab == nullptr) return SXD_ERR_DEVICE;
  if (state == nullptr) return SXD_ERR_INVALID_ARGUMENT;
  const auto pair_kernel = up.substep < 0 ? &gh_pair_kernel<true, false, false>
                                          : &gh_pair_kernel<true, false, true>;
  for (const RaggedClass& c : classes) {
    const int lds = (kPairStride * c.np_max + c.d_doubles) * 8;
    if (!allow_lds(reinterpret_cast<const void*>(pair_kernel), lds)) return SXD_ERR_UNSUPPORTED;
    const int threads = c.np_max > 910 ? 512 : c.np_max > 128 ? 256 : 128;
    const int limit = launch_limit(10, threads);
    for (int first = 0; first < c.count; first += limit) {
      const int count = std::min(limit, c.count - first);
      hipLaunchKernelGGL(pair_kernel, dim3((count + kNumXcds - 1) / kNumXcds * kNumXcds * 10),
                         dim3(threads), lds, stream, count, 0, 0, 0, el, list + c.begin + first,
                         nullptr, u, gammas, inv_jac, state, nullptr, nullptr, dt, dtab, table,
                         corr, up);
      if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
    }
  }
  return SXD_OK;
}

}  // namespace sxd
