// Face part of the GH adjoint on ragged domains: the transposed mortar coupling,
// both sides of a mortar in one workgroup per symmetric pair.
//
// For each side, with c its corrections on the face and gbar the adjoint of dt:
// the forward is recomputed up to c (mortar_side.hpp), then
//   seeds   gbar * lift factor on the face, and gbar . c for the adjoint of |n|;
//   P^T     the seeds through the transposed projection, dimension b, then a;
//   weights the adjoint of the side's package on the mortar, interior for its own
//           correction and exterior for the other side's, from the upwind
//           weights of the mortar speeds;
//   I^T     transposed interpolation onto the face, dimension b, then a;
//   package reverse at the face points: the pair's 5 components of the side's
//           contribution, and the adjoints of its normals and speeds.
// Contributions go to a slot per record ([50][nf], added by the transposed
// sweeps), the adjoints of normals, speeds and |n| to 11 values per pair and
// face point, which gh_adjoint_sides_kernel sums over the pairs and takes to g.
//
// Bound by LDS traffic and the barriers between the steps, as the forward's
// corrections.  One workgroup per (element, face side, pair) took each mortar
// twice, formed both sides' packages in each, and updated ubar in three
// launches: 257 us per dimension on 300 elements of extents 6 .. 10, where the
// mortars here take 203 us in all and the whole adjoint 742 us instead of 1284.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_common.hpp"
#include "gh_adjoint.hpp"
#include "gh_point.hpp"
#include "kernels.hpp"
#include "mortar_side.hpp"

namespace sxd {
namespace {

// LDS (doubles) beyond the forward's: the seeds of both sides; the corrections'
// room also holds 10 values per mortar point, and the staged values' room one
// side's package adjoint on the mortar and with dimension b transposed.
struct AdjointLds {
  int bc, staged, seeds;
  __host__ __device__ AdjointLds(int na0, int nb0, int ka0, int na1, int nb1, int ka1, int km,
                                 const SideLds& l0, const SideLds& l1) {
    bc = corrections_doubles(km, l0, l1);
    const int t0 = ka0 * nb0 > na0 * nb0 ? ka0 * nb0 : na0 * nb0;
    const int t1 = ka1 * nb1 > na1 * nb1 ? ka1 * nb1 : na1 * nb1;
    const int fwd = l0.staged + l1.staged, back = kPk * (km + (t0 > t1 ? t0 : t1));
    staged = fwd > back ? fwd : back;
    seeds = 5 * (na0 * nb0 + na1 * nb1);
  }
  __host__ __device__ AdjointLds(const MortarSide& r0, const MortarSide& r1, const SideLds& l0,
                                 const SideLds& l1)
      : AdjointLds(r0.na, r0.nb, r0.ka, r1.na, r1.nb, r1.ka, r0.ka * r0.kb, l0, l1) {}
};

// out[i] (5 of 13 values from c0) = sum over r of w[r ws] in[r] at stride `step`.
__device__ __forceinline__ void transposed_line(double s[5], const double* in, int step,
                                                const double* w, int ws, int n) {
#pragma unroll
  for (int c = 0; c < 5; ++c) s[c] = w[0] * in[c];
#pragma unroll 2
  for (int r = 1; r < n; ++r) {
    in += step;
    const double a = w[r * ws];
#pragma unroll
    for (int c = 0; c < 5; ++c) s[c] = fma(a, in[c], s[c]);
  }
}

// Steps from the seeds on the mortar (own: this side's, other: the other
// side's) to the face for one side.  own_first: the side is the job's first, so
// its mortar points are numbered as `gather` is indexed.
__device__ __forceinline__ void side_adjoint(const MortarSide& r, const SideLds& l, bool own_first,
                                             const double* own, const double* other,
                                             const double* ma, const double* mb, double* s_b,
                                             const int32_t* gather, int pr, const double* u,
                                             const double* sides, const double* speeds,
                                             double* contrib, double* side_adj) {
  const int km = r.ka * r.kb, t = threadIdx.x, T = blockDim.x;
  double* s_w = s_b + kPk * km;
  const unsigned by_ka = divisor(r.ka), by_na = divisor(r.na);
  for (int k = t; k < km; k += T) {
    const int q = gather[k];
    const int mine = own_first ? k : q, theirs = own_first ? q : k;
    double lam[4], B[13];
#pragma unroll
    for (int c = 0; c < 4; ++c) lam[c] = speeds[4 * r.rec_off + c * km + mine];
    gh_package_seed(lam, own + 5 * mine, other + 5 * theirs, B);
#pragma unroll
    for (int c = 0; c < kPk; ++c) s_b[kPk * mine + c] = B[c];
  }
  __syncthreads();
  const double* w = s_b;  // dimension b transposed: [face b][mortar a]
  if (l.mat_b > 0) {
    const int items = r.ka * r.nb;
    for (int x = t; x < 3 * items; x += T) {
      const int g = (x >= items) + (x >= 2 * items), y = x - g * items;
      const int lb = divide(y, by_ka), ra = y - lb * r.ka;
      double s[5];
      transposed_line(s, s_b + kPk * ra + 4 * g, kPk * r.ka, mb + lb, r.nb, r.kb);
#pragma unroll
      for (int c = 0; c < 5; ++c) s_w[kPk * y + 4 * g + c] = s[c];
    }
    __syncthreads();
    w = s_w;
  }
  const double* x_face = w;
  if (l.mat_a > 0) {
    double* out = l.mat_b > 0 ? s_b : s_w;
    const int items = r.na * r.nb;
    for (int x = t; x < 3 * items; x += T) {
      const int g = (x >= items) + (x >= 2 * items), y = x - g * items;
      const int lb = divide(y, by_na), la = y - lb * r.na;
      double s[5];
      transposed_line(s, w + kPk * r.ka * lb + 4 * g, kPk, ma + la, r.na, r.ka);
#pragma unroll
      for (int c = 0; c < 5; ++c) out[kPk * y + 4 * g + c] = s[c];
    }
    __syncthreads();
    x_face = out;
  }
  const int nf = r.nf;
  for (int f = t; f < nf; f += T) {
    const int b = divide(f, by_na), a = f - b * r.na;
    const int p = r.base + a * r.step_a + b * r.step_b;
    const double* sd = sides + 12 * r.pt_off + f;
    double n[3], nv[3], lam[4], B[13], fields[5], out[5];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      n[i] = sd[i * nf];
      nv[i] = sd[(3 + i) * nf];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) lam[c] = sd[(6 + c) * nf];
    const double gamma2 = sd[10 * nf];
    const double* ue = u + 50 * r.off + p;
    const int comp[5] = {pr, 10 + pr, 20 + 3 * pr, 21 + 3 * pr, 22 + 3 * pr};
#pragma unroll
    for (int c = 0; c < 5; ++c) fields[c] = ue[comp[c] * r.np];
#pragma unroll
    for (int c = 0; c < kPk; ++c) B[c] = x_face[kPk * f + c];
    double adj[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    gh_package_vjp(n, nv, lam, gamma2, fields, B, out, adj, adj + 3, adj + 6);
    double* to = contrib + 50 * r.corr_off + f;
#pragma unroll
    for (int c = 0; c < 5; ++c) to[comp[c] * nf] = out[c];
    double* so = side_adj + 110 * r.corr_off + 11 * pr * nf + f;
#pragma unroll
    for (int c = 0; c < 10; ++c) so[c * nf] = adj[c];
  }
  __syncthreads();  // the LDS is free for the other side
}

// Grid as mortar_corrections_kernel<true>.
__global__ void __launch_bounds__(256)
gh_adjoint_mortar_kernel(int count, const MortarJob* __restrict__ jobs,
                         const int32_t* __restrict__ gather, const double* __restrict__ u,
                         const double* __restrict__ params, const double* __restrict__ inv_jac,
                         const double* __restrict__ gbar, const double* __restrict__ sides,
                         const double* __restrict__ speeds, double* __restrict__ contrib,
                         double* __restrict__ side_adj, const double* __restrict__ full,
                         const double* __restrict__ half) {
  extern __shared__ double s_lds[];
  const int xcd = blockIdx.x % kNumXcds, slot = blockIdx.x / kNumXcds;
  const int at = slot / 10 * kNumXcds + xcd, pr = slot % 10;
  if (at >= count) return;
  const MortarSide& r0 = jobs[at].side[0];
  const MortarSide& r1 = jobs[at].side[1];
  const SideLds l0(r0, true), l1(r1, true);
  const AdjointLds la(r0, r1, l0, l1);
  const int km = r0.ka * r0.kb;
  const MortarLds sh(s_lds, km, l0, l1, la.bc, la.staged);
  double* const s_seed0 = sh.end;
  double* const s_seed1 = s_seed0 + 5 * r0.nf;
  const int comp[5] = {pr, 10 + pr, 20 + 3 * pr, 21 + 3 * pr, 22 + 3 * pr};
  mortar_terms<true>(r0, r1, l0, l1, sh, comp, gather, u, params, inv_jac, sides, speeds, full,
                     half);
  const int t = threadIdx.x, T = blockDim.x;
  const unsigned by_na0 = divisor(r0.na), by_na1 = divisor(r1.na);
  // corrections on the faces; seeds, and the pair's part of the |n| adjoint
  for (int x = t; x < r0.nf + r1.nf; x += T) {
    const bool second = x >= r0.nf;
    const MortarSide& r = second ? r1 : r0;
    const int f = second ? x - r0.nf : x, nf = r.nf;
    const int fb = divide(f, second ? by_na1 : by_na0), fa = f - fb * r.na;
    double v[5];
    mortar_face_value(v, r, second ? l1.mat_a > 0 : l0.mat_a > 0,
                      second ? l1.mat_b > 0 : l0.mat_b > 0, sh, second, fa, fb);
    const double lift = lift_factor(r.extent, 1.0);
    const double fac = lift * sides[12 * r.pt_off + 11 * nf + f];
    const double* ge = gbar + 50 * r.off + r.base + fa * r.step_a + fb * r.step_b;
    double* seed = MortarLds::pick(second, s_seed1, s_seed0) + 5 * f;
    double fac_b = 0.0;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const double gb = ge[comp[c] * r.np];
      fac_b += gb * v[c];
      seed[c] = gb * fac;
    }
    side_adj[110 * r.corr_off + (11 * pr + 10) * nf + f] = lift * fac_b;
  }
  __syncthreads();
  // transposed projection of both sides' seeds: dimension b into the staged
  // values' room, then dimension a into the corrections' room
  if (l0.mat_b + l1.mat_b > 0) {
    const int items0 = l0.mat_b > 0 ? r0.na * r0.kb : 0;
    const int items1 = l1.mat_b > 0 ? r1.na * r1.kb : 0;
    for (int x = t; x < items0 + items1; x += T) {
      const bool second = x >= items0;
      const MortarSide& r = second ? r1 : r0;
      const int y = second ? x - items0 : x;
      const int rb = divide(y, second ? by_na1 : by_na0), fa = y - rb * r.na;
      double s[5];
      transposed_line(s, MortarLds::pick(second, s_seed1, s_seed0) + 5 * fa, 5 * r.na,
                      sh.mb(second) + r.nb * r.kb + rb, r.kb, r.nb);
      double* o = sh.st(second) + 5 * y;
#pragma unroll
      for (int c = 0; c < 5; ++c) o[c] = s[c];
    }
    __syncthreads();
  }
  const unsigned by_ka0 = divisor(r0.ka), by_ka1 = divisor(r1.ka);
  double* const z0 = MortarLds::pick(l0.mat_b > 0, sh.st0, s_seed0);
  double* const z1 = MortarLds::pick(l1.mat_b > 0, sh.st1, s_seed1);
  for (int x = t; x < 2 * km; x += T) {
    const bool second = x >= km;
    const MortarSide& r = second ? r1 : r0;
    const int y = second ? x - km : x;
    const int rb = divide(y, second ? by_ka1 : by_ka0), ra = y - rb * r.ka;
    const double* src = MortarLds::pick(second, z1, z0);
    double s[5];
    if (second ? l1.mat_a > 0 : l0.mat_a > 0) {
      transposed_line(s, src + 5 * r.na * rb, 5, sh.ma(second) + r.na * r.ka + ra,
                      r.ka, r.na);
    } else {
#pragma unroll
      for (int c = 0; c < 5; ++c) s[c] = src[5 * y + c];
    }
    double* o = sh.bc(second) + 5 * y;
#pragma unroll
    for (int c = 0; c < 5; ++c) o[c] = s[c];
  }
  __syncthreads();
  const int32_t* to_second = gather + r0.rec_off;
  side_adjoint(r0, l0, true, sh.bc0, sh.bc1, sh.ma0, sh.mb0, sh.st0, to_second, pr, u, sides,
               speeds, contrib, side_adj);
  side_adjoint(r1, l1, false, sh.bc1, sh.bc0, sh.ma1, sh.mb1, sh.st0, to_second, pr, u, sides,
               speeds, contrib, side_adj);
}

// The adjoints of a face's normals, speeds and |n|, summed over its mortars and
// the ten pairs, to g: added to the g components of its first mortar's slot.
// One workgroup per face.
__global__ void __launch_bounds__(128)
gh_adjoint_sides_kernel(const MixedElement* __restrict__ el, const MortarFace* __restrict__ faces,
                        const MortarRecord* __restrict__ recs, const double* __restrict__ u,
                        const double* __restrict__ params, const double* __restrict__ inv_jac,
                        const double* __restrict__ side_adj, double* __restrict__ contrib) {
  const MortarFace fr = faces[blockIdx.x];
  const MixedElement m = el[fr.e];
  const int d = fr.dir >> 1, side = fr.dir & 1;
  const int n0 = m.n[0], n1 = m.n[1], na = d == 0 ? n1 : n0, nf = fr.nf;
  const int nd = d == 0 ? n0 : (d == 1 ? n1 : m.n[2]);
  const int64_t slot = recs[fr.rec_begin].corr_off;
  for (int f = threadIdx.x; f < nf; f += blockDim.x) {
    const int b = f / na, a = f - b * na, fixed = side == 0 ? 0 : nd - 1;
    const int p = d == 0 ? fixed + n0 * (a + n1 * b)
                  : d == 1 ? a + n0 * (fixed + n1 * b) : a + n0 * (b + n1 * fixed);
    double n[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      n[i] = inv_jac[9 * m.off + ij3(d, i) * m.np + p];
      if (side == 0) n[i] = n[i] * -1.0;
    }
    const double gamma1 = params[3 * m.off + m.np + p];
    GhSideFwd s;
    gh_side_forward(s, u + 50 * m.off + p, m.np, gamma1, n);
    double sum[11] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int q = 0; q < fr.rec_count; ++q) {
      const double* in = side_adj + 110 * (slot + static_cast<int64_t>(q) * nf) + f;
#pragma unroll 2
      for (int pr = 0; pr < 10; ++pr)
#pragma unroll
        for (int c = 0; c < 11; ++c) sum[c] += in[(11 * pr + c) * nf];
    }
    double gm[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    gh_side_vjp(s, gamma1, sum, sum + 3, sum + 6, sum[10], gm);
    double* out = contrib + 50 * slot + f;
#pragma unroll
    for (int c = 0; c < 10; ++c) out[c * nf] += gm[c];
  }
}

}  // namespace

int gh_adjoint_mortar_lds_bytes(const MortarRecord& r, const MortarRecord& partner) {
  auto side = [](const MortarRecord& m) {
    return SideLds(m.size_a != kChildFull || m.na != m.ka, m.size_b != kChildFull || m.nb != m.kb,
                   m.na, m.nb, m.ka, m.kb, true);
  };
  const SideLds a = side(r), b = side(partner);
  const AdjointLds l(r.na, r.nb, r.ka, partner.na, partner.nb, partner.ka, r.ka * r.kb, a, b);
  return 8 * (l.bc + l.staged + l.seeds + a.mat_a + a.mat_b + b.mat_a + b.mat_b);
}

GhAdjointFacesWork::GhAdjointFacesWork(const MortarPlan& plan, double* work) {
  contrib = work;
  side_adj = contrib + 50 * plan.corr_points;
  sides = side_adj + 110 * plan.corr_points;
  speeds = sides + 12 * plan.face_points;
  doubles = 160 * plan.corr_points + 12 * plan.face_points + 4 * plan.record_points;
}

int launch_gh_adjoint_faces(const MortarPlan& plan, const MixedElement* el, const double* u,
                            const double* gammas, const double* inv_jac, const double* gbar,
                            double* work, hipStream_t stream) {
  const double* full = device_mortar_matrices();
  const double* half = device_half_mortar_matrices();
  if (full == nullptr || half == nullptr) return SXD_ERR_DEVICE;
  if (work == nullptr || plan.num_remote > 0) return SXD_ERR_INVALID_ARGUMENT;
  const GhAdjointFacesWork w(plan, work);
  int rc = launch_gh_mortar_sides(plan, el, u, gammas, inv_jac, w.sides, w.speeds, stream);
  if (rc != SXD_OK) return rc;
  for (const MortarClass& c : plan.classes[1]) {
    if (!allow_lds(reinterpret_cast<const void*>(&gh_adjoint_mortar_kernel), c.adjoint_lds_bytes))
      return SXD_ERR_UNSUPPORTED;
    const int limit = launch_limit(10, 192);
    for (int first = 0; first < c.count; first += limit) {
      const int count = std::min(limit, c.count - first);
      hipLaunchKernelGGL(gh_adjoint_mortar_kernel,
                         dim3((count + kNumXcds - 1) / kNumXcds * kNumXcds * 10), dim3(192),
                         c.adjoint_lds_bytes, stream, count, plan.d_jobs + c.begin + first,
                         plan.d_gather, u, gammas, inv_jac, gbar, w.sides, w.speeds, w.contrib,
                         w.side_adj, full, half);
      if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
    }
  }
  hipLaunchKernelGGL(gh_adjoint_sides_kernel, dim3(plan.num_faces), dim3(128), 0, stream, el,
                     plan.d_faces, plan.d_records, u, gammas, inv_jac, w.side_adj, w.contrib);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

}  // namespace sxd
