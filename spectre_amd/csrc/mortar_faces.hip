// Boundary corrections of mortar domains without remote mortars: every mortar
// taken from its two elements' fields to both elements' lifted corrections in
// one workgroup (GH: one per symmetric pair).  The volume kernels add the
// corrections where they write dt, each point's faces in direction order and
// a face's mortars in record order.
//
// mortar.hip keeps the steps apart (packages, projection, boundary terms, lift)
// around the exchange of boundary messages.  There every step is a pass over
// HBM: 134 packaged values per GH mortar point written and read, 50
// corrections written and read, and dt read and written once per face, against
// the two faces' fields read and 50 corrections per face point written here.
//
// Steps of a workgroup, each over both sides, with a barrier in between (the
// arithmetic and its order are mortar.hip's):
//   1. packages of the face points (13 values) into LDS, next to each other;
//   2. dimension-a interpolation onto the mortar where the mesh differs;
//   3. per mortar point and group of outputs: dimension-b interpolation of the
//      3 or 4 values the group needs, boundary terms of both sides;
//   4. dimension-a projection back; 5. dimension-b projection, lift, write.
// A mortar's LDS is laid out by its own extents; GH mortars are launched in
// classes of similar LDS size, since a launch reserves its largest for all.
// What bounds it is latency: the phases of a workgroup are short and 12 to 18
// waves per CU hide them only in part (vector units busy 40 %, LDS 30 %).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_common.hpp"
#include "gh_point.hpp"
#include "kernels.hpp"
#include "mortar_side.hpp"

namespace sxd {
namespace {

__device__ __forceinline__ int volume_index(const MixedElement& m, int d, int side, int a,
                                            int b) {
  const int n0 = m.n[0], n1 = m.n[1];
  const int nd = d == 0 ? n0 : (d == 1 ? n1 : m.n[2]);
  const int fixed = side == 0 ? 0 : nd - 1;
  if (d == 0) return fixed + n0 * (a + n1 * b);
  if (d == 1) return a + n0 * (fixed + n1 * b);
  return a + n0 * (b + n1 * fixed);
}

__device__ __forceinline__ const double* matrix_block(const double* full, const double* half,
                                                      int nf, int nm, int size) {
  const double* table = size == kChildFull ? full
                        : size == kChildUpperHalf ? half : half + kPackedMortarSize;
  return table + mortar_table_offset(nf, nm);
}

// Normals, speeds, gamma2 and |n| of every face point ([12][nf] at 12 pt_off)
// and the speeds on each of the face's mortars ([4][km] at 4 rec_off), one
// workgroup per face: they are the same for the ten pairs.
__global__ void __launch_bounds__(128)
gh_mortar_sides_kernel(const MixedElement* __restrict__ el, const MortarFace* __restrict__ faces,
                       const MortarRecord* __restrict__ recs, const double* __restrict__ u,
                       const double* __restrict__ params, const double* __restrict__ inv_jac,
                       double* __restrict__ sides, double* __restrict__ speeds,
                       const double* __restrict__ full, const double* __restrict__ half,
                       int kf) {
  extern __shared__ double s_lam[];  // [4][nf], then [4][ka nb]
  double* s_tmp = s_lam + 4 * kf;
  const MortarFace fr = faces[blockIdx.x];
  const MixedElement m = el[fr.e];
  const int d = fr.dir >> 1, side = fr.dir & 1;
  const int na = d == 0 ? m.n[1] : m.n[0];
  const int nf = fr.nf, np = m.np;
  double* out = sides + 12 * fr.pt_off;
  for (int f = threadIdx.x; f < nf; f += blockDim.x) {
    const int p = volume_index(m, d, side, f % na, f / na);
    const double* ue = u + 50 * m.off + p;
    double g[10], lapse, shift[3], inv_sp[6], mag;
#pragma unroll
    for (int c = 0; c < 10; ++c) g[c] = ue[c * np];
    GhFaceSide s;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      s.n[i] = inv_jac[9 * m.off + ij3(d, i) * np + p];
      if (side == 0) s.n[i] = s.n[i] * -1.0;
    }
    gh_lapse_shift(&lapse, shift, inv_sp, g);
    const double* ga = params + 3 * m.off + p;
    gh_normalize(s.n, s.nv, &mag, inv_sp);
    gh_char_speeds(s.lam, ga[np], lapse, shift, s.n);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      out[i * nf + f] = s.n[i];
      out[(3 + i) * nf + f] = s.nv[i];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      out[(6 + c) * nf + f] = s.lam[c];
      s_lam[c * nf + f] = s.lam[c];
    }
    out[10 * nf + f] = ga[2 * np];
    out[11 * nf + f] = mag;
  }
  for (int t = fr.rec_begin; t < fr.rec_begin + fr.rec_count; ++t) {
    const MortarRecord r = recs[t];
    const int km = r.ka * r.kb;
    const double* src = s_lam;
    __syncthreads();
    if (r.size_a != kChildFull || r.na != r.ka) {
      const double* Ma = matrix_block(full, half, r.na, r.ka, r.size_a);
      for (int x = threadIdx.x; x < 4 * r.ka * r.nb; x += blockDim.x) {
        const int c = x / (r.ka * r.nb), y = x % (r.ka * r.nb), lb = y / r.ka, ra = y % r.ka;
        const double* v = s_lam + c * nf + r.na * lb;
        double s = Ma[ra * r.na] * v[0];
        for (int l = 1; l < r.na; ++l) s = fma(Ma[ra * r.na + l], v[l], s);
        s_tmp[x] = s;
      }
      src = s_tmp;
      __syncthreads();
    }
    const double* Mb = matrix_block(full, half, r.nb, r.kb, r.size_b);
    for (int x = threadIdx.x; x < 4 * km; x += blockDim.x) {
      const int c = x / km, k = x % km, rb = k / r.ka, ra = k % r.ka;
      const double* v = src + c * r.ka * r.nb + ra;
      double s;
      if (r.size_b != kChildFull || r.nb != r.kb) {
        s = Mb[rb * r.nb] * v[0];
        for (int l = 1; l < r.nb; ++l) s = fma(Mb[rb * r.nb + l], v[r.ka * l], s);
      } else {
        s = v[r.ka * rb];
      }
      speeds[4 * r.rec_off + x] = s;
    }
  }
}

// Grid: GH 10 workgroups per job, one per symmetric pair (next to each other on
// one XCD, padded to a multiple of 8 jobs); ScalarWave one workgroup per job.
// corr: [NC][nf] per side at NC corr_off, the lifted corrections of the side's
// own face.
template <bool GH>
__global__ void __launch_bounds__(256)
mortar_corrections_kernel(int count, const MortarJob* __restrict__ jobs,
                          const int32_t* __restrict__ gather, const double* __restrict__ u,
                          const double* __restrict__ params, const double* __restrict__ inv_jac,
                          const double* __restrict__ sides, const double* __restrict__ speeds,
                          double* __restrict__ corr, const double* __restrict__ full,
                          const double* __restrict__ half) {
  constexpr int NC = GH ? 50 : 5;
  extern __shared__ double s_lds[];
  int at = blockIdx.x, pr = 0;
  if constexpr (GH) {
    const int x = blockIdx.x % kNumXcds, slot = blockIdx.x / kNumXcds;
    at = slot / 10 * kNumXcds + x;
    pr = slot % 10;
    if (at >= count) return;
  }
  const MortarSide& r0 = jobs[at].side[0];
  const MortarSide& r1 = jobs[at].side[1];
  const SideLds l0(r0, GH), l1(r1, GH);
  const int km = r0.ka * r0.kb;
  const MortarLds sh(s_lds, km, l0, l1, corrections_doubles(km, l0, l1), l0.staged + l1.staged);
  const int comp[5] = {pr, GH ? 10 + pr : 1, GH ? 20 + 3 * pr : 2, GH ? 21 + 3 * pr : 3,
                       GH ? 22 + 3 * pr : 4};
  mortar_terms<GH>(r0, r1, l0, l1, sh, comp, gather, u, params, inv_jac, sides, speeds, full,
                   half);
  // 5. dimension b back to the face, and lift
  const unsigned by_na0 = divisor(r0.na), by_na1 = divisor(r1.na);
  for (int x = threadIdx.x; x < r0.nf + r1.nf; x += blockDim.x) {
    const bool second = x >= r0.nf;
    const MortarSide& r = second ? r1 : r0;
    const int f = second ? x - r0.nf : x, nf = r.nf;
    const int fb = divide(f, second ? by_na1 : by_na0), fa = f - fb * r.na;
    double v[5];
    mortar_face_value(v, r, second ? l1.mat_a > 0 : l0.mat_a > 0,
                      second ? l1.mat_b > 0 : l0.mat_b > 0, sh, second, fa, fb);
    double mag;
    if constexpr (GH)
      mag = sides[12 * r.pt_off + 11 * nf + f];
    else
      mag = sh.mag(second)[f];
    const double fac = lift_factor(r.extent, mag);
    double* out = corr + NC * r.corr_off + f;
#pragma unroll
    for (int c = 0; c < 5; ++c) out[comp[c] * nf] = v[c] * fac;
  }
}

}  // namespace

int mortar_corrections_lds_bytes(bool gh, const MortarRecord& r, const MortarRecord& partner) {
  auto side = [gh](const MortarRecord& m) {
    return SideLds(m.size_a != kChildFull || m.na != m.ka, m.size_b != kChildFull || m.nb != m.kb,
                   m.na, m.nb, m.ka, m.kb, gh);
  };
  const SideLds a = side(r), b = side(partner);
  return 8 * (corrections_doubles(r.ka * r.kb, a, b) + a.staged + b.staged + a.mat_a + a.mat_b +
              b.mat_a + b.mat_b + a.mag + b.mag);
}

MortarCorrectionsWork::MortarCorrectionsWork(bool gh, const MortarPlan& plan, double* work) {
  corr = work;
  sides = corr + (gh ? 50 : 5) * plan.corr_points;
  speeds = sides + (gh ? 12 * plan.face_points : 0);
  doubles = (gh ? 50 : 5) * plan.corr_points +
            (gh ? 12 * plan.face_points + 4 * plan.record_points : 0);
}

int launch_gh_mortar_sides(const MortarPlan& plan, const MixedElement* el, const double* u,
                           const double* params, const double* inv_jac, double* sides,
                           double* speeds, hipStream_t stream) {
  const double* full = device_mortar_matrices();
  const double* half = device_half_mortar_matrices();
  if (full == nullptr || half == nullptr) return SXD_ERR_DEVICE;
  hipLaunchKernelGGL(gh_mortar_sides_kernel, dim3(plan.num_faces), dim3(128),
                     8 * 4 * (plan.kf + plan.tmp_max), stream, el, plan.d_faces, plan.d_records, u,
                     params, inv_jac, sides, speeds, full, half, plan.kf);
  return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
}

int launch_mortar_lifted_corrections(bool gh, const MortarPlan& plan, const MixedElement* el,
                                     const double* u, const double* params,
                                     const double* inv_jac, double* work, hipStream_t stream) {
  const double* full = device_mortar_matrices();
  const double* half = device_half_mortar_matrices();
  if (full == nullptr || half == nullptr) return SXD_ERR_DEVICE;
  if (work == nullptr || plan.num_remote > 0) return SXD_ERR_INVALID_ARGUMENT;
  const MortarCorrectionsWork w(gh, plan, work);
  if (gh) {
    const int rc = launch_gh_mortar_sides(plan, el, u, params, inv_jac, w.sides, w.speeds, stream);
    if (rc != SXD_OK) return rc;
  }
  for (const MortarClass& c : plan.classes[gh ? 1 : 0]) {
    const void* kernel = gh ? reinterpret_cast<const void*>(&mortar_corrections_kernel<true>)
                            : reinterpret_cast<const void*>(&mortar_corrections_kernel<false>);
    const int lds = c.lds_bytes;
    if (!allow_lds(kernel, lds)) return SXD_ERR_DEVICE;
    // threads, measured on 1000 elements of extents 4 .. 12 with 64 / 128 / 192 /
    // 256: whole GH RHS 1055 / 912 / 864 / 864 us (768 refined and rotated elements
    // 448 / 403 / 401 / 412), 12 ScalarWave RHS 2155 / 1837 / 1728 / 1673 us
    const int limit = gh ? launch_limit(10, 192) : launch_limit(1, 256);
    for (int first = 0; first < c.count; first += limit) {
      const int count = std::min(limit, c.count - first);
      const MortarJob* jobs = plan.d_jobs + c.begin + first;
      if (gh)
        hipLaunchKernelGGL(mortar_corrections_kernel<true>,
                           dim3((count + kNumXcds - 1) / kNumXcds * kNumXcds * 10), dim3(192),
                           lds, stream, count, jobs, plan.d_gather, u, params, inv_jac, w.sides,
                           w.speeds, w.corr, full, half);
      else
        hipLaunchKernelGGL(mortar_corrections_kernel<false>, dim3(count), dim3(256), lds, stream,
                           count, jobs, plan.d_gather, u, params, inv_jac, nullptr, nullptr,
                           w.corr, full, half);
      if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
    }
  }
  return SXD_OK;
}

}  // namespace sxd
