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
#include "sw_point.hpp"

namespace sxd {
namespace {

constexpr int kPk = 13;  // packaged values of a point and pair

// A dimension is the identity where the mortar covers all of it (matrix in the
// Full table) with the face's extent.
__host__ __device__ inline bool projects_a(const MortarSide& r) {
  return r.mat_a < 0 || r.na != r.ka;
}
__host__ __device__ inline bool projects_b(const MortarSide& r) {
  return r.mat_b < 0 || r.nb != r.kb;
}

// LDS of one side (doubles): the face package where dimension a is projected,
// the staged values (dimension a done; later the corrections with dimension a
// projected back), and the side's matrices (face to mortar, then mortar to
// face, per projected dimension).
struct SideLds {
  int face, staged, mat_a, mat_b, mag;
  __host__ __device__ SideLds(bool proj_a, bool proj_b, int na, int nb, int ka, int kb, bool gh) {
    const int fwd = kPk * ka * nb, back = 5 * na * kb;
    face = proj_a ? kPk * na * nb : 0;
    staged = fwd > back ? fwd : back;
    mat_a = proj_a ? 2 * na * ka : 0;
    mat_b = proj_b ? 2 * nb * kb : 0;
    mag = gh ? 0 : na * nb;
  }
  __host__ __device__ SideLds(const MortarSide& r, bool gh)
      : SideLds(projects_a(r), projects_b(r), r.na, r.nb, r.ka, r.kb, gh) {}
};

// The corrections of both sides lie over the face packages.
__host__ __device__ inline int corrections_doubles(int km, const SideLds& a, const SideLds& b) {
  const int faces = a.face + b.face, bc = 10 * km;
  return faces > bc ? faces : bc;
}

// x / n for x < 8000 and n <= 20 with one multiplication.
__device__ __forceinline__ unsigned divisor(int n) {
  return ((1u << 20) + static_cast<unsigned>(n) - 1) / static_cast<unsigned>(n);
}
__device__ __forceinline__ int divide(int x, unsigned m) {
  return static_cast<int>((static_cast<unsigned>(x) * m) >> 20);
}

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

// v[j] of the packaged values OFF[j] at mortar point (ra, rb) of a side:
// dimension b of the interpolation (row: the matrix row of rb, null for the
// identity) from the staged values.
template <int O0, int O1, int O2, int O3>
__device__ __forceinline__ void mortar_values(double v[4], const double* staged, const double* row,
                                              int nb, int ka, int ra, int rb) {
  const double* at = staged + kPk * ra;
  if (row == nullptr) {
    at += kPk * ka * rb;
    v[0] = at[O0], v[1] = at[O1], v[2] = at[O2], v[3] = at[O3];
    return;
  }
  double w = row[0];
  v[0] = w * at[O0], v[1] = w * at[O1], v[2] = w * at[O2], v[3] = w * at[O3];
#pragma unroll 2
  for (int l = 1; l < nb; ++l) {
    at += kPk * ka;
    w = row[l];
    v[0] = fma(w, at[O0], v[0]);
    v[1] = fma(w, at[O1], v[1]);
    v[2] = fma(w, at[O2], v[2]);
    v[3] = fma(w, at[O3], v[3]);
  }
}

template <bool GH>
__device__ __forceinline__ void boundary_terms(double bc[5], const double in[13],
                                               const double lam_in[4], const double ex[13],
                                               const double lam_ex[4]) {
  if constexpr (GH)
    gh_boundary_terms_pair(bc, in, lam_in, ex, lam_ex);
  else
    sw_boundary_terms(bc, in, ex);
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
  const int nf0 = r0.nf, nf1 = r1.nf, km = r0.ka * r0.kb;
  double* s_face0 = s_lds;
  double* s_face1 = s_face0 + l0.face;
  double* s_bc0 = s_lds;
  double* s_bc1 = s_bc0 + 5 * km;
  double* s_st0 = s_lds + corrections_doubles(km, l0, l1);
  double* s_st1 = s_st0 + l0.staged;
  double* s_ma0 = s_st1 + l1.staged;
  double* s_mb0 = s_ma0 + l0.mat_a;
  double* s_ma1 = s_mb0 + l0.mat_b;
  double* s_mb1 = s_ma1 + l1.mat_a;
  double* s_mag0 = s_mb1 + l1.mat_b;
  double* s_mag1 = s_mag0 + l0.mag;
  const int t = threadIdx.x, T = blockDim.x;
  const unsigned by_na0 = divisor(r0.na), by_na1 = divisor(r1.na);
  const unsigned by_ka0 = divisor(r0.ka), by_ka1 = divisor(r1.ka);
  {
    auto block = [&](int mat) { return mat >= 0 ? full + mat : half + (-1 - mat); };
    const double* a0 = block(r0.mat_a);
    const double* b0 = block(r0.mat_b);
    const double* a1 = block(r1.mat_a);
    const double* b1 = block(r1.mat_b);
    for (int x = t; x < l0.mat_a; x += T) s_ma0[x] = a0[x];
    for (int x = t; x < l0.mat_b; x += T) s_mb0[x] = b0[x];
    for (int x = t; x < l1.mat_a; x += T) s_ma1[x] = a1[x];
    for (int x = t; x < l1.mat_b; x += T) s_mb1[x] = b1[x];
  }
  const int comp[5] = {pr, GH ? 10 + pr : 1, GH ? 20 + 3 * pr : 2, GH ? 21 + 3 * pr : 3,
                       GH ? 22 + 3 * pr : 4};
  // 1. packages
  for (int x = t; x < nf0 + nf1; x += T) {
    const bool second = x >= nf0;
    const MortarSide& r = second ? r1 : r0;
    const int f = second ? x - nf0 : x;
    const int nf = second ? nf1 : nf0, np = r.np;
    const int b = divide(f, second ? by_na1 : by_na0), a = f - b * r.na;
    const int p = r.base + a * r.step_a + b * r.step_b;
    double pk[kPk];
    if constexpr (GH) {
      const double* sd = sides + 12 * r.pt_off + f;
      GhFaceSide s;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        s.n[i] = sd[i * nf];
        s.nv[i] = sd[(3 + i) * nf];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) s.lam[c] = sd[(6 + c) * nf];
      s.gamma2 = sd[10 * nf];
      const double* ue = u + 50 * r.off + p;
      double phi[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) phi[i] = ue[comp[2 + i] * np];
      gh_package_pair(pk, ue[comp[0] * np], ue[comp[1] * np], phi, s);
    } else {
      double n[3], up[5], mag;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        n[i] = inv_jac[9 * r.off + ij3(r.dim, i) * np + p];
        if (r.side == 0) n[i] = n[i] * -1.0;
      }
#pragma unroll
      for (int c = 0; c < 5; ++c) up[c] = u[5 * r.off + c * np + p];
      flat_normalize(n, &mag);
      sw_package(pk, up, params[r.off + p], n);
      (second ? s_mag1 : s_mag0)[f] = mag;
    }
    double* out = (second ? (l1.face > 0 ? s_face1 : s_st1) : (l0.face > 0 ? s_face0 : s_st0)) +
                  kPk * f;
#pragma unroll
    for (int c = 0; c < kPk; ++c) out[c] = pk[c];
  }
  __syncthreads();
  // 2. dimension a onto the mortar: a work item is two output points of one
  // line for 5 of the 13 values (groups from 0, 4 and 8)
  if (l0.face + l1.face > 0) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const MortarSide& r = s == 0 ? r0 : r1;
      if ((s == 0 ? l0.face : l1.face) == 0) continue;
      const double* in = s == 0 ? s_face0 : s_face1;
      const double* M = s == 0 ? s_ma0 : s_ma1;
      double* out = s == 0 ? s_st0 : s_st1;
      const int half_ka = (r.ka + 1) / 2, items = half_ka * r.nb;
      const unsigned by_half = divisor(half_ka);
      for (int x = t; x < 3 * items; x += T) {
        const int g = (x >= items) + (x >= 2 * items), y = x - g * items;
        const int lb = divide(y, by_half), ra = 2 * (y - lb * half_ka);
        const bool two = ra + 1 < r.ka;
        const double* v = in + kPk * r.na * lb + 4 * g;
        const double* w0 = M + ra * r.na;
        const double* w1 = two ? w0 + r.na : w0;
        double s0[5], s1[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) {
          s0[c] = w0[0] * v[c];
          s1[c] = w1[0] * v[c];
        }
  #pragma unroll 2
      for (int l = 1; l < r.na; ++l) {
          v += kPk;
          const double a = w0[l], b = w1[l];
#pragma unroll
          for (int c = 0; c < 5; ++c) {
            s0[c] = fma(a, v[c], s0[c]);
            s1[c] = fma(b, v[c], s1[c]);
          }
        }
        double* o = out + kPk * (r.ka * lb + ra) + 4 * g;
#pragma unroll
        for (int c = 0; c < 5; ++c) o[c] = s0[c];
        if (two) {
#pragma unroll
          for (int c = 0; c < 5; ++c) o[kPk + c] = s1[c];
        }
      }
    }
    __syncthreads();
  }
  // 3. boundary terms: groups 0..2 the Phi_g output (values 1 + g, 6 + g,
  // 9 + g), group 3 the g and Pi outputs (values 0, 4, 5, 12)
  for (int x = t; x < 4 * km; x += T) {
    const int g = (x >= km) + (x >= 2 * km) + (x >= 3 * km), k = x - g * km;
    const int q = gather[r0.rec_off + k];
    const int rb0 = divide(k, by_ka0), ra0 = k - rb0 * r0.ka;
    const int rb1 = divide(q, by_ka1), ra1 = q - rb1 * r1.ka;
    const double* row0 = l0.mat_b > 0 ? s_mb0 + rb0 * r0.nb : nullptr;
    const double* row1 = l1.mat_b > 0 ? s_mb1 + rb1 * r1.nb : nullptr;
    double lam0[4] = {0, 0, 0, 0}, lam1[4] = {0, 0, 0, 0};
    if constexpr (GH) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        lam0[c] = speeds[4 * r0.rec_off + c * km + k];
        lam1[c] = speeds[4 * r1.rec_off + c * km + q];
      }
    }
    double p0[13], p1[13], bc[5], v[4];
    if (g < 3) {
      mortar_values<1, 6, 9, 9>(v, s_st0 + g, row0, r0.nb, r0.ka, ra0, rb0);
      p0[1] = v[0], p0[6] = v[1], p0[9] = v[2];
      mortar_values<1, 6, 9, 9>(v, s_st1 + g, row1, r1.nb, r1.ka, ra1, rb1);
      p1[1] = v[0], p1[6] = v[1], p1[9] = v[2];
      boundary_terms<GH>(bc, p0, lam0, p1, lam1);
      s_bc0[5 * k + 2 + g] = bc[2];
      boundary_terms<GH>(bc, p1, lam1, p0, lam0);
      s_bc1[5 * q + 2 + g] = bc[2];
    } else {
      mortar_values<0, 4, 5, 12>(v, s_st0, row0, r0.nb, r0.ka, ra0, rb0);
      p0[0] = v[0], p0[4] = v[1], p0[5] = v[2], p0[12] = v[3];
      mortar_values<0, 4, 5, 12>(v, s_st1, row1, r1.nb, r1.ka, ra1, rb1);
      p1[0] = v[0], p1[4] = v[1], p1[5] = v[2], p1[12] = v[3];
      boundary_terms<GH>(bc, p0, lam0, p1, lam1);
      s_bc0[5 * k] = bc[0];
      s_bc0[5 * k + 1] = bc[1];
      boundary_terms<GH>(bc, p1, lam1, p0, lam0);
      s_bc1[5 * q] = bc[0];
      s_bc1[5 * q + 1] = bc[1];
    }
  }
  __syncthreads();
  // 4. dimension a back to the face, both sides' lines as one list
  if (l0.mat_a + l1.mat_a > 0) {
    const int items0 = l0.mat_a > 0 ? r0.na * r0.kb : 0;
    const int items1 = l1.mat_a > 0 ? r1.na * r1.kb : 0;
    for (int x = t; x < items0 + items1; x += T) {
      const bool second = x >= items0;
      const int y = second ? x - items0 : x;
      const int na = second ? r1.na : r0.na, ka = second ? r1.ka : r0.ka;
      const int lb = divide(y, second ? by_na1 : by_na0), ra = y - lb * na;
      const double* v = (second ? s_bc1 : s_bc0) + 5 * ka * lb;
      const double* w = (second ? s_ma1 : s_ma0) + na * ka + ra * ka;
      double s[5];
#pragma unroll
      for (int c = 0; c < 5; ++c) s[c] = w[0] * v[c];
#pragma unroll 2
      for (int l = 1; l < ka; ++l) {
        v += 5;
        const double a = w[l];
#pragma unroll
        for (int c = 0; c < 5; ++c) s[c] = fma(a, v[c], s[c]);
      }
      double* o = (second ? s_st1 : s_st0) + 5 * y;
#pragma unroll
      for (int c = 0; c < 5; ++c) o[c] = s[c];
    }
    __syncthreads();
  }
  // 5. dimension b back to the face, and lift
  for (int x = t; x < nf0 + nf1; x += T) {
    const bool second = x >= nf0;
    const MortarSide& r = second ? r1 : r0;
    const int f = second ? x - nf0 : x;
    const int nf = second ? nf1 : nf0, na = r.na;
    const int fb = divide(f, second ? by_na1 : by_na0), fa = f - fb * na;
    const double* v =
        (second ? (l1.mat_a > 0 ? s_st1 : s_bc1) : (l0.mat_a > 0 ? s_st0 : s_bc0)) + 5 * fa;
    double s[5];
    if ((second ? l1.mat_b : l0.mat_b) > 0) {
      const int nb = r.nb, kb = r.kb;
      const double* w = (second ? s_mb1 : s_mb0) + nb * kb + fb * kb;
#pragma unroll
      for (int c = 0; c < 5; ++c) s[c] = w[0] * v[c];
#pragma unroll 2
      for (int l = 1; l < kb; ++l) {
        v += 5 * na;
        const double a = w[l];
#pragma unroll
        for (int c = 0; c < 5; ++c) s[c] = fma(a, v[c], s[c]);
      }
    } else {
#pragma unroll
      for (int c = 0; c < 5; ++c) s[c] = v[5 * na * fb + c];
    }
    double mag;
    if constexpr (GH)
      mag = sides[12 * r.pt_off + 11 * nf + f];
    else
      mag = (second ? s_mag1 : s_mag0)[f];
    const double fac = lift_factor(r.extent, mag);
    double* out = corr + NC * r.corr_off + f;
#pragma unroll
    for (int c = 0; c < 5; ++c) out[comp[c] * nf] = s[c] * fac;
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

int launch_mortar_lifted_corrections(bool gh, const MortarPlan& plan, const MixedElement* el,
                                     const double* u, const double* params,
                                     const double* inv_jac, double* work, hipStream_t stream) {
  const double* full = device_mortar_matrices();
  const double* half = device_half_mortar_matrices();
  if (full == nullptr || half == nullptr) return SXD_ERR_DEVICE;
  if (work == nullptr || plan.num_remote > 0) return SXD_ERR_INVALID_ARGUMENT;
  const MortarCorrectionsWork w(gh, plan, work);
  if (gh) {
    const int lds = 8 * 4 * (plan.kf + plan.tmp_max);
    hipLaunchKernelGGL(gh_mortar_sides_kernel, dim3(plan.num_faces), dim3(128), lds, stream, el,
                       plan.d_faces, plan.d_records, u, params, inv_jac, w.sides, w.speeds, full,
                       half, plan.kf);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  for (const MortarClass& c : plan.classes[gh ? 1 : 0]) {
    const void* kernel = gh ? reinterpret_cast<const void*>(&mortar_corrections_kernel<true>)
                            : reinterpret_cast<const void*>(&mortar_corrections_kernel<false>);
    const int lds = c.lds_bytes;
    if (!allow_lds(kernel, lds)) return SXD_ERR_DEVICE;
    const MortarJob* jobs = plan.d_jobs + c.begin;
    // threads, measured on 1000 elements of extents 4 .. 12 with 64 / 128 / 192 /
    // 256: whole GH RHS 1055 / 912 / 864 / 864 us (768 refined and rotated elements
    // 448 / 403 / 401 / 412), 12 ScalarWave RHS 2155 / 1837 / 1728 / 1673 us
    if (gh)
      hipLaunchKernelGGL(mortar_corrections_kernel<true>,
                         dim3((c.count + kNumXcds - 1) / kNumXcds * kNumXcds * 10),
                         dim3(192), lds, stream, c.count, jobs, plan.d_gather, u, params, inv_jac,
                         w.sides, w.speeds, w.corr, full, half);
    else
      hipLaunchKernelGGL(mortar_corrections_kernel<false>, dim3(c.count), dim3(256), lds,
                         stream, c.count, jobs, plan.d_gather, u, params, inv_jac, nullptr,
                         nullptr, w.corr, full, half);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  return SXD_OK;
}

}  // namespace sxd
