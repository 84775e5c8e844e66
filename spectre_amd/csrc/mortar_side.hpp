// One local mortar in a workgroup: LDS layout and the steps from the fields of
// its two elements to the boundary corrections of both sides with dimension a
// projected back to the faces (shared by the corrections and their adjoint).
#pragma once

#include "device_common.hpp"
#include "gh_point.hpp"
#include "kernels.hpp"
#include "sw_point.hpp"

namespace sxd {

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

// The workgroup's LDS: corrections (over the face packages), staged values,
// matrices, and |n| of the face points (ScalarWave).
struct MortarLds {
  double *face0, *face1, *bc0, *bc1, *st0, *st1, *ma0, *mb0, *ma1, *mb1, *mag0, *mag1, *end;
  // bc_doubles, st_doubles: room for the corrections and for the staged values
  // of both sides, at least corrections_doubles and the sides' own.
  __device__ __forceinline__ MortarLds(double* lds, int km, const SideLds& l0, const SideLds& l1,
                                       int bc_doubles, int st_doubles) {
    face0 = lds;
    face1 = face0 + l0.face;
    bc0 = lds;
    bc1 = bc0 + 5 * km;
    st0 = lds + bc_doubles;
    st1 = st0 + l0.staged;
    ma0 = st0 + st_doubles;
    mb0 = ma0 + l0.mat_a;
    ma1 = mb0 + l0.mat_b;
    mb1 = ma1 + l1.mat_a;
    mag0 = mb1 + l1.mat_b;
    mag1 = mag0 + l0.mag;
    end = mag1 + l1.mag;
  }
  // By value: a choice between the members themselves would keep the struct in
  // scratch memory.
  static __device__ __forceinline__ double* pick(bool second, double* b, double* a) {
    return second ? b : a;
  }
  __device__ __forceinline__ double* bc(bool second) const { return pick(second, bc1, bc0); }
  __device__ __forceinline__ double* st(bool second) const { return pick(second, st1, st0); }
  __device__ __forceinline__ double* ma(bool second) const { return pick(second, ma1, ma0); }
  __device__ __forceinline__ double* mb(bool second) const { return pick(second, mb1, mb0); }
  __device__ __forceinline__ double* mag(bool second) const { return pick(second, mag1, mag0); }
};

// Steps 1 to 4 of mortar_faces.hip for the fields comp[] of the two elements: on
// return (after a barrier) a side's corrections with dimension a projected back
// are [mortar b][face a][5], for mortar_face_value.
template <bool GH>
__device__ __forceinline__ void mortar_terms(const MortarSide& r0, const MortarSide& r1,
                                             const SideLds& l0, const SideLds& l1,
                                             const MortarLds& sh, const int comp[5],
                                             const int32_t* __restrict__ gather,
                                             const double* __restrict__ u,
                                             const double* __restrict__ params,
                                             const double* __restrict__ inv_jac,
                                             const double* __restrict__ sides,
                                             const double* __restrict__ speeds,
                                             const double* __restrict__ full,
                                             const double* __restrict__ half) {
  const int nf0 = r0.nf, nf1 = r1.nf, km = r0.ka * r0.kb;
  const int t = threadIdx.x, T = blockDim.x;
  const unsigned by_na0 = divisor(r0.na), by_na1 = divisor(r1.na);
  const unsigned by_ka0 = divisor(r0.ka), by_ka1 = divisor(r1.ka);
  {
    auto block = [&](int mat) { return mat >= 0 ? full + mat : half + (-1 - mat); };
    const double* a0 = block(r0.mat_a);
    const double* b0 = block(r0.mat_b);
    const double* a1 = block(r1.mat_a);
    const double* b1 = block(r1.mat_b);
    for (int x = t; x < l0.mat_a; x += T) sh.ma0[x] = a0[x];
    for (int x = t; x < l0.mat_b; x += T) sh.mb0[x] = b0[x];
    for (int x = t; x < l1.mat_a; x += T) sh.ma1[x] = a1[x];
    for (int x = t; x < l1.mat_b; x += T) sh.mb1[x] = b1[x];
  }
  // 1. packages
  double* to0 = MortarLds::pick(l0.face > 0, sh.face0, sh.st0);
  double* to1 = MortarLds::pick(l1.face > 0, sh.face1, sh.st1);
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
      sh.mag(second)[f] = mag;
    }
    double* out = MortarLds::pick(second, to1, to0) + kPk * f;
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
      const double* in = MortarLds::pick(s == 1, sh.face1, sh.face0);
      const double* M = sh.ma(s == 1);
      double* out = sh.st(s == 1);
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
    const double* row0 = l0.mat_b > 0 ? sh.mb0 + rb0 * r0.nb : nullptr;
    const double* row1 = l1.mat_b > 0 ? sh.mb1 + rb1 * r1.nb : nullptr;
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
      mortar_values<1, 6, 9, 9>(v, sh.st0 + g, row0, r0.nb, r0.ka, ra0, rb0);
      p0[1] = v[0], p0[6] = v[1], p0[9] = v[2];
      mortar_values<1, 6, 9, 9>(v, sh.st1 + g, row1, r1.nb, r1.ka, ra1, rb1);
      p1[1] = v[0], p1[6] = v[1], p1[9] = v[2];
      boundary_terms<GH>(bc, p0, lam0, p1, lam1);
      sh.bc0[5 * k + 2 + g] = bc[2];
      boundary_terms<GH>(bc, p1, lam1, p0, lam0);
      sh.bc1[5 * q + 2 + g] = bc[2];
    } else {
      mortar_values<0, 4, 5, 12>(v, sh.st0, row0, r0.nb, r0.ka, ra0, rb0);
      p0[0] = v[0], p0[4] = v[1], p0[5] = v[2], p0[12] = v[3];
      mortar_values<0, 4, 5, 12>(v, sh.st1, row1, r1.nb, r1.ka, ra1, rb1);
      p1[0] = v[0], p1[4] = v[1], p1[5] = v[2], p1[12] = v[3];
      boundary_terms<GH>(bc, p0, lam0, p1, lam1);
      sh.bc0[5 * k] = bc[0];
      sh.bc0[5 * k + 1] = bc[1];
      boundary_terms<GH>(bc, p1, lam1, p0, lam0);
      sh.bc1[5 * q] = bc[0];
      sh.bc1[5 * q + 1] = bc[1];
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
      const double* v = sh.bc(second) + 5 * ka * lb;
      const double* w = sh.ma(second) + na * ka + ra * ka;
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
      double* o = sh.st(second) + 5 * y;
#pragma unroll
      for (int c = 0; c < 5; ++c) o[c] = s[c];
    }
    __syncthreads();
  }
}

// Dimension b of the projection back at face point (fa, fb) of a side: back are
// the corrections with dimension a projected back (staged, or the corrections
// themselves where dimension a is the identity).
__device__ __forceinline__ void mortar_face_value(double v[5], const MortarSide& r, bool mat_a,
                                                  bool mat_b, const MortarLds& sh, bool second,
                                                  int fa, int fb) {
  const double* at = MortarLds::pick(mat_a, sh.st(second), sh.bc(second)) + 5 * fa;
  if (!mat_b) {
#pragma unroll
    for (int c = 0; c < 5; ++c) v[c] = at[5 * r.na * fb + c];
    return;
  }
  const double* w = sh.mb(second) + r.nb * r.kb + fb * r.kb;
#pragma unroll
  for (int c = 0; c < 5; ++c) v[c] = w[0] * at[c];
#pragma unroll 2
  for (int l2 = 1; l2 < r.kb; ++l2) {
    at += 5 * r.na;
    const double a = w[l2];
#pragma unroll
    for (int c = 0; c < 5; ++c) v[c] = fma(a, at[c], v[c]);
  }
}

}  // namespace sxd
