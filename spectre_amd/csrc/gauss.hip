// ScalarWave DG right-hand side on Legendre-Gauss points (CDNA4, FP64).
//
// On Gauss points no grid point lies on a face
// (NumericalAlgorithms/DiscontinuousGalerkin/ProjectToBoundary.hpp:54-147,
// Evolution/DiscontinuousGalerkin/Actions/ApplyBoundaryCorrections.hpp:
// 939-986, NumericalAlgorithms/DiscontinuousGalerkin/LiftFromBoundary.cpp:
// 140-180):
//   * u and gamma2 on a face are interpolated along the normal pencil with
//     the boundary interpolation row l_j(+-1) (first term a product, then
//     fused multiply-adds);
//   * the face normal is the face's inverse-Jacobian row d (the map
//     evaluated on the face), negated on the lower face, normalised flat;
//   * the face det J is the boundary interpolation of the volume det J =
//     1 / det(inverse Jacobian);
//   * the UpwindPenalty correction bc of a face point is lifted onto every
//     point l of its pencil: dt_c(l) += -(((detinvJ(l) lift_l) faceDetJ) |n|)
//     bc_c, lift_l = l_l(+-1) / w_l, one face after another in direction
//     order.
// Two launches: sw_gauss_face_values_kernel interpolates every element's own
// values to its six faces, so that each pencil is summed once and a neighbour
// reads face values; sw_gauss_rhs_kernel takes an element through volume terms
// and lifts in one workgroup and writes dt once.  Both are bound by HBM
// traffic: u, gamma2 and det_inv_jac twice, the rest once, 35 doubles per point
// at 8^3.  Elements whose fields and corrections exceed the LDS take separate
// volume kernels and one sw_gauss_face_kernel launch per dimension: a thread
// per (element, face point) owns the pencil through that point, interpolates
// both sides itself and lifts its lower face, then its upper one.  512
// elements of 8^3: 184 us that way (149 us of it the face launches, which read
// each neighbour's whole pencils and update dt three times), 32 us with the
// two launches.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "kernels.hpp"
#include "sw_point.hpp"

namespace sxd {
namespace {

// Offset of face `dir` (2 d + side) in an element's block of face data with
// `per_point` doubles per face point (the six faces back to back in direction
// order), and the block size.
__host__ __device__ inline int64_t gauss_face_offset(int n0, int n1, int n2, int dir,
                                                     int per_point) {
  const int nf[3] = {n1 * n2, n0 * n2, n0 * n1};
  int64_t off = 0;
  for (int f = 0; f < dir; ++f) off += static_cast<int64_t>(per_point) * nf[f / 2];
  return off;
}

__global__ void __launch_bounds__(128)
sw_gauss_face_kernel(int d, int num_elements, int n0, int n1, int n2,
                     const int32_t* __restrict__ nbr, const double* __restrict__ u,
                     const double* __restrict__ gamma2, const double* __restrict__ det_inv_jac,
                     const double* __restrict__ face_inv_jac, double* __restrict__ dt,
                     const double* __restrict__ gtab) {
  const int ext[3] = {n0, n1, n2};
  const int nd = ext[d];
  const int na = ext[d == 0 ? 1 : 0], nb = ext[d == 2 ? 1 : 2];
  const int nf = na * nb;
  const int64_t x = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (x >= static_cast<int64_t>(num_elements) * nf) return;
  const int64_t e = x / nf;
  const int f = static_cast<int>(x % nf);
  const int a = f % na, b = f / na;
  const int np = n0 * n1 * n2;
  const int64_t fblock = gauss_face_offset(n0, n1, n2, 6, 3);
  // pencil through face point (a, b): volume index base + l * stride
  int stride, base;
  if (d == 0) {
    stride = 1;
    base = n0 * (a + n1 * b);
  } else if (d == 1) {
    stride = n0;
    base = a + n0 * n1 * b;
  } else {
    stride = n0 * n1;
    base = a + n0 * b;
  }
  const double* B = gtab + kPackedDSize + packed_gauss_boundary_offset(nd);
  auto interp = [&](const double* field, int side) {
    const double* row = B + side * nd;
    double s = row[0] * field[base];
    for (int l = 1; l < nd; ++l) s = fma(row[l], field[base + l * stride], s);
    return s;
  };
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {
    const int dir = 2 * d + side;
    const int64_t en = nbr[6 * e + dir];
    double ui[5], ue[5], n[3], nn[3], mag, magn;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      ui[c] = interp(u + (e * 5 + c) * np, side);
      ue[c] = interp(u + (en * 5 + c) * np, 1 - side);
    }
    const double g2i = interp(gamma2 + e * np, side);
    const double g2e = interp(gamma2 + en * np, 1 - side);
    const double* fij = face_inv_jac + e * fblock + gauss_face_offset(n0, n1, n2, dir, 3);
    const double* fijn = face_inv_jac + en * fblock + gauss_face_offset(n0, n1, n2, dir ^ 1, 3);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      n[i] = fij[i * nf + f];
      if (side == 0) n[i] = n[i] * -1.0;
      nn[i] = fijn[i * nf + f];
      if (side == 1) nn[i] = nn[i] * -1.0;  // the neighbour's face is its lower one
    }
    flat_normalize(n, &mag);
    flat_normalize(nn, &magn);
    double pki[13], pke[13], bc[5];
    sw_package(pki, ui, g2i, n);
    sw_package(pke, ue, g2e, nn);
    sw_boundary_terms(bc, pki, pke);
    // face det J: boundary interpolation of the volume det J
    const double* dij = det_inv_jac + e * np;
    const double* row = B + side * nd;
    double fdj = row[0] * (1.0 / dij[base]);
    for (int l = 1; l < nd; ++l) fdj = fma(row[l], 1.0 / dij[base + l * stride], fdj);
    const double* lift = B + (2 + side) * nd;
    for (int l = 0; l < nd; ++l) {
      const int p = base + l * stride;
      const double scale = ((dij[p] * lift[l]) * fdj) * mag;
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        double& target = dt[(e * 5 + c) * np + p];
        target = target + fma(-scale, bc[c], 0.0);
      }
    }
  }
}

// Own face values of every element: u (5), gamma2 and the face det J
// interpolated along the normal pencils, face_values [E][7][face points in
// direction order].  Grid (E, 7): a workgroup per field, a thread per pencil
// for both of its ends.
constexpr int kGaussFaceFields = 7;

__global__ void __launch_bounds__(256)
sw_gauss_face_values_kernel(int n0, int n1, int n2, const double* __restrict__ u,
                            const double* __restrict__ gamma2,
                            const double* __restrict__ det_inv_jac,
                            double* __restrict__ face_values, const double* __restrict__ gtab) {
  const int64_t e = blockIdx.x;
  const int c = blockIdx.y;
  const int np = n0 * n1 * n2;
  const int nf0 = n1 * n2, nf1 = n0 * n2, nf2 = n0 * n1;
  const int pencils = nf0 + nf1 + nf2;
  const double* field = c < 5 ? u + (e * 5 + c) * np
                              : c == 5 ? gamma2 + e * np : det_inv_jac + e * np;
  double* out = face_values + (e * kGaussFaceFields + c) * 2 * pencils;
  for (int x = threadIdx.x; x < pencils; x += blockDim.x) {
    int d, f, base, stride, nd;
    if (x < nf0) {
      d = 0, f = x, nd = n0, stride = 1, base = n0 * f;
    } else if (x < nf0 + nf1) {
      d = 1, f = x - nf0, nd = n1, stride = n0, base = f % n0 + n0 * n1 * (f / n0);
    } else {
      d = 2, f = x - nf0 - nf1, nd = n2, stride = n0 * n1, base = f;
    }
    const double* row = gtab + kPackedDSize + packed_gauss_boundary_offset(nd);
    double v = field[base];
    if (c == 6) v = 1.0 / v;
    double lower = row[0] * v, upper = row[nd] * v;
    for (int l = 1; l < nd; ++l) {
      v = field[base + l * stride];
      if (c == 6) v = 1.0 / v;
      lower = fma(row[l], v, lower);
      upper = fma(row[nd + l], v, upper);
    }
    out[face_begin(n0, n1, n2, 2 * d) + f] = lower;
    out[face_begin(n0, n1, n2, 2 * d + 1) + f] = upper;
  }
}

// Corrections kept per face point: bc (5), the face det J and |n|.
constexpr int kGaussLiftFields = 7;

__host__ __device__ inline int gauss_rhs_lds_doubles(int n0, int n1, int n2) {
  return n0 * n0 + n1 * n1 + n2 * n2 + 5 * n0 * n1 * n2 +
         kGaussLiftFields * 2 * (n1 * n2 + n0 * n2 + n0 * n1);
}

// One workgroup per element.  Dynamic LDS (gauss_rhs_lds_doubles): the D
// matrices, the element's fields, and the corrections of its face points.
__global__ void __launch_bounds__(512)
sw_gauss_rhs_kernel(int n0, int n1, int n2, const int32_t* __restrict__ nbr,
                    const double* __restrict__ u, const double* __restrict__ gamma2,
                    const double* __restrict__ inv_jac, const double* __restrict__ det_inv_jac,
                    const double* __restrict__ face_inv_jac,
                    const double* __restrict__ face_values, double* __restrict__ dt,
                    const double* __restrict__ gtab) {
  extern __shared__ double s_lds[];
  const int64_t e = xcd_local_element(blockIdx.x, gridDim.x);
  const int n[3] = {n0, n1, n2};
  const int np = n0 * n1 * n2;
  const int nf0 = n1 * n2, nf1 = n0 * n2, nf2 = n0 * n1;
  const int points = 2 * (nf0 + nf1 + nf2);
  const double* D[3];
  stage_diff_matrices(gtab, n, s_lds, D);
  double* s_u = s_lds + n0 * n0 + n1 * n1 + n2 * n2;
  double* s_bc = s_u + 5 * np;
  const double* ue = u + e * 5 * np;
  for (int x = threadIdx.x; x < 5 * np; x += blockDim.x) s_u[x] = ue[x];
  for (int x = threadIdx.x; x < points; x += blockDim.x) {
    const int d = x < 2 * nf0 ? 0 : x < 2 * (nf0 + nf1) ? 1 : 2;
    const int nf = d == 0 ? nf0 : d == 1 ? nf1 : nf2;
    const int first = face_begin(n0, n1, n2, 2 * d);
    const int side = x - first >= nf ? 1 : 0;
    const int f = x - first - side * nf;
    const int64_t en = nbr[6 * e + 2 * d + side];
    const int xn = first + (1 - side) * nf + f;
    const double* own = face_values + e * kGaussFaceFields * points;
    const double* other = face_values + en * kGaussFaceFields * points;
    double ui[5], uo[5], ni[3], no[3], mag, magn, pki[13], pke[13], bc[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      ui[c] = own[c * points + x];
      uo[c] = other[c * points + xn];
    }
    const double* fij = face_inv_jac + 3 * (e * points + first + side * nf);
    const double* fijn = face_inv_jac + 3 * (en * points + first + (1 - side) * nf);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      ni[i] = fij[i * nf + f];
      if (side == 0) ni[i] = ni[i] * -1.0;
      no[i] = fijn[i * nf + f];
      if (side == 1) no[i] = no[i] * -1.0;  // the neighbour's face is its lower one
    }
    flat_normalize(ni, &mag);
    flat_normalize(no, &magn);
    sw_package(pki, ui, own[5 * points + x], ni);
    sw_package(pke, uo, other[5 * points + xn], no);
    sw_boundary_terms(bc, pki, pke);
#pragma unroll
    for (int c = 0; c < 5; ++c) s_bc[c * points + x] = bc[c];
    s_bc[5 * points + x] = own[6 * points + x];
    s_bc[6 * points + x] = mag;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < np; p += blockDim.x) {
    const int i = p % n0, j = (p / n0) % n1, k = p / (n0 * n1);
    double ij[9], up[5], dup[15], dtp[5];
#pragma unroll
    for (int c = 0; c < 9; ++c) ij[c] = inv_jac[(e * 9 + c) * np + p];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const double* sc = s_u + c * np;
      up[c] = sc[p];
      const double* x0 = sc + n0 * (j + n1 * k);
      const double* x1 = sc + i + n0 * n1 * k;
      const double* x2 = sc + i + n0 * j;
      double d0 = D[0][i * n0] * x0[0];
      for (int l = 1; l < n0; ++l) d0 = fma(D[0][i * n0 + l], x0[l], d0);
      double d1 = D[1][j * n1] * x1[0];
      for (int l = 1; l < n1; ++l) d1 = fma(D[1][j * n1 + l], x1[n0 * l], d1);
      double d2 = D[2][k * n2] * x2[0];
      for (int l = 1; l < n2; ++l) d2 = fma(D[2][k * n2 + l], x2[n0 * n1 * l], d2);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        double s = ij[ij3(0, a)] * d0;
        s = fma(ij[ij3(1, a)], d1, s);
        s = fma(ij[ij3(2, a)], d2, s);
        dup[3 * c + a] = s;
      }
    }
    sw_time_derivative(dtp, up, dup, gamma2[e * np + p]);
    const double dij = det_inv_jac[e * np + p];
#pragma unroll
    for (int dir = 0; dir < 6; ++dir) {
      const int d = dir / 2, side = dir % 2;
      const int nd = d == 0 ? n0 : d == 1 ? n1 : n2;
      const int f = d == 0 ? j + n1 * k : d == 1 ? i + n0 * k : i + n0 * j;
      const int l = d == 0 ? i : d == 1 ? j : k;
      const int x = face_begin(n0, n1, n2, dir) + f;
      const double lift =
          gtab[kPackedDSize + packed_gauss_boundary_offset(nd) + (2 + side) * nd + l];
      const double scale = ((dij * lift) * s_bc[5 * points + x]) * s_bc[6 * points + x];
#pragma unroll
      for (int c = 0; c < 5; ++c) dtp[c] = dtp[c] + fma(-scale, s_bc[c * points + x], 0.0);
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) dt[(e * 5 + c) * np + p] = dtp[c];
  }
}

}  // namespace

int launch_sw_rhs_gauss(int num_elements, const int32_t ext[3], const int32_t* nbr,
                        const double* u, const double* gamma2, const double* inv_jac,
                        const double* det_inv_jac, const double* face_inv_jac, double* dt,
                        double* scratch_du, hipStream_t stream) {
  const double* gtab = device_gauss_tables();
  if (gtab == nullptr) return SXD_ERR_DEVICE;
  if (scratch_du == nullptr) return SXD_ERR_INVALID_ARGUMENT;
  const int64_t np = static_cast<int64_t>(ext[0]) * ext[1] * ext[2];
  // Two launches where the element's fields and corrections fit the LDS (up
  // to 13^3) and its face values the work array (from 3^3 on).
  const int lds = gauss_rhs_lds_doubles(ext[0], ext[1], ext[2]) * 8;
  const int64_t pencils = np / ext[0] + np / ext[1] + np / ext[2];
  if (lds <= 160 * 1024 && 2 * kGaussFaceFields * pencils <= 15 * np) {
    if (!allow_lds(reinterpret_cast<const void*>(&sw_gauss_rhs_kernel), lds))
      return SXD_ERR_DEVICE;
    hipLaunchKernelGGL(sw_gauss_face_values_kernel, dim3(num_elements, kGaussFaceFields),
                       dim3(pencils > 128 ? 256 : 128), 0, stream, ext[0], ext[1], ext[2], u,
                       gamma2, det_inv_jac, scratch_du, gtab);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
    const int threads = np > 256 ? 512 : np > 128 ? 256 : 128;
    hipLaunchKernelGGL(sw_gauss_rhs_kernel, dim3(num_elements), dim3(threads), lds, stream,
                       ext[0], ext[1], ext[2], nbr, u, gamma2, inv_jac, det_inv_jac, face_inv_jac,
                       scratch_du, dt, gtab);
    return hipGetLastError() == hipSuccess ? SXD_OK : SXD_ERR_DEVICE;
  }
  int rc = launch_partial_derivatives(num_elements, ext, 5, u, inv_jac, scratch_du, nullptr,
                                      stream, gtab);
  if (rc != SXD_OK) return rc;
  rc = launch_sw_volume_batched(np, static_cast<int64_t>(num_elements) * np, u, scratch_du,
                                gamma2, dt, stream);
  if (rc != SXD_OK) return rc;
  for (int d = 0; d < 3; ++d) {
    const int64_t threads = static_cast<int64_t>(num_elements) * (np / ext[d]);
    hipLaunchKernelGGL(sw_gauss_face_kernel, dim3(static_cast<unsigned>((threads + 127) / 128)),
                       dim3(128), 0, stream, d, num_elements, ext[0], ext[1], ext[2], nbr, u,
                       gamma2, det_inv_jac, face_inv_jac, dt, gtab);
    if (hipGetLastError() != hipSuccess) return SXD_ERR_DEVICE;
  }
  return SXD_OK;
}

}  // namespace sxd
