// readbr's arithmetic on the GPU: the photospheric Br map interpolated onto
// the solver's theta/phi half mesh, made periodic in phi, given its m=0 pole
// ghosts, flux balanced, and (option 'open') replaced by |Br|.
//
//   intrp2d + interp   src/pot3d.F90:6830-6910, 7028-7072 (bilinear)
//   readbr             src/pot3d.F90:6751-6829 (seam, poles, flux balance)
//   set_flux           src/pot3d.F90:3806-3833 (|Br| for option 'open')
//
// The driver keeps the HDF5 read (rdhdf_2d) and hands over the map and its
// scales.  Interpolation, seam and pole values follow the reference's
// expression order with FMA contraction off, so they are bit-identical to a
// plain FP64 evaluation; the three flux sums are FP64 in a fixed parallel
// order, so br00err can differ from a sequential sum in its last bits.
//
// What bounds it: latency.  Three launches (interpolation and seam; poles and
// flux partials; balance) between two copies in, the map and one block of
// tables, and two out.  The reference's interval searches over the axes, a few
// hundred bisections, are made on the host with the range checks.  A call for
// 91x181 points of a 1-degree map 311 -> 181 us (seven launches, eight copies
// in and the pole sums one load at a time before).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "../../include/pot3d_hip.h"

namespace p3d {
int set_error(int code, const char* msg);
}

namespace {

constexpr int kFluxLanes = 1024;  // lanes that add the fluxes
constexpr int kFluxBlocks = 16;   // blocks they are spread over
constexpr int kFluxThreads = kFluxLanes / kFluxBlocks;
constexpr int kPoleChunk = 1024;   // terms of the pole sums in LDS at a time

// interp (src/pot3d.F90:7028-7072): the first interval i with
// x[i] <= v <= x[i+1], alpha = (v - x[i]) / (x[i+1] - x[i]).  With x strictly
// increasing and x[0] <= v <= x[n-1] (checked before) that interval is the
// smallest i with x[i+1] >= v, found here by bisection.
void axis_entry(int n, const double* x, double v, int* idx, double* alpha) {
  int lo = 0, hi = n - 2;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (x[mid + 1] >= v)
      hi = mid;
    else
      lo = mid + 1;
  }
  *idx = lo;
  *alpha = (v - x[lo]) / (x[lo + 1] - x[lo]);
}

// intrp2d's bilinear formula (src/pot3d.F90:6891-6892) on the interior
// (j = 2..nt-1, k = 2..np-1 in the reference's 1-based indices), and the phi
// seam of the interior rows (br0(:,1) = br0(:,np-1), br0(:,np) = br0(:,2),
// :6777-6778); br0 is (nt, np) in Fortran order, bn (ntn, npn).
__global__ void k_intrp2d(int nt, int np, int ntn, const double* __restrict__ bn,
                          const int* __restrict__ it, const double* __restrict__ at,
                          const int* __restrict__ ip, const double* __restrict__ ap,
                          double* __restrict__ br0) {
#pragma clang fp contract(off)
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = nt - 2, c = np - 2;
  if (q >= b * c) return;
  const int j = q % b, k = q / b;
  const int ii = it[j], jj = ip[k];
  const double ax = at[j], ay = ap[k];
  const double f00 = bn[ii + (size_t)ntn * jj], f01 = bn[ii + (size_t)ntn * (jj + 1)];
  const double f10 = bn[ii + 1 + (size_t)ntn * jj], f11 = bn[ii + 1 + (size_t)ntn * (jj + 1)];
  const double v =
      (1.0 - ax) * ((1.0 - ay) * f00 + ay * f01) + ax * ((1.0 - ay) * f10 + ay * f11);
  br0[(j + 1) + (size_t)nt * (k + 1)] = v;
  if (k == c - 1) br0[j + 1] = v;
  if (k == 0) br0[(j + 1) + (size_t)nt * (np - 1)] = v;
}

// Block 0: m=0 pole ghosts (src/pot3d.F90:6784-6788): sum0/sum1 = sum over
// k=2..np-1 of br0(2,k)*dph(k) (resp. row nt-1), in k order, times pl_i; then
// br0(1,:) = 2 sum0 - br0(2,:), br0(nt,:) = 2 sum1 - br0(nt-1,:).  All lanes
// form the terms, two lanes add them in order from LDS (read by the two lanes
// one after the other from memory they took 44 us of 180 terms).
// Blocks 1..16: positive flux, negative flux and area over the interior
// (src/pot3d.F90:6792-6804), da = sth(j)*dth(j)*dph(k).  1024 lanes each add a
// strided subset in order, then a tree pairs lanes 512, 256, ... 1 apart;
// block f has the lanes f, f + 16, ..., so the levels down to 16 stay inside
// it and part[f + {0, 1, 2} kFluxBlocks] enters the last four.
__global__ void __launch_bounds__(kFluxThreads)
    k_poles_flux(int nt, int np, const double* __restrict__ sth, const double* __restrict__ dth,
                 const double* __restrict__ dph, double pl_i, double* __restrict__ br0,
                 double* __restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double sh[2 * kPoleChunk];
  __shared__ double sums[2];
  const int t = threadIdx.x;
  if (blockIdx.x == 0) {
    double s = 0.0;
    for (int k0 = 1; k0 < np - 1; k0 += kPoleChunk) {
      const int n = min(kPoleChunk, np - 1 - k0);
      for (int e = t; e < 2 * n; e += kFluxThreads) {
        const int k = k0 + (e >> 1), row = e & 1 ? nt - 2 : 1;
        sh[e] = br0[row + (size_t)nt * k] * dph[k];
      }
      __syncthreads();
      if (t < 2) {
#pragma unroll 8
        for (int e = 0; e < n; e++) s = s + sh[2 * e + t];
      }
      __syncthreads();
    }
    if (t < 2) sums[t] = s * pl_i;
    __syncthreads();
    for (int k = t; k < np; k += kFluxThreads) {
      br0[(size_t)nt * k] = 2.0 * sums[0] - br0[1 + (size_t)nt * k];
      br0[nt - 1 + (size_t)nt * k] = 2.0 * sums[1] - br0[nt - 2 + (size_t)nt * k];
    }
    return;
  }
  const int b = nt - 2, c = np - 2, f = (int)blockIdx.x - 1;
  double fp = 0.0, fm = 0.0, ar = 0.0;
#pragma unroll 4
  for (int q = f + kFluxBlocks * t; q < b * c; q += kFluxLanes) {
    const int j = 1 + q % b, k = 1 + q / b;
    const double da = sth[j] * dth[j] * dph[k];
    const double v = br0[j + (size_t)nt * k];
    if (v > 0.0)
      fp = fp + v * da;
    else
      fm = fm + v * da;
    ar = ar + da;
  }
  sh[t] = fp;
  sh[kFluxThreads + t] = fm;
  sh[2 * kFluxThreads + t] = ar;
  __syncthreads();
  for (int w = kFluxThreads / 2; w > 0; w >>= 1) {
    if (t < w)
#pragma unroll
      for (int e = t; e < 3 * kFluxThreads; e += kFluxThreads) sh[e] = sh[e] + sh[e + w];
    __syncthreads();
  }
  if (t < 3) part[t * kFluxBlocks + f] = sh[t * kFluxThreads];
}

// The last levels of the three sums, then br0 -= br00err with br00err = (fluxp +
// fluxm)/area when balancing (src/pot3d.F90:6812-6823), then |br0| for option
// 'open' (set_flux, :3832).  out: fluxp, fluxm, area, br00err (0 when not
// balanced).
__global__ void __launch_bounds__(256)
    k_balance(int n, int balance, int abs_br, const double* __restrict__ part,
              double* __restrict__ out, double* __restrict__ br0) {
  __shared__ double sums[3];
  const int t = threadIdx.x, q = blockIdx.x * 256 + t;
  double v = q < n ? br0[q] : 0.0;
  if (t < 3) {
    double s[kFluxBlocks];
#pragma unroll
    for (int f = 0; f < kFluxBlocks; f++) s[f] = part[t * kFluxBlocks + f];
#pragma unroll
    for (int w = kFluxBlocks / 2; w > 0; w >>= 1)
#pragma unroll
      for (int f = 0; f < w; f++) s[f] = s[f] + s[f + w];
    sums[t] = s[0];
  }
  __syncthreads();
  const double e = balance ? (sums[0] + sums[1]) / sums[2] : 0.0;
  if (q < 3) out[q] = sums[q];
  if (q == 3) out[3] = e;
  if (q >= n) return;
  if (balance) v = v - e;
  br0[q] = abs_br ? fabs(v) : v;
}

inline int nblk(long long n, int t) { return (int)((n + t - 1) / t); }

int fail(int code, const char* msg) { return p3d::set_error(code, msg); }

}  // namespace

extern "C" int p3d_readbr(int nt, int np, const double* th, const double* ph,
                          const double* sth, const double* dth, const double* dph, double pl,
                          int ntn, int npn, const double* tn, const double* pn, const double* bn,
                          int balance_flux, int abs_br, double* br0, double* flux) {
  if (!th || !ph || !sth || !dth || !dph || !tn || !pn || !bn || !br0)
    return fail(P3D_EINVAL, "null argument");
  if (nt < 3 || np < 3 || ntn < 2 || npn < 2 || !(pl > 0.0))
    return fail(P3D_EINVAL, "bad sizes (need nt, np >= 3, map scales of >= 2 points, pl > 0)");
  if ((long long)nt * np >= (1LL << 31) || (long long)ntn * npn >= (1LL << 31))
    return fail(P3D_EINVAL, "arrays too large for 32-bit indices");
  // intrp2d's checks (src/pot3d.F90:6870-6889): increasing scales, and every
  // mesh point inside them
  for (int i = 0; i + 1 < ntn; i++)
    if (!(tn[i + 1] > tn[i]))
      return fail(P3D_EINVAL, "theta scale of the Br map is not monotonically increasing");
  for (int i = 0; i + 1 < npn; i++)
    if (!(pn[i + 1] > pn[i]))
      return fail(P3D_EINVAL, "phi scale of the Br map is not monotonically increasing");
  for (int j = 1; j < nt - 1; j++)
    if (!(th[j] >= tn[0] && th[j] <= tn[ntn - 1]))
      return fail(P3D_EINVAL, "theta mesh point outside the range of the Br map's scale");
  for (int k = 1; k < np - 1; k++)
    if (!(ph[k] >= pn[0] && ph[k] <= pn[npn - 1]))
      return fail(P3D_EINVAL, "phi mesh point outside the range of the Br map's scale");

  // one device block: bn | tables | br0 | out[4] | flux partials.  Tables, one
  // copy: alpha_t | alpha_p | sth | dth | dph | index_t, index_p (ints)
  const size_t nb = (size_t)nt * np, nm = (size_t)ntn * npn;
  const size_t b = (size_t)nt - 2, c = (size_t)np - 2;
  const size_t ntab = b + c + 2 * (size_t)nt + np + (b + c + 1) / 2;
  std::vector<double> tab(ntab);
  double* h_at = tab.data();
  double* h_ap = h_at + b;
  double* h_sth = h_ap + c;
  double* h_dth = h_sth + nt;
  double* h_dph = h_dth + nt;
  int* h_it = reinterpret_cast<int*>(h_dph + np);
  int* h_ip = h_it + b;
  // tables for the interior points th(2:nt-1), ph(2:np-1)
  for (size_t j = 0; j < b; j++) axis_entry(ntn, tn, th[j + 1], h_it + j, h_at + j);
  for (size_t k = 0; k < c; k++) axis_entry(npn, pn, ph[k + 1], h_ip + k, h_ap + k);
  std::copy(sth, sth + nt, h_sth);
  std::copy(dth, dth + nt, h_dth);
  std::copy(dph, dph + np, h_dph);
  double* d = nullptr;
  if (hipMalloc((void**)&d, (nm + ntab + nb + 4 + 3 * kFluxBlocks) * 8) != hipSuccess)
    return fail(P3D_ENOMEM, "allocation failed");
  double* d_at = d + nm;
  double* d_ap = d_at + b;
  double* d_sth = d_ap + c;
  double* d_dth = d_sth + nt;
  double* d_dph = d_dth + nt;
  const int* d_it = reinterpret_cast<const int*>(d_dph + np);
  double* d_br = d_at + ntab;
  double* d_out = d_br + nb;
  double* d_part = d_out + 4;
  hipStream_t st = nullptr;
  bool ok = hipStreamCreateWithFlags(&st, hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipMemcpyAsync(d, bn, nm * 8, hipMemcpyHostToDevice, st) == hipSuccess &&
       hipMemcpyAsync(d_at, h_at, ntab * 8, hipMemcpyHostToDevice, st) == hipSuccess;
  if (ok) {
    k_intrp2d<<<nblk((long long)(b * c), 256), 256, 0, st>>>(nt, np, ntn, d, d_it, d_at,
                                                             d_it + b, d_ap, d_br);
    k_poles_flux<<<1 + kFluxBlocks, kFluxThreads, 0, st>>>(nt, np, d_sth, d_dth, d_dph, 1.0 / pl, d_br,
                                                  d_part);
    k_balance<<<nblk((long long)nb, 256), 256, 0, st>>>((int)nb, balance_flux != 0,
                                                        abs_br != 0, d_part, d_out, d_br);
    ok = hipGetLastError() == hipSuccess;
  }
  double out[4] = {0, 0, 0, 0};
  ok = ok && hipMemcpyAsync(br0, d_br, nb * 8, hipMemcpyDeviceToHost, st) == hipSuccess;
  ok = ok && hipMemcpyAsync(out, d_out, 32, hipMemcpyDeviceToHost, st) == hipSuccess;
  ok = ok && hipStreamSynchronize(st) == hipSuccess;
  if (st) hipStreamDestroy(st);
  hipFree(d);
  if (!ok) return fail(P3D_EHIP, "readbr kernels failed");
  if (flux)
    for (int q = 0; q < 4; q++) flux[q] = out[q];
  return P3D_OK;
}
