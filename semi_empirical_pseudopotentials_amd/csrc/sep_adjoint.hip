// sep_adjoint.hip -- Hellmann-Feynman adjoint of V(r): contractions of state
// densities rho_p(g) = psi_i(g) psi_j(g) against the derivatives of the local
// potential V(g) = sum_a s_a interp_{t(a)}(|r_g - R_a|) (filter/init.c:161-182,
// filter/interpolate.c:11-23, strain scale of filterStrainCube/interpolate.c:20-21)
// with respect to the atom positions R_a, the per-atom scales s_a and the
// tabulated values pot_t[k]:
//
//   dR[p][a]    = dv sum_g rho_p(g) dV(g)/dR_a
//               = dv sum_g rho_p(g) (-aa_a(g)) (r_g - R_a) / |r_g - R_a|
//   dscale[p][a]= dv sum_g rho_p(g) interp_{t(a)}(|r_g - R_a|)
//   dtab[p][t][k] = dv sum_g rho_p(g) dV(g)/dpot_t[k]
//
// With rho_n = psi_n^2 these are dE_n/d(.) for a converged eigenpair
// (Hellmann-Feynman); with i != j the couplings <psi_i|dV/dR_a|psi_j> of
// nonAdiabaticCoupling/nonadiabatic.c:143-301.  The derivative is that of the
// forward model: segment k = (long)(del / dr_t), zero beyond row npot_t - 2,
// linear interp = (1 - w) pot[k] + w pot[k+1] with w = (del - vr[k]) /
// (vr[k+1] - vr[k]), or (SEP_INTERP_CUBIC) the cubic Hermite interpolant of
// cubic_weights()/cubic_rows() on rows k-1 .. k+2, whose derivative in del
// is continuous.
//
// Work split: an item is a slice of one atom's bounding box of grid points
// within the table range (as many slices as make the runs of items even, a few
// long ones for few atoms: hf_slices); a persistent grid of two workgroups per CU takes
// contiguous runs of items, atoms sorted by type.  An item's partial sums go
// to a work array, summed in slice order by a second kernel.  The table
// histogram accumulates in LDS over all of a workgroup's items of one type and
// is flushed with global atomic adds (so dtab is reproducible to rounding
// only).  Bound by the FP64 divisions and square root of a point, its LDS
// atomics and the few waves that the histogram's LDS leaves on a CU (77 KB
// for 8 pairs of 1201 rows).  693 atoms on 96^3, linear tables: one density
// 178 us (539 with a workgroup per slice), 3 pairs 232 (730), 8 pairs 381
// (1179; 748 before the row weights were specialised by interpolation and the
// densities loaded ahead of the geometry), 8 pairs of cubic tables 693.
#include <hip/hip_runtime.h>

#include <cmath>

#include "sep_internal.h"

namespace sep {

constexpr int HF_THREADS = 512;
constexpr int HF_BLOCKS = 512;  // persistent workgroups: two per CU

// order: atom of each item group (atoms sorted by type), items it =
// group * nsplit + slice
template <int PB, bool CUBIC>
__global__ void __launch_bounds__(HF_THREADS, 4) k_hf_atom(
    int nx, int ny, int nz, double xmin, double ymin, double zmin, double dx, double dy,
    double dz, const double *__restrict__ xyz, const int *__restrict__ type,
    const int *__restrict__ order, const double *__restrict__ scale,
    const long *__restrict__ npot, const double *__restrict__ vr, const double *__restrict__ pot,
    long stride, const double *__restrict__ dr, const double *__restrict__ rho, long N, int np,
    int p0, int ntype, int nitems, int nsplit, double *__restrict__ work,
    double *__restrict__ htab) {
  extern __shared__ double hist[];  // [PB][npot_t] of the current type
  __shared__ double red[HF_THREADS / 64][PB * 4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int it0 = (int)((long)nitems * blockIdx.x / gridDim.x);
  const int it1 = (int)((long)nitems * (blockIdx.x + 1) / gridDim.x);
  int cur = -1;  // type whose histogram is in LDS
  long nt = 0;
  // table histogram -> global (only rows the items touched are non-zero)
  auto flush = [&]() {
    for (int k = threadIdx.x; k < PB * (int)nt; k += HF_THREADS) {
      const int q = k / (int)nt;
      const double v = hist[k];
      if (v != 0.0 && p0 + q < np)
        atomicAdd(&htab[((long)(p0 + q) * ntype + cur) * stride + (k - q * (int)nt)], v);
    }
  };
  for (int it = it0; it < it1; it++) {
    const int a = order[it / nsplit], split = it % nsplit;
    const int t = type[a];
    if (t != cur) {
      if (cur >= 0) {
        __syncthreads();
        flush();
        __syncthreads();
      }
      cur = t;
      nt = npot[t];
      for (int k = threadIdx.x; k < PB * (int)nt; k += HF_THREADS) hist[k] = 0.0;
      __syncthreads();
    }
    const double drt = dr[t];
    const double rmax = (double)(nt - 1) * drt;
    const double Rx = xyz[3 * a], Ry = xyz[3 * a + 1], Rz = xyz[3 * a + 2];
    const double sa = scale ? scale[a] : 1.0;
    const double *vt = vr + t * stride, *pt = pot + t * stride;
    // bounding box of grid points within rmax of the atom
    auto lo = [](double c, double r, double o, double d) { return (int)ceil((c - r - o) / d); };
    auto hi = [](double c, double r, double o, double d) { return (int)floor((c + r - o) / d); };
    const int x0 = max(0, lo(Rx, rmax, xmin, dx)), x1 = min(nx - 1, hi(Rx, rmax, xmin, dx));
    const int y0 = max(0, lo(Ry, rmax, ymin, dy)), y1 = min(ny - 1, hi(Ry, rmax, ymin, dy));
    const int z0 = max(0, lo(Rz, rmax, zmin, dz)), z1 = min(nz - 1, hi(Rz, rmax, zmin, dz));
    const int Lx = x1 >= x0 ? x1 - x0 + 1 : 0, Ly = y1 >= y0 ? y1 - y0 + 1 : 0,
              Lz = z1 >= z0 ? z1 - z0 + 1 : 0;
    const int tot = Lx * Ly * Lz;
    const int chunk = (tot + nsplit - 1) / nsplit;
    const int b0 = min(tot, split * chunk), b1 = min(tot, b0 + chunk);
    double acc[PB][4];
#pragma unroll
    for (int q = 0; q < PB; q++) acc[q][0] = acc[q][1] = acc[q][2] = acc[q][3] = 0.0;
    int b = b0 + threadIdx.x;
    if (b < b1) {
      // position in the box, advanced by the workgroup's size with carries
      // (a division per point otherwise)
      int ix = b % Lx, iy = b / Lx % Ly, iz = b / (Lx * Ly);
      const int sx = HF_THREADS % Lx, sy = HF_THREADS / Lx % Ly, sz = HF_THREADS / (Lx * Ly);
      for (; b < b1; b += HF_THREADS) {
        const int gx = x0 + ix, gy = y0 + iy, gz = z0 + iz;
        ix += sx;
        iy += sy;
        iz += sz;
        if (ix >= Lx) {
          ix -= Lx;
          iy++;
        }
        if (iy >= Ly) {
          iy -= Ly;
          iz++;
        }
        const double ddx = (xmin + gx * dx) - Rx, ddy = (ymin + gy * dy) - Ry,
                     ddz = (zmin + gz * dz) - Rz;
        const double del = sqrt(ddx * ddx + ddy * ddy + ddz * ddz);
        const long kl = (long)(del / drt);
        if (kl > nt - 2) continue;
        const int k = (int)kl;
        // the pairs' densities first, in flight under the geometry (loads
        // between the LDS atomics would each wait for the one before)
        const unsigned go = (unsigned)((gz * ny + gy) * nx + gx) * (unsigned)sizeof(double);
        double rq[PB];
#pragma unroll
        for (int q = 0; q < PB; q++)
          rq[q] = p0 + q < np ? *reinterpret_cast<const double *>(
                                    reinterpret_cast<const char *>(rho + (long)(p0 + q) * N) + go)
                              : 0.0;
        const double v0 = vt[k];
        const double span = vt[k + 1] - v0;
        const double w = (del - v0) / span;
        // value, d(value)/d(del) without the scale, and the table-row weights:
        // rows k, k + 1 (linear), or four rows (cubic)
        constexpr int NR = CUBIC ? 4 : 2;
        int rows[NR];
        double wr[NR];
        double val, dval;
        if constexpr (CUBIC) {
          double cw[4], cd[4], dr4[4];
          long r4[4];
          cubic_weights(w, cw, cd);
          cubic_rows(k, nt, cw, r4, wr);
          cubic_rows(k, nt, cd, r4, dr4);
          val = dval = 0.0;
#pragma unroll
          for (int c = 0; c < 4; c++) {
            rows[c] = (int)r4[c];
            val += wr[c] * pt[rows[c]];
            dval += dr4[c] * pt[rows[c]];
          }
          dval /= span;
        } else {
          rows[0] = k;
          rows[1] = k + 1;
          wr[0] = 1.0 - w;
          wr[1] = w;
          const double pa = pt[k], pb = pt[k + 1];
          val = wr[0] * pa + w * pb;
          dval = (pb - pa) / span;
        }
        const double g = del > 0.0 ? -sa * dval / del : 0.0;
        const double fx = g * ddx, fy = g * ddy, fz = g * ddz;
#pragma unroll
        for (int c = 0; c < NR; c++) wr[c] *= sa;
#pragma unroll
        for (int q = 0; q < PB; q++) {
          if (p0 + q >= np) break;
          const double r = rq[q];
          acc[q][0] += r * fx;
          acc[q][1] += r * fy;
          acc[q][2] += r * fz;
          acc[q][3] += r * val;
          double *h = hist + q * (int)nt;
#pragma unroll
          for (int c = 0; c < NR; c++)
            if (wr[c] != 0.0) atomicAdd(&h[rows[c]], r * wr[c]);
        }
      }
    }
    // partial sums of the item (wave shuffles, then LDS across waves)
#pragma unroll
    for (int q = 0; q < PB; q++)
#pragma unroll
      for (int c = 0; c < 4; c++) {
        double v = acc[q][c];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (lane == 0) red[wv][q * 4 + c] = v;
      }
    __syncthreads();
    if (threadIdx.x < PB * 4) {
      double v = 0.0;
      for (int w2 = 0; w2 < HF_THREADS / 64; w2++) v += red[w2][threadIdx.x];
      work[((long)a * nsplit + split) * PB * 4 + threadIdx.x] = v;
    }
    __syncthreads();  // red is free for the next item
  }
  if (cur >= 0) flush();
}

// Sum the per-split partials in split order and scale by dv.
template <int PB>
__global__ void k_hf_reduce(const double *__restrict__ work, int natom, int nsplit, int np, int p0,
                            double dv, double *__restrict__ dR, double *__restrict__ dscale) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;  // (atom, q)
  if (i >= (long)natom * PB) return;
  const int a = (int)(i / PB), q = (int)(i % PB);
  if (p0 + q >= np) return;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  for (int sp = 0; sp < nsplit; sp++)
    for (int c = 0; c < 4; c++) s[c] += work[((long)a * nsplit + sp) * PB * 4 + q * 4 + c];
  const long o = (long)(p0 + q) * natom + a;
  if (dR)
    for (int c = 0; c < 3; c++) dR[o * 3 + c] = s[c] * dv;
  if (dscale) dscale[o] = s[3] * dv;
}

// rho_p(g) = psi_i(g) psi_j(g) for np pairs, or, with weights, the single
// density rho(g) = sum_p w_p psi_i(g) psi_j(g) (summed in pair order).
__global__ void k_pair_density(const double *__restrict__ states, long N,
                               const long *__restrict__ pairs, const double *__restrict__ wts,
                               int np, double *__restrict__ rho) {
  for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < N;
       g += (long)gridDim.x * blockDim.x) {
    if (wts) {
      double s = 0.0;
      for (int p = 0; p < np; p++)
        s += wts[p] * states[pairs[2 * p] * N + g] * states[pairs[2 * p + 1] * N + g];
      rho[g] = s;
    } else {
      for (int p = 0; p < np; p++)
        rho[(long)p * N + g] = states[pairs[2 * p] * N + g] * states[pairs[2 * p + 1] * N + g];
    }
  }
}

int pair_density_dev(const double *states, long N, const long *pairs_d, const double *w_d, int np,
                     double *rho, hipStream_t st) {
  hipLaunchKernelGGL(k_pair_density, dim3(2048), dim3(256), 0, st, states, N, pairs_d, w_d, np, rho);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

template <int PB>
static int hf_pass(const GridDev &gd, double xmin, double ymin, double zmin, double dx, double dy,
                   double dz, double dv, int natom, const double *xyz, const int *type,
                   const int *order, const double *scale, const long *npot, long maxnpot, const double *vr,
                   const double *pot, long stride, const double *dr, int ntype, const double *rho,
                   int np, int p0, int nsplit, int interp, double *work, double *htab, double *dR,
                   double *dscale, hipStream_t st) {
  const size_t lds = sizeof(double) * PB * (size_t)maxnpot;
  const int nitems = natom * nsplit;
  auto launch = [&](auto *kernel, bool *attr) {
    if (!*attr) {
      hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                          160 * 1024 - 4096);
      *attr = true;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)(nitems < HF_BLOCKS ? nitems : HF_BLOCKS)),
                       dim3(HF_THREADS), lds, st, gd.nx, gd.ny, gd.nz, xmin, ymin, zmin, dx, dy, dz,
                       xyz, type, order, scale, npot, vr, pot, stride, dr, rho, gd.N, np, p0, ntype,
                       nitems, nsplit, work, htab);
  };
  static bool attr[2] = {false, false};
  if (interp == SEP_INTERP_CUBIC)
    launch(k_hf_atom<PB, true>, &attr[1]);
  else
    launch(k_hf_atom<PB, false>, &attr[0]);
  const long nthr = (long)natom * PB;
  hipLaunchKernelGGL(k_hf_reduce<PB>, dim3((unsigned)((nthr + 255) / 256)), dim3(256), 0, st, work,
                     natom, nsplit, np, p0, dv, dR, dscale);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// Slices per atom of about `box` points, for passes of pb pairs: the least of
// the persistent grid's work, halfway between its longest workgroup's share (x
// rounded up) and the average (x).  A slice's reduction costs as much as some
// 512 (pb + 1) points (3.5 us at one pair, 19 at eight), so that many slices
// help a few atoms only: 100 atoms on 64^3 with 1 / 5 / 20 / 64 slices, whole
// call: 8 pairs 334 / 306 / 361 / 543 us, one 253 / 228 / 233 / 272; 693 atoms
// and 8 pairs with 1 / 2 / 4 / 64 448 / 471 / 521 / 2083; 10 atoms and 8 pairs
// with 1 / 5 / 20 / 64 315 / 260 / 252 / 287.
int hf_slices(long natom, double box, int pb) {
  int best = 1;
  double least = 0.0;
  for (int n = 1; n <= 64; n++) {
    const double x = (double)natom * n / HF_BLOCKS;
    const double cost = (x + std::ceil(x)) * (box / n + 512.0 * (pb + 1));
    if (n == 1 || cost < least) {
      best = n;
      least = cost;
    }
  }
  return best;
}

// Pairs of one pass: the largest batch whose LDS histogram (pairs x maxnpot
// doubles) fits 152 KB, no larger than np needs (a single density would pay
// the registers and LDS of eight); 0 if one does not fit.
int hf_pairs_per_pass(long maxnpot, long np) {
  const long cap = (160 * 1024 - 8192) / 8;
  int pb = 8;
  while (pb > 1 && ((long)pb * maxnpot > cap || pb / 2 >= np)) pb /= 2;
  return (long)pb * maxnpot <= cap ? pb : 0;
}

int hf_adjoint_dev(const GridDev &gd, double xmin, double ymin, double zmin, double dx, double dy,
                   double dz, double dv, int natom, const double *xyz, const int *type,
                   const int *order, const double *scale, const long *npot, long maxnpot, const double *vr,
                   const double *pot, long stride, const double *dr, int ntype, const double *rho,
                   int np, int nsplit, int interp, double *work, double *htab, double *dR,
                   double *dscale, hipStream_t st) {
  if (hf_pairs_per_pass(maxnpot, np) == 0) return SEP_ERR_ARG;
  // the last pass at the width of what is left
  for (int p0 = 0, pb = 0; p0 < np; p0 += pb) {
    pb = hf_pairs_per_pass(maxnpot, np - p0);
    int rc;
    switch (pb) {
      case 8:
        rc = hf_pass<8>(gd, xmin, ymin, zmin, dx, dy, dz, dv, natom, xyz, type, order, scale, npot,
                        maxnpot, vr, pot, stride, dr, ntype, rho, np, p0, nsplit, interp, work, htab,
                        dR, dscale, st);
        break;
      case 4:
        rc = hf_pass<4>(gd, xmin, ymin, zmin, dx, dy, dz, dv, natom, xyz, type, order, scale, npot,
                        maxnpot, vr, pot, stride, dr, ntype, rho, np, p0, nsplit, interp, work, htab,
                        dR, dscale, st);
        break;
      case 2:
        rc = hf_pass<2>(gd, xmin, ymin, zmin, dx, dy, dz, dv, natom, xyz, type, order, scale, npot,
                        maxnpot, vr, pot, stride, dr, ntype, rho, np, p0, nsplit, interp, work, htab,
                        dR, dscale, st);
        break;
      default:
        rc = hf_pass<1>(gd, xmin, ymin, zmin, dx, dy, dz, dv, natom, xyz, type, order, scale, npot,
                        maxnpot, vr, pot, stride, dr, ntype, rho, np, p0, nsplit, interp, work, htab,
                        dR, dscale, st);
    }
    if (rc != SEP_OK) return rc;
  }
  return SEP_OK;
}

}  // namespace sep
