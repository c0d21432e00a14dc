// sep_kernels.hip -- non-FFT kernels of libsep: V(r) assembly, deterministic
// per-state reductions, row scaling and precision conversion.
#include <hip/hip_runtime.h>

#include "fft_core.h"
#include "sep_internal.h"

namespace sep {

// ------------------------------------------------------------ V(r) assembly
// filter/init.c:161-182 (sum over atoms in file order, + expot), interpolate
// of filter/interpolate.c:11-23 with the per-atom scale of
// filterStrainCube/interpolate.c:20-21.  Contraction is off so each term is
// rounded exactly as the reference source writes it.  interp = SEP_INTERP_CUBIC
// replaces the linear segment by the cubic Hermite interpolant of
// cubic_weights() (same segment, same cutoff), a C^1 function of |r - R|.
//
// One workgroup per brick of 8 x 8 x 4 points, a cube of 4 per wave.  Each 256 atoms are tested
// against the brick (distance to its box against the table's range) and the
// survivors gathered in LDS in file order, so a point meets the atoms near
// its brick only; the skipped ones add nothing in the reference either, so
// the sum is the same bit for bit.  Bound by the FP64 divisions and square
// roots of the pairs in range: 1667 atoms on 128^3 (CdSe, 4 nm) 5.73 ms with
// every atom at every point, 0.31 ms in bricks of 16 x 4 x 4 with rows of 16 a
// wave, 0.28 with cubes of 4 (more of an atom's waves are skipped whole), 0.26
// in the more compact bricks (cubic tables 0.40, 0.35 and 0.34).
constexpr int VB_X = 8, VB_Y = 8, VB_Z = 4;
__global__ void __launch_bounds__(256) k_build_potential(
    int nx, int ny, int nz, double xmin, double ymin, double zmin, double dx, double dy, double dz,
    long natom, const double *__restrict__ xyz, const int *__restrict__ type,
    const double *__restrict__ scale, const long *__restrict__ npot, const double *__restrict__ vr,
    const double *__restrict__ pot, long stride, const double *__restrict__ dr, double ex_e,
    double ex_x0, double ex_t, int interp, double *__restrict__ potl) {
#pragma clang fp contract(off)
  static_assert(VB_X * VB_Y * VB_Z == 256, "one thread per point of the brick");
  __shared__ double sx[256], sy[256], sz[256], ss[256], sc[256];
  __shared__ int st[256];
  __shared__ double ax[VB_X + VB_Y + VB_Z];
  __shared__ int wcount[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int bx = blockIdx.x * VB_X, by = blockIdx.y * VB_Y, bz = blockIdx.z * VB_Z;
  // grid coordinates by repeated addition (filter/init.c:157-159), each of the
  // brick's once
  if (t < VB_X) {
    double p = xmin;
    for (int i = 0; i < bx + t; i++) p += dx;
    ax[t] = p;
  } else if (t >= 64 && t < 64 + VB_Y) {
    double p = ymin;
    for (int i = 0; i < by + t - 64; i++) p += dy;
    ax[VB_X + t - 64] = p;
  } else if (t >= 128 && t < 128 + VB_Z) {
    double p = zmin;
    for (int i = 0; i < bz + t - 128; i++) p += dz;
    ax[VB_X + VB_Y + t - 128] = p;
  }
  __syncthreads();
  const int qx = 4 * (wave % 2) + lane % 4, qy = 4 * (wave / 2) + lane / 4 % 4, qz = lane / 16;
  const double px = ax[qx], py = ax[VB_X + qy], pz = ax[VB_X + VB_Y + qz];
  const double xa = ax[0], xb = ax[VB_X - 1], ya = ax[VB_X], yb = ax[VB_X + VB_Y - 1],
               za = ax[VB_X + VB_Y], zb = ax[VB_X + VB_Y + VB_Z - 1];
  const double x0 = fmin(xa, xb), x1 = fmax(xa, xb), y0 = fmin(ya, yb), y1 = fmax(ya, yb),
               z0 = fmin(za, zb), z1 = fmax(za, zb);
  const bool act = bx + qx < nx && by + qy < ny && bz + qz < nz;
  double sum = 0.0;
  for (long a0 = 0; a0 < natom; a0 += 256) {
    const long a = a0 + t;
    double x = 0.0, y = 0.0, z = 0.0, rc2 = 0.0;
    int ty = 0;
    bool keep = false;
    if (a < natom) {
      x = xyz[3 * a];
      y = xyz[3 * a + 1];
      z = xyz[3 * a + 2];
      ty = type[a];
      // beyond the last segment a pair adds nothing; the margin covers the
      // rounding of the distance, the segment index below decides.  An atom with
      // a NaN coordinate is at no distance from any point: it is kept in every
      // brick and makes all of V NaN
      const double rc = (double)(npot[ty] - 1) * dr[ty];
      rc2 = rc * rc * (1.0 + 1.0e-9);
      const double ex = fmax(fmax(x0 - x, x - x1), 0.0), ey = fmax(fmax(y0 - y, y - y1), 0.0),
                   ez = fmax(fmax(z0 - z, z - z1), 0.0);
      keep = !(ex * ex + ey * ey + ez * ez > rc2) || x != x || y != y || z != z;
    }
    const unsigned long mask = __ballot(keep);
    __syncthreads();  // the previous atoms are consumed
    if (lane == 0) wcount[wave] = __popcll(mask);
    __syncthreads();
    int na = 0, at = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (w == wave) at = na;
      na += wcount[w];
    }
    if (keep) {
      at += __popcll(mask & ((1UL << lane) - 1));
      sx[at] = x;
      sy[at] = y;
      sz[at] = z;
      ss[at] = scale ? scale[a] : 1.0;
      sc[at] = rc2;
      st[at] = ty;
    }
    __syncthreads();
    if (act) {
      for (int k = 0; k < na; k++) {
        double ddx = px - sx[k], ddy = py - sy[k], ddz = pz - sz[k];
        const double d2 = ddx * ddx + ddy * ddy + ddz * ddz;
        if (d2 > sc[k]) continue;
        double del = sqrt(d2);
        const int tk = st[k];
        const double drt = dr[tk];
        long i = (long)(del / drt);
        if (i > npot[tk] - 2) continue;  // adds 0.0 in the reference
        const double *p = pot + tk * stride, *v = vr + tk * stride;
        if (interp == SEP_INTERP_CUBIC) {
          double w[4], dw[4];
          cubic_weights((del - v[i]) / (v[i + 1] - v[i]), w, dw);
          const long n = npot[tk];
          sum += ss[k] * (w[0] * p[i > 0 ? i - 1 : 0] + w[1] * p[i] + w[2] * p[i + 1] +
                          w[3] * p[i + 2 < n ? i + 2 : n - 1] + cubic_edge(i, n, w, p));
          continue;
        }
        double aa = ss[k] * (p[i + 1] - p[i]) / (v[i + 1] - v[i]);
        double bb = ss[k] * p[i] - v[i] * aa;
        sum += aa * del + bb;
      }
    }
  }
  if (act) {
    double rex = sqrt(px * px + py * py + pz * pz);
    double potEx = ex_e * (1.0 / (exp((rex - ex_x0) / ex_t) + 1.0) - 1.0);
    potl[((long)(bz + qz) * ny + by + qy) * nx + bx + qx] = sum + potEx;
  }
}

int build_potential_dev(const GridDev &gd, double xmin, double ymin, double zmin, double dx,
                        double dy, double dz, long natom, const double *xyz_d, const int *type_d,
                        const double *scale_d, const long *npot_d, const double *vr_d,
                        const double *pot_d, long stride, const double *dr_d, double ex_e,
                        double ex_x0, double ex_t, int interp, double *potl_d, hipStream_t st) {
  dim3 grid((unsigned)((gd.nx + VB_X - 1) / VB_X), (unsigned)((gd.ny + VB_Y - 1) / VB_Y),
            (unsigned)((gd.nz + VB_Z - 1) / VB_Z));
  hipLaunchKernelGGL(k_build_potential, grid, dim3(256), 0, st, gd.nx, gd.ny, gd.nz, xmin, ymin,
                     zmin, dx, dy, dz, natom, xyz_d, type_d, scale_d, npot_d, vr_d, pot_d, stride,
                     dr_d, ex_e, ex_x0, ex_t, interp, potl_d);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// V in FP32 beside the FP64 one, and each workgroup's extrema of V
// (part[2 b], part[2 b + 1]; filter/init.c:116-117,196-199 on its points), one
// pass over V.
__global__ void __launch_bounds__(256) k_finish_potential(const double *__restrict__ v,
                                                          float *__restrict__ f, long n,
                                                          double *__restrict__ part) {
  double lo = 1.0e10, hi = -1.0e10;
  for (long g = (long)blockIdx.x * 256 + threadIdx.x; g < n; g += (long)gridDim.x * 256) {
    const double x = v[g];
    f[g] = (float)x;
    if (hi < x) hi = x;
    if (lo > x) lo = x;
  }
  __shared__ double red[2][4];
  for (int off = 32; off > 0; off >>= 1) {
    const double a = __shfl_down(lo, off, 64), b = __shfl_down(hi, off, 64);
    if (lo > a) lo = a;
    if (hi < b) hi = b;
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = lo;
    red[1][threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; w++) {
      if (lo > red[0][w]) lo = red[0][w];
      if (hi < red[1][w]) hi = red[1][w];
    }
    part[2 * blockIdx.x] = lo;
    part[2 * blockIdx.x + 1] = hi;
  }
}
long finish_potential_blocks(long n) { return n > 512 * 1024 ? 512 : (n + 1023) / 1024; }
int finish_potential_dev(const double *v, float *f, long n, double *part, hipStream_t st) {
  hipLaunchKernelGGL(k_finish_potential, dim3((unsigned)finish_potential_blocks(n)), dim3(256), 0,
                     st, v, f, n, part);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// ------------------------------------------------ deterministic row dots
// stage 1: part[i*nb + b] = sum over block b's chunk; stage 2: fixed-order sum
template <typename R>
__global__ void __launch_bounds__(256) k_dot_part(const R *a, long lda, const R *b, long ldb,
                                                  long n, long chunk, double *part) {
  const long i = blockIdx.y;
  const long b0 = (long)blockIdx.x * chunk;
  long b1 = b0 + chunk;
  if (b1 > n) b1 = n;
  double s = 0.0;
  for (long g = b0 + threadIdx.x; g < b1; g += 256) s += (double)a[i * lda + g] * (double)b[i * ldb + g];
  __shared__ double red[4];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[i * gridDim.x + blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ void k_dot_final(const double *part, long nb, long m, double *out) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  double s = 0.0;
  for (long b = 0; b < nb; b++) s += part[i * nb + b];
  out[i] = s;
}

template <typename R>
static int dots_impl(const R *a, long lda, const R *b, long ldb, long m, long n, double *out_d,
                     double *scratch, long scratch_len, hipStream_t st) {
  long chunk = 16384;
  long nb = (n + chunk - 1) / chunk;
  if (nb * m > scratch_len) return SEP_ERR_NOMEM;
  hipLaunchKernelGGL(k_dot_part<R>, dim3((unsigned)nb, (unsigned)m), dim3(256), 0, st, a, lda, b,
                     ldb, n, chunk, scratch);
  hipLaunchKernelGGL(k_dot_final, dim3((unsigned)((m + 127) / 128)), dim3(128), 0, st, scratch, nb,
                     m, out_d);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}
int dots_dev(const double *a, long lda, const double *b, long ldb, long m, long n, double *out_d,
             double *scratch, long scratch_len, hipStream_t st) {
  return dots_impl<double>(a, lda, b, ldb, m, n, out_d, scratch, scratch_len, st);
}
int dots_dev_f(const float *a, long lda, const float *b, long ldb, long m, long n, double *out_d,
               double *scratch, long scratch_len, hipStream_t st) {
  return dots_impl<float>(a, lda, b, ldb, m, n, out_d, scratch, scratch_len, st);
}

__global__ void k_scale_rows(double *x, long ld, long n, const double *s) {
  const long i = blockIdx.y;
  const double f = s[i];
  for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x)
    x[i * ld + g] *= f;
}
int scale_rows_dev(double *x, long ld, long m, long n, const double *s_d, hipStream_t st) {
  unsigned nbx = (unsigned)((n + 255) / 256);
  if (nbx > 4096) nbx = 4096;
  hipLaunchKernelGGL(k_scale_rows, dim3(nbx, (unsigned)m), dim3(256), 0, st, x, ld, n, s_d);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// y_i -= s_i x_i for m rows of n points (residuals H psi - e psi)
// out_i = y_i - s_i x_i for the m rows (out may be y)
__global__ void k_sub_scaled_rows(double *out, long ldo, const double *y, long ldy,
                                  const double *x, long ldx, long n, const double *s) {
  const long i = blockIdx.y;
  const double f = s[i];
  for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x)
    out[i * ldo + g] = y[i * ldy + g] - f * x[i * ldx + g];
}
int diff_scaled_rows_dev(double *out, long ldo, const double *y, long ldy, const double *x,
                         long ldx, long m, long n, const double *s_d, hipStream_t st) {
  unsigned nbx = (unsigned)((n + 255) / 256);
  if (nbx > 4096) nbx = 4096;
  hipLaunchKernelGGL(k_sub_scaled_rows, dim3(nbx, (unsigned)m), dim3(256), 0, st, out, ldo, y, ldy,
                     x, ldx, n, s_d);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}
int sub_scaled_rows_dev(double *y, long ldy, const double *x, long ldx, long m, long n,
                        const double *s_d, hipStream_t st) {
  return diff_scaled_rows_dev(y, ldy, y, ldy, x, ldx, m, n, s_d, st);
}

__global__ void k_d2f(const double *in, float *out, long n) {
  for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x)
    out[g] = (float)in[g];
}
__global__ void k_f2d(const float *in, double *out, long n) {
  for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x)
    out[g] = (double)in[g];
}
int convert_d2f(const double *in, float *out, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_d2f, dim3(4096), dim3(256), 0, st, in, out, n);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}
int convert_f2d(const float *in, double *out, long n, hipStream_t st) {
  hipLaunchKernelGGL(k_f2d, dim3(4096), dim3(256), 0, st, in, out, n);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// ---- small dense matrices of the subspace stage (n <= a few thousand)

// A <- scale * (A + A^T) / 2 for an n x n row-major matrix; the (i > j)
// thread of each pair writes both entries, the diagonal is only scaled
// A <- scale (A + A^T) / 2 for a row-major n x n matrix.  With blk > 0 only
// the blk x blk blocks on and above the block diagonal hold values: an
// element of a block below it takes its mirror above, unaveraged.
__global__ void k_symmetrize(double *A, long n, double scale, long blk) {
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long i = (long)blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= n || j >= n || j > i) return;
  if (i == j) {
    A[i * n + i] *= scale;
    return;
  }
  const double a = (blk > 0 && i / blk != j / blk) ? A[j * n + i] * scale
                                                   : 0.5 * (A[i * n + j] + A[j * n + i]) * scale;
  A[i * n + j] = a;
  A[j * n + i] = a;
}
int symmetrize_dev(double *A, long n, double scale, hipStream_t st, long blk) {
  const dim3 blk2(32, 8), grd((unsigned)((n + 31) / 32), (unsigned)((n + 7) / 8));
  hipLaunchKernelGGL(k_symmetrize, grd, blk2, 0, st, A, n, scale, blk);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// M[i * k + j] = V[c(j) * n + i] * (sc ? sc[j] : 1), c(j) = j or n - 1 - j:
// eigenvector columns (column-major V, as the eigensolver leaves them) to the
// row-major coefficient matrix of combine_dev, through a 32 x 32 LDS tile
__global__ void k_eigvec_cols(const double *V, long n, long k, const double *sc, int reverse,
                              double *M) {
  __shared__ double t[32][33];
  const long i0 = (long)blockIdx.x * 32, j0 = (long)blockIdx.y * 32;
  for (int r = threadIdx.y; r < 32; r += blockDim.y) {  // r: output column j0 + r
    const long j = j0 + r, i = i0 + threadIdx.x;
    if (j < k && i < n) t[r][threadIdx.x] = V[(reverse ? n - 1 - j : j) * n + i];
  }
  __syncthreads();
  for (int r = threadIdx.y; r < 32; r += blockDim.y) {  // r: row i0 + r
    const long i = i0 + r, j = j0 + threadIdx.x;
    if (i < n && j < k) M[i * k + j] = t[threadIdx.x][r] * (sc ? sc[j] : 1.0);
  }
}
int eigvec_cols_dev(const double *V, long n, long k, const double *sc_d, bool reverse, double *M,
                    hipStream_t st) {
  const dim3 blk(32, 8), grd((unsigned)((n + 31) / 32), (unsigned)((k + 31) / 32));
  hipLaunchKernelGGL(k_eigvec_cols, grd, blk, 0, st, V, n, k, sc_d, reverse ? 1 : 0, M);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// zero the strictly lower triangle (i > j) of an n x n row-major matrix
__global__ void k_zero_lower(double *A, long n) {
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long i = (long)blockIdx.y * blockDim.y + threadIdx.y;
  if (i < n && j < i) A[i * n + j] = 0.0;
}
int zero_lower_dev(double *A, long n, hipStream_t st) {
  const dim3 blk(32, 8), grd((unsigned)((n + 31) / 32), (unsigned)((n + 7) / 8));
  hipLaunchKernelGGL(k_zero_lower, grd, blk, 0, st, A, n);
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

}  // namespace sep
