// sep_box.hip -- H.psi of grids whose vector fits one CU's LDS, in one kernel.
//
// The two-kernel form of sep_split.h needs three launches for one application
// (forward rows, tiles, backward rows), each 3 us of latency on data that a
// single CU holds.  Here a workgroup takes one complex vector through the whole
// application: y lines from memory, x lines, z lines with the kinetic factor, x
// lines back, y lines back with the epilogue.  A thread owns a whole line in
// registers in every pass and writes it back to the LDS places it read, so the
// passes exchange through one copy of the box with one barrier each.  Rows of
// the box have an odd pitch: lanes along y fall on different banks.
//
// Bound by its serial chain (five passes of LDS reads, a 16- or 24-point
// transform and LDS writes on 4 to 6 waves).  The kernel takes 7.6 us for one
// vector of 16^3 in FP64 and 8.7 for 64 (8.4 and 9.2 without psi and V kept in
// registers and the kinetic terms loaded at the start; a loop over the axes
// instead of straight code: 13.5).  An application call, in us for the three
// kernels and this one: 16^3 FP64 20.4 -> 18.6 (1 vector), 24.8 -> 19.8 (64);
// FP32 20.1 -> 18.0, 22.7 -> 18.3; 24x16x16 FP32 20.9 -> 19.7, 25.3 -> 20.7.
// It stops paying where a vector is longer: FP64 24x16x16 20.7 -> 21.8, FP32
// 24x24x16 20.9 -> 22.6 at one vector.
#include <hip/hip_runtime.h>

#include "sep_internal.h"
#include "sep_split.h"

namespace sep {

template <int r, int S, typename R>
__device__ __forceinline__ void dft_line(cx<R> *v) {
  if constexpr (r == 24) dft_pfa<S, 3, 8>(v);
  else dft<r, S>(v);
}

template <typename R, int NX, int NY, int NZ>
struct BoxCfg {
  static constexpr int LX = NY * NZ, LY = NX * NZ, LZ = NX * NY;  // lines along x, y, z
  static constexpr int M = LX > LY ? (LX > LZ ? LX : LZ) : (LY > LZ ? LY : LZ);
  static constexpr int T = (M + 63) / 64 * 64;
  static constexpr int PX = NX + 1;  // 16 and 24: an odd pitch
  static constexpr int E = NX > NY ? (NX > NZ ? NX : NZ) : (NY > NZ ? NY : NZ);
  static constexpr size_t LDS = sizeof(cx<R>) * PX * NY * NZ;
};

template <typename R, int NX, int NY, int NZ>
__global__ void __launch_bounds__((BoxCfg<R, NX, NY, NZ>::T))
    k_box(VecView<R> in, VecView<R> out, Epi<R> epi, const double *kxx, const double *kyy,
          const double *kzz, double ekin, double kscale, double pden) {
  using C = BoxCfg<R, NX, NY, NZ>;
  constexpr int PX = C::PX, T = C::T;
  extern __shared__ __align__(16) char smem_b[];
  __shared__ double kz[NZ];
  cx<R> *box = reinterpret_cast<cx<R> *>(smem_b);  // (x, y, z) at x + PX (y + NY z)
  const int t = threadIdx.x;
  const long vec = blockIdx.x;
  cx<R> v[C::E];
  cx<R> p[NY];  // psi and V of the thread's y line, kept for the epilogue
  R V[NY];
  const int zx = t % NX, zy = t / NX;  // z lines
  const bool za = T == C::LZ || t < C::LZ;
  // ---- y lines: thread = (x fastest, z)
  const bool ya = T == C::LY || t < C::LY;
  const int yx = t % NX, yz = t / NX;
  const unsigned g0 = (unsigned)(yz * NY * NX + yx);
  cx<R> *yl = box + yx + PX * NY * yz;
  if (ya) {
    auto load = [&](auto form) {
#pragma unroll
      for (int k = 0; k < NY; k++) v[k] = ld_row<form.value>(in, vec, (long)k * NX, g0);
    };
    const int form = view_form(in);
    if (form == VIEW_CX) load(std::integral_constant<int, VIEW_CX>{});
    else if (form == VIEW_PLANES) load(std::integral_constant<int, VIEW_PLANES>{});
    else load(std::integral_constant<int, VIEW_REAL>{});
#pragma unroll
    for (int k = 0; k < NY; k++) {
      p[k] = v[k];
      V[k] = at_bytes(epi.pot + k * NX, g0 * (unsigned)sizeof(R));
    }
    dft_line<NY, -1>(v);
#pragma unroll
    for (int k = 0; k < NY; k++) yl[PX * k] = v[k];
  }
  const double kxy = za ? kxx[zx] + kyy[zy] : 0.0;
  for (int i = t; i < NZ; i += T) kz[i] = kzz[i];
  lds_sync();
  // ---- x lines: thread = (y, z)
  const bool xa = T == C::LX || t < C::LX;
  cx<R> *xl = box + PX * t;
  auto x_lines = [&](auto sign) {
    if (xa) {
#pragma unroll
      for (int k = 0; k < NX; k++) v[k] = xl[k];
      dft_line<NX, sign.value>(v);
#pragma unroll
      for (int k = 0; k < NX; k++) xl[k] = v[k];
    }
    lds_sync();
  };
  x_lines(std::integral_constant<int, -1>{});
  // ---- z lines: thread = (x fastest, y)
  if (za) {
    cx<R> *zl = box + zx + PX * zy;
#pragma unroll
    for (int k = 0; k < NZ; k++) v[k] = zl[PX * NY * k];
    dft_line<NZ, -1>(v);
    // filter/init.c:138-144 order: (kx + ky) + kz, clamp
#pragma unroll
    for (int k = 0; k < NZ; k++) {
      const double kin = fmin(kxy + kz[k], ekin);
      v[k] = cscale(v[k], (R)(pden > 0.0 ? kscale / (kin + pden) : kin));
    }
    dft_line<NZ, 1>(v);
#pragma unroll
    for (int k = 0; k < NZ; k++) zl[PX * NY * k] = v[k];
  }
  lds_sync();
  x_lines(std::integral_constant<int, 1>{});
  // ---- y lines back, epilogue
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  if (ya) {
#pragma unroll
    for (int k = 0; k < NY; k++) v[k] = yl[PX * k];
    dft_line<NY, 1>(v);
    auto finish = [&](auto form) {
#pragma unroll
      for (int k = 0; k < NY; k++)
        st_row<form.value>(out, vec, (long)k * NX, g0, epilogue(epi, v[k], p[k], V[k], s));
    };
    const int form = view_form(out);  // in and out have one form
    if (form == VIEW_CX) finish(std::integral_constant<int, VIEW_CX>{});
    else if (form == VIEW_PLANES) finish(std::integral_constant<int, VIEW_PLANES>{});
    else finish(std::integral_constant<int, VIEW_REAL>{});
  }
  if (epi.part) block_sum4_any<T>(s, epi.part, vec, reinterpret_cast<double *>(smem_b));
}

template <typename R, int NX, int NY, int NZ>
static void box_launch(const GridDev &gd, const VecView<R> &in, const VecView<R> &out,
                       const Epi<R> &epi, int nvec, hipStream_t st) {
  using C = BoxCfg<R, NX, NY, NZ>;
  static_assert(C::LDS + sizeof(double) * NZ <= 160 * 1024, "box exceeds a CU's LDS");
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute((const void *)k_box<R, NX, NY, NZ>,
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS);
    attr = true;
  }
  if (nvec == 0) return;  // attribute only (before graph capture)
  hipLaunchKernelGGL((k_box<R, NX, NY, NZ>), dim3((unsigned)nvec), dim3(C::T), C::LDS, st, in, out,
                     epi, gd.kxx, gd.kyy, gd.kzz, gd.ekin, gd.pden > 0.0 ? gd.pnum : 1.0, gd.pden);
}

template <typename R>
bool box_apply(const GridDev &gd, const VecView<R> &in, const VecView<R> &out, const Epi<R> &epi,
               int nvec, hipStream_t st) {
  const int n[3] = {gd.nx, gd.ny, gd.nz};
  if (!box_supported<R>(n[0], n[1], n[2])) return false;
  if constexpr (sizeof(R) == 4) {
    if (n[0] == 24) return box_launch<R, 24, 16, 16>(gd, in, out, epi, nvec, st), true;
    if (n[1] == 24) return box_launch<R, 16, 24, 16>(gd, in, out, epi, nvec, st), true;
    if (n[2] == 24) return box_launch<R, 16, 16, 24>(gd, in, out, epi, nvec, st), true;
  }
  box_launch<R, 16, 16, 16>(gd, in, out, epi, nvec, st);
  return true;
}
template bool box_apply<double>(const GridDev &, const VecView<double> &, const VecView<double> &,
                                const Epi<double> &, int, hipStream_t);
template bool box_apply<float>(const GridDev &, const VecView<float> &, const VecView<float> &,
                               const Epi<float> &, int, hipStream_t);

}  // namespace sep
