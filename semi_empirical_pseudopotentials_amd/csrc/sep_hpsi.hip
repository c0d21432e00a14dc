// sep_hpsi.hip -- the H.psi operator of the reference (filter/hamiltonian.c:11-44,
// filter/hnorm.c:11-39) as hand-written CDNA4 kernels.
//
// One application on a batch of complex vectors v (in the filter each complex
// vector carries two real states, re and im, because H is real) computes
//           out = alpha (T psi + V psi) - beta psi
// alpha = 1, beta = 0 is hamiltonian(); alpha = dE_1 = 4/dE,
// beta = 2 + z_{j-1} + Vmin dE_1 is the Newton step of hnorm().
// Every grid runs the two-kernel form of sep_split.h.  Measured against the
// forms kept here (filter loop, us per Newton step, MI355X): complex128 36^3
// x 8 vectors 17.6 (xy planes 33.8), 64^3 x 8 45.2 (47.5), 96^3 x 16 299
// (434), 128^3 x 4 160 (rows + lines 239), 80 x 64 x 64 x 5 39 (68);
// complex64 64^3 x 8 26.4 (29.7), 128^3 x 8 171 (190), 160^3 x 8 386 (631).
// Selectable beside it (sep_set_hpsi_family) are
//   rows + lines   x rows, strided y lines, z pencils (k_rows_*, k_lines,
//                  k_pencil): five passes over the spectrum
//   xy planes      complex64 128^2: pass A (x, y forward), pass B (k_pencil),
//                  pass C (y, x backward + epilogue), C fused with the next A
//                  through a whole plane of LDS (swizzled) or half (chunked)
#include <hip/hip_runtime.h>

#include "fft_core.h"
#include "sep_internal.h"
#include "sep_split.h"

namespace sep {

// block reduction of 4 doubles; writes part[blk*4 + q]
template <int T>
__device__ __forceinline__ void block_sum4(double s[4], double *part, long blk) {
  __shared__ double red[4][T / 64];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    double x = s[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double x = 0.0;
    for (int w = 0; w < (int)(blockDim.x + 63) / 64; w++) x += red[threadIdx.x][w];
    part[blk * 4 + threadIdx.x] = x;
  }
}

template <typename R, int N>
__device__ __forceinline__ void load_tw(cx<R> *dst, const cx<R> *src) {
  for (int i = threadIdx.x; i < N; i += blockDim.x) dst[i] = src[i];
}

// ======================================================= row kernels (x lines)
// forward: view -> Tbuf (interleaved)
template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_rows_fwd(VecView<R> in, cx<R> *tb, long nrows, long N,
                                                const cx<R> *twx) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, ROWS = T / G, P = PL::P, PN = lds_line<NX>();
  __shared__ cx<R> buf[ROWS][PN];
  __shared__ cx<R> tw[NX];
  load_tw<R, NX>(tw, twx);
  __syncthreads();
  const long vec = blockIdx.y;
  const int rl = threadIdx.x / G;
  const int g = threadIdx.x % G;
  const long row = (long)blockIdx.x * ROWS + rl;
  const bool act = (rl < ROWS) && (row < nrows);
  const int rls = rl < ROWS ? rl : 0;
  TwFor<NX, -1, R> tc;
  tc.init(g, tw);
  cx<R> v[E];
  constexpr int r0 = Pass<NX, -1>::radix(0);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / r0; b++)
#pragma unroll
      for (int k = 0; k < r0; k++) v[b * r0 + k] = in.ld(vec, row * NX + in_idx<NX, -1, 0>(g, b, k));
  }
  run_passes_c<NX, -1, 0, P>(v, g, act, tc, [&](int i) -> cx<R> & { return buf[rls][lds_pad(i)]; });
  constexpr int rl_ = Pass<NX, -1>::radix(P - 1);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++)
        tb[vec * N + row * NX + out_idx<NX, -1, P - 1>(g, b, k)] = v[b * rl_ + k];
  }
}

// backward + epilogue: Tbuf -> view (psi_in read from `pin`)
template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_rows_bwd(const cx<R> *tb, VecView<R> pin, VecView<R> out,
                                                Epi<R> epi, long nrows, long N, const cx<R> *twx) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, ROWS = T / G, P = PL::P, PN = lds_line<NX>();
  __shared__ cx<R> buf[ROWS][PN];
  __shared__ cx<R> tw[NX];
  load_tw<R, NX>(tw, twx);
  __syncthreads();
  const long vec = blockIdx.y;
  const int rl = threadIdx.x / G;
  const int g = threadIdx.x % G;
  const long row = (long)blockIdx.x * ROWS + rl;
  const bool act = (rl < ROWS) && (row < nrows);
  const int rls = rl < ROWS ? rl : 0;
  TwFor<NX, 1, R> tc;
  tc.init(g, tw);
  cx<R> v[E];
  constexpr int r0 = Pass<NX, 1>::radix(0);
  constexpr int rl_ = Pass<NX, 1>::radix(P - 1);
  cx<R> p[E];
  R V[E];
  if (act) {
#pragma unroll
    for (int b = 0; b < E / r0; b++)
#pragma unroll
      for (int k = 0; k < r0; k++) v[b * r0 + k] = tb[vec * N + row * NX + in_idx<NX, 1, 0>(g, b, k)];
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++) {
        const long gi = row * NX + out_idx<NX, 1, P - 1>(g, b, k);
        p[b * rl_ + k] = pin.ld(vec, gi);
        V[b * rl_ + k] = epi.pot[gi];
      }
  }
  run_passes_c<NX, 1, 0, P>(v, g, act, tc, [&](int i) -> cx<R> & { return buf[rls][lds_pad(i)]; });
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++) {
        const long gi = row * NX + out_idx<NX, 1, P - 1>(g, b, k);
        out.st(vec, gi, epilogue(epi, v[b * rl_ + k], p[b * rl_ + k], V[b * rl_ + k], s));
      }
  }
  if (epi.part) block_sum4<T>(s, epi.part, (long)blockIdx.y * gridDim.x + blockIdx.x);
}

// The row + line family's counterpart of k_plane_bwd_fwd_w: the inverse x
// FFT and epilogue of Newton step j (k_rows_bwd) and the forward x FFT of the
// resulting psi_j row for step j+1 (k_rows_fwd) in one kernel; the row of tb
// read at the start is rewritten at the end by the same threads.  Saves the
// forward kernel's read of psi_j.
template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_rows_bwd_fwd(cx<R> *tb, VecView<R> pin, VecView<R> out,
                                                    Epi<R> epi, long nrows, long N,
                                                    const cx<R> *twx) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, ROWS = T / G, P = PL::P, PN = lds_line<NX>();
  __shared__ cx<R> buf[ROWS][PN];
  __shared__ cx<R> tw[NX];
  load_tw<R, NX>(tw, twx);
  __syncthreads();
  const long vec = blockIdx.y;
  const int rl = threadIdx.x / G;
  const int g = threadIdx.x % G;
  const long row = (long)blockIdx.x * ROWS + rl;
  const bool act = (rl < ROWS) && (row < nrows);
  const int rls = rl < ROWS ? rl : 0;
  TwFor<NX, 1, R> tcb;
  tcb.init(g, tw);
  cx<R> v[E];
  constexpr int r0 = Pass<NX, 1>::radix(0);
  constexpr int rl_ = Pass<NX, 1>::radix(P - 1);
  constexpr int rlf = Pass<NX, -1>::radix(P - 1);
  cx<R> p[E];
  R V[E];
  if (act) {
#pragma unroll
    for (int b = 0; b < E / r0; b++)
#pragma unroll
      for (int k = 0; k < r0; k++) v[b * r0 + k] = tb[vec * N + row * NX + in_idx<NX, 1, 0>(g, b, k)];
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++) {
        const long gi = row * NX + out_idx<NX, 1, P - 1>(g, b, k);
        p[b * rl_ + k] = pin.ld(vec, gi);
        V[b * rl_ + k] = epi.pot[gi];
      }
  }
  auto at = [&](int i) -> cx<R> & { return buf[rls][lds_pad(i)]; };
  run_passes_c<NX, 1, 0, P>(v, g, act, tcb, at);
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++) {
        const long gi = row * NX + out_idx<NX, 1, P - 1>(g, b, k);
        v[b * rl_ + k] = epilogue(epi, v[b * rl_ + k], p[b * rl_ + k], V[b * rl_ + k], s);
        out.st(vec, gi, v[b * rl_ + k]);
      }
  }
  // psi_j's row through the row buffer into the forward input order
  __syncthreads();
  write_out<NX, 1, P - 1>(v, g, act, at);
  __syncthreads();
  read_in<NX, -1, 0>(v, g, act, at);
  TwFor<NX, -1, R> tcf;
  tcf.init(g, tw);
  run_passes_c<NX, -1, 0, P>(v, g, act, tcf, at);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rlf; b++)
#pragma unroll
      for (int k = 0; k < rlf; k++)
        tb[vec * N + row * NX + out_idx<NX, -1, P - 1>(g, b, k)] = v[b * rlf + k];
  }
}

// =============================================== strided lines (y, fallback)
// Lines of length N along an axis with element stride `es`; the block takes W
// consecutive x positions.  Line base for (x, outer) = outer*os + x.
template <typename R, int NL, int W, int S>
__global__ void __launch_bounds__(W * FftPlan<NL>::G) k_lines(cx<R> *tb, long N, int nx, long es,
                                                              long os, const cx<R> *twl) {
  using PL = FftPlan<NL>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  __shared__ cx<R> buf[NL][W];
  __shared__ cx<R> tw[NL];
  load_tw<R, NL>(tw, twl);
  __syncthreads();
  const int p = threadIdx.x % W;
  const int g = threadIdx.x / W;
  const long x = (long)blockIdx.x * W + p;
  const long outer = blockIdx.y;
  const long vec = blockIdx.z;
  const bool act = x < nx;
  cx<R> *base = tb + vec * N + outer * os + x;
  cx<R> v[E];
  constexpr int r0 = Pass<NL, S>::radix(0);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / r0; b++)
#pragma unroll
      for (int k = 0; k < r0; k++) v[b * r0 + k] = base[(long)in_idx<NL, S, 0>(g, b, k) * es];
  }
  run_passes<NL, S, 0, P>(v, g, act, tw, [&](int i) -> cx<R> & { return buf[i][p]; });
  constexpr int rl_ = Pass<NL, S>::radix(P - 1);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rl_; b++)
#pragma unroll
      for (int k = 0; k < rl_; k++) base[(long)out_idx<NL, S, P - 1>(g, b, k) * es] = v[b * rl_ + k];
  }
}

// ======================================== z pencils: forward, * k^2, backward
// PRE: the factor is kscale / (kin + pden) (kinetic preconditioner) instead
// of kin * kscale
template <typename R, int NZ, int W, bool PRE = false>
__global__ void __launch_bounds__(W * FftPlan<NZ>::G) k_pencil(cx<R> *tb, long N, int nx, int ny,
                                                               const cx<R> *twz,
                                                               const double *kxx,
                                                               const double *kyy,
                                                               const double *kzz, double ekin,
                                                               double kscale, double pden) {
  using PL = FftPlan<NZ>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  __shared__ cx<R> buf[NZ][W];
  __shared__ cx<R> tw[NZ];
  __shared__ double kz_s[NZ];
  load_tw<R, NZ>(tw, twz);
  for (int i = threadIdx.x; i < NZ; i += blockDim.x) kz_s[i] = kzz[i];
  __syncthreads();
  const int p = threadIdx.x % W;
  const int g = threadIdx.x / W;
  const long x = (long)blockIdx.x * W + p;
  const long y = blockIdx.y;
  const long vec = blockIdx.z;
  const bool act = x < nx;
  const long es = (long)nx * ny;
  cx<R> *base = tb + vec * N + y * nx + x;
  cx<R> v[E];
  constexpr int r0 = Pass<NZ, -1>::radix(0);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / r0; b++)
#pragma unroll
      for (int k = 0; k < r0; k++) v[b * r0 + k] = base[(long)in_idx<NZ, -1, 0>(g, b, k) * es];
  }
  auto at = [&](int i) -> cx<R> & { return buf[i][p]; };
  run_passes<NZ, -1, 0, P>(v, g, act, tw, at);
  // kinetic factor, filter/init.c:138-144 order: (kx + ky) + kz, clamp
  const double kxy = act ? (kxx[x] + kyy[y]) : 0.0;
  constexpr int rl_ = Pass<NZ, -1>::radix(P - 1);
#pragma unroll
  for (int b = 0; b < E / rl_; b++)
#pragma unroll
    for (int k = 0; k < rl_; k++) {
      int z = out_idx<NZ, -1, P - 1>(g, b, k);
      double kin = kxy + kz_s[z];
      if (kin > ekin) kin = ekin;
      if constexpr (PRE)
        v[b * rl_ + k] = cscale(v[b * rl_ + k], (R)(kscale / (kin + pden)));
      else
        v[b * rl_ + k] = cscale(v[b * rl_ + k], (R)(kin * kscale));
    }
  // backward: pass 0 reads exactly the registers the forward last pass wrote
  run_passes<NZ, 1, 0, P>(v, g, act, tw, at);
  constexpr int rb = Pass<NZ, 1>::radix(P - 1);
  if (act) {
#pragma unroll
    for (int b = 0; b < E / rb; b++)
#pragma unroll
      for (int k = 0; k < rb; k++) base[(long)out_idx<NZ, 1, P - 1>(g, b, k) * es] = v[b * rb + k];
  }
}

// ------------------------------------------- wave-local plane kernels
// When the threads of one line fit a wavefront (64 % G == 0), every FFT
// exchange of a row or a column stays inside one wavefront; only the
// row <-> column transpose needs block barriers.  Line positions in LDS are
// placed by PlaneLds (below) so the strided exchange patterns spread over the
// banks; FP32 threads keep their twiddles in registers (TwFor).
// The spectrum of a plane is stored column-major, Tbuf[z][kx][ky], so that
// the column phase writes (and the backward column phase reads) contiguous
// ky runs.

// LDS placement of one plane in the wave-local plane kernels: row y of the
// (transposed) plane starts at rowbase(y); during the row FFTs element x of
// a row sits at rowbase(y) + xpos(x).  Generic lengths: pitch NX/NH + 1,
// rows and in-row positions xor-swizzled.  Complex64 at 128 (G = 16 threads
// per line, two lines per half-wave): pitch 150 with per-row offsets and an
// in-row permutation that make every access of the row and column phases
// free of bank conflicts for 8-byte accesses on gfx950 (64 banks of 4 B, 32
// lanes served per cycle): the two rows (columns) of a half-wave start
// 16 mod 32 elements apart, and the 16 positions of every access pattern of
// the radix-8/8/2 passes are distinct mod 16.
template <typename R, int NX, int NH>
struct PlaneLds {
  static constexpr int LDc = NX / NH + 1;
  static __device__ __forceinline__ int rowbase(int y) { return lds_swz(y) * LDc; }
  static __device__ __forceinline__ int xpos(int x) { return lds_swz(x); }
};
template <>
struct PlaneLds<float, 128, 1> {
  static constexpr int LDc = 150;
  static __device__ __forceinline__ int rowbase(int y) {
    const int d = 3 + 2 * ((y >> 5) & 3) + ((((y >> 3) ^ (y >> 4)) & 1) ^ ((y >> 6) & 1)) -
                  3 * (y & 1);
    return y * LDc + 2 * d;
  }
  static __device__ __forceinline__ int xpos(int x) {
    const int u = x >> 4;
    return x ^ (((9 * u) ^ (8 * (u >> 2))) & 15);
  }
};

template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_plane_fwd_w(VecView<R> in, cx<R> *tb, long N, int nz,
                                                   const cx<R> *twg) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  static_assert(64 % G == 0 && NX % 8 == 0, "lines must not straddle wavefronts");
  using L = PlaneLds<R, NX, 1>;
  constexpr int LDc = L::LDc;
  constexpr int RX = T / G;               // lines per round
  constexpr int NR = (NX + RX - 1) / RX;  // row rounds, column rounds
  extern __shared__ char smem_raw[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem_raw);  // [NX][LDc], row y at L::rowbase(y)
  cx<R> *tw = buf + NX * LDc;
  const long vec = blockIdx.x / nz;
  const long z = blockIdx.x % nz;
  const long pbase = z * (long)NX * NX;
  const int tl = threadIdx.x / G, g = threadIdx.x % G;
  constexpr int r0 = Pass<NX, -1>::radix(0);
  constexpr int rl_ = Pass<NX, -1>::radix(P - 1);
  cx<R> v[NR][E];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int row = r * RX + tl;
    if (row < NX) {
#pragma unroll
      for (int b = 0; b < E / r0; b++)
#pragma unroll
        for (int k = 0; k < r0; k++)
          v[r][b * r0 + k] = in.ld(vec, pbase + row * NX + in_idx<NX, -1, 0>(g, b, k));
    }
  }
  load_tw<R, NX>(tw, twg);
  __syncthreads();
  TwFor<NX, -1, R> tc;
  tc.init(g, tw);
  // ---- rows: x FFT, exchanged in the row's own buffer row; the results stay
  // in registers
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int row = r * RX + tl;
    const bool act = row < NX;
    const int base = L::rowbase(act ? row : 0);
    auto at = [&](int i) -> cx<R> & { return buf[base + L::xpos(i)]; };
    run_passes_c<NX, -1, 0, P, WaveSync>(v[r], g, act, tc, at);
  }
  // ---- columns
  __syncthreads();  // the row exchanges are done
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int row = r * RX + tl;
    if (row < NX) {
#pragma unroll
      for (int b = 0; b < E / rl_; b++)
#pragma unroll
        for (int k = 0; k < rl_; k++)
          buf[L::rowbase(row) + out_idx<NX, -1, P - 1>(g, b, k)] = v[r][b * rl_ + k];
    }
  }
  __syncthreads();  // the transpose
#pragma unroll
  for (int cr = 0; cr < NR; cr++) {
    const int cl = cr * RX + tl;
    const bool act = cl < NX;
    const int cs = act ? cl : 0;
    cx<R> w[E];
    auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
    read_in<NX, -1, 0>(w, g, act, at);
    run_passes_c<NX, -1, 0, P, WaveSync>(w, g, act, tc, at);
    if (act) {
      cx<R> *dst = tb + vec * N + pbase + (long)cs * NX;
#pragma unroll
      for (int b = 0; b < E / rl_; b++)
#pragma unroll
        for (int k = 0; k < rl_; k++) dst[out_idx<NX, -1, P - 1>(g, b, k)] = w[b * rl_ + k];
    }
  }
}

// At 1024 threads the register budget is 128: twiddles come from LDS, and of
// the epilogue's operands only V is loaded before the row's FFT.
template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_plane_bwd_w(const cx<R> *tb, VecView<R> pin,
                                                   VecView<R> out, Epi<R> epi, long N, int nz,
                                                   const cx<R> *twg) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  static_assert(64 % G == 0 && NX % 8 == 0, "lines must not straddle wavefronts");
  using L = PlaneLds<R, NX, 1>;
  constexpr int LDc = L::LDc;
  constexpr int RX = T / G;
  constexpr int NR = (NX + RX - 1) / RX;
  extern __shared__ char smem_raw[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem_raw);
  cx<R> *tw = buf + NX * LDc;
  const long vec = blockIdx.x / nz;
  const long z = blockIdx.x % nz;
  const long pbase = z * (long)NX * NX;
  const int tl = threadIdx.x / G, g = threadIdx.x % G;
  constexpr int r0 = Pass<NX, 1>::radix(0);
  constexpr int rl_ = Pass<NX, 1>::radix(P - 1);
  TwTable<NX, 1, R> tc;
  // ---- columns: load, y FFT, into the buffer
  {
    cx<R> w[NR][E];
#pragma unroll
    for (int cr = 0; cr < NR; cr++) {
      const int cl = cr * RX + tl;
      if (cl < NX) {
        const cx<R> *src = tb + vec * N + pbase + (long)cl * NX;
#pragma unroll
        for (int b = 0; b < E / r0; b++)
#pragma unroll
          for (int k = 0; k < r0; k++) w[cr][b * r0 + k] = src[in_idx<NX, 1, 0>(g, b, k)];
      }
    }
    load_tw<R, NX>(tw, twg);
    __syncthreads();
    tc.init(g, tw);
#pragma unroll
    for (int cr = 0; cr < NR; cr++) {
      const int cl = cr * RX + tl;
      const bool act = cl < NX;
      const int cs = act ? cl : 0;
      auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
      run_passes_c<NX, 1, 0, P, WaveSync>(w[cr], g, act, tc, at);
      WaveSync::sync();
      write_out<NX, 1, P - 1>(w[cr], g, act, at);
    }
  }
  __syncthreads();  // the transpose
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int row = r * RX + tl;
    const bool act = row < NX;
    const int rs = act ? row : 0;
    cx<R> p[E];
    R V[E];
    if (act) {
#pragma unroll
      for (int b = 0; b < E / rl_; b++)
#pragma unroll
        for (int k = 0; k < rl_; k++)
          V[b * rl_ + k] = epi.pot[pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k)];
    }
    // the row is in the buffer (at L::rowbase(y), x in natural order); the
    // exchanges then run in place in that row at the permuted positions
    cx<R> x[E];
    auto at0 = [&](int i) -> cx<R> & { return buf[L::rowbase(rs) + i]; };
    read_in<NX, 1, 0>(x, g, act, at0);
    auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(rs) + L::xpos(i)]; };
    run_passes_c<NX, 1, 0, P, WaveSync>(x, g, act, tc, at);
    if (act) {
#pragma unroll
      for (int b = 0; b < E / rl_; b++)
#pragma unroll
        for (int k = 0; k < rl_; k++)
          p[b * rl_ + k] = pin.ld(vec, pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k));
#pragma unroll
      for (int b = 0; b < E / rl_; b++)
#pragma unroll
        for (int k = 0; k < rl_; k++) {
          const long gi = pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k);
          out.st(vec, gi, epilogue(epi, x[b * rl_ + k], p[b * rl_ + k], V[b * rl_ + k], s));
        }
    }
  }
  if (epi.part) block_sum4<T>(s, epi.part, blockIdx.x);
}

// An int the compiler must treat as unknown: index and LDS address math
// derived from it is recomputed where it is used instead of being kept live
// in registers across the phases of a kernel.
__device__ __forceinline__ int opaque_int(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Pass C of Newton step j fused with pass A of step j+1 (whole-plane buffer).
// The epilogue's psi_j is stored (the ring slot the accumulation
// reads) and, still in registers, transformed forward -- x rows in each row's
// own buffer row, then y columns -- into plane z of the spectrum buffer,
// which this block alone read at its start.  Saves pass A's read of psi_j;
// the arithmetic is that of k_plane_bwd_w followed by k_plane_fwd_w.
template <typename R, int NX, int T>
__global__ void __launch_bounds__(T) k_plane_bwd_fwd_w(cx<R> *tb, VecView<R> pin, VecView<R> out,
                                                       Epi<R> epi, long N, int nz,
                                                       const cx<R> *twg) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  static_assert(64 % G == 0 && NX % 8 == 0, "lines must not straddle wavefronts");
  using L = PlaneLds<R, NX, 1>;
  constexpr int LDc = L::LDc;
  constexpr int RX = T / G;
  constexpr int NR = (NX + RX - 1) / RX;
  extern __shared__ char smem_raw[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem_raw);
  cx<R> *tw = buf + NX * LDc;
  const long vec = blockIdx.x / nz;
  const long z = blockIdx.x % nz;
  const long pbase = z * (long)NX * NX;
  const int tl = threadIdx.x / G, g0 = threadIdx.x % G;
  const int g = g0;
  constexpr int r0b = Pass<NX, 1>::radix(0);
  constexpr int rlb = Pass<NX, 1>::radix(P - 1);
  constexpr int rlf = Pass<NX, -1>::radix(P - 1);
  // psi_{j-1} is loaded after the row FFT (before it, it fits the registers but
  // measured 5 % slower: 138 against 132 us at 128^3)
  TwTable<NX, 1, R> tcb;
  TwTable<NX, -1, R> tcf;
  // ---- inverse y FFT of the columns (pass C)
  {
    cx<R> w[NR][E];
#pragma unroll
    for (int cr = 0; cr < NR; cr++) {
      const int cl = cr * RX + tl;
      if (cl < NX) {
        const cx<R> *src = tb + vec * N + pbase + (long)cl * NX;
#pragma unroll
        for (int b = 0; b < E / r0b; b++)
#pragma unroll
          for (int k = 0; k < r0b; k++) w[cr][b * r0b + k] = src[in_idx<NX, 1, 0>(g, b, k)];
      }
    }
    load_tw<R, NX>(tw, twg);
    __syncthreads();
    tcb.init(g, tw);
    tcf.init(g, tw);
#pragma unroll
    for (int cr = 0; cr < NR; cr++) {
      const int cl = cr * RX + tl;
      const bool act = cl < NX;
      const int cs = act ? cl : 0;
      auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
      run_passes_c<NX, 1, 0, P, WaveSync>(w[cr], g, act, tcb, at);
      WaveSync::sync();
      write_out<NX, 1, P - 1>(w[cr], g, act, at);
    }
  }
  __syncthreads();  // the transpose
  // ---- rows: inverse x FFT, epilogue, store psi_j, forward x FFT of psi_j
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int g = opaque_int(g0);  // per-round index math (see opaque_int)
    tcb.init(g, tw);
    tcf.init(g, tw);
    const int row = r * RX + tl;
    const bool act = row < NX;
    const int rs = act ? row : 0;
    cx<R> p[E];
    R V[E];
    if (act) {
#pragma unroll
      for (int b = 0; b < E / rlb; b++)
#pragma unroll
        for (int k = 0; k < rlb; k++)
          V[b * rlb + k] = epi.pot[pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k)];
    }
    cx<R> x[E];
    auto at0 = [&](int i) -> cx<R> & { return buf[L::rowbase(rs) + i]; };
    read_in<NX, 1, 0>(x, g, act, at0);
    auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(rs) + L::xpos(i)]; };
    run_passes_c<NX, 1, 0, P, WaveSync>(x, g, act, tcb, at);
    if (act) {
#pragma unroll
      for (int b = 0; b < E / rlb; b++)
#pragma unroll
        for (int k = 0; k < rlb; k++)
          p[b * rlb + k] = pin.ld(vec, pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k));
#pragma unroll
      for (int b = 0; b < E / rlb; b++)
#pragma unroll
        for (int k = 0; k < rlb; k++) {
          const long gi = pbase + rs * NX + out_idx<NX, 1, P - 1>(g, b, k);
          x[b * rlb + k] = epilogue(epi, x[b * rlb + k], p[b * rlb + k], V[b * rlb + k], s);
          out.st(vec, gi, x[b * rlb + k]);
        }
    }
    // psi_j's row back through the row buffer into the forward input order
    WaveSync::sync();
    write_out<NX, 1, P - 1>(x, g, act, at);
    WaveSync::sync();
    read_in<NX, -1, 0>(x, g, act, at);
    run_passes_c<NX, -1, 0, P, WaveSync>(x, g, act, tcf, at);
    WaveSync::sync();
    if (act) {
#pragma unroll
      for (int b = 0; b < E / rlf; b++)
#pragma unroll
        for (int k = 0; k < rlf; k++)
          buf[L::rowbase(rs) + out_idx<NX, -1, P - 1>(g, b, k)] = x[b * rlf + k];
    }
  }
  __syncthreads();  // the transpose
  // ---- forward y FFT of the columns (pass A of step j+1) into plane z of tb
#pragma unroll
  for (int cr = 0; cr < NR; cr++) {
    const int g = opaque_int(g0);
    tcf.init(g, tw);
    const int cl = cr * RX + tl;
    const bool act = cl < NX;
    const int cs = act ? cl : 0;
    cx<R> y[E];
    auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
    read_in<NX, -1, 0>(y, g, act, at);
    run_passes_c<NX, -1, 0, P, WaveSync>(y, g, act, tcf, at);
    if (act) {
      cx<R> *dst = tb + vec * N + pbase + (long)cs * NX;
#pragma unroll
      for (int b = 0; b < E / rlf; b++)
#pragma unroll
        for (int k = 0; k < rlf; k++) dst[out_idx<NX, -1, P - 1>(g, b, k)] = y[b * rlf + k];
    }
  }
}

// Pass C fused with the next pass A, with the plane held in registers and
// transposed through a buffer of NX/NH columns, same arithmetic as
// k_plane_bwd_fwd_w.  The buffer is 1/NH of a plane, so NH = 2 at complex64
// 128^2 (67 KB) lets two workgroups share a CU and one's HBM phases run
// under the other's FFTs; waves_per_eu holds the register budget to what two
// resident workgroups leave (T / 128 waves per SIMD: 128 VGPRs at T = 512).
template <typename R, int NX, int T, int NH>
__global__ void __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T / 128)))
k_plane_bwd_fwd_h(cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi, long N, int nz,
                  const cx<R> *twg) {
  using PL = FftPlan<NX>;
  constexpr int G = PL::G, E = PL::E, P = PL::P;
  static_assert(64 % G == 0 && NX % 8 == 0, "lines must not straddle wavefronts");
  static_assert(NH > 1 && NX % NH == 0, "the chunked kernel splits the plane into NH chunks");
  constexpr int W = NX / NH;
  using L = PlaneLds<R, NX, NH>;
  constexpr int LDc = L::LDc;
  constexpr int RX = T / G;
  constexpr int NR = (NX + RX - 1) / RX;
  constexpr int NCR = (W + RX - 1) / RX;
  constexpr int RS = NX + 1;
  static_assert(RX * RS <= NX * LDc, "row exchange slices exceed the chunk buffer");
  extern __shared__ char smem_raw[];
  cx<R> *buf = reinterpret_cast<cx<R> *>(smem_raw);
  cx<R> *tw = buf + NX * LDc;
  const long vec = blockIdx.x / nz;
  const long z = blockIdx.x % nz;
  const long pbase = z * (long)NX * NX;
  const int tl = threadIdx.x / G, g0 = threadIdx.x % G;
  const int g = g0;
  constexpr int r0b = Pass<NX, 1>::radix(0);
  constexpr int rlb = Pass<NX, 1>::radix(P - 1);
  constexpr int rlf = Pass<NX, -1>::radix(P - 1);
  TwTable<NX, 1, R> tcb;
  TwTable<NX, -1, R> tcf;
  cx<R> v[NR][E];  // the plane's rows, x in registers
  // ---- inverse y FFT of the columns, chunk by chunk; each thread gathers
  // the chunk's x positions of the rows it owns
#pragma unroll
  for (int c = 0; c < NH; c++) {
    cx<R> w[NCR][E];
#pragma unroll
    for (int cr = 0; cr < NCR; cr++) {
      const int cl = cr * RX + tl;
      if (cl < W) {
        const cx<R> *src = tb + vec * N + pbase + (long)(c * W + cl) * NX;
#pragma unroll
        for (int b = 0; b < E / r0b; b++)
#pragma unroll
          for (int k = 0; k < r0b; k++) w[cr][b * r0b + k] = src[in_idx<NX, 1, 0>(g, b, k)];
      }
    }
    if (c == 0) load_tw<R, NX>(tw, twg);
    __syncthreads();  // twiddles loaded / the previous chunk's gather is done
    tcb.init(g, tw);
#pragma unroll
    for (int cr = 0; cr < NCR; cr++) {
      const int cl = cr * RX + tl;
      const bool act = cl < W;
      const int cs = act ? cl : 0;
      auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
      run_passes_c<NX, 1, 0, P, WaveSync>(w[cr], g, act, tcb, at);
      WaveSync::sync();
      write_out<NX, 1, P - 1>(w[cr], g, act, at);
    }
    __syncthreads();  // the transpose
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int row = r * RX + tl;
      if (row < NX) {
#pragma unroll
        for (int b = 0; b < E / r0b; b++)
#pragma unroll
          for (int k = 0; k < r0b; k++) {
            const int x = in_idx<NX, 1, 0>(g, b, k);
            if (x / W == c) v[r][b * r0b + k] = buf[L::rowbase(row) + (x - c * W)];
          }
      }
    }
  }
  __syncthreads();  // the buffer is free for the row exchanges
  // ---- rows: inverse x FFT, epilogue, store psi_j, forward x FFT of psi_j.
  // Exchanges use slice tl of the buffer.  V and psi_{j-1} are loaded after
  // the FFT (the other workgroup on the CU covers the latency); psi is in
  // planar form (re and im arrays), and no partial sums are formed (the
  // filter loop asks for none).
  const R alpha = (R)epi.alpha, beta = (R)epi.beta;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int g = opaque_int(g0);  // per-round index math (see opaque_int)
    tcb.init(g, tw);
    tcf.init(g, tw);
    const int row = r * RX + tl;
    const bool act = row < NX;
    const int rs = act ? row : 0;
    auto at = [&](int i) -> cx<R> & { return buf[tl * RS + lds_swz(i)]; };
    run_passes_c<NX, 1, 0, P, WaveSync>(v[r], g, act, tcb, at);
    if (act) {
      const long ro = pbase + (long)rs * NX;
      const R *pr = pin.re + vec * pin.vstride + ro, *pi = pin.im + vec * pin.vstride + ro;
      R *qr = out.re + vec * out.vstride + ro, *qi = out.im + vec * out.vstride + ro;
      const R *vp = epi.pot + ro;
      R V[E], pre[E], pim[E];
#pragma unroll
      for (int b = 0; b < E / rlb; b++)
#pragma unroll
        for (int k = 0; k < rlb; k++) {
          const int x = out_idx<NX, 1, P - 1>(g, b, k);
          V[b * rlb + k] = vp[x];
          pre[b * rlb + k] = pr[x];
          pim[b * rlb + k] = pi[x];
        }
#pragma unroll
      for (int b = 0; b < E / rlb; b++)
#pragma unroll
        for (int k = 0; k < rlb; k++) {
          const int e = b * rlb + k, x = out_idx<NX, 1, P - 1>(g, b, k);
          cx<R> o;  // the arithmetic of epilogue()
          o.re = alpha * (v[r][e].re + V[e] * pre[e]) - beta * pre[e];
          o.im = alpha * (v[r][e].im + V[e] * pim[e]) - beta * pim[e];
          qr[x] = o.re;
          qi[x] = o.im;
          v[r][e] = o;
        }
    }
    // psi_j's row back through the slice into the forward input order
    WaveSync::sync();
    write_out<NX, 1, P - 1>(v[r], g, act, at);
    WaveSync::sync();
    read_in<NX, -1, 0>(v[r], g, act, at);
    run_passes_c<NX, -1, 0, P, WaveSync>(v[r], g, act, tcf, at);
  }
  // ---- forward y FFT of the columns (pass A of step j+1), chunk by chunk
#pragma unroll
  for (int c = 0; c < NH; c++) {
    __syncthreads();  // row exchanges / the previous chunk's columns are done
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int row = r * RX + tl;
      if (row < NX) {
#pragma unroll
        for (int b = 0; b < E / rlf; b++)
#pragma unroll
          for (int k = 0; k < rlf; k++) {
            const int kx = out_idx<NX, -1, P - 1>(g, b, k);
            if (kx / W == c) buf[L::rowbase(row) + (kx - c * W)] = v[r][b * rlf + k];
          }
      }
    }
    __syncthreads();  // the transpose
#pragma unroll
    for (int cr = 0; cr < NCR; cr++) {
      const int g = opaque_int(g0);
      tcf.init(g, tw);
      const int cl = cr * RX + tl;
      const bool act = cl < W;
      const int cs = act ? cl : 0;
      cx<R> y[E];
      auto at = [&](int i) -> cx<R> & { return buf[L::rowbase(i) + cs]; };
      read_in<NX, -1, 0>(y, g, act, at);
      run_passes_c<NX, -1, 0, P, WaveSync>(y, g, act, tcf, at);
      if (act) {
        cx<R> *dst = tb + vec * N + pbase + (long)(c * W + cs) * NX;
#pragma unroll
        for (int b = 0; b < E / rlf; b++)
#pragma unroll
          for (int k = 0; k < rlf; k++) dst[out_idx<NX, -1, P - 1>(g, b, k)] = y[b * rlf + k];
      }
    }
  }
}

// ================================================================= dispatch
template <typename R, int NX>
constexpr size_t plane_lds() {
  return sizeof(cx<R>) * ((size_t)NX * PlaneLds<R, NX, 1>::LDc + NX);
}

template <typename R>
struct HOps {
  // returns false if size unsupported
  static bool rows_fwd(int nx, VecView<R> in, cx<R> *tb, long nrows, long N, int nvec,
                       const cx<R> *tw, hipStream_t st);
  static bool rows_bwd(int nx, const cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi,
                       long nrows, long N, int nvec, const cx<R> *tw, hipStream_t st,
                       long *nblk);
  static bool lines(int nl, int S, cx<R> *tb, long N, int nx, long es, long os, int nouter,
                    int nvec, const cx<R> *tw, hipStream_t st);
  static bool pencil(int nz, cx<R> *tb, long N, int nx, int ny, int nvec, const cx<R> *tw,
                     const double *kxx, const double *kyy, const double *kzz, double ekin,
                     double kscale, double pden, hipStream_t st);
  // k_rows_bwd + the next step's k_rows_fwd in one kernel
  static bool rows_bwd_fwd(int nx, cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi,
                           long nrows, long N, int nvec, const cx<R> *tw, hipStream_t st);
};

#define SEP_LINE_SIZES(X) X(16) X(24) X(32) X(36) X(48) X(64) X(80) X(96) X(128) X(160)

template <typename R>
bool HOps<R>::rows_fwd(int nx, VecView<R> in, cx<R> *tb, long nrows, long N, int nvec,
                       const cx<R> *tw, hipStream_t st) {
  switch (nx) {
#define C(n)                                                                              \
  case n: {                                                                               \
    constexpr int T = 256, ROWS = T / FftPlan<n>::G;                                      \
    dim3 grid((unsigned)((nrows + ROWS - 1) / ROWS), (unsigned)nvec);                     \
    hipLaunchKernelGGL((k_rows_fwd<R, n, T>), grid, dim3(T), 0, st, in, tb, nrows, N, tw); \
    return true;                                                                          \
  }
    SEP_LINE_SIZES(C)
#undef C
  }
  return false;
}

template <typename R>
bool HOps<R>::rows_bwd(int nx, const cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi,
                       long nrows, long N, int nvec, const cx<R> *tw, hipStream_t st,
                       long *nblk) {
  switch (nx) {
#define C(n)                                                                                \
  case n: {                                                                                 \
    constexpr int T = 256, ROWS = T / FftPlan<n>::G;                                        \
    dim3 grid((unsigned)((nrows + ROWS - 1) / ROWS), (unsigned)nvec);                       \
    if (nblk) *nblk = (long)grid.x * grid.y;                                                \
    hipLaunchKernelGGL((k_rows_bwd<R, n, T>), grid, dim3(T), 0, st, tb, pin, out, epi, nrows, \
                       N, tw);                                                              \
    return true;                                                                            \
  }
    SEP_LINE_SIZES(C)
#undef C
  }
  return false;
}

template <typename R>
bool HOps<R>::rows_bwd_fwd(int nx, cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi,
                           long nrows, long N, int nvec, const cx<R> *tw, hipStream_t st) {
  switch (nx) {
#define C(n)                                                                                 \
  case n: {                                                                                  \
    constexpr int T = 256, ROWS = T / FftPlan<n>::G;                                         \
    dim3 grid((unsigned)((nrows + ROWS - 1) / ROWS), (unsigned)nvec);                        \
    hipLaunchKernelGGL((k_rows_bwd_fwd<R, n, T>), grid, dim3(T), 0, st, tb, pin, out, epi,    \
                       nrows, N, tw);                                                        \
    return true;                                                                             \
  }
    SEP_LINE_SIZES(C)
#undef C
  }
  return false;
}

template <typename R>
bool HOps<R>::lines(int nl, int S, cx<R> *tb, long N, int nx, long es, long os, int nouter,
                    int nvec, const cx<R> *tw, hipStream_t st) {
  constexpr int W = sizeof(R) == 8 ? 16 : 32;
  dim3 grid((unsigned)((nx + W - 1) / W), (unsigned)nouter, (unsigned)nvec);
  switch (nl) {
#define C(n)                                                                                   \
  case n:                                                                                      \
    if (S < 0)                                                                                 \
      hipLaunchKernelGGL((k_lines<R, n, W, -1>), grid, dim3(W * FftPlan<n>::G), 0, st, tb, N, nx, \
                         es, os, tw);                                                          \
    else                                                                                       \
      hipLaunchKernelGGL((k_lines<R, n, W, 1>), grid, dim3(W * FftPlan<n>::G), 0, st, tb, N, nx,  \
                         es, os, tw);                                                          \
    return true;
    SEP_LINE_SIZES(C)
#undef C
  }
  return false;
}

// pden > 0: preconditioner factor kscale / (kin + pden), FP64 only
template <typename R>
bool HOps<R>::pencil(int nz, cx<R> *tb, long N, int nx, int ny, int nvec, const cx<R> *tw,
                     const double *kxx, const double *kyy, const double *kzz, double ekin,
                     double kscale, double pden, hipStream_t st) {
  constexpr int W = sizeof(R) == 8 ? 16 : 32;
  dim3 grid((unsigned)((nx + W - 1) / W), (unsigned)ny, (unsigned)nvec);
  if (pden > 0.0 && sizeof(R) != 8) return false;
  switch (nz) {
#define C(n)                                                                                  \
  case n:                                                                                     \
    if constexpr (sizeof(R) == 8) {                                                           \
      if (pden > 0.0) {                                                                       \
        hipLaunchKernelGGL((k_pencil<R, n, W, true>), grid, dim3(W * FftPlan<n>::G), 0, st, tb, \
                           N, nx, ny, tw, kxx, kyy, kzz, ekin, kscale, pden);                 \
        return true;                                                                          \
      }                                                                                       \
    }                                                                                         \
    hipLaunchKernelGGL((k_pencil<R, n, W>), grid, dim3(W * FftPlan<n>::G), 0, st, tb, N, nx, ny, \
                       tw, kxx, kyy, kzz, ekin, kscale, 0.0);                                 \
    return true;
    SEP_LINE_SIZES(C)
#undef C
  }
  return false;
}

// The xy-plane kernels: complex64 128^2 only, 1024 threads (16 waves on the CU
// that one plane buffer occupies).
constexpr int kPlaneN = 128, kPlaneT = 1024;

template <typename K>
static void lds_attr(K *kernel, size_t lds, bool *done) {
  if (*done) return;
  hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  *done = true;
}
// nvec == 0: kernel attributes only (before graph capture)
static void plane_fwd(VecView<float> in, cx<float> *tb, long N, int nz, int nvec,
                      const cx<float> *tw, hipStream_t st) {
  constexpr size_t lds = plane_lds<float, kPlaneN>();
  static_assert(lds <= 160 * 1024, "plane buffer exceeds the LDS of a gfx950 workgroup");
  static bool attr = false;
  lds_attr(k_plane_fwd_w<float, kPlaneN, kPlaneT>, lds, &attr);
  if (nvec == 0) return;
  hipLaunchKernelGGL((k_plane_fwd_w<float, kPlaneN, kPlaneT>), dim3((unsigned)(nz * nvec)),
                     dim3(kPlaneT), lds, st, in, tb, N, nz, tw);
}
static void plane_bwd(const cx<float> *tb, VecView<float> pin, VecView<float> out, Epi<float> epi,
                      long N, int nz, int nvec, const cx<float> *tw, hipStream_t st, long *nblk) {
  constexpr size_t lds = plane_lds<float, kPlaneN>();
  static bool attr = false;
  if (nblk) *nblk = (long)nz * nvec;
  lds_attr(k_plane_bwd_w<float, kPlaneN, kPlaneT>, lds, &attr);
  if (nvec == 0) return;
  hipLaunchKernelGGL((k_plane_bwd_w<float, kPlaneN, kPlaneT>), dim3((unsigned)(nz * nvec)),
                     dim3(kPlaneT), lds, st, tb, pin, out, epi, N, nz, tw);
}
// pass C fused with the next pass A; form SEP_FUSED_CHUNKED or _SWIZZLED
static void plane_bwd_fwd(cx<float> *tb, VecView<float> pin, VecView<float> out, Epi<float> epi,
                          long N, int nz, int nvec, const cx<float> *tw, hipStream_t st, int form) {
  if (form == SEP_FUSED_CHUNKED) {
    constexpr int T = 512, NH = 2;
    constexpr size_t lds = sizeof(cx<float>) * ((size_t)kPlaneN * PlaneLds<float, kPlaneN, NH>::LDc + kPlaneN);
    static_assert(2 * lds <= 160 * 1024, "two chunk buffers must share the LDS of a CU");
    static bool attr = false;
    lds_attr(k_plane_bwd_fwd_h<float, kPlaneN, T, NH>, lds, &attr);
    if (nvec == 0) return;
    hipLaunchKernelGGL((k_plane_bwd_fwd_h<float, kPlaneN, T, NH>), dim3((unsigned)(nz * nvec)),
                       dim3(T), lds, st, tb, pin, out, epi, N, nz, tw);
    return;
  }
  constexpr size_t lds = plane_lds<float, kPlaneN>();
  static bool attr = false;
  lds_attr(k_plane_bwd_fwd_w<float, kPlaneN, kPlaneT>, lds, &attr);
  if (nvec == 0) return;
  hipLaunchKernelGGL((k_plane_bwd_fwd_w<float, kPlaneN, kPlaneT>), dim3((unsigned)(nz * nvec)),
                     dim3(kPlaneT), lds, st, tb, pin, out, epi, N, nz, tw);
}

bool plane_fused_form_supported(int n, int prec, int form) {
  return form == SEP_FUSED_PLANE || (n == kPlaneN && prec == SEP_PREC_FP32);
}

// ----------------------------------------------------------------- public
bool hop_supported(int n) {
  switch (n) {
#define C(x) case x:
    SEP_LINE_SIZES(C)
#undef C
    return true;
  }
  return false;
}

// Grids on which the default form goes by the name SEP_HPSI_PLANE (square xy
// planes of these lengths); elsewhere it is SEP_HPSI_SPLIT only.
bool plane_supported(int nx, int ny, int prec) {
  if (nx != ny) return false;
  switch (nx) {
    case 16: case 24: case 32: case 36: case 48: case 64: case 96:
      return true;
    case 128:
      return prec == SEP_PREC_FP32;
  }
  return false;
}

// Whether this grid's H.psi runs the xy-plane kernels: the chunked or swizzled
// family was asked for.
static bool use_plane(const GridDev &gd, int prec) {
  return !gd.force_lines[prec] && gd.fused_form[prec] != SEP_FUSED_PLANE;
}
// Whether it runs the two-kernel form of sep_split.h (every grid does unless
// another family was asked for).
static bool use_split(const GridDev &gd, int prec) {
  return !gd.force_lines[prec] && gd.fused_form[prec] == SEP_FUSED_PLANE;
}
// Whether one application is one kernel (the filter's fused steps run the
// two-kernel form: their first kernel also starts the next step).
template <typename R>
static bool use_box(const GridDev &gd) {
  return use_split(gd, sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32) &&
         box_supported<R>(gd.nx, gd.ny, gd.nz);
}
template <typename R>
static const cx<R> *twid(const GridDev &gd, int axis) {
  return reinterpret_cast<const cx<R> *>(sizeof(R) == 8 ? gd.tw64[axis] : gd.tw32[axis]);
}
// The passes around the kinetic factor, in place on tb: the split form's
// tiles, or z pencils (a column-major plane spectrum swaps the roles of x
// and y).  nvec == 0: kernel attributes only.
template <typename R>
static bool spectral(const GridDev &gd, cx<R> *tb, int nvec, hipStream_t st) {
  const int prec = sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32;
  const double kscale = gd.pden > 0.0 ? gd.pnum : 1.0;
  if (use_split(gd, prec))
    return SplitOps<R>::tile(gd.nx, gd.ny, gd.nz, tb, nvec, twid<R>(gd, 1), twid<R>(gd, 2), gd.kxx,
                             gd.kyy, gd.kzz, gd.ekin, kscale, gd.pden, st);
  const bool cm = use_plane(gd, prec);
  return HOps<R>::pencil(gd.nz, tb, gd.N, cm ? gd.ny : gd.nx, cm ? gd.nx : gd.ny, nvec,
                         twid<R>(gd, 2), cm ? gd.kyy : gd.kxx, cm ? gd.kxx : gd.kyy, gd.kzz,
                         gd.ekin, kscale, gd.pden, st);
}

// One H application (see file header) on nvec complex vectors.  With ev,
// events are recorded before the first kernel, after the forward pass (pass
// A; the split form's forward rows), after the spectral passes and at the
// end (ev[0..3]).
template <typename R>
int hpsi_apply(const GridDev &gd, const VecView<R> &in, const VecView<R> &out, cx<R> *tb,
               const R *pot, int nvec, double alpha, double beta, double *part, long *nblk,
               hipStream_t st, hipEvent_t *ev) {
  const int nx = gd.nx, ny = gd.ny, nz = gd.nz;
  const long N = gd.N;
  const int prec = sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32;
  const cx<R> *twx = twid<R>(gd, 0), *twy = twid<R>(gd, 1);
  Epi<R> epi{pot, alpha, beta, part};
  bool ok = true;
  if (ev) hipEventRecord(ev[0], st);
  if (use_box<R>(gd)) {
    // the whole kernel counts as the spectral passes
    if (ev) hipEventRecord(ev[1], st);
    ok = box_apply<R>(gd, in, out, epi, nvec, st);
    if (nblk) *nblk = nvec;
    if (ev) {
      hipEventRecord(ev[2], st);
      hipEventRecord(ev[3], st);
    }
    if (!ok) return SEP_ERR_UNSUPPORTED;
    return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
  }
  if (use_split(gd, prec)) {
    ok = SplitOps<R>::rows_fwd(nx, ny, nz, in, tb, nvec, twx, st);
  } else if (use_plane(gd, prec)) {
    if constexpr (sizeof(R) == 4) plane_fwd(in, tb, N, nz, nvec, twx, st);
  } else {
    ok = HOps<R>::rows_fwd(nx, in, tb, (long)ny * nz, N, nvec, twx, st) &&
         HOps<R>::lines(ny, -1, tb, N, nx, nx, (long)nx * ny, nz, nvec, twy, st);
  }
  if (ev) hipEventRecord(ev[1], st);
  ok = ok && spectral<R>(gd, tb, nvec, st);
  if (ev) hipEventRecord(ev[2], st);
  if (use_split(gd, prec)) {
    ok = ok && SplitOps<R>::rows_bwd(nx, ny, nz, tb, in, out, epi, nvec, twx, twy, false, st, nblk);
  } else if (use_plane(gd, prec)) {
    if constexpr (sizeof(R) == 4) plane_bwd(tb, in, out, epi, N, nz, nvec, twx, st, nblk);
  } else {
    ok = ok && HOps<R>::lines(ny, 1, tb, N, nx, nx, (long)nx * ny, nz, nvec, twy, st) &&
         HOps<R>::rows_bwd(nx, tb, in, out, epi, (long)ny * nz, N, nvec, twx, st, nblk);
  }
  if (ev) hipEventRecord(ev[3], st);
  if (!ok) return SEP_ERR_UNSUPPORTED;
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// Split Newton step: the filter loop transforms psi_0 forward once
// (hpsi_fwd), then each step runs the spectral passes and one kernel that
// finishes psi_j and transforms it forward for the next step (hpsi_step with
// fwd_next); the spectrum of psi_j stays in tb between steps.  Rows + lines:
// the forward y lines move to the start of the next step.  Both planes of the
// vectors must exist (the fused kernels keep the imaginary plane that a
// real-only view would drop).
template <typename R>
bool hpsi_fused_supported(const GridDev &gd) {
  return !(gd.pden > 0.0) && hop_supported(gd.nx) && hop_supported(gd.ny);
}

template <typename R>
int hpsi_fwd(const GridDev &gd, const VecView<R> &in, cx<R> *tb, int nvec, hipStream_t st) {
  const int prec = sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32;
  const cx<R> *twx = twid<R>(gd, 0);
  if (!hpsi_fused_supported<R>(gd) || !in.im) return SEP_ERR_UNSUPPORTED;
  bool ok = true;
  if (use_split(gd, prec)) {
    ok = SplitOps<R>::rows_fwd(gd.nx, gd.ny, gd.nz, in, tb, nvec, twx, st);
  } else if (use_plane(gd, prec)) {
    if constexpr (sizeof(R) == 4) plane_fwd(in, tb, gd.N, gd.nz, nvec, twx, st);
  } else {
    ok = HOps<R>::rows_fwd(gd.nx, in, tb, (long)gd.ny * gd.nz, gd.N, nvec, twx, st);
  }
  if (!ok) return SEP_ERR_UNSUPPORTED;
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}

// tb holds the spectrum of in (psi_{j-1}; for the row + line family its x
// transform only); out <- alpha (T + V) in - beta in and, with fwd_next, tb
// <- the same transform of out.  Events as hpsi_apply's ev[1..3]: before the
// spectral passes (with the row + line family's y lines), after them, after
// the last kernel; ev[0] is not recorded.
template <typename R>
int hpsi_step(const GridDev &gd, const VecView<R> &in, const VecView<R> &out, cx<R> *tb,
              const R *pot, int nvec, double alpha, double beta, bool fwd_next, hipStream_t st,
              hipEvent_t *ev, const SoEpi *so) {
  const int nx = gd.nx, ny = gd.ny, nz = gd.nz;
  const long N = gd.N;
  const int prec = sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32;
  const cx<R> *twx = twid<R>(gd, 0), *twy = twid<R>(gd, 1);
  if (!hpsi_fused_supported<R>(gd) || !in.im || !out.im) return SEP_ERR_UNSUPPORTED;
  const bool split = use_split(gd, prec), plane = use_plane(gd, prec);
  // the spin-orbit add rides only in the split form's FP64 row kernel
  if (so && (sizeof(R) != 8 || !split || !fwd_next)) return SEP_ERR_UNSUPPORTED;
  bool ok = true;
  if (ev) hipEventRecord(ev[1], st);
  if (!split && !plane) ok = HOps<R>::lines(ny, -1, tb, N, nx, nx, (long)nx * ny, nz, nvec, twy, st);
  ok = ok && spectral<R>(gd, tb, nvec, st);
  if (!split && !plane)
    ok = ok && HOps<R>::lines(ny, 1, tb, N, nx, nx, (long)nx * ny, nz, nvec, twy, st);
  if (ev) hipEventRecord(ev[2], st);
  Epi<R> epi{pot, alpha, beta, nullptr};
  if (so) {
    epi.so_map = so->map;
    epi.so_g = so->g;
    epi.so_nsp = so->nsp;
    epi.so_alpha = so->alpha;
  }
  if (split) {
    ok = ok &&
         SplitOps<R>::rows_bwd(nx, ny, nz, tb, in, out, epi, nvec, twx, twy, fwd_next, st, nullptr);
  } else if (plane) {
    if constexpr (sizeof(R) == 4) {
      if (fwd_next)
        plane_bwd_fwd(tb, in, out, epi, N, nz, nvec, twx, st, gd.fused_form[prec]);
      else
        plane_bwd(tb, in, out, epi, N, nz, nvec, twx, st, nullptr);
    }
  } else if (fwd_next) {
    ok = ok && HOps<R>::rows_bwd_fwd(nx, tb, in, out, epi, (long)ny * nz, N, nvec, twx, st);
  } else {
    ok = ok && HOps<R>::rows_bwd(nx, tb, in, out, epi, (long)ny * nz, N, nvec, twx, st, nullptr);
  }
  if (ev) hipEventRecord(ev[3], st);
  if (!ok) return SEP_ERR_UNSUPPORTED;
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}
template bool hpsi_fused_supported<double>(const GridDev &);
template bool hpsi_fused_supported<float>(const GridDev &);
template int hpsi_fwd<double>(const GridDev &, const VecView<double> &, cx<double> *, int,
                              hipStream_t);
template int hpsi_fwd<float>(const GridDev &, const VecView<float> &, cx<float> *, int, hipStream_t);
template int hpsi_step<double>(const GridDev &, const VecView<double> &, const VecView<double> &,
                               cx<double> *, const double *, int, double, double, bool,
                               hipStream_t, hipEvent_t *, const SoEpi *);
template int hpsi_step<float>(const GridDev &, const VecView<float> &, const VecView<float> &,
                              cx<float> *, const float *, int, double, double, bool, hipStream_t,
                              hipEvent_t *, const SoEpi *);
bool hpsi_so_fused(const GridDev &gd) { return use_split(gd, SEP_PREC_FP64); }

// Kernel attributes of this grid's H.psi kernels, set outside any stream
// capture (hipFuncSetAttribute is not a stream operation).
template <typename R>
int hpsi_prepare(const GridDev &gd) {
  const int prec = sizeof(R) == 8 ? SEP_PREC_FP64 : SEP_PREC_FP32;
  if (use_split(gd, prec)) {
    if (!spectral<R>(gd, nullptr, 0, nullptr)) return SEP_ERR_UNSUPPORTED;
    const VecView<R> none{nullptr, nullptr, nullptr, 0};
    if (use_box<R>(gd)) box_apply<R>(gd, none, none, Epi<R>{}, 0, nullptr);
  } else if (use_plane(gd, prec)) {
    if constexpr (sizeof(R) == 4) {
      VecView<R> none{nullptr, nullptr, nullptr, 0};
      Epi<R> epi{nullptr, 0.0, 0.0, nullptr};
      plane_fwd(none, nullptr, gd.N, gd.nz, 0, nullptr, nullptr);
      plane_bwd(nullptr, none, none, epi, gd.N, gd.nz, 0, nullptr, nullptr, nullptr);
      plane_bwd_fwd(nullptr, none, none, epi, gd.N, gd.nz, 0, nullptr, nullptr, gd.fused_form[prec]);
    }
  }
  return hipGetLastError() == hipSuccess ? SEP_OK : SEP_ERR_HIP;
}
template int hpsi_prepare<double>(const GridDev &);
template int hpsi_prepare<float>(const GridDev &);

template int hpsi_apply<double>(const GridDev &, const VecView<double> &, const VecView<double> &,
                                cx<double> *, const double *, int, double, double, double *,
                                long *, hipStream_t, hipEvent_t *);
template int hpsi_apply<float>(const GridDev &, const VecView<float> &, const VecView<float> &,
                               cx<float> *, const float *, int, double, double, double *, long *,
                               hipStream_t, hipEvent_t *);

}  // namespace sep
