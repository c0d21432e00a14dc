// sep_split.h -- H.psi in two kernels per Newton step, for boxes of any shape.
//
// A line of N = A B points is transformed by one radix-A and one radix-B
// pass (radices up to 16).  The y transform is split between the kernels:
//
//   k_xrows  one (z, jy): the A_y rows y = jy + k B_y.  Inverse radix-A_y
//            pass of y and inverse x FFT, epilogue psi_j, forward radix-A_y
//            pass of y and forward x FFT
//   k_tile   one kx and W of the A_y y-residues, all z: forward radix-B_y
//            pass of y, z FFT, * min(k^2/2, Ekin)/N, inverse z FFT, inverse
//            radix-B_y pass, in place
//
// so that each kernel works on a few thousand points that stay in registers
// and go through LDS four times, several workgroups share a CU, and a step
// moves the three-pass minimum of (6c + r) bytes per point and complex
// vector (c complex, r real bytes) whatever the box: 104 B at FP64 128^3,
// where a 128 x 128 plane (262 KB) fits no CU and the row + line kernels
// move 168 B.
//
// Spectrum buffer: T[z / 2][jy][kx][q / W][z % 2][q % W], q < A_y the y
// residue.  A row workgroup owns both z of a pair and so reads and writes
// contiguous chunks of T; a tile workgroup reads and writes runs of 2 W
// elements (128 bytes in FP64).  With single z (runs of W elements) the
// loads and stores of a W = 4 tile alone took 55 us at FP64 128^3 x 4 vectors
// (268 MB), runs of 128 bytes 34 us.
#pragma once
#include "fft_core.h"
#include "sep_internal.h"

namespace sep {

// Operands of the epilogue out = alpha (T psi + V psi) - beta psi.
template <typename R>
struct Epi {
  const R *pot;   // V on the grid
  double alpha, beta;
  double *part;   // per-block partial sums (4 per block) or nullptr
  // spinor filter (FP64 backward rows that start the next step): psi_j += so_alpha *
  // (V_so psi_{j-1}) at the grid points in a spin-orbit list, so_map[g] the
  // point's row of so_g (4 doubles per spinor: up re, im, dn re, im) or -1
  const int *so_map = nullptr;
  const double *so_g = nullptr;
  long so_nsp = 0;
  double so_alpha = 0.0;
};

template <typename R>
__device__ __forceinline__ cx<R> epilogue(const Epi<R> &e, cx<R> t, cx<R> p, R V, double s[4]) {
  R a = (R)e.alpha, b = (R)e.beta;
  cx<R> o;
  o.re = a * (t.re + V * p.re) - b * p.re;
  o.im = a * (t.im + V * p.im) - b * p.im;
  if (e.part) {  // uniform: the FP64 sums only when a reduction was asked for
    s[0] += (double)p.re * (double)o.re;
    s[1] += (double)p.im * (double)o.im;
    s[2] += (double)o.re * (double)o.re;
    s[3] += (double)o.im * (double)o.im;
  }
  return o;
}

// ---------------------------------------------------------- butterflies
// Prime-factor forms (no twiddles): with N = P Q, P and Q coprime, input
// n = (Q n1 + P n2) mod N and output k = (k mod P, k mod Q).
template <int S, int P, int Q, typename R>
__device__ __forceinline__ void dft_pfa(cx<R> *v) {
  constexpr int N = P * Q;
  cx<R> a[Q][P];
#pragma unroll
  for (int n2 = 0; n2 < Q; n2++) {
#pragma unroll
    for (int n1 = 0; n1 < P; n1++) a[n2][n1] = v[(Q * n1 + P * n2) % N];
    dft<P, S>(a[n2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < P; k1++) {
    cx<R> b[Q];
#pragma unroll
    for (int n2 = 0; n2 < Q; n2++) b[n2] = a[n2][k1];
    dft<Q, S>(b);
#pragma unroll
    for (int k = 0; k < N; k++)
      if (k % P == k1) v[k] = b[k % Q];
  }
}
template <int r, int S, typename R>
__device__ __forceinline__ void dft_x(cx<R> *v) {
  if constexpr (r == 6) dft_pfa<S, 2, 3>(v);
  else if constexpr (r == 10) dft_pfa<S, 2, 5>(v);
  else if constexpr (r == 12) dft_pfa<S, 3, 4>(v);
  else dft<r, S>(v);
}

// ---------------------------------------------------------- plans
// x and z lines: N = A B.  Forward: radix A on butterflies j < B (inputs
// j + k B, outputs A j + k), exchange, radix B on j < A (inputs and outputs
// j + k A, twiddles w_N^(j k)).  Inverse: the same backwards (radix B, then
// A), so that its first pass reads the registers the forward one ended with.
// GZ threads share a z line: as many as leave few of them idle in either pass
// and few points a thread; at 160 ten keep 20 points a thread, which fit FP32's
// registers (16 threads: 80 -> 98 us, 4 vectors) but not FP64's (166 -> 180).
// At 80 ten for eight 33.2 -> 31.7 us FP64, 21.9 -> 20.7 FP32 (8 vectors).
template <int N>
struct LinePlan;
#define SEP_LINE_PLAN(N_, A_, B_, GZ64_, GZ32_)               \
  template <>                                                 \
  struct LinePlan<N_> {                                       \
    static constexpr int N = N_, A = A_, B = B_;              \
    static constexpr int GZ64 = GZ64_, GZ32 = GZ32_;          \
    static_assert(A_ * B_ == N_, "two-pass plan");            \
  };
SEP_LINE_PLAN(16, 4, 4, 4, 4)
SEP_LINE_PLAN(24, 6, 4, 4, 4)
SEP_LINE_PLAN(32, 8, 4, 4, 4)
SEP_LINE_PLAN(36, 6, 6, 6, 6)
SEP_LINE_PLAN(48, 6, 8, 8, 8)
SEP_LINE_PLAN(64, 8, 8, 8, 8)
SEP_LINE_PLAN(80, 10, 8, 10, 10)
SEP_LINE_PLAN(96, 16, 6, 8, 8)
SEP_LINE_PLAN(128, 16, 8, 8, 8)
SEP_LINE_PLAN(160, 16, 10, 16, 10)
#undef SEP_LINE_PLAN

// y lines: AY rows per group of k_xrows (register-local pass), BY points per
// thread in k_tile, W = y_width(AY) of the AY residues per tile: small tiles,
// so that several workgroups share a CU and one's memory phases run under
// another's transforms (FP64 128^3 x 4 vectors: W = 8 72 us, W = 4 61 us).
#define SEP_Y_PLANS(X)                                              \
  X(16, 4, 4) X(24, 6, 4) X(32, 8, 4) X(36, 6, 6) X(48, 8, 6)       \
  X(64, 8, 8) X(80, 16, 5) X(96, 16, 6) X(128, 16, 8) X(160, 16, 10)
constexpr int y_width(int ay) { return ay % 4 == 0 ? 4 : ay; }
// distinct (BY, W)
#define SEP_Y_TILES(X) X(4, 4) X(4, 6) X(5, 4) X(6, 4) X(6, 6) X(8, 4) X(10, 4)
#define SEP_SPLIT_LENGTHS(X) X(16) X(24) X(32) X(36) X(48) X(64) X(80) X(96) X(128) X(160)

// LDS barrier: orders LDS accesses only, so that global loads and stores in
// flight are not waited for.
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f(i, j, k) for element k of butterfly j = g + G b (register i), the NB
// butterflies of radix RAD below LIM that thread g owns.
template <int NB, int RAD, int LIM, int G, typename F>
__device__ __forceinline__ void each_el(int g, bool act, F f) {
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int j = g + G * b;
    if (act && (NB * G == LIM || j < LIM)) {
#pragma unroll
      for (int k = 0; k < RAD; k++) f(b * RAD + k, j, k);
    }
  }
}

// Twiddle table of a line plan in LDS: w_N^(j k) for j < A, k < B at
// k (A + 1) + j, so that both directions read at a thread base plus constant
// offsets (forward: j the thread's, stride A + 1; inverse: k the thread's,
// stride 1) without bank conflicts.
template <int N>
struct LineTw {
  static constexpr int A = LinePlan<N>::A, B = LinePlan<N>::B, P = A + 1, WORDS = B * P;
  template <typename R>
  static __device__ __forceinline__ void load(cx<R> *tab, const cx<R> *tw, int t, int T) {
    for (int i = t; i < N; i += T) tab[(i / A) * P + i % A] = tw[(i / A) * (i % A)];
  }
};

// One pass: twiddles of the table at tab + (thread's index) JS + k KS
// (conjugated for S > 0; JS == 0: none) and butterflies.
template <int S, int NB, int RAD, int LIM, int G, int JS, int KS, typename R>
__device__ __forceinline__ void radix_pass(cx<R> *v, int g, bool act, const cx<R> *tab) {
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int j = g + G * b;
    if (act && (NB * G == LIM || j < LIM)) {
      if constexpr (JS > 0) {
#pragma unroll
        for (int k = 1; k < RAD; k++) {
          cx<R> w = tab[j * JS + k * KS];
          if constexpr (S > 0) w.im = -w.im;
          v[b * RAD + k] = cmul(v[b * RAD + k], w);
          if constexpr (RAD > 8) {
            if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      dft_x<RAD, S>(v + b * RAD);
      if constexpr (NB > 1 && NB * RAD > 12) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Exchange through LDS: put(f) calls f(register, address) for the elements
// a thread holds, get(f) for those it reads.  SPLIT moves the real and the
// imaginary parts one after the other through half the space.  The barrier
// before the first write lets the buffer's last readers finish.
template <bool SPLIT, typename R, typename Put, typename Get>
__device__ __forceinline__ void exchange(cx<R> *v, void *lds, Put put, Get get) {
  if constexpr (SPLIT) {
    R *s = static_cast<R *>(lds);
    lds_sync();
    put([&](int i, int a) { s[a] = v[i].re; });
    lds_sync();
    get([&](int i, int a) { v[i].re = s[a]; });
    lds_sync();
    put([&](int i, int a) { s[a] = v[i].im; });
    lds_sync();
    get([&](int i, int a) { v[i].im = s[a]; });
  } else {
    cx<R> *s = static_cast<cx<R> *>(lds);
    lds_sync();
    put([&](int i, int a) { s[a] = v[i]; });
    lds_sync();
    get([&](int i, int a) { v[i] = s[a]; });
  }
}

// Element at a wave-uniform pointer plus a 32-bit byte offset of the lane: the
// uniform part stays in scalar registers and one vector register addresses
// all of a thread's elements (64-bit addresses per element cost 2 VGPRs each
// from the first load to the last store: 32 of 128 in k_tile).
template <typename T>
__device__ __forceinline__ T &at_bytes(T *p, unsigned b) {
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + b);
}
template <typename T>
__device__ __forceinline__ const T &at_bytes(const T *p, unsigned b) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + b);
}
// Makes the compiler forget a uniform pointer and a lane offset, so that the
// addresses of the stores at a kernel's end are formed there instead of being
// kept from the loads at its start.
template <typename T>
__device__ __forceinline__ void forget(T *&p, unsigned &b) {
  asm volatile("" : "+s"(p), "+v"(b));
}
// Forms of a view: interleaved, two real planes, or one real plane (the
// imaginary part reads as 0 and is not written).
enum { VIEW_CX = 0, VIEW_PLANES = 1, VIEW_REAL = 2 };
template <typename R>
__device__ __forceinline__ int view_form(const VecView<R> &v) {
  return v.c ? VIEW_CX : v.im ? VIEW_PLANES : VIEW_REAL;
}
// Element `lane` of a view past a wave-uniform offset (vec, off).
template <int FORM, typename R>
__device__ __forceinline__ cx<R> ld_row(const VecView<R> &v, long vec, long off, unsigned lane) {
  const long u = vec * v.vstride + off;
  if constexpr (FORM == VIEW_CX) {
    return at_bytes<const cx<R>>(v.c + u, lane * (unsigned)sizeof(cx<R>));
  } else {
    const unsigned b = lane * (unsigned)sizeof(R);
    cx<R> x;
    x.re = at_bytes<const R>(v.re + u, b);
    x.im = FORM == VIEW_PLANES ? at_bytes<const R>(v.im + u, b) : (R)0;
    return x;
  }
}
template <int FORM, typename R>
__device__ __forceinline__ void st_row(const VecView<R> &v, long vec, long off, unsigned lane,
                                       cx<R> x) {
  const long u = vec * v.vstride + off;
  if constexpr (FORM == VIEW_CX) {
    at_bytes(v.c + u, lane * (unsigned)sizeof(cx<R>)) = x;
  } else {
    const unsigned b = lane * (unsigned)sizeof(R);
    at_bytes(v.re + u, b) = x.re;
    if constexpr (FORM == VIEW_PLANES) at_bytes(v.im + u, b) = x.im;
  }
}

// ---------------------------------------------------------- x rows
template <typename R, int NX, int AY>
struct XRows {
  using PL = LinePlan<NX>;
  static constexpr int A = PL::A, B = PL::B;
  // one thread per x in row order; in the x passes G threads share each of
  // the AY rows
  static constexpr int G0 = NX / AY > 0 ? NX / AY : 1;
  static constexpr int GM = A > B ? A : B;
  static constexpr int G = G0 < GM ? G0 : GM;
  static constexpr int W = y_width(AY);
  static constexpr int TG = AY * G > NX ? AY * G : NX;  // threads of one group of rows
  // pairs of groups (z even and odd, one jy) per workgroup
  static constexpr int MP = 2 * TG >= 128 ? 1 : 128 / (2 * TG);
  static constexpr int T = MP * 2 * TG;
  static constexpr int NB0 = (B + G - 1) / G, NB1 = (A + G - 1) / G;
  static constexpr int E1 = NB0 * A > NB1 * B ? NB0 * A : NB1 * B;
  static constexpr int E = E1 > AY ? E1 : AY;
  static constexpr int LD = AY + 1;  // odd pitch: no bank conflicts across x
  static constexpr bool SPLIT = sizeof(cx<R>) * NX * LD * 2 * MP > 40 * 1024;
  static constexpr int LDSG = NX * LD;  // elements per group
  static constexpr int LDS = (SPLIT ? (int)sizeof(R) : (int)sizeof(cx<R>)) * LDSG * 2 * MP;
  // waves per SIMD the register budget must allow
  static constexpr int WPE = E * sizeof(cx<R>) > 128 ? 3 : 4;

  // Thread's place: its pair; in row order its z of the pair and x; in the x
  // passes its line of the pair (w2, the order of T) and index g.
  int pr, zz, x, w2, g, rbase, xbase;
  bool xact, fact;
  __device__ __forceinline__ XRows(int t) {
    pr = t / (2 * TG);
    const int tt = t % (2 * TG);
    zz = tt / TG;
    x = tt % TG;
    w2 = tt % (2 * AY);
    g = tt / (2 * AY);
    xact = TG == NX || x < NX;
    fact = TG == AY * G || g < G;
    rbase = (2 * pr + zz) * LDSG + x * LD;
    xbase = (2 * pr + (w2 / W) % 2) * LDSG + w2 / (2 * W) * W + w2 % W;
  }
  template <typename F>
  __device__ __forceinline__ void each_row(F f) const {  // f(register, LDS address)
    if (xact) {
#pragma unroll
      for (int k = 0; k < AY; k++) f(k, rbase + k);
    }
  }
  template <int NB, int RAD, int LIM, typename Pos, typename F>
  __device__ __forceinline__ void each_x(Pos pos, F f) const {
    each_el<NB, RAD, LIM, G>(
        g, fact, [&](int i, int j, int k) { f(i, xbase + pos(j, k) * LD); });
  }
  // Forward y pass (radix AY, in registers) and x FFT of the rows in row
  // order, into the pair's chunk of T (at go of tv).
  __device__ __forceinline__ void fwd(cx<R> *v, void *lds, const cx<R> *tw, cx<R> *tv,
                                      unsigned go, bool gact) const {
    dft_x<AY, -1>(v);
    exchange<SPLIT>(
        v, lds, [&](auto f) { each_row(f); },
        [&](auto f) { each_x<NB0, A, B>([](int j, int k) { return j + k * B; }, f); });
    radix_pass<-1, NB0, A, B, G, 0, 0>(v, g, fact, tw);
    exchange<SPLIT>(
        v, lds, [&](auto f) { each_x<NB0, A, B>([](int j, int k) { return j * A + k; }, f); },
        [&](auto f) { each_x<NB1, B, A>([](int j, int k) { return j + k * A; }, f); });
    radix_pass<-1, NB1, B, A, G, 1, A + 1>(v, g, fact, tw);
    unsigned o = (go + g * (2 * AY) + w2) * (unsigned)sizeof(cx<R>);
    forget(tv, o);
    each_el<NB1, B, A, G>(g, fact && gact,
                          [&](int i, int j, int k) { at_bytes(tv + (j - g + k * A) * (2 * AY), o) = v[i]; });
  }
  // Inverse x FFT of the pair's chunk, left in row order, and the inverse y
  // pass: twiddles conj(wy[k jy]), radix AY.
  __device__ __forceinline__ void bwd(cx<R> *v, void *lds, const cx<R> *tw, const cx<R> *tv,
                                      unsigned go, bool gact, const cx<R> *wy, int jy) const {
    const unsigned o = (go + g * (2 * AY) + w2) * (unsigned)sizeof(cx<R>);
    each_el<NB1, B, A, G>(g, fact && gact,
                          [&](int i, int j, int k) { v[i] = at_bytes(tv + (j - g + k * A) * (2 * AY), o); });
    radix_pass<1, NB1, B, A, G, 0, 0>(v, g, fact, tw);
    exchange<SPLIT>(
        v, lds, [&](auto f) { each_x<NB1, B, A>([](int j, int k) { return j * B + k; }, f); },
        [&](auto f) { each_x<NB0, A, B>([](int j, int k) { return j + k * B; }, f); });
    radix_pass<1, NB0, A, B, G, A + 1, 1>(v, g, fact, tw);
    exchange<SPLIT>(
        v, lds, [&](auto f) { each_x<NB0, A, B>([](int j, int k) { return j + k * B; }, f); },
        [&](auto f) { each_row(f); });
#pragma unroll
    for (int k = 1; k < AY; k++) {
      cx<R> y = wy[k * jy];
      y.im = -y.im;
      v[k] = cmul(v[k], y);
    }
    dft_x<AY, 1>(v);
  }
};

// Pairs of row groups of one vector: pi = (z / 2) BY + jy; row k of a group is
// y = jy + k BY.
template <typename R, int NX, int AY>
__global__ void __launch_bounds__((XRows<R, NX, AY>::T), (XRows<R, NX, AY>::WPE))
k_xrows_fwd(VecView<R> in, cx<R> *tb, int npair, int by, long N, const cx<R> *twx) {
  using X = XRows<R, NX, AY>;
  __shared__ __align__(16) char lds[X::LDS];
  __shared__ cx<R> tw[LineTw<NX>::WORDS];
  const X q(threadIdx.x);
  const long vec = blockIdx.y;
  const int pi = (int)blockIdx.x * X::MP + q.pr;
  const bool gact = X::MP == 1 || pi < npair;
  const int z = pi / by * 2 + q.zz, jy = pi % by;
  const unsigned g0 = (unsigned)((z * by * AY + jy) * NX + q.x);
  cx<R> v[X::E];
  auto load = [&](auto form) {
#pragma unroll
    for (int k = 0; k < AY; k++) v[k] = ld_row<form.value>(in, vec, (long)k * by * NX, g0);
  };
  if (q.xact && gact) {
    const int form = view_form(in);
    if (form == VIEW_CX) load(std::integral_constant<int, VIEW_CX>{});
    else if (form == VIEW_PLANES) load(std::integral_constant<int, VIEW_PLANES>{});
    else load(std::integral_constant<int, VIEW_REAL>{});
  }
  LineTw<NX>::load(tw, twx, threadIdx.x, X::T);
  q.fwd(v, lds, tw, tb + vec * N, (unsigned)pi * (2 * AY * NX), gact);
}

// Sums of a workgroup's four partial sums per thread (T threads, 64 or more:
// one whole wave adds them up) in fixed order: part[blk * 4 + q].
template <int T>
__device__ __forceinline__ void block_sum4_any(const double s[4], double *part, long blk,
                                               double *red) {
  static_assert(T >= 64, "one whole wave adds the sums");
  lds_sync();
#pragma unroll
  for (int q = 0; q < 4; q++) red[q * T + threadIdx.x] = s[q];
  lds_sync();
  if (threadIdx.x < 64) {
    const int q = threadIdx.x >> 4, l = threadIdx.x & 15;
    double x = 0.0;
    for (int i = l; i < T; i += 16) x += red[q * T + i];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) x += __shfl_down(x, off, 16);
    if (l == 0) part[blk * 4 + q] = x;
  }
}

// Inverse x rows and y pass of T and the epilogue out = alpha (t + V p) -
// beta p; FWD: then the forward y pass and x rows of out back into T (the next
// Newton step's), SO: with the spin-orbit term of Epi added to out first.
template <typename R, int NX, int AY, bool FWD, bool SO>
__global__ void __launch_bounds__((XRows<R, NX, AY>::T), (XRows<R, NX, AY>::WPE - (SO ? 1 : 0)))
k_xrows_bwd(cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi, int npair, int by, long N,
            const cx<R> *twx, const cx<R> *twy) {
  using X = XRows<R, NX, AY>;
  constexpr int RED = FWD ? 1 : (int)(4 * X::T * sizeof(double));
  __shared__ __align__(16) char lds[X::LDS > RED ? X::LDS : RED];
  __shared__ cx<R> tw[LineTw<NX>::WORDS];
  const X q(threadIdx.x);
  const long vec = blockIdx.y;
  const int pi = (int)blockIdx.x * X::MP + q.pr;
  const bool gact = X::MP == 1 || pi < npair;
  const int z = pi / by * 2 + q.zz, jy = pi % by;
  const unsigned g0 = (unsigned)((z * by * AY + jy) * NX + q.x);
  cx<R> *tv = tb + vec * N;
  const unsigned go = (unsigned)pi * (2 * AY * NX);
  LineTw<NX>::load(tw, twx, threadIdx.x, X::T);
  cx<R> v[X::E];
  q.bwd(v, lds, tw, tv, go, gact, twy, gact ? jy : 0);
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  auto finish = [&](auto form) {
    constexpr int FORM = form.value;
    // psi and V a chunk of rows at a time, so that their registers and the
    // transform's fit the budget
    constexpr int CH = AY > 8 ? 8 : AY;
#pragma unroll
    for (int c = 0; c < AY; c += CH) {
      cx<R> p[CH];
      R V[CH];
#pragma unroll
      for (int k = 0; k < CH; k++) {
        p[k] = ld_row<FORM>(pin, vec, (long)(c + k) * by * NX, g0);
        V[k] = at_bytes(epi.pot + (long)(c + k) * by * NX, g0 * (unsigned)sizeof(R));
      }
#pragma unroll
      for (int k = 0; k < CH; k++) {
        v[c + k] = epilogue(epi, v[c + k], p[k], V[k], s);
        if constexpr (SO) {  // vector v: spinor v / 2, up (v even) or down
          const int u = at_bytes(epi.so_map + (long)(c + k) * by * NX, g0 * 4u);
          if (u >= 0) {
            const double *gq = epi.so_g + ((long)u * epi.so_nsp + (vec >> 1)) * 4 + 2 * (vec & 1);
            v[c + k].re = fma(epi.so_alpha, gq[0], (double)v[c + k].re);
            v[c + k].im = fma(epi.so_alpha, gq[1], (double)v[c + k].im);
          }
        }
        st_row<FORM>(out, vec, (long)(c + k) * by * NX, g0, v[c + k]);
      }
      if constexpr (AY > CH) __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (q.xact && gact) {  // pin and out have one form; FWD: two planes
    const int form = FWD ? (int)VIEW_PLANES : view_form(out);
    if (form == VIEW_PLANES) finish(std::integral_constant<int, VIEW_PLANES>{});
    else if (form == VIEW_CX) finish(std::integral_constant<int, VIEW_CX>{});
    else finish(std::integral_constant<int, VIEW_REAL>{});
  }
  if constexpr (FWD) {
    q.fwd(v, lds, tw, tv, go, gact);
  } else {
    if (epi.part)
      block_sum4_any<X::T>(s, epi.part, vec * gridDim.x + blockIdx.x, reinterpret_cast<double *>(lds));
  }
}

// ---------------------------------------------------------- y, z tiles
template <typename R, int BY, int W, int NZ>
struct TileCfg {
  using PZ = LinePlan<NZ>;
  static constexpr int G = sizeof(R) == 8 ? PZ::GZ64 : PZ::GZ32, A = PZ::A, B = PZ::B;
  static constexpr int L = W * BY;  // z lines of the tile
  static constexpr int T = L * G;
  static_assert(T % (2 * W) == 0, "whole runs of T");
  static constexpr int NB0 = (B + G - 1) / G, NB1 = (A + G - 1) / G;
  static constexpr int RY = (W * NZ + T - 1) / T;  // y butterflies per thread
  static constexpr int E0 = NB0 * A > NB1 * B ? NB0 * A : NB1 * B;
  static constexpr int E = E0 > RY * BY ? E0 : RY * BY;
  // pitch of a z row in LDS: at least L, and an odd multiple of W modulo the
  // elements that one cycle of the LDS serves (W itself where W does not divide
  // them), so that the W-element runs of consecutive z fall on different banks
  static constexpr int pitch(int slots) {
    int p = L;
    while (slots % W == 0 ? p % (2 * W) != W : p % slots != W % slots) p++;
    return p;
  }
  // halves above 36 KB, so that at least four workgroups share a CU: FP64 96^3
  // x 8 vectors (28-element rows) 57 us with two workgroups, 50 now; halving
  // further sizes costs the extra barriers' time (128^3 x 8 FP32 54 -> 55.5)
  static constexpr bool SPLIT =
      sizeof(cx<R>) * NZ * pitch((int)(256 / sizeof(cx<R>))) > 36 * 1024;
  static constexpr size_t ES = SPLIT ? sizeof(R) : sizeof(cx<R>);
  static constexpr int P = pitch((int)(256 / ES));
  static constexpr size_t BUF = (ES * (size_t)NZ * P + 15) / 16 * 16;
  static constexpr size_t LDS = BUF + sizeof(cx<R>) * LineTw<NZ>::WORDS + sizeof(double) * NZ;
  // waves per SIMD the register budget must allow: 16 and more FP64 points a
  // thread spill at 4; 20 FP32 points run better held to 5 (160^3 x 4: 80 ->
  // 73 us; six-residue tiles 31.4 -> 32), 16 spill there (128^3 x 8: 53 -> 67)
  static constexpr int WPE =
      E * sizeof(cx<R>) > 192 ? 3 : sizeof(R) == 4 && E > 16 && W == 4 ? 5 : 4;
};

// pden > 0: the factor is kscale / (kin + pden) instead of kin * kscale.
template <typename R, int BY, int W, int NZ>
__global__ void __launch_bounds__((TileCfg<R, BY, W, NZ>::T), (TileCfg<R, BY, W, NZ>::WPE))
k_tile(cx<R> *tb, long N, int nx, int ay, const cx<R> *twy, const cx<R> *twz, const double *kxx,
       const double *kyy, const double *kzz, double ekin, double kscale, double pden) {
  using C = TileCfg<R, BY, W, NZ>;
  constexpr int G = C::G, A = C::A, B = C::B, L = C::L, P = C::P, T = C::T, RY = C::RY;
  extern __shared__ __align__(16) char smem_t[];
  void *lds = smem_t;
  cx<R> *tw = reinterpret_cast<cx<R> *>(smem_t + C::BUF);
  double *kz_s = reinterpret_cast<double *>(tw + LineTw<NZ>::WORDS);
  const int t = threadIdx.x;
  // tiles of one kx 8 workgroups apart, on one XCD (workgroup b runs on XCD
  // b mod 8): they share 128-byte lines of T where a run is shorter, which
  // that XCD's L2 then reads and writes once (complex64 128^3 x 8: 66 -> 54 us)
  const int nw = ay / W, bi = blockIdx.x, full = nx / 8 * 8 * nw;
  const long vec = blockIdx.y;
  const int x = bi < full ? bi / (8 * nw) * 8 + bi % 8 : bi / nw;
  const int q0 = (bi < full ? bi / 8 % nw : bi % nw) * W;
  cx<R> *base = tb + vec * N + 2 * (x * ay + q0);
  const int sj = 2 * nx * ay, sz = sj * BY;  // strides of jy and z / 2 in T
  cx<R> v[C::E];
  // y order: butterfly t + T r is run element t % (2 W) (z parity, residue) of
  // z pair t / (2 W) + ..., its BY points along jy
  const int w = t % W, zp = t / W % 2, zt = t / (2 * W);
  unsigned o = (unsigned)(zt * sz + t % (2 * W)) * (unsigned)sizeof(cx<R>);
  auto each_y = [&](auto f) {  // f(register, LDS address, uniform offset in T past o)
#pragma unroll
    for (int r = 0; r < RY; r++) {
      if (RY * T == W * NZ || zt + (T / (2 * W)) * r < NZ / 2) {
#pragma unroll
        for (int m = 0; m < BY; m++)
          f(r * BY + m, (2 * zt + zp + (T / W) * r) * P + m * W + w,
            (long)((T / (2 * W)) * r) * sz + (long)m * sj);
      }
    }
  };
  // z passes: line l = w + W m (fastest), G threads each
  const int l = t % L, g = t / L;
  auto z0 = [&](auto f, auto pos) {
    each_el<C::NB0, A, B, G>(g, true, [&](int i, int j, int k) { f(i, pos(j, k) * P + l); });
  };
  auto z1 = [&](auto f, auto pos) {
    each_el<C::NB1, B, A, G>(g, true, [&](int i, int j, int k) { f(i, pos(j, k) * P + l); });
  };
  auto nA = [](int j, int k) { return j + k * B; };
  auto nB = [](int j, int k) { return j + k * A; };
  auto mA = [](int j, int k) { return j * A + k; };
  auto mB = [](int j, int k) { return j * B + k; };
  each_y([&](int i, int, long u) { v[i] = at_bytes(base + u, o); });
  LineTw<NZ>::load(tw, twz, t, T);
  for (int i = t; i < NZ; i += T) kz_s[i] = kzz[i];
  // ---- forward y: twiddles w^(m q), radix BY
#pragma unroll
  for (int r = 0; r < RY; r++) {
#pragma unroll
    for (int m = 1; m < BY; m++) v[r * BY + m] = cmul(v[r * BY + m], twy[m * (q0 + w)]);
    dft_x<BY, -1>(v + r * BY);
  }
  auto ya = [&](auto f) { each_y([&](int i, int a, long) { f(i, a); }); };
  exchange<C::SPLIT>(v, lds, ya, [&](auto f) { z0(f, nA); });
  // ---- forward z, kinetic factor, inverse z
  radix_pass<-1, C::NB0, A, B, G, 0, 0>(v, g, true, tw);
  exchange<C::SPLIT>(v, lds, [&](auto f) { z0(f, mA); }, [&](auto f) { z1(f, nB); });
  const double kxy = kxx[x] + kyy[q0 + l % W + (l / W) * ay];
  // one butterfly at a time through its last forward pass, the factor and its
  // first inverse pass (few registers beyond its B points)
#pragma unroll
  for (int b = 0; b < C::NB1; b++) {
    const int j = g + G * b;
    if (C::NB1 * G == A || j < A) {
      cx<R> *u = v + b * B;
#pragma unroll
      for (int k = 1; k < B; k++) u[k] = cmul(u[k], tw[j + k * (A + 1)]);
      dft_x<B, -1>(u);
      // filter/init.c:138-144 order: (kx + ky) + kz, clamp
      if (pden > 0.0) {
#pragma unroll
        for (int k = 0; k < B; k++) {
          const double kin = fmin(kxy + kz_s[j + k * A], ekin);
          u[k] = cscale(u[k], (R)(kscale / (kin + pden)));
        }
      } else {
#pragma unroll
        for (int k = 0; k < B; k++) {
          const double kin = fmin(kxy + kz_s[j + k * A], ekin);
          u[k] = cscale(u[k], (R)kin);  // kscale = 1 without a preconditioner
        }
      }
      dft_x<B, 1>(u);
    }
    if constexpr (C::NB1 > 1) __builtin_amdgcn_sched_barrier(0);
  }
  exchange<C::SPLIT>(v, lds, [&](auto f) { z1(f, mB); }, [&](auto f) { z0(f, nA); });
  radix_pass<1, C::NB0, A, B, G, A + 1, 1>(v, g, true, tw);
  exchange<C::SPLIT>(v, lds, [&](auto f) { z0(f, nA); }, ya);
  // ---- inverse y: radix BY (its twiddles belong to the row kernel's pass)
#pragma unroll
  for (int r = 0; r < RY; r++) dft_x<BY, 1>(v + r * BY);
  forget(base, o);
  each_y([&](int i, int, long u) { at_bytes(base + u, o) = v[i]; });
}

// ---------------------------------------------------------- dispatch
struct YPlan {
  int ay, by;  // ay = 0: no plan
};
inline YPlan y_plan(int ny) {
  switch (ny) {
#define C(n, a, b) \
  case n:          \
    return {a, b};
    SEP_Y_PLANS(C)
#undef C
  }
  return {0, 0};
}

template <typename R>
struct SplitOps {
  // whether every axis has a plan
  static bool supported(int nx, int ny, int nz);
  static bool rows_fwd(int nx, int ny, int nz, VecView<R> in, cx<R> *tb, int nvec,
                       const cx<R> *twx, hipStream_t st);
  static bool tile(int nx, int ny, int nz, cx<R> *tb, int nvec, const cx<R> *twy, const cx<R> *twz,
                   const double *kxx, const double *kyy, const double *kzz, double ekin,
                   double kscale, double pden, hipStream_t st);
  // fwd_next: with the next step's forward rows
  static bool rows_bwd(int nx, int ny, int nz, cx<R> *tb, VecView<R> pin, VecView<R> out,
                       Epi<R> epi, int nvec, const cx<R> *twx, const cx<R> *twy, bool fwd_next,
                       hipStream_t st, long *nblk);
};

// Definitions of SplitOps<R>, instantiated once per precision
// (sep_split64.hip, sep_split32.hip).
template <typename R>
bool SplitOps<R>::supported(int nx, int ny, int nz) {
  return y_plan(nx).ay > 0 && y_plan(ny).ay > 0 && y_plan(nz).ay > 0;
}

template <typename R, int NX, int AY>
static void xrows_fwd_launch(VecView<R> in, cx<R> *tb, int npair, int by, long N, int nvec,
                             const cx<R> *twx, hipStream_t st) {
  using X = XRows<R, NX, AY>;
  const dim3 grid((unsigned)((npair + X::MP - 1) / X::MP), (unsigned)nvec);
  hipLaunchKernelGGL((k_xrows_fwd<R, NX, AY>), grid, dim3(X::T), 0, st, in, tb, npair, by, N, twx);
}
template <typename R, int NX, int AY>
static bool xrows_bwd_launch(cx<R> *tb, VecView<R> pin, VecView<R> out, Epi<R> epi, int npair,
                             int by, long N, int nvec, const cx<R> *twx, const cx<R> *twy,
                             bool fwd_next, hipStream_t st, long *nblk) {
  using X = XRows<R, NX, AY>;
  const dim3 grid((unsigned)((npair + X::MP - 1) / X::MP), (unsigned)nvec);
  if (nblk) *nblk = (long)grid.x * grid.y;
  if constexpr (sizeof(R) == 8) {
    if (fwd_next && epi.so_map) {
      hipLaunchKernelGGL((k_xrows_bwd<R, NX, AY, true, true>), grid, dim3(X::T), 0, st, tb, pin,
                         out, epi, npair, by, N, twx, twy);
      return true;
    }
  }
  if (epi.so_map) return false;
  if (fwd_next)
    hipLaunchKernelGGL((k_xrows_bwd<R, NX, AY, true, false>), grid, dim3(X::T), 0, st, tb, pin,
                       out, epi, npair, by, N, twx, twy);
  else
    hipLaunchKernelGGL((k_xrows_bwd<R, NX, AY, false, false>), grid, dim3(X::T), 0, st, tb, pin,
                       out, epi, npair, by, N, twx, twy);
  return true;
}

// AY of the y plan, then NX
#define SEP_ROWS_SWITCH(CALL)                                     \
  switch (yp.ay) {                                                \
    case 4: switch (nx) { SEP_SPLIT_LENGTHS(CALL##_4) } break;    \
    case 6: switch (nx) { SEP_SPLIT_LENGTHS(CALL##_6) } break;    \
    case 8: switch (nx) { SEP_SPLIT_LENGTHS(CALL##_8) } break;    \
    case 16: switch (nx) { SEP_SPLIT_LENGTHS(CALL##_16) } break;  \
  }

template <typename R>
bool SplitOps<R>::rows_fwd(int nx, int ny, int nz, VecView<R> in, cx<R> *tb, int nvec,
                           const cx<R> *twx, hipStream_t st) {
  const YPlan yp = y_plan(ny);
  const long N = (long)nx * ny * nz;
  if (nvec == 0) return true;
#define F(n, a)                                                                      \
  case n:                                                                            \
    xrows_fwd_launch<R, n, a>(in, tb, nz / 2 * yp.by, yp.by, N, nvec, twx, st);          \
    return true;
#define F_4(n) F(n, 4)
#define F_6(n) F(n, 6)
#define F_8(n) F(n, 8)
#define F_16(n) F(n, 16)
  SEP_ROWS_SWITCH(F)
#undef F
#undef F_4
#undef F_6
#undef F_8
#undef F_16
  return false;
}

template <typename R>
bool SplitOps<R>::rows_bwd(int nx, int ny, int nz, cx<R> *tb, VecView<R> pin, VecView<R> out,
                           Epi<R> epi, int nvec, const cx<R> *twx, const cx<R> *twy,
                           bool fwd_next, hipStream_t st, long *nblk) {
  const YPlan yp = y_plan(ny);
  const long N = (long)nx * ny * nz;
  if (nvec == 0) return true;
#define F(n, a)                                                                            \
  case n:                                                                                  \
    return xrows_bwd_launch<R, n, a>(tb, pin, out, epi, nz / 2 * yp.by, yp.by, N, nvec, twx, twy, \
                                     fwd_next, st, nblk);
#define F_4(n) F(n, 4)
#define F_6(n) F(n, 6)
#define F_8(n) F(n, 8)
#define F_16(n) F(n, 16)
  SEP_ROWS_SWITCH(F)
#undef F
#undef F_4
#undef F_6
#undef F_8
#undef F_16
  return false;
}
#undef SEP_ROWS_SWITCH

template <typename R, int BY, int W, int NZ>
static void tile_launch(int nx, int ay, cx<R> *tb, long N, int nvec, const cx<R> *twy,
                        const cx<R> *twz, const double *kxx, const double *kyy, const double *kzz,
                        double ekin, double kscale, double pden, hipStream_t st) {
  using C = TileCfg<R, BY, W, NZ>;
  static_assert(C::LDS <= 160 * 1024 && C::T <= 1024, "tile exceeds a gfx950 workgroup");
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute((const void *)k_tile<R, BY, W, NZ>,
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS);
    attr = true;
  }
  if (nvec == 0) return;  // attribute only (before graph capture)
  hipLaunchKernelGGL((k_tile<R, BY, W, NZ>), dim3((unsigned)(nx * (ay / W)), (unsigned)nvec),
                     dim3(C::T), C::LDS, st, tb, N, nx, ay, twy, twz, kxx, kyy, kzz, ekin, kscale,
                     pden);
}

template <typename R>
bool SplitOps<R>::tile(int nx, int ny, int nz, cx<R> *tb, int nvec, const cx<R> *twy,
                       const cx<R> *twz, const double *kxx, const double *kyy, const double *kzz,
                       double ekin, double kscale, double pden, hipStream_t st) {
  const YPlan yp = y_plan(ny);
  const long N = (long)nx * ny * nz;
#define Z(n)                                                                                   \
  case n:                                                                                      \
    tile_launch<R, TB, TW, n>(nx, yp.ay, tb, N, nvec, twy, twz, kxx, kyy, kzz, ekin, kscale, pden, \
                              st);                                                             \
    return true;
#define C(nb, nw)                      \
  if (yp.by == nb && y_width(yp.ay) == nw) { \
    constexpr int TB = nb, TW = nw;    \
    switch (nz) { SEP_SPLIT_LENGTHS(Z) } \
  }
  SEP_Y_TILES(C)
#undef C
#undef Z
  return false;
}

// Grids whose application runs in one kernel (sep_box.hip): all sides 16, or
// in FP32 one of them 24.
template <typename R>
inline bool box_supported(int nx, int ny, int nz) {
  const bool sides = (nx == 16 || nx == 24) && (ny == 16 || ny == 24) && (nz == 16 || nz == 24);
  return sides && (long)nx * ny * nz <= (sizeof(R) == 8 ? 4096 : 6144);
}
// That application; the sums of a vector go to part[4 vec].  false: no such
// form.  nvec == 0: kernel attributes only.
template <typename R>
bool box_apply(const GridDev &gd, const VecView<R> &in, const VecView<R> &out, const Epi<R> &epi,
               int nvec, hipStream_t st);

// compiled in sep_split64.hip and sep_split32.hip
extern template struct SplitOps<double>;
extern template struct SplitOps<float>;

}  // namespace sep
