// LDS-resident FP64 FFT building blocks for gfx950.
//
// Lines of length N (N = 2^a 3^b 5^c 7^d) are transformed in place in LDS by a
// mixed-radix Stockham schedule (radix 8, then 4, 2, 3, 5, 7).  Each pass loads
// every butterfly's inputs into registers, synchronises the workgroup, then
// writes the outputs to their Stockham positions, so a pass needs no second
// buffer.  Sign convention: SIGN = -1 is the forward transform
// X[k] = sum_n x[n] e^{-2 pi i k n / N}, SIGN = +1 the inverse; both are
// unnormalised, matching the FFTW calls of the reference (src/fft3_mod.f90:85-122).
//
// Twiddles come from a per-length table tw[m] = exp(-2 pi i m / N), m < N,
// built on the host; SIGN = +1 uses its conjugate.
#pragma once
#include <hip/hip_runtime.h>

#include "tuned.hpp"

namespace pscf {

// ---------------------------------------------------------------- complex ops
// a b + c, rounded once on the device.  Where two products are added it is
// written out which one is fused: kernels that must agree bit for bit (one
// system alone, many in one launch) may not leave that to the compiler.  Host
// code (the CPU emulation of the kernels) rounds twice rather than call the C
// library.
__device__ __forceinline__ double mad(double a, double b, double c) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_fma(a, b, c);
#else
  return a * b + c;
#endif
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(mad(a.x, b.x, -(a.y * b.y)), mad(a.x, b.y, a.y * b.x));
}
// a * b + c
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
  return make_double2(mad(a.x, b.x, mad(-a.y, b.y, c.x)), mad(a.x, b.y, mad(a.y, b.x, c.y)));
}
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
// multiply by s*i, s = +-1
template <int S> __device__ __forceinline__ double2 cmul_si(double2 a) {
  return S > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// ------------------------------------------------------ compile-time factoring
// Per-length kernel plan: the tuned table (tuned.hpp) or, for lengths it does
// not list, radix 8, no padding, separate plane buffers, k_step_a's
// workgroups per plane chosen at launch, the default register-line
// factorisation and 128 lanes per z workgroup.  PSCF_MAX_RADIX, PSCF_XPAD,
// PSCF_ALIAS, PSCF_AJOBS and PSCF_ZLANES, when defined, override the plan for
// every length (the variants the autotuner builds and times; PSCF_LPV, the
// line factorisation, is in fft_reg.hpp).
constexpr TunedPlan plan_for(int n) {
  for (const TunedPlan& p : kTunedPlans)
    if (p.n == n) return p;
  return TunedPlan{n, 8, 0, 0, 0, 0, 128};
}
constexpr int plan_ajobs(int n) {
#ifdef PSCF_AJOBS
  return PSCF_AJOBS;
#else
  return plan_for(n).ajobs;
#endif
}
constexpr int plan_alias(int n) {
#ifdef PSCF_ALIAS
  return PSCF_ALIAS;
#else
  return plan_for(n).alias;
#endif
}
constexpr int plan_max_radix(int n) {
#ifdef PSCF_MAX_RADIX
  return PSCF_MAX_RADIX;
#else
  return plan_for(n).max_radix;
#endif
}
constexpr int plan_xpad(int n) {
#ifdef PSCF_XPAD
  return PSCF_XPAD;
#else
  return plan_for(n).xpad;
#endif
}
constexpr int plan_zl(int n) {
#ifdef PSCF_ZLANES
  return PSCF_ZLANES;
#else
  return plan_for(n).zl;
#endif
}
constexpr int fft_nfac(int n) {
  int c = 0;
  const bool r8 = plan_max_radix(n) >= 8;
  while (r8 && n > 1 && n % 8 == 0) { n /= 8; ++c; }
  while (n % 4 == 0) { n /= 4; ++c; }
  while (n % 2 == 0) { n /= 2; ++c; }
  while (n % 3 == 0) { n /= 3; ++c; }
  while (n % 5 == 0) { n /= 5; ++c; }
  while (n % 7 == 0) { n /= 7; ++c; }
  return n == 1 ? c : -1;
}
constexpr int fft_fac(int n, int p) {
  int c = 0;
  const bool r8 = plan_max_radix(n) >= 8;
  while (r8 && n > 1 && n % 8 == 0) { if (c == p) return 8; n /= 8; ++c; }
  while (n % 4 == 0) { if (c == p) return 4; n /= 4; ++c; }
  while (n % 2 == 0) { if (c == p) return 2; n /= 2; ++c; }
  while (n % 3 == 0) { if (c == p) return 3; n /= 3; ++c; }
  while (n % 5 == 0) { if (c == p) return 5; n /= 5; ++c; }
  while (n % 7 == 0) { if (c == p) return 7; n /= 7; ++c; }
  return 0;
}

// ------------------------------------------------------------ radix kernels
template <int R, int S> struct Dft;

template <int S> struct Dft<2, S> {
  static __device__ __forceinline__ void run(double2* v) {
    double2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};

template <int S> struct Dft<4, S> {
  static __device__ __forceinline__ void run(double2* v) {
    double2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    double2 t2 = cadd(v[1], v[3]), t3 = cmul_si<S>(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
  }
};

template <int S> struct Dft<8, S> {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr double h = 0.70710678118654752440;  // 1/sqrt(2)
    double2 e[4] = {v[0], v[2], v[4], v[6]};
    double2 o[4] = {v[1], v[3], v[5], v[7]};
    Dft<4, S>::run(e);
    Dft<4, S>::run(o);
    // o[q] *= w8^q, w8 = (1 + S i)/sqrt(2)
    double2 o1 = make_double2(h * (o[1].x - S * o[1].y), h * (o[1].y + S * o[1].x));
    double2 o2 = cmul_si<S>(o[2]);
    double2 o3 = make_double2(h * (-o[3].x - S * o[3].y), h * (-o[3].y + S * o[3].x));
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);
    v[7] = csub(e[3], o3);
  }
};

template <int S> struct Dft<3, S> {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr double r3 = 0.86602540378443864676;  // sqrt(3)/2
    double2 t = cadd(v[1], v[2]);
    double2 d = csub(v[1], v[2]);
    double2 m = make_double2(v[0].x - 0.5 * t.x, v[0].y - 0.5 * t.y);
    double2 sd = cmul_si<S>(cscale(d, r3));
    v[0] = cadd(v[0], t);
    v[1] = cadd(m, sd);
    v[2] = csub(m, sd);
  }
};

template <int S> struct Dft<5, S> {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    double2 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
    double2 d1 = csub(v[1], v[4]), d2 = csub(v[2], v[3]);
    double2 a1 = make_double2(v[0].x + c1 * t1.x + c2 * t2.x, v[0].y + c1 * t1.y + c2 * t2.y);
    double2 a2 = make_double2(v[0].x + c2 * t1.x + c1 * t2.x, v[0].y + c2 * t1.y + c1 * t2.y);
    double2 b1 = make_double2(mad(s1, d1.x, s2 * d2.x), mad(s1, d1.y, s2 * d2.y));
    double2 b2 = make_double2(mad(s2, d1.x, -s1 * d2.x), mad(s2, d1.y, -s1 * d2.y));
    double2 ib1 = cmul_si<S>(b1), ib2 = cmul_si<S>(b2);
    v[0] = cadd(v[0], cadd(t1, t2));
    v[1] = cadd(a1, ib1);
    v[4] = csub(a1, ib1);
    v[2] = cadd(a2, ib2);
    v[3] = csub(a2, ib2);
  }
};

// 7: X_k = x0 + sum_m cos(2 pi k m/7) t_m + S i sum_m sin(2 pi k m/7) d_m with
// t_m = x_m + x_{7-m}, d_m = x_m - x_{7-m} (m = 1..3); X_{7-k} takes -S.
template <int S> struct Dft<7, S> {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr double c1 = 0.62348980185873353053, c2 = -0.22252093395631440429;
    constexpr double c3 = -0.90096886790241912624;
    constexpr double s1 = 0.78183148246802980871, s2 = 0.97492791218182360702;
    constexpr double s3 = 0.43388373911755812048;
    const double2 t1 = cadd(v[1], v[6]), t2 = cadd(v[2], v[5]), t3 = cadd(v[3], v[4]);
    const double2 d1 = csub(v[1], v[6]), d2 = csub(v[2], v[5]), d3 = csub(v[3], v[4]);
    const double2 x0 = v[0];
    auto lin = [](double2 a, double ca, double2 b, double cb, double2 c, double cc) {
      return make_double2(mad(cc, c.x, mad(cb, b.x, ca * a.x)), mad(cc, c.y, mad(cb, b.y, ca * a.y)));
    };
    const double2 a1 = cadd(x0, lin(t1, c1, t2, c2, t3, c3));
    const double2 a2 = cadd(x0, lin(t1, c2, t2, c3, t3, c1));
    const double2 a3 = cadd(x0, lin(t1, c3, t2, c1, t3, c2));
    const double2 b1 = cmul_si<S>(lin(d1, s1, d2, s2, d3, s3));
    const double2 b2 = cmul_si<S>(lin(d1, s2, d2, -s3, d3, -s1));
    const double2 b3 = cmul_si<S>(lin(d1, s3, d2, -s1, d3, s2));
    v[0] = cadd(x0, cadd(t1, cadd(t2, t3)));
    v[1] = cadd(a1, b1);
    v[6] = csub(a1, b1);
    v[2] = cadd(a2, b2);
    v[5] = csub(a2, b2);
    v[3] = cadd(a3, b3);
    v[4] = csub(a3, b3);
  }
};

// ----------------------------------------------------------- Stockham pass
// LINES lines of length N in `buf`; element n of line l sits at
// buf[l*LS + n*ES].  JFAST selects the thread mapping: consecutive threads
// take consecutive butterflies of one line (rows, ES == 1) or the same
// butterfly of consecutive lines (columns, LS == 1), so LDS addresses of a
// wavefront are consecutive either way.
template <int N, int R, int NS, int SIGN, int LINES, int LS, int ES, bool JFAST, int NT>
__device__ __forceinline__ void stockham_pass(double2* buf, const double2* __restrict__ tw, int tid) {
  constexpr int NB = N / R;
  constexpr int TOT = LINES * NB;
  constexpr int PER = (TOT + NT - 1) / NT;
  constexpr int TSTEP = N / (NS * R);
  double2 v[PER][R];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int bf = tid + p * NT;
    if (bf < TOT) {
      const int j = JFAST ? bf % NB : bf / LINES;
      const int line = JFAST ? bf / NB : bf % LINES;
      const double2* base = buf + line * LS;
#pragma unroll
      for (int r = 0; r < R; ++r) v[p][r] = base[(j + r * NB) * ES];
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int bf = tid + p * NT;
    if (bf < TOT) {
      const int j = JFAST ? bf % NB : bf / LINES;
      const int line = JFAST ? bf / NB : bf % LINES;
      const int k = j % NS;
      if (NS > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          double2 w = tw[k * r * TSTEP];
          if (SIGN > 0) w.y = -w.y;
          v[p][r] = cmul(v[p][r], w);
        }
      }
      Dft<R, SIGN>::run(v[p]);
      double2* base = buf + line * LS;
      const int idx = (j / NS) * NS * R + k;
#pragma unroll
      for (int q = 0; q < R; ++q) base[(idx + q * NS) * ES] = v[p][q];
    }
  }
  __syncthreads();
}

template <int N, int P, int NS, int SIGN, int LINES, int LS, int ES, bool JFAST, int NT>
__device__ __forceinline__ void fft_passes(double2* buf, const double2* __restrict__ tw, int tid) {
  if constexpr (P < fft_nfac(N)) {
    constexpr int R = fft_fac(N, P);
    stockham_pass<N, R, NS, SIGN, LINES, LS, ES, JFAST, NT>(buf, tw, tid);
    fft_passes<N, P + 1, NS * R, SIGN, LINES, LS, ES, JFAST, NT>(buf, tw, tid);
  }
}

// In-place FFT of LINES lines of length N in LDS (a no-op for N == 1).
template <int N, int SIGN, int LINES, int LS, int ES, bool JFAST, int NT>
__device__ __forceinline__ void fft_lines(double2* buf, const double2* __restrict__ tw, int tid) {
  static_assert(fft_nfac(N) >= 0, "FFT length must be 2^a 3^b 5^c 7^d");
  fft_passes<N, 0, 1, SIGN, LINES, LS, ES, JFAST, NT>(buf, tw, tid);
}

// ----------------------------------------------------------- plane helpers
// A real plane of N1 x N2 points (x fastest) is packed two rows per complex
// line: P[pl*N1 + x] = row(2 pl)[x] + i row(2 pl + 1)[x] (the odd partner of
// an odd last row is 0).  After the forward x-transform each pair is split
// into the two half spectra (k = 0..N1/2) of a half plane
// H[y*(N1/2+1) + k]; the inverse rebuilds the pairs from the Hermitian
// extension, using only the real parts at k = 0 and k = N1/2 as a c2r
// transform does.
template <int N1, int N2> struct Plane {
  static constexpr int N1H = N1 / 2 + 1;
  static constexpr int NP = (N2 + 1) / 2;        // packed row pairs
  static constexpr int PLS = N1 + plan_xpad(N1);  // LDS stride of a packed row
  static constexpr int PSIZE = PLS * NP;         // complex words in P
  static constexpr int HSIZE = N1H * N2;         // complex words in H
  static constexpr bool XJFAST = plan_xpad(N1) == 0;  // thread mapping of the x passes
  // P and H share one LDS buffer (the plan's choice, or forced where the two
  // would not fit the 160 KB of a CU together, as from 128 x 128 planes on)
  static constexpr bool ALIAS = plan_alias(N1) != 0 || (PSIZE + HSIZE) * 16 > 120 * 1024;
  static constexpr int USIZE = ALIAS ? (PSIZE > HSIZE ? PSIZE : HSIZE) : PSIZE + HSIZE;
  static_assert(N1 % 2 == 0, "first grid dimension must be even");
  // LDS index of element x of packed row pl, given i = pl*N1 + x
  static __device__ __forceinline__ int pidx(int i) { return (i / N1) * PLS + i % N1; }
  static __device__ __forceinline__ double2* Pbuf(double2* U) { return U; }
  static __device__ __forceinline__ double2* Hbuf(double2* U) { return ALIAS ? U : U + PSIZE; }
};

// P (x-transformed pairs) -> H (half rows)
template <int N1, int N2, int NT>
__device__ __forceinline__ void split_pairs(const double2* P, double2* H, int tid) {
  using PL = Plane<N1, N2>;
  constexpr int TOT = PL::NP * PL::N1H;
  constexpr int PER = (TOT + NT - 1) / NT;
  double2 z[PER], zc[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = tid + p * NT;
    if (i < TOT) {
      const int pl = i / PL::N1H, k = i % PL::N1H;
      z[p] = P[pl * PL::PLS + k];
      zc[p] = cconj(P[pl * PL::PLS + (N1 - k) % N1]);
    }
  }
  if (PL::ALIAS) __syncthreads();                           // H overwrites P
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = tid + p * NT;
    if (i < TOT) {
      const int pl = i / PL::N1H, k = i % PL::N1H;
      H[(2 * pl) * PL::N1H + k] = make_double2(0.5 * (z[p].x + zc[p].x), 0.5 * (z[p].y + zc[p].y));
      if (2 * pl + 1 < N2) {
        const double2 d = csub(z[p], zc[p]);               // (z - zc) / (2i)
        H[(2 * pl + 1) * PL::N1H + k] = make_double2(0.5 * d.y, -0.5 * d.x);
      }
    }
  }
  __syncthreads();
}

// H (half rows, after the inverse y-transform) -> P (pairs ready for the inverse x-transform)
template <int N1, int N2, int NT>
__device__ __forceinline__ void join_pairs(const double2* H, double2* P, int tid) {
  using PL = Plane<N1, N2>;
  constexpr int TOT = PL::NP * N1;
  constexpr int PER = (TOT + NT - 1) / NT;
  double2 v[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = tid + p * NT;
    if (i < TOT) {
      const int pl = i / N1, x = i % N1;
      const bool hi = x > N1 / 2;
      const int k = hi ? N1 - x : x;
      double2 a = H[(2 * pl) * PL::N1H + k];
      double2 b = (2 * pl + 1 < N2) ? H[(2 * pl + 1) * PL::N1H + k] : make_double2(0.0, 0.0);
      if (k == 0 || k == N1 / 2) { a.y = 0.0; b.y = 0.0; }
      if (hi) { a.y = -a.y; b.y = -b.y; }
      v[p] = make_double2(a.x - b.y, a.y + b.x);           // a + i b
    }
  }
  if (PL::ALIAS) __syncthreads();                           // P overwrites H
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = tid + p * NT;
    if (i < TOT) P[(i / N1) * PL::PLS + i % N1] = v[p];
  }
  __syncthreads();
}

// Forward r2c of the plane held in P (pairs, already filled): x then y.
template <int N1, int N2, int NT>
__device__ __forceinline__ void plane_forward(double2* P, double2* H, const double2* tw1,
                                              const double2* tw2, int tid) {
  using PL = Plane<N1, N2>;
  fft_lines<N1, -1, PL::NP, PL::PLS, 1, PL::XJFAST, NT>(P, tw1, tid);
  split_pairs<N1, N2, NT>(P, H, tid);
  fft_lines<N2, -1, PL::N1H, 1, PL::N1H, false, NT>(H, tw2, tid);
}

// Inverse c2r of the half plane held in H: y then x; result pairs in P.
template <int N1, int N2, int NT>
__device__ __forceinline__ void plane_inverse(double2* H, double2* P, const double2* tw1,
                                              const double2* tw2, int tid) {
  using PL = Plane<N1, N2>;
  fft_lines<N2, +1, PL::N1H, 1, PL::N1H, false, NT>(H, tw2, tid);
  join_pairs<N1, N2, NT>(H, P, tid);
  fft_lines<N1, +1, PL::NP, PL::PLS, 1, PL::XJFAST, NT>(P, tw1, tid);
}

}  // namespace pscf
