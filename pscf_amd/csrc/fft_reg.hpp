// Register-resident FP64 line transforms for gfx950.
//
// A line of length N = P*Q is transformed by P threads that each hold Q of
// its points in registers.  Two layouts of a line's points over its threads:
//   layout A: thread t holds a[r]     = x[t + P r],                r < Q
//   layout B: thread t holds b[u][k2] = x[(t + P u) + Q k2],  k2 < P,
//             for the rounds u with t + P u < Q (U = ceil(Q/P) rounds)
// line_fwd (A -> B) and line_inv (B -> A) each compute an unnormalised DFT
// of sign S (X[k] = sum_n x[n] e^{S 2 pi i n k / N}) with one exchange of the
// line through LDS:
//   line_fwd: DFT_Q over r in registers, twiddle w_N^{S t k1}, exchange,
//             DFT_P over t (n = t + P r, k = k1 + Q k2);
//   line_inv: DFT_P over k2 in registers, twiddle w_N^{S n1 k1}, exchange,
//             DFT_Q over k1 (k = k1 + Q k2, n = n1 + P n2).
// Both are the two-factor Cooley-Tukey decomposition; a transform of data in
// layout A ends in layout B and vice versa, so a chain of transforms and
// pointwise products never reshuffles its data.  Twiddles come from the
// per-length table tw[m] = exp(-2 pi i m / N) (conjugated for S = +1).
//
// Exchange buffers: element i of a line's exchange order is stored at
// E[eoff(i)], where the caller picks the layout for its lane mapping.  With
// WAVE (default) the P threads of a line are lanes of one wavefront and the
// exchange synchronises only that wavefront; otherwise the workgroup.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_lds.hpp"

namespace pscf {

template <int S> struct Dft<1, S> {
  static __device__ __forceinline__ void run(double2*) {}
};

// 6 = 2 x 3 (prime-factor algorithm, no twiddles): n = (3 n1 + 2 n2) mod 6,
// k = (3 k1 + 4 k2) mod 6, DFT_3 over n2 then DFT_2 over n1.
template <int S> struct Dft<6, S> {
  static __device__ __forceinline__ void run(double2* v) {
    double2 a0[3] = {v[0], v[2], v[4]};   // n1 = 0: n = 2 n2
    double2 a1[3] = {v[3], v[5], v[1]};   // n1 = 1: n = 3 + 2 n2 (mod 6)
    Dft<3, S>::run(a0);
    Dft<3, S>::run(a1);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) {
      const double2 p = cadd(a0[k2], a1[k2]), m = csub(a0[k2], a1[k2]);
      v[(4 * k2) % 6] = p;          // k1 = 0
      v[(3 + 4 * k2) % 6] = m;      // k1 = 1
    }
  }
};

// 10 = 2 x 5 (prime-factor): n = (5 n1 + 2 n2) mod 10, k = (5 k1 + 6 k2) mod 10.
template <int S> struct Dft<10, S> {
  static __device__ __forceinline__ void run(double2* v) {
    double2 a0[5], a1[5];
#pragma unroll
    for (int n2 = 0; n2 < 5; ++n2) {
      a0[n2] = v[(2 * n2) % 10];
      a1[n2] = v[(5 + 2 * n2) % 10];
    }
    Dft<5, S>::run(a0);
    Dft<5, S>::run(a1);
#pragma unroll
    for (int k2 = 0; k2 < 5; ++k2) {
      v[(6 * k2) % 10] = cadd(a0[k2], a1[k2]);
      v[(5 + 6 * k2) % 10] = csub(a0[k2], a1[k2]);
    }
  }
};

// 12 = 3 x 4 (prime-factor): n = (4 n1 + 3 n2) mod 12, k = (4 k1 + 9 k2) mod 12,
// DFT_4 over n2 then DFT_3 over n1.
template <int S> struct Dft<12, S> {
  static __device__ __forceinline__ void run(double2* v) {
    double2 a[3][4];
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) {
#pragma unroll
      for (int n2 = 0; n2 < 4; ++n2) a[n1][n2] = v[(4 * n1 + 3 * n2) % 12];
      Dft<4, S>::run(a[n1]);
    }
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) {
      double2 c[3] = {a[0][k2], a[1][k2], a[2][k2]};
      Dft<3, S>::run(c);
#pragma unroll
      for (int k1 = 0; k1 < 3; ++k1) v[(4 * k1 + 9 * k2) % 12] = c[k1];
    }
  }
};

// 16 = 4 x 4 (Cooley-Tukey): n = 4 n1 + n2, k = k1 + 4 k2,
// X[k1 + 4 k2] = sum_n2 w4^{n2 k2} w16^{n2 k1} sum_n1 x[4 n1 + n2] w4^{n1 k1}.
template <int S> __device__ __forceinline__ double2 rot(double2 a, double c, double s) {
  return make_double2(mad(a.x, c, -(S * s) * a.y), mad(a.y, c, (S * s) * a.x));   // a e^{S i theta}
}
template <int S> struct Dft<16, S> {
  static __device__ __forceinline__ void run(double2* v) {
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;  // cos, sin pi/8
    constexpr double h = 0.70710678118654752440;
    double2 a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) a[n2][n1] = v[4 * n1 + n2];
      Dft<4, S>::run(a[n2]);                       // a[n2][k1]
    }
    a[1][1] = rot<S>(a[1][1], c1, s1);             // w16^1
    a[1][2] = rot<S>(a[1][2], h, h);               // w16^2
    a[1][3] = rot<S>(a[1][3], s1, c1);             // w16^3
    a[2][1] = rot<S>(a[2][1], h, h);               // w16^2
    a[2][2] = cmul_si<S>(a[2][2]);                 // w16^4
    a[2][3] = rot<S>(a[2][3], -h, h);              // w16^6
    a[3][1] = rot<S>(a[3][1], s1, c1);             // w16^3
    a[3][2] = rot<S>(a[3][2], -h, h);              // w16^6
    a[3][3] = rot<S>(a[3][3], -c1, -s1);           // w16^9
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      double2 c[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
      Dft<4, S>::run(c);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = c[k2];
    }
  }
};

// ------------------------------------------------------------- line plans
struct LinePlan {
  int p, q;
};
// lengths with a register DFT (Dft<n>)
constexpr bool dft_ok(int n) {
  return n == 1 || n == 2 || n == 3 || n == 4 || n == 5 || n == 6 || n == 7 || n == 8 ||
         n == 10 || n == 12 || n == 16;
}
// Candidate factorisations N = P*Q of a supported length, P threads per line
// holding Q points each; variant 0 is the default.  Variants past a length's
// list fall back to the default.
constexpr LinePlan line_alt(int n, int v) {
  int ps[6] = {0, 0, 0, 0, 0, 0};
  switch (n) {
    case 1: ps[0] = 1; break;
    case 8: ps[0] = 2; ps[1] = 4; break;
    case 12: ps[0] = 3; ps[1] = 4; ps[2] = 2; ps[3] = 6; break;
    case 16: ps[0] = 4; ps[1] = 2; ps[2] = 8; break;
    case 20: ps[0] = 4; ps[1] = 5; ps[2] = 2; ps[3] = 10; break;
    case 24: ps[0] = 3; ps[1] = 8; ps[2] = 4; ps[3] = 6; ps[4] = 2; ps[5] = 12; break;
    case 28: ps[0] = 4; ps[1] = 7; break;
    case 32: ps[0] = 4; ps[1] = 8; ps[2] = 2; ps[3] = 16; break;
    case 40: ps[0] = 5; ps[1] = 8; ps[2] = 4; ps[3] = 10; break;
    case 48: ps[0] = 6; ps[1] = 8; ps[2] = 4; ps[3] = 12; ps[4] = 3; ps[5] = 16; break;
    case 56: ps[0] = 7; ps[1] = 8; break;
    case 64: ps[0] = 8; ps[1] = 4; ps[2] = 16; break;
    case 96: ps[0] = 8; ps[1] = 12; ps[2] = 6; ps[3] = 16; break;
    case 128: ps[0] = 8; break;          // 16 x 8 needs 65 x 16 > 1024 y-role threads
    default: return {0, 0};
  }
  const int p = (v >= 0 && v < 6 && ps[v] > 0) ? ps[v] : ps[0];
  return {p, n / p};
}
// threads per line P and points per thread Q of each supported length: the
// tuned factorisation (tuned.hpp lp), PSCF_LPV's variant in tuning builds,
// else the default
constexpr LinePlan line_plan(int n) {
#ifdef PSCF_LPV
  return line_alt(n, PSCF_LPV);
#else
  const int p = plan_for(n).lp;
  if (p > 0 && n % p == 0 && dft_ok(p) && dft_ok(n / p)) return {p, n / p};
  return line_alt(n, 0);
#endif
}

constexpr int pow2ceil(int n) {
  int p = 1;
  while (p < n) p *= 2;
  return p;
}

// A line of N points on PP threads (default: the length's plan).
template <int LEN, int PP = line_plan(LEN).p> struct Line {
  static constexpr int N = LEN;
  static constexpr int P = PP;
  static constexpr int Q = N / P;
  static_assert(P > 0 && P * Q == N && dft_ok(P) && dft_ok(Q), "no register line plan for this length");
  static constexpr int U = (Q + P - 1) / P;       // rounds of layout B
  // every thread holds a point set in every round of layout B (P divides
  // Q); otherwise only the threads t + P u < Q do (all of t < Q when P > Q)
  static constexpr bool FULLB = Q % P == 0;
  // lanes reserved per line: a power of two, so that the P threads of a
  // line always sit in one wavefront (lanes P..PS-1 of a slot idle)
  static constexpr int PS = pow2ceil(P);
  static_assert(PS <= 64, "a line must fit in one wavefront");
  // index of layout-B point (u, k2) of thread t, and whether t holds round u
  static __device__ __forceinline__ int at(int t, int u, int k2) { return t + P * u + Q * k2; }
  static __device__ __forceinline__ bool has(int t, int u) { return FULLB || t + P * u < Q; }
};

// The threads of a line are lanes of one wavefront, which execute in
// lockstep and see their own LDS accesses in order: the exchange of a line
// needs only a wavefront-scope fence (no workgroup barrier), so the waves of
// a workgroup run their lines' LDS and arithmetic phases independently.
// Called by every thread of the workgroup (inactive ones too).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the value of lane ^ 8: a DPP rotation by half a row of 16 lanes, no LDS.
// Called by every lane of the wavefront.
__device__ __forceinline__ double lane_swap(double v) {
#ifdef __HIP_DEVICE_COMPILE__
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x128, 0xF, 0xF, true);          // row_ror:8
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x128, 0xF, 0xF, true);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
#else
  return __shfl_xor(v, 8, 64);
#endif
}
__device__ __forceinline__ double2 lane_swap(double2 v) { return make_double2(lane_swap(v.x), lane_swap(v.y)); }

template <int S> __device__ __forceinline__ double2 twid(const double2* tw, int m) {
  double2 w = tw[m];
  if (S > 0) w.y = -w.y;
  return w;
}

// The twiddles of a line's two transforms, w_N^{t k1} (line_fwd) and
// w_N^{n1 (t + P u)} (line_inv), read from a table in LDS:
template <class L> struct TwTable {
  const double2* tw;
  template <int S> __device__ __forceinline__ double2 f(int t, int k1) const {
    return twid<S>(tw, (t * k1) % L::N);
  }
  template <int S> __device__ __forceinline__ double2 i(int t, int u, int n1) const {
    return twid<S>(tw, (n1 * (t + L::P * u)) % L::N);
  }
};
// or held in registers by the thread (a thread's t never changes), which
// frees a line transform of a third of its LDS reads.  INV: line_inv's too.
// COUNT complex values.
template <class L, bool INV> struct TwRegs {
  static constexpr int P = L::P, Q = L::Q, U = L::U;
  static constexpr bool SHARED = P == Q;      // both transforms use the same values
  static constexpr bool OWN = INV && !SHARED;
  static constexpr int COUNT = Q - 1 + (OWN ? U * (P - 1) : 0);
  double2 wf[Q], wi[OWN ? U : 1][OWN ? P : 1];
  __device__ __forceinline__ void load(const double2* __restrict__ g, int t) {
#pragma unroll
    for (int k1 = 1; k1 < Q; ++k1) wf[k1] = g[(t * k1) % L::N];
    if constexpr (OWN) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int n1 = 1; n1 < P; ++n1) wi[u][n1] = g[(n1 * (t + P * u)) % L::N];
    }
  }
  template <int S> __device__ __forceinline__ double2 f(int, int k1) const { return twid<S>(wf, k1); }
  template <int S> __device__ __forceinline__ double2 i(int, int u, int n1) const {
    if constexpr (SHARED) return twid<S>(wf, n1);
    else return twid<S>(wi[u], n1);
  }
};

template <bool WAVE> __device__ __forceinline__ void line_sync() {
  if constexpr (WAVE) wave_sync();
  else __syncthreads();
}

// The two transforms for M lines per thread at once.
//
// Layout A -> layout B, DFT of sign S.  eoff(m, i): exchange slot of element
// i of line m (i = k1 P + t on write, (t + P u) P + tt on read); a line's
// slots are its own, so only its threads touch them.  The caller separates
// other uses of the same LDS words by workgroup barriers.
template <class L, int S, int M, bool WAVE = true, class EOff, class Tw>
__device__ __forceinline__ void line_fwd(double2 (&a)[M][L::Q], double2 (&b)[M][L::U][L::P], double2* E,
                                         EOff eoff, int t, const Tw& tw, bool active) {
  constexpr int P = L::P, Q = L::Q, U = L::U;
  if constexpr (P == 1) {           // one thread per line: no exchange
    if (active) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        Dft<Q, S>::run(a[m]);
#pragma unroll
        for (int k1 = 0; k1 < Q; ++k1) b[m][k1][0] = a[m][k1];
      }
    }
    return;
  }
  line_sync<WAVE>();                // the lines' earlier reads of their slots are done
  if (active) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      Dft<Q, S>::run(a[m]);
#pragma unroll
      for (int k1 = 1; k1 < Q; ++k1) a[m][k1] = cmul(a[m][k1], tw.template f<S>(t, k1));
#pragma unroll
      for (int k1 = 0; k1 < Q; ++k1) E[eoff(m, k1 * P + t)] = a[m][k1];
    }
  }
  line_sync<WAVE>();
  if (active) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (L::has(t, u)) {
          const int k1 = t + P * u;
#pragma unroll
          for (int tt = 0; tt < P; ++tt) b[m][u][tt] = E[eoff(m, k1 * P + tt)];
          Dft<P, S>::run(b[m][u]);
        }
  }
}

// Layout B -> layout A, DFT of sign S.  eoff(m, i): exchange slot of element
// i of line m (i = n1 Q + k1 on write, t Q + k1 on read); slots as in line_fwd.
template <class L, int S, int M, bool WAVE = true, class EOff, class Tw>
__device__ __forceinline__ void line_inv(double2 (&b)[M][L::U][L::P], double2 (&a)[M][L::Q], double2* E,
                                         EOff eoff, int t, const Tw& tw, bool active) {
  constexpr int P = L::P, Q = L::Q, U = L::U;
  if constexpr (P == 1) {
    if (active) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
#pragma unroll
        for (int k1 = 0; k1 < Q; ++k1) a[m][k1] = b[m][k1][0];
        Dft<Q, S>::run(a[m]);
      }
    }
    return;
  }
  line_sync<WAVE>();
  if (active) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (L::has(t, u)) {
          const int k1 = t + P * u;
          Dft<P, S>::run(b[m][u]);
#pragma unroll
          for (int n1 = 0; n1 < P; ++n1) {
            double2 v = b[m][u][n1];
            if (Q > 1 && n1 > 0) v = cmul(v, tw.template i<S>(t, u, n1));
            E[eoff(m, n1 * Q + k1)] = v;
          }
        }
  }
  line_sync<WAVE>();
  if (active) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
#pragma unroll
      for (int k1 = 0; k1 < Q; ++k1) a[m][k1] = E[eoff(m, t * Q + k1)];
      Dft<Q, S>::run(a[m]);
    }
  }
}

}  // namespace pscf
