// gfx950 kernels of the SCFT inner loop (FP64).
//
// Data layout in HBM follows the reference's Fortran arrays (x fastest):
//   real grid      r(x, y, z)            at x + N1*(y + N2*z)             M  = N1*N2*N3
//   half spectrum  k(kx, ky, kz), kx<=N1/2 at kx + N1H*(ky + N2*kz)       Mk = N1H*N2*N3
//   contour slab   q(:, s), s = 0..Ns    at s*M (one slab per chain and direction)
// A 3D transform is one XY-plane pass (x and y transforms in LDS, one workgroup
// per z plane) and one Z-column pass.  The pointwise factors of the contour
// step are fused into those passes, and the z forward transform, the
// reciprocal-space factor and the z inverse transform of one sub-step share a
// single pass.  The sweeps' own fields and spectra have the packed-row layout
// (below, at StepPlane); what enters and leaves them has the layout above.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fft_lds.hpp"
#include "fft_reg.hpp"

namespace pscf {

constexpr int MAXBLK = 16;     // blocks per chain

// Workgroup size of a kernel: enough threads for every butterfly of the first
// (radix-8) transform pass to run at once -- e.g. 33 half-spectrum lines of
// 64 points have 264 radix-8 butterflies, so 320 threads rather than 256,
// which would leave one wave doing a second butterfly alone in every pass.
constexpr int round64(int n) { return ((n + 63) / 64) * 64; }
constexpr int clampnt(int n) { return n < 64 ? 64 : (n > 1024 ? 1024 : n); }
constexpr int plane_nt(int n1, int n2) {
  const int x = ((n2 + 1) / 2) * (n1 / fft_fac(n1, 0));
  const int y = n2 > 1 ? (n1 / 2 + 1) * (n2 / fft_fac(n2, 0)) : 0;
  return clampnt(round64(x > y ? x : y));
}
constexpr int zcol_nt(int w, int n3) { return n3 > 1 ? clampnt(round64(w * (n3 / fft_fac(n3, 0)))) : 64; }
constexpr int c2c_nt(int n1, int n2) {
  const int x = n2 * (n1 / fft_fac(n1, 0));
  const int y = n2 > 1 ? n1 * (n2 / fft_fac(n2, 0)) : 0;
  return clampnt(round64(x > y ? x : y));
}

// One contour sweep (a chain's q or q-dagger) advanced by the step kernels.
// Step j maps contour index in(j) -> out(j): forward in = j, backward
// in = ns - j.  The step interval [lo, lo+1] (lo = min(in, out)) belongs to
// block b with bnd[b] <= lo < bnd[b+1].  A task takes the steps
// jbeg <= j < jend of its sweep, step j during the launch with index
// j - jofs; its first step reads its input from `start` (if set) or from its
// slab.  Contour point s lives at slab + slot(s)*M, slot(s) = pmap[s] (pmap
// set; -1: the point is not stored) or s.
struct StepTask {
  // What every step kernel reads, within the first cache lines: one scalar
  // load latency lies between a launch and its first global load.
  double* slab;                 // stored contour points
  const double* fac;            // propagator factors of the blocks (task_e1 ... task_k2)
  double2* A;                   // full-step spectrum        (Mk)
  double2* B;                   // first half-step spectrum  (Mk)
  double2* C;                   // second half-step spectrum (Mk)
  double* q1;                   // full-step result          (M)
  const int* pmap;              // contour point -> slot of slab (length ns+1), or null
  const double* start;          // input of step jbeg (M), or null
  long fm, fk;                  // points of a block's e1 and e2 (M) and of its k1 and k2 (z_factors)
  int ns;
  int jofs, jbeg, jend;         // launch offset and active step window
  int dir;                      // +1 forward sweep, -1 backward sweep
  int init_one;                 // 1: the first point is the constant 1 (and is written)
  int skip;                     // 1: inactive (converged instance of a batch): every kernel returns
  int rev;                      // 1: step j is the step j' = ns-1-j (adjoint recomputation)
  int reload;                   // 1: every step reads its input from the slab (no carry)
  int add_src;                  // 1: adjoint sweep, out = T in + g(out), g computed in place
  int src_end;                  // contour point that also receives scal[1] (-1: none)
  int nostore;                  // 1: step outputs are not written to the slab
  int sym;                      // symmetric planes (sym_planes), 0: every plane is stored
  int nblk;
  int bnd[MAXBLK + 1];          // block starts; entries past nblk hold ns
  // adjoint support: pre-factor fields of the step kept for the gradient,
  // U = C1[e1 q], V = C2[e2 q], W = C2[e1 V] (C: normalised convolutions)
  double* keepA;                // step inputs, two buffers by step parity (2 M)
  double* keepU;
  double* keepV;
  double* keepW;
  double2* keepK[3];            // spectra FFT[e1 q], FFT[e2 q], FFT[e1 V] (Mk, before the k factor)
  // adjoint sources g(s) = scal[0] sum_b (ds_b/3) w_b(s) lam_b oth(s) [+ scal[1] at src_end],
  // w_b: Simpson weights of block b (1 at its ends, 4 odd, 2 even interior points)
  const double* oth;            // the other sweep's q points
  const int* omap;              // their slots (as pmap), or null
  const double* lam[MAXBLK];    // dL/drho of each block's monomer (M)
  const double* scal;           // coefficient, end term
  double ds[MAXBLK];            // block step sizes (adjoint gradient)
  double bsq[MAXBLK];           // squared statistical segment length of the block's monomer
  double* grad[MAXBLK];         // omega gradient of the block (M)
  double* kgrad[MAXBLK];        // |k|^2 gradient of the block on the half grid (Mk)
};

// Propagator factors of block b, stored per block as e1, e2, k1, k2:
// exp(-ds/2 w) and exp(-ds/4 w) (fm points each), exp(-ds b^2 |k|^2 / 6) and
// exp(-ds b^2 |k|^2 / 12) (fk each), these times the transforms' scale: 1/M,
// and 1/2 for packed rows (their transforms scale by M/2, k_step_z's split and
// merge by 4).
__device__ __forceinline__ const double* task_e1(const StepTask& t, int b) {
  return t.fac + b * (2 * t.fm + 2 * t.fk);
}
__device__ __forceinline__ const double* task_e2(const StepTask& t, int b) { return task_e1(t, b) + t.fm; }
__device__ __forceinline__ const double* task_k1(const StepTask& t, int b) { return task_e1(t, b) + 2 * t.fm; }
__device__ __forceinline__ const double* task_k2(const StepTask& t, int b) {
  return task_e1(t, b) + 2 * t.fm + t.fk;
}

__device__ __forceinline__ int task_slot(const StepTask& t, int sp) { return t.pmap ? t.pmap[sp] : sp; }
__device__ __forceinline__ int task_j(const StepTask& t, int j) { return t.rev ? t.ns - 1 - j : j; }
__device__ __forceinline__ int task_in(const StepTask& t, int j) {
  j = task_j(t, j);
  return t.dir > 0 ? j : t.ns - j;
}
__device__ __forceinline__ int task_out(const StepTask& t, int j) {
  j = task_j(t, j);
  return t.dir > 0 ? j + 1 : t.ns - j - 1;
}
__device__ __forceinline__ int task_block(const StepTask& t, int j) {
  j = task_j(t, j);
  const int lo = t.dir > 0 ? j : t.ns - j - 1;
  // the first four blocks without a chain of dependent loads (lo < ns, so the
  // entries past nblk never count)
  int b = (lo >= t.bnd[1]) + (lo >= t.bnd[2]) + (lo >= t.bnd[3]);
  if (t.nblk > 4)
    while (b + 1 < t.nblk && lo >= t.bnd[b + 1]) ++b;
  return b;
}

// x / c, rounded as the division: one Newton step on the residual of
// x * (1/c) (Markstein); r is 1/c rounded.  Three FMAs where a division is a
// chain of ten FP64 instructions.
__device__ __forceinline__ double div_by(double x, double c, double r) {
#ifdef __HIP_DEVICE_COMPILE__
  const double q = x * r;
  const double e = mad(-c, q, x);
  return e == e ? mad(e, r, q) : q;       // x infinite or NaN: q is the quotient
#else
  (void)r;
  return x / c;
#endif
}

// Copy n complex words global -> LDS (no barrier).
template <int N, int NT>
__device__ __forceinline__ void stage(double2* dst, const double2* __restrict__ src, int tid) {
#pragma unroll
  for (int p = 0; p < (N + NT - 1) / NT; ++p) {
    const int i = tid + p * NT;
    if (i < N) dst[i] = src[i];
  }
}

template <int N, int NT>
__device__ __forceinline__ void stage_tw(double2* dst, const double2* __restrict__ src, int tid) {
  for (int i = tid; i < N; i += NT) dst[i] = src[i];
}
constexpr int imax(int a, int b) { return a > b ? a : b; }

// ----------------------------------------------------------------------------
// Packed rows.  The contour sweeps hold a real plane of N1 x N2 points as NL =
// N2/2 complex rows, row l = grid row 2l + i (grid row 2l+1), interleaved in
// memory: grid point (x, 2l + h) at 2 (x + N1 (l + NL z)) + h (N2 = 1: one row,
// no partner).  All fields of a sweep (q, e1, e2, q1, kept fields) have this
// layout; it loads 16 bytes per lane.  A plane's transform is the complex
// transform of the packed rows, C(kx, l), N1 x NL: it needs no split of the
// pairs, no extra Nyquist column, and its rows are whole cache lines.  With
// ky = l or l + NL and w = exp(-2 pi i / N2), the real plane's spectrum F is
//   E = (C(kx,l) + C*(-kx,-l))/2,  O = (C(kx,l) - C*(-kx,-l))/(2i),
//   F(kx, l) = E + w^l O,   F(kx, l+NL) = E - w^l O,
// linear at every z, so only the z kernel splits and merges, where it applies
// the reciprocal-space factor.
// ----------------------------------------------------------------------------
// ----------------------------------------------------------------------------
// Symmetric planes.  The fields of a space group whose operations map z to
// +-z + c and (x, y) to +-(x, y) + tau determine all planes from the first NP:
// for an operation (x,y,z) -> (a (x,y) + tau, s z + c), a and s = +-1,
//   f(x, y, s z + c) = f(a ((x,y) - tau), z),  and for the plane spectra
//   F(k, s z + c) = (-1)^{2 k tau} F(a k, z),  F(-k, z) = conj F(k, z)
// (tau and c are 0 or half an edge).  The sweeps then store and transform the
// first NP planes only -- N3/4 + 1 of them where the group has both z -> -z
// and z -> z + N3/2, as every body-centred centrosymmetric group has -- and the
// z kernel makes the whole column from them.  Code of a system (0: none):
//   bit 0: z -> -z (R); bit 1: z -> z + N3/2 (T); then three bits each for T
//   (2), R (5) and T R (8): a = -1, tau_x = N1/2, tau_y = N2/2.
// ----------------------------------------------------------------------------
constexpr int SYM_R = 1, SYM_T = 2;
__host__ __device__ __forceinline__ int sym_planes(int sym, int n3) {
  const int l = (sym & SYM_T) ? n3 / 2 : n3;
  return (sym & SYM_R) ? l / 2 + 1 : l;
}
// plane z: its stored plane u, and the three bits of the operation from u to z
__host__ __device__ __forceinline__ int sym_source(int sym, int n3, int z, int& u) {
  const int l = (sym & SYM_T) ? n3 / 2 : n3;
  int q = 0;
  if ((sym & SYM_T) && z >= l) {
    q = 1;
    z -= l;
  }
  const bool r = (sym & SYM_R) && 2 * z > l;
  u = r ? l - z : z;
  // z = l (q + 1) - u: T R where l (q + 1) is half the edge, R where it is 0
  const int op = r ? ((sym & SYM_T) && q == 0 ? 8 : 5) : (q ? 2 : -1);
  return op < 0 ? 0 : (sym >> op) & 7;
}
// how many planes a stored plane stands for
__host__ __device__ __forceinline__ int sym_weight(int sym, int n3, int u) {
  const int np = sym_planes(sym, n3);
  return ((sym & SYM_T) ? 2 : 1) * ((sym & SYM_R) && u != 0 && u != np - 1 ? 2 : 1);
}
// the point of a plane that operation `op` takes to (x, y)
__host__ __device__ __forceinline__ int sym_in_plane(int op, int n1, int n2, int x, int y) {
  if (op & 2) x = x >= n1 / 2 ? x - n1 / 2 : x + n1 / 2;
  if (op & 4) y = y >= n2 / 2 ? y - n2 / 2 : y + n2 / 2;
  if (op & 1) {
    x = x ? n1 - x : 0;
    y = y ? n2 - y : 0;
  }
  return x + n1 * y;
}
// grid index of the stored point with the value of grid point g (planes n1 x n2)
__host__ __device__ __forceinline__ long sym_point(int sym, int n1, int n2, int n3, long g) {
  int u;
  const int op = sym_source(sym, n3, (int)(g / ((long)n1 * n2)), u);
  return sym_in_plane(op, n1, n2, (int)(g % n1), (int)(g / n1 % n2)) + (long)n1 * n2 * u;
}
// a point that the symmetry gives the value of grid point g, so that a field
// is symmetric if all these pairs are equal: the stored point, or on the first
// and last stored plane, which z -> -z maps onto themselves, the image there;
// g itself on the others
__host__ __device__ __forceinline__ long sym_partner(int sym, int n1, int n2, int n3, long g) {
  const int z = (int)(g / ((long)n1 * n2)), np = sym_planes(sym, n3);
  if (z >= np) return sym_point(sym, n1, n2, n3, g);
  if (!(sym & SYM_R) || (z != 0 && z != np - 1)) return g;
  const int op = sym >> (z != 0 && (sym & SYM_T) ? 8 : 5) & 7;
  return sym_in_plane(op, n1, n2, (int)(g % n1), (int)(g / n1 % n2)) + (long)n1 * n2 * z;
}
// flip the sign of v where bit 31 of m is set
__device__ __forceinline__ double sign_flip(double v, int m) {
  return __builtin_bit_cast(double, __builtin_bit_cast(long long, v) ^ ((long long)(m & 0x80000000) << 32));
}

// 16-byte accesses at a uniform base plus a 32-bit byte offset (scalar base,
// immediate steps: no 64-bit address arithmetic per lane and point)
__device__ __forceinline__ double2 ld16(const void* base, unsigned off) {
  return *reinterpret_cast<const double2*>(static_cast<const char*>(base) + off);
}
__device__ __forceinline__ void st16(void* base, unsigned off, double2 v) {
  *reinterpret_cast<double2*>(static_cast<char*>(base) + off) = v;
}
// packed index -> grid index
__host__ __device__ __forceinline__ long unpack_index(long i, int n1, int n2) {
  if (n2 == 1) return i;
  const int h = (int)(i & 1);
  const long p = i >> 1;
  const int nl = n2 / 2;
  const long x = p % n1, row = p / n1;            // row = l + NL z
  return x + n1 * (2 * (row % nl) + h + n2 * (row / nl));
}
// grid index -> packed index
__host__ __device__ __forceinline__ long pack_index(long g, int n1, int n2) {
  if (n2 == 1) return g;
  const long x = g % n1, yz = g / n1;
  const int nl = n2 / 2, y = (int)(yz % n2);
  return 2 * (x + n1 * (y / 2 + nl * (yz / n2))) + (y & 1);
}
// Columns are stored in groups of eight, four kx and their four -kx (half a
// cache line each); kx = 0 and N1/2, which are their own partners, share a
// place.  Position of column kx in a row:
__host__ __device__ __forceinline__ constexpr int col_pos(int kx, int n1) {
  const bool neg = 2 * kx >= n1;
  const int p = 2 * kx == n1 ? 0 : (neg ? n1 - kx : kx);
  const int left = n1 / 2 - p / 4 * 4;
  return p / 4 * 8 + (neg ? (left < 4 ? left : 4) : 0) + p % 4;
}

// The z kernels' column slots.  A slot is the pair of packed columns (kx, l)
// and (-kx, -l), kx <= N1/2: words o[0] and o[1] of a plane, from which the
// spectrum's columns ky = l and l + NL are split.  A tile of zw slots (one
// workgroup) is zw/2 pairs of columns of rows l and -l (or 0 and NL/2, their
// own partners): whole groups of storage columns, so whole cache lines, which
// no other tile touches.  Eight slots are four kx of row l, then of row -l.
// At kx = 0 and N1/2 slots l and -l are one; the tiles' first pair has one of
// each, and a last tile the kx = N1/2 of rows 0 and NL/2.
struct ZSlot {
  int kx, l, o[2];
  bool ok;
};
__host__ __device__ __forceinline__ int z_tiles(int n1, int nl, int zw) {
  return (n1 / 2 + zw / 2 - 1) / (zw / 2) * (nl > 1 ? nl / 2 : 1) + 1;
}
__host__ __device__ __forceinline__ ZSlot z_slot(int tile, int c, int n1, int nl, int zw) {
  const int kp = zw / 2, ntx = (n1 / 2 + kp - 1) / kp, nlp = nl > 1 ? nl / 2 : 1;
  const int i = c / 8 * 4 + c % 4, sg = c / 4 % 2;
  const bool last = tile == ntx * nlp;
  const int lp = last ? 0 : tile / ntx, p = last ? i : tile % ntx * kp + i;
  ZSlot s;
  s.l = lp == 0 ? (sg ? nl / 2 : 0) : (sg ? nl - lp : lp);
  s.ok = p < n1 / 2 && (sg == 0 || nl > 1) && (!last || i == 0);
  s.kx = p;
  if (last || (p == 0 && lp > 0 && sg)) {
    s.kx = n1 / 2;
    if (lp > 0) s.l = lp;
  }
  s.o[0] = s.l * n1 + col_pos(s.kx, n1);
  s.o[1] = (s.l ? nl - s.l : 0) * n1 + col_pos(s.kx ? n1 - s.kx : 0, n1);
  return s;
}
// Lanes of a tile: 16 for eight slots, first their o[0] and ky = l (h = 0),
// then their o[1] and ky = l + NL (h = 1), so that four lanes share 64 bytes.
__host__ __device__ __forceinline__ int z_lane_slot(int lane) { return lane / 16 * 8 + lane % 8; }
__host__ __device__ __forceinline__ int z_lane_h(int lane) { return lane / 8 % 2; }
// Reciprocal-space factors in the lanes' order, (kz tiles + tile) 2 zw + lane
// (N2 = 1: both h alike).  -> half-grid index, or -1 where the slot is empty
__host__ __device__ __forceinline__ long z_factors(int n1, int n2, int n3, int zw) {
  return (long)n3 * z_tiles(n1, n2 > 1 ? n2 / 2 : 1, zw) * 2 * zw;
}
__host__ __device__ __forceinline__ long unpack_kindex(long i, int n1, int n2, int zw) {
  const int nl = n2 > 1 ? n2 / 2 : 1, tiles = z_tiles(n1, nl, zw);
  const int lane = (int)(i % (2 * zw));
  const long row = i / (2 * zw);
  const ZSlot s = z_slot((int)(row % tiles), z_lane_slot(lane), n1, nl, zw);
  if (!s.ok) return -1;
  const int h = n2 > 1 ? z_lane_h(lane) : 0;
  return s.kx + (n1 / 2 + 1) * (s.l + h * nl + n2 * (row / tiles));
}

// ... and back, for one plane (N3 = 1): the place of the factor of column kx
// (any kx < N1) at ky = l + h NL.  |k| of k and -k are one, so a column kx >
// N1/2 takes the factor of (-kx, -ky), and of the columns kx = 0 and N1/2 one
// of l and -l is held.
__host__ __device__ __forceinline__ int z_factor_at(int kx, int l, int h, int n1, int nl, int zw) {
  const int kp = zw / 2, ntx = (n1 / 2 + kp - 1) / kp, nlp = nl > 1 ? nl / 2 : 1;
  const bool edge = kx == 0 || 2 * kx == n1;
  if (edge ? 2 * l > nl : 2 * kx > n1) {           // -> (-kx, -ky)
    kx = edge ? kx : n1 - kx;
    if (l) {
      l = nl - l;
      h = 1 - h;
    }
  }
  int lp = 0, sg = 0, p = kx;
  if (nl > 1) {
    if (l == 0 || 2 * l == nl) {
      sg = l != 0;
    } else {
      sg = 2 * l > nl;
      lp = sg ? nl - l : l;
    }
  }
  int tile = lp * ntx + p / kp;
  if (2 * kx == n1) {                              // the last tile, or beside kx = 0
    p = 0;
    tile = lp ? lp * ntx : ntx * nlp;
    if (lp) sg = 1;
  }
  const int i = p % kp, c = i / 4 * 8 + sg * 4 + i % 4;
  return tile * 2 * zw + c / 8 * 16 + h * 8 + c % 8;
}

// Words between the planes of a packed spectrum: an odd multiple of 16 (256
// bytes), so that a z column's values go to all memory channels in turn.  At
// 64^3 whole rows alone are 32 KB per plane, one channel for a whole column:
// k_step_z 14.8 instead of 7.0 us.
constexpr int plane_words(int n1, int nl) { return ((n1 * nl + 15) / 16 | 1) * 16; }

// lanes per y line: the factorisation of NL whose workgroup (N1 columns) is
// nearest the x role's, so that both roles use all threads; ties to fewer lanes
constexpr int y_lanes(int n1, int nl, int ntx) {
  int best = 0, cost = 1 << 30;
  for (int p = 1; p <= 16; ++p) {
    if (nl % p || !dft_ok(p) || !dft_ok(nl / p)) continue;
    const int nt = n1 * pow2ceil(p);
    if (nt > 1024) continue;
    const int c = nt > ntx ? nt - ntx : ntx - nt;
    if (c < cost) {
      cost = c;
      best = p;
    }
  }
  return best;
}

// An XY plane on one workgroup.  x role: the threads of packed row l (Line<N1>,
// layout A over x), consecutive lanes; y role: the threads of column kx (a
// line of NL), CW columns per wavefront, consecutive columns on consecutive
// lanes.  In both roles a line's threads are lanes of one wavefront (a
// power-of-two slot per line), so its exchange needs no workgroup barrier, and
// global and LDS accesses are contiguous over lanes.
// The spectra pass between the roles through the plane buffer PL.
//   forward: x role layout A over x   -> y role layout B over l
//   inverse: y role layout A over l   -> x role layout A over x
// LDS: exchange buffer E and plane buffer PL (one shared buffer, with more
// barriers, where both together would exceed LDSCAP: the default leaves room
// for two workgroups per CU, the stress transform's for four at 64 x 64).
// YINV: the kernel also takes the y lines from layout B to A (line_inv).
template <int N1, int N2, int LDSCAP = 80 * 1024, bool FEWREGS = false, bool YINV = false> struct StepPlane {
  static constexpr bool ROWS = N2 > 1;
  static constexpr int NL = ROWS ? N2 / 2 : 1;
  using LX = Line<N1>;
  using LY = Line<NL, y_lanes(N1, NL, NL * LX::PS)>;
  static constexpr int PX = LX::P, QX = LX::Q, UX = LX::U, SX = LX::PS;
  static constexpr int PY = LY::P, QY = LY::Q, UY = LY::U, SY = LY::PS;
  static constexpr int CW = 64 / SY;
  static constexpr int NTX = NL * SX, NTY = (N1 + CW - 1) / CW * 64;
  static constexpr int NT = clampnt(round64(imax(NTX, NTY)));
  // x exchange slots: per line, contiguous, one padding word every G words
  // (G = min(P, Q)) so that the strided half of the exchange is free of LDS
  // bank conflicts; y exchange slots: an odd stride between columns
  static constexpr int GX = PX < QX ? PX : QX;
  static constexpr int EXW = N1 + N1 / GX + 1;
  static constexpr int EYW = NL | 1;
  static constexpr int ESIZE = imax(NL * EXW, PY > 1 || YINV ? N1 * EYW : 1);
  static constexpr int PLS = N1;                    // row stride in PL
  static constexpr int PSIZE = NL * PLS;
  static constexpr bool ALIAS = (ESIZE + PSIZE + N1 + NL) * 16 > LDSCAP;
  static constexpr int EBUF = ALIAS ? imax(ESIZE, PSIZE) : ESIZE;
  static constexpr int PBUF = ALIAS ? 1 : PSIZE;
  static constexpr size_t LDS = sizeof(double2) * (EBUF + PBUF + N1 + NL);   // at most
  // Twiddles in registers where they are few and the kernel has registers
  // left (FEWREGS: it has not; a smaller LDSCAP is for launches whose
  // workgroups share a CU, where registers decide how many fit)
  static constexpr bool TWREG =
      !FEWREGS && LDSCAP >= 80 * 1024 && TwRegs<LX, true>::COUNT <= 12 &&
      (YINV ? !ROWS || TwRegs<LX, true>::COUNT + TwRegs<LY, YINV>::COUNT <= 16 : TwRegs<LY, false>::COUNT <= 8);
  using TwX = std::conditional_t<TWREG, TwRegs<LX, true>, TwTable<LX>>;
  using TwY = std::conditional_t<TWREG, TwRegs<LY, YINV>, TwTable<LY>>;
  static constexpr int TWN = TWREG ? 1 : N1 + NL;   // LDS words of the tables
  static_assert(N1 % 2 == 0, "the first grid dimension must be even");
  static_assert(N2 == 1 || N2 % 4 == 0, "the second grid dimension must be 1 or a multiple of 4");
  static_assert(NTX <= 1024 && NTY <= 1024, "plane too large for one workgroup");

  struct Roles {
    int xl, xt, yk, yt, yp;           // yp: storage position of column yk
    bool xact, yact;
    __device__ explicit Roles(int tid)
        : xl(tid / SX), xt(tid % SX), yk(tid / 64 * CW + tid % CW), yt(tid % 64 / CW),
          yp(col_pos(yk, N1)), xact(xl < NL && xt < PX), yact(yk < N1 && yt < PY) {}
    __device__ int ey(int i) const { return yk * EYW + i; }
    __device__ int ex(int i) const { return xl * EXW + i + i / GX; }
  };

  struct Tw {
    TwX x;
    TwY y;
    // registers from the global tables (lengths N1 and NL), or the tables
    // into LDS (T, TWN words; sync() publishes them)
    __device__ __forceinline__ void load(const double2* __restrict__ g1, const double2* __restrict__ gl,
                                         double2* T, const Roles& R, int tid) {
      if constexpr (TWREG) {
        x.load(g1, R.xt);
        y.load(gl, R.yt);
      } else {
        stage_tw<N1, NT>(T, g1, tid);
        stage_tw<NL, NT>(T + N1, gl, tid);
        x.tw = T;
        y.tw = T + N1;
      }
    }
    static __device__ __forceinline__ void sync() {
      if constexpr (!TWREG) __syncthreads();
    }
  };

  // x-role point r of a thread: packed row pair (ROWS) or single value of a
  // field whose plane starts at `base`
  static __device__ __forceinline__ double2 get(const double* __restrict__ base, const Roles& R, int r) {
    const unsigned o = R.xl * N1 + R.xt;
    if constexpr (ROWS) return ld16(base, o * 16 + PX * r * 16);
    else return make_double2(base[o + PX * r], 0.0);
  }
  static __device__ __forceinline__ void put(double* __restrict__ base, const Roles& R, int r, double2 v) {
    const unsigned o = R.xl * N1 + R.xt;
    if constexpr (ROWS) st16(base, o * 16 + PX * r * 16, v);
    else base[o + PX * r] = v.x;
  }
  static __device__ __forceinline__ void get_all(const double* __restrict__ base, const Roles& R,
                                                 double2 (&v)[QX]) {
#pragma unroll
    for (int r = 0; r < QX; ++r) v[r] = get(base, R, r);
  }

  // the y role's spectrum values (layout A over l) of the plane at base
  static __device__ __forceinline__ void load_cols(const double2* __restrict__ base, double2 (&c)[1][QY],
                                                   const Roles& R) {
    if (!R.yact) return;
#pragma unroll
    for (int r = 0; r < QY; ++r) c[0][r] = ld16(base, unsigned(R.yt * N1 + R.yp) * 16 + PY * r * N1 * 16);
  }
  // the y role's spectrum values (layout B over l) into the plane at base
  static __device__ __forceinline__ void store_cols(double2* __restrict__ base,
                                                    const double2 (&h)[1][UY][PY], const Roles& R) {
    if (!R.yact) return;
#pragma unroll
    for (int u = 0; u < UY; ++u)
      if (LY::has(R.yt, u)) {
#pragma unroll
        for (int k2 = 0; k2 < PY; ++k2) st16(base, unsigned(R.yt * N1 + R.yp) * 16 + (PY * u + QY * k2) * N1 * 16, h[0][u][k2]);
      }
  }

  // packed rows a (x role, layout A) -> spectrum h (y role, layout B over l)
  static __device__ __forceinline__ void fwd(double2 (&a)[1][QX], double2 (&h)[1][UY][PY], double2* E,
                                             double2* PL, const Tw& tw, const Roles& R) {
    double2 b[1][UX][PX];
    line_fwd<LX, -1, 1>(a, b, E, [&](int, int i) { return R.ex(i); }, R.xt, tw.x, R.xact);
    if (ALIAS) __syncthreads();
    if (R.xact) {
#pragma unroll
      for (int u = 0; u < UX; ++u)
        if (LX::has(R.xt, u)) {
#pragma unroll
          for (int k2 = 0; k2 < PX; ++k2) PL[R.xl * PLS + LX::at(R.xt, u, k2)] = b[0][u][k2];
        }
    }
    __syncthreads();
    double2 c[1][QY];
    if (R.yact) {
#pragma unroll
      for (int r = 0; r < QY; ++r) c[0][r] = PL[(R.yt + PY * r) * PLS + R.yk];
    }
    if (ALIAS) __syncthreads();
    line_fwd<LY, -1, 1>(c, h, E, [&](int, int i) { return R.ey(i); }, R.yt, tw.y, R.yact);
  }

  // spectrum c (y role, layout A over l, from load_cols) -> packed rows a (x
  // role, layout A), in two stages: inv_y (y transforms into PL) and inv_x
  static __device__ __forceinline__ void inv_y(double2 (&c)[1][QY], double2* E, double2* PL, const Tw& tw,
                                               const Roles& R) {
    double2 h[1][UY][PY];
    line_fwd<LY, +1, 1>(c, h, E, [&](int, int i) { return R.ey(i); }, R.yt, tw.y, R.yact);
    if (ALIAS) __syncthreads();
    if (R.yact) {
#pragma unroll
      for (int u = 0; u < UY; ++u)
        if (LY::has(R.yt, u)) {
#pragma unroll
          for (int k2 = 0; k2 < PY; ++k2) PL[LY::at(R.yt, u, k2) * PLS + R.yk] = h[0][u][k2];
        }
    }
    __syncthreads();
  }
  static __device__ __forceinline__ void inv_x(double2 (&a)[1][QX], double2* E, double2* PL, const Tw& tw,
                                               const Roles& R) {
    double2 b[1][UX][PX];
    if (R.xact) {
#pragma unroll
      for (int u = 0; u < UX; ++u)
        if (LX::has(R.xt, u)) {
#pragma unroll
          for (int k2 = 0; k2 < PX; ++k2) b[0][u][k2] = PL[R.xl * PLS + LX::at(R.xt, u, k2)];
        }
    }
    if (ALIAS) __syncthreads();
    line_inv<LX, +1, 1>(b, a, E, [&](int, int i) { return R.ex(i); }, R.xt, tw.x, R.xact);
  }

  // v[r] += the adjoint source at contour point sp (see StepTask)
  static __device__ __forceinline__ void add_source(const StepTask& t, int sp, long M, long pbase,
                                                    const Roles& R, double2 (&v)[QX]) {
    double2 s[QX];
#pragma unroll
    for (int r = 0; r < QX; ++r) s[r] = make_double2(0.0, 0.0);
    for (int b = 0; b < t.nblk; ++b) {
      const int lo = t.bnd[b], hi = t.bnd[b + 1];
      if (sp < lo || sp > hi) continue;
      const double w = t.ds[b] / 3.0 * ((sp == lo || sp == hi) ? 1.0 : (((sp - lo) & 1) ? 4.0 : 2.0));
      const double* lam = t.lam[b] + pbase;
#pragma unroll
      for (int r = 0; r < QX; ++r) {
        const double2 l = get(lam, R, r);
        s[r].x += w * l.x;
        s[r].y += w * l.y;
      }
    }
    const double* oth = t.oth + (long)(t.omap ? t.omap[sp] : sp) * M + pbase;
    const double c = t.scal[0], end = sp == t.src_end ? t.scal[1] : 0.0;
#pragma unroll
    for (int r = 0; r < QX; ++r) {
      const double2 o = get(oth, R, r);
      v[r].x += c * s[r].x * o.x + end;
      v[r].y += c * s[r].y * o.y + end;
    }
  }
};

// ----------------------------------------------------------------------------
// Step kernel A (ONEJOB false: two workgroups per z plane and sweep; true: one
// workgroup does both jobs, one inverse transform fewer).  Both finish step
// j-1: x,y inverse transform of the second half step's spectrum C, times
// exp(-ds w/4), Richardson q = (4 q2 - q1)/3 (job 0 stores it to the slab).
// Then step j starts: job 0 transforms exp(-ds w/2) q into A, job 1
// exp(-ds w/4) q into B.  Reference: src/step_mod.f90:156-174.
// ADJ: with what adjoint and recomputed sweeps need besides (reload, sources,
// kept fields), which would only cost the plain sweeps code and scalar loads.
// Every global input is requested at kernel entry, the start factors after
// the y stage (their registers are free then).
// ----------------------------------------------------------------------------
template <int N1, int N2, bool ONEJOB, bool ADJ>
__global__ void __launch_bounds__((StepPlane<N1, N2>::NT)) k_step_a(const StepTask* __restrict__ tasks, int jl,
                                                               const double2* __restrict__ tw1g,
                                                               const double2* __restrict__ twlg) {
  using SP = StepPlane<N1, N2, 80 * 1024, ONEJOB || ADJ>;
  constexpr int QX = SP::QX, QY = SP::QY, PY = SP::PY, UY = SP::UY;
  __shared__ double2 TWS[SP::TWN];
  __shared__ double2 EB[SP::EBUF];
  __shared__ double2 PB[SP::PBUF];
  double2* const E = EB;
  double2* const PL = SP::ALIAS ? EB : PB;
  const int tid = threadIdx.x, z = blockIdx.x, job = ONEJOB ? 0 : blockIdx.z;
  const StepTask& t = tasks[blockIdx.y];
  const int j = jl + t.jofs;
  if (t.skip || j < t.jbeg || j > t.jend || (job == 1 && j == t.jend)) return;
  const typename SP::Roles R(tid);
  const long M = t.fm;
  const double i3 = 1.0 / 3.0;
  const long pbase = (long)z * N1 * N2;
  const long hbase = (long)z * plane_words(N1, SP::NL);
  const bool start = j < t.jend;
  const bool first = j == t.jbeg;
  typename SP::Tw tw;
  tw.load(tw1g, twlg, TWS, R, tid);
  double2 c[1][QY];
  if (!first) SP::load_cols(t.C + hbase, c, R);
  // factors: e2 of step j-1 (finish) with q1, loaded at entry; the start
  // factors of step j (e1 for job 0, e2 for job 1) after the y stage of the
  // inverse transform.  Job 1 (and ONEJOB's second start) reuse the finish e2
  // when steps j-1 and j share a block.
  const int bj = start ? task_block(t, j) : 0;
  const int bp = first ? -1 : task_block(t, j - 1);
  const bool reuse = !first && bp == bj;
  const int s_out = first ? 0 : task_out(t, j - 1);
  const int so = first || (ADJ && (t.nostore || !t.slab)) ? -1 : task_slot(t, s_out);
  double2 q[QX], e2[QX], q1[QX];
#pragma unroll
  for (int r = 0; r < QX; ++r) q[r] = e2[r] = q1[r] = make_double2(0.0, 0.0);
  if (R.xact && !first) {
    SP::get_all(task_e2(t, bp) + pbase, R, e2);
    SP::get_all(t.q1 + pbase, R, q1);
  }
  // start factors: f (e1 for job 0, e2 for job 1), g (ONEJOB: e2)
  double2 f[QX], g[ONEJOB ? QX : 1];
  const auto load_start = [&] {
    if (!start || !R.xact) {
#pragma unroll
      for (int r = 0; r < QX; ++r) {
        f[r] = make_double2(0.0, 0.0);
        if constexpr (ONEJOB) g[r] = f[r];
      }
      return;
    }
    const double* fe2 = task_e2(t, bj) + pbase;
    const double* fe1 = task_e1(t, bj) + pbase;
    if (job == 1 && reuse) {
#pragma unroll
      for (int r = 0; r < QX; ++r) f[r] = e2[r];
    } else {
      SP::get_all(job == 1 ? fe2 : fe1, R, f);
    }
    if constexpr (ONEJOB) {
      if (reuse) {
#pragma unroll
        for (int r = 0; r < QX; ++r) g[r] = e2[r];
      } else {
        SP::get_all(fe2, R, g);
      }
    }
  };
  if (ADJ && R.xact && t.reload && start && !first)
    SP::get_all(t.slab + (long)task_slot(t, task_in(t, j)) * M + pbase, R, q);
  SP::Tw::sync();
  if (first) {
    load_start();
    if (R.xact) {
      const int s_in = task_in(t, j);
      const int sl = t.slab ? task_slot(t, s_in) : -1;
      double* qin = sl >= 0 ? t.slab + (long)sl * M + pbase : nullptr;
      const bool keep = job == 0 && qin && !t.nostore;
      if (t.init_one) {
#pragma unroll
        for (int r = 0; r < QX; ++r) q[r] = make_double2(1.0, SP::ROWS ? 1.0 : 0.0);
      } else if (ADJ && t.add_src) {
        SP::add_source(t, s_in, M, pbase, R, q);
      } else {
        SP::get_all(t.start ? t.start + pbase : qin, R, q);
      }
      if (keep && (t.init_one || t.start)) {
#pragma unroll
        for (int r = 0; r < QX; ++r) SP::put(qin, R, r, q[r]);
      }
    }
  } else {
    SP::inv_y(c, E, PL, tw, R);
    load_start();
    double2 a[1][QX];
    SP::inv_x(a, E, PL, tw, R);
    if (R.xact) {
      double2 v[QX];
#pragma unroll
      for (int r = 0; r < QX; ++r) {
        const double2 q2 = make_double2(e2[r].x * a[0][r].x, e2[r].y * a[0][r].y);
        v[r] = make_double2(div_by(4.0 * q2.x - q1[r].x, 3.0, i3), div_by(4.0 * q2.y - q1[r].y, 3.0, i3));
      }
      if (ADJ && t.add_src) SP::add_source(t, s_out, M, pbase, R, v);
      if (!(ADJ && t.reload)) {
#pragma unroll
        for (int r = 0; r < QX; ++r) q[r] = v[r];
      }
      if (job == 0) {
        if (so >= 0) {
          double* qo = t.slab + (long)so * M + pbase;
#pragma unroll
          for (int r = 0; r < QX; ++r) SP::put(qo, R, r, v[r]);
        }
        if (ADJ && t.keepW) {
#pragma unroll
          for (int r = 0; r < QX; ++r) SP::put(t.keepW + pbase, R, r, a[0][r]);
        }
      }
    }
    __syncthreads();                // PL is reused by the forward transform
  }
  if (!start) return;
  double2 p[1][QX];
#pragma unroll
  for (int r = 0; r < QX; ++r) p[0][r] = make_double2(f[r].x * q[r].x, f[r].y * q[r].y);
  if (ADJ && t.keepA && job == 0 && R.xact) {
    double* ka = t.keepA + (j & 1) * M + pbase;
#pragma unroll
    for (int r = 0; r < QX; ++r) SP::put(ka, R, r, q[r]);
  }
  double2 h[1][UY][PY];
  SP::fwd(p, h, E, PL, tw, R);
  SP::store_cols((job == 0 ? t.A : t.B) + hbase, h, R);
  if constexpr (ONEJOB) {          // the half-step start: exp(-ds w/4) q -> B
#pragma unroll
    for (int r = 0; r < QX; ++r) p[0][r] = make_double2(g[r].x * q[r].x, g[r].y * q[r].y);
    __syncthreads();
    SP::fwd(p, h, E, PL, tw, R);
    SP::store_cols(t.B + hbase, h, R);
  }
}

// ----------------------------------------------------------------------------
// Step kernel C (two workgroups per z plane and sweep): job 0 turns the full
// step spectrum into q1 = exp(-ds w/2) IFFT[.]; job 1 ends the first half step
// and starts the second: exp(-ds w/2) IFFT[.], then the x,y forward transform
// into C (1/M is in the reciprocal-space factors).  Reference: src/step_mod.f90:159-167.  ADJ: keeps U and V.
// ----------------------------------------------------------------------------
template <int N1, int N2, bool ADJ, int LDSCAP = 80 * 1024, int WPE = 1>
__global__ void __launch_bounds__((StepPlane<N1, N2>::NT)) __attribute__((amdgpu_waves_per_eu(WPE)))
k_step_c(const StepTask* __restrict__ tasks, int jl, const double2* __restrict__ tw1g,
         const double2* __restrict__ twlg) {
  using SP = StepPlane<N1, N2, LDSCAP>;
  constexpr int QX = SP::QX, QY = SP::QY, PY = SP::PY, UY = SP::UY;
  __shared__ double2 TWS[SP::TWN];
  __shared__ double2 EB[SP::EBUF];
  __shared__ double2 PB[SP::PBUF];
  double2* const E = EB;
  double2* const PL = SP::ALIAS ? EB : PB;
  const int tid = threadIdx.x, z = blockIdx.x, job = blockIdx.z;
  const StepTask& t = tasks[blockIdx.y];
  const int j = jl + t.jofs;
  if (t.skip || j < t.jbeg || j >= t.jend) return;
  const typename SP::Roles R(tid);
  const long pbase = (long)z * N1 * N2;
  const long hbase = (long)z * plane_words(N1, SP::NL);
  typename SP::Tw tw;
  tw.load(tw1g, twlg, TWS, R, tid);
  double2 c[1][QY];
  SP::load_cols((job == 0 ? t.A : t.B) + hbase, c, R);
  double2 f[QX];
#pragma unroll
  for (int r = 0; r < QX; ++r) f[r] = make_double2(0.0, 0.0);
  if (R.xact) SP::get_all(task_e1(t, task_block(t, j)) + pbase, R, f);
  SP::Tw::sync();
  double2 a[1][QX];
  SP::inv_y(c, E, PL, tw, R);
  SP::inv_x(a, E, PL, tw, R);
  double* keep = !ADJ ? nullptr : (job == 0 ? t.keepU : t.keepV);
  if (ADJ && keep && R.xact) {
#pragma unroll
    for (int r = 0; r < QX; ++r) SP::put(keep + pbase, R, r, a[0][r]);
  }
#pragma unroll
  for (int r = 0; r < QX; ++r)
    a[0][r] = make_double2(f[r].x * a[0][r].x, f[r].y * a[0][r].y);
  if (job == 0) {
    if (R.xact) {
#pragma unroll
      for (int r = 0; r < QX; ++r) SP::put(t.q1 + pbase, R, r, a[0][r]);
    }
    return;
  }
  __syncthreads();                  // PL is reused by the forward transform
  double2 h[1][UY][PY];
  SP::fwd(a, h, E, PL, tw, R);
  SP::store_cols(t.C + hbase, h, R);
}

// ----------------------------------------------------------------------------
// Packed real planes -> x,y transformed packed planes C(kx, l), kept on
// selected columns: entry l N1 + (position of kx) goes to out[b][z][cpos[.]] when
// that is >= 0 (ncol entries per plane).  Two input sets per launch
// (blockIdx.z: in, in2, each of gridDim.y arrays); the second set's outputs
// follow the first's.  scf_stress transforms every stored contour point of
// both sweeps this way and reads one wave per star
// (src/scf_mod.fp.f90:451-550).
// ----------------------------------------------------------------------------
template <int N1, int N2>
__global__ void __launch_bounds__((StepPlane<N1, N2>::NT)) k_plane_r2c_cols(
    const double* __restrict__ in, const double* __restrict__ in2, long istride,
    double2* __restrict__ out, long ostride, const double2* __restrict__ tw1g,
    const double2* __restrict__ twlg, const int* __restrict__ cpos, int ncol) {
  using SP = StepPlane<N1, N2, 40 * 1024>;   // four workgroups per CU at 64 x 64
  constexpr int QX = SP::QX, PY = SP::PY, UY = SP::UY;
  __shared__ double2 TWS[SP::TWN];
  __shared__ double2 EB[SP::EBUF];
  __shared__ double2 PB[SP::PBUF];
  double2* const E = EB;
  double2* const PL = SP::ALIAS ? EB : PB;
  const int tid = threadIdx.x, z = blockIdx.x;
  const typename SP::Roles R(tid);
  typename SP::Tw tw;
  tw.load(tw1g, twlg, TWS, R, tid);
  double2 p[1][QX];
#pragma unroll
  for (int r = 0; r < QX; ++r) p[0][r] = make_double2(0.0, 0.0);
  if (R.xact)
    SP::get_all((blockIdx.z ? in2 : in) + blockIdx.y * istride + (long)z * N1 * N2, R, p[0]);
  SP::Tw::sync();
  double2 h[1][UY][PY];
  SP::fwd(p, h, E, PL, tw, R);
  double2* dst = out + ((long)blockIdx.z * gridDim.y + blockIdx.y) * ostride + (long)z * ncol;
  if (!R.yact) return;
#pragma unroll
  for (int u = 0; u < UY; ++u)
    if (SP::LY::has(R.yt, u)) {
#pragma unroll
      for (int k2 = 0; k2 < PY; ++k2) {
        const int c = cpos[SP::LY::at(R.yt, u, k2) * N1 + R.yp];
        if (c >= 0) dst[c] = h[0][u][k2];
      }
    }
}

// ----------------------------------------------------------------------------
// Z-column convolution: forward z transform, multiply by the reciprocal-space
// factor, inverse z transform, in place; one tile of column slots (z_slot) per
// workgroup.  The spectrum's columns ky = l and l + NL are split from the
// packed pair at every z, and merged into it at the end: lanes eight apart (h =
// 0, 1) hold the two packed columns and then the two spectrum columns, and
// trade values by a lane swap.  2 P lanes per slot (Line<N3>), the slots of a
// tile fastest across lanes.  Jobs: kind 0 -> (A, k1) and (B, k2); kind 1 ->
// (C, k2).  Z_ADJ: keeps the spectrum before the factor.  Z_SYM: symmetric
// planes; loads a column from its stored planes (each up to four times, from
// the cache) and stores those.
// ----------------------------------------------------------------------------
// LEN: points of the lines, N3 or (Z_HALF) N3/2.
template <int N3, int LEN = N3> struct StepZ {
  using L = Line<LEN>;
  static constexpr int P = L::P, Q = L::Q, U = L::U;
  static constexpr int ZW = imax(1, plan_zl(N3) / Line<N3>::P / 8) * 8;   // slots per workgroup
  static constexpr int NT = clampnt(round64(2 * ZW * P));
  static constexpr int NTC = clampnt(round64(ZW * P));  // of k_zfwd_cols
  // twiddles in registers where they are few, else a table in LDS
  static constexpr bool TWREG = TwRegs<L, true>::COUNT <= 12;
  using Tw = std::conditional_t<TWREG, TwRegs<L, true>, TwTable<L>>;
  static constexpr int TWN = TWREG ? 1 : LEN;
  template <int T> static __device__ __forceinline__ void load_tw(Tw& tw, const double2* __restrict__ g,
                                                                  double2* lds, int tz, int tid) {
    if constexpr (TWREG) {
      tw.load(g, tz);
    } else {
      stage_tw<LEN, T>(lds, g, tid);
      tw.tw = lds;
    }
  }
};

enum { Z_PLAIN = 0, Z_ADJ = 1, Z_SYM = 2, Z_HALF = 4 };    // flags
// Z_HALF (with Z_SYM): the translation z -> z + N3/2 without a rotation in the
// plane (body, face and base centring).  A column is then periodic or
// antiperiodic over half the edge, and only its even or its odd kz are not
// zero: lines of N3/2 points, twiddled by w_N3^z where antiperiodic.
// Half the points, LDS words and butterflies of the whole lines; density() +
// scf_stress() before and now: gyroid 64^3 6125 -> 5649 us, 96^3 13640 ->
// 12250 us, 32 body-centred 32^3 fields 7293 -> 6652 us.  Reverse-mode sweeps
// keep whole lines: their kept spectra need the zeros too.
constexpr bool sym_half(int sym) { return (sym & SYM_T) != 0 && !(sym >> 2 & 1); }
constexpr bool z_half_ok(int n3) { return n3 % 2 == 0 && line_plan(n3 / 2).p > 0; }
// twiddle tables of length n, then n/2 (Z_HALF's lines)
constexpr int z_tables(int n3) { return n3 + n3 / 2; }
template <int N1, int N3, int MODE>
__global__ void __launch_bounds__((StepZ<N3, (MODE & Z_HALF) ? N3 / 2 : N3>::NT)) k_step_z(const StepTask* __restrict__ tasks, int jl, int N2,
                                                       int kind, const double2* __restrict__ tw2g,
                                                       const double2* __restrict__ tw3g) {
  constexpr bool HALF = (MODE & Z_HALF) != 0;
  constexpr int NZ = HALF ? N3 / 2 : N3;
  using SZ = StepZ<N3, NZ>;
  constexpr bool ADJ = (MODE & Z_ADJ) != 0, SYM = (MODE & Z_SYM) != 0;
  using L = typename SZ::L;
  constexpr int P = SZ::P, Q = SZ::Q, U = SZ::U, ZW = SZ::ZW;
  constexpr int N1H = N1 / 2 + 1;
  __shared__ double2 E[NZ > 1 ? 2 * NZ * ZW : 1];
  __shared__ double2 TWS[SZ::TWN];
  const int tid = threadIdx.x, hc = tid % (2 * ZW), tz = tid / (2 * ZW);
  const int h = z_lane_h(hc), c = z_lane_slot(hc);
  const int job = blockIdx.z;
  const StepTask& t = tasks[blockIdx.y];
  const int j = jl + t.jofs;
  if (t.skip || j < t.jbeg || j >= t.jend) return;
  const bool rows = N2 > 1;
  const int nl = rows ? N2 / 2 : 1;
  const ZSlot sl = z_slot(blockIdx.x, c, N1, nl, ZW);
  const bool act = tz < P && sl.ok;
  const int io = h ? sl.o[1] : sl.o[0];            // this lane's packed column
  const unsigned pb = 16 * plane_words(N1, nl);    // bytes per plane
  const unsigned ob = 16 * io + tz * pb;
  const int np = SYM ? sym_planes(t.sym, N3) : N3;
  const int b = task_block(t, j);
  double2* arr = kind == 0 ? (job == 0 ? t.A : t.B) : t.C;
  const double* kf = kind == 0 && job == 0 ? task_k1(t, b) : task_k2(t, b);
  // antiperiodic columns (HALF): odd kz
  const int odd = HALF ? ((t.sym & 8 ? sl.kx : 0) ^ (t.sym & 16 ? sl.l + h * nl : 0)) & 1 : 0;
  double2 v[1][Q], wl = make_double2(1.0, 0.0);
  double f[U][P];
  int op[SYM ? Q : 1];
#pragma unroll
  for (int r = 0; r < Q; ++r) {
    v[0][r] = make_double2(0.0, 0.0);
    if constexpr (SYM) op[r] = 0;
  }
  if (act) {
#pragma unroll
    for (int r = 0; r < Q; ++r) {
      if constexpr (SYM) {
        int u;
        op[r] = sym_source(t.sym, N3, tz + P * r, u);
        v[0][r] = ld16(arr, 16 * io + u * pb);
      } else {
        v[0][r] = ld16(arr, ob + P * r * pb);
      }
    }
    wl = tw2g[sl.l];
    const unsigned kz = gridDim.x * (2 * ZW), k0 = blockIdx.x * (2 * ZW) + hc + tz * kz;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (L::has(tz, u)) {
#pragma unroll
        for (int k2 = 0; k2 < P; ++k2) {
          if constexpr (HALF) f[u][k2] = 2.0 * kf[k0 - tz * kz + (2 * (tz + P * u + Q * k2) + odd) * kz];
          else f[u][k2] = kf[k0 + (P * u + Q * k2) * kz];
        }
      }
  }
  double2 wz[HALF ? Q : 1];
  if constexpr (HALF) {
#pragma unroll
    for (int r = 0; r < Q; ++r) wz[r] = odd && act ? tw3g[tz + P * r] : make_double2(1.0, 0.0);
  }
  typename SZ::Tw tw;
  SZ::template load_tw<SZ::NT>(tw, HALF ? tw3g + N3 : tw3g, TWS, tz, tid);
  if constexpr (!SZ::TWREG) __syncthreads();
  // split: v = 2 F(ky = l + h NL) = a + m + (-1)^h w^l (a - m)/i with a =
  // C(kx,l), m = C*(-kx,-l), written in the sums and differences of this
  // lane's column and the other's, so that no lane has to select
  const double sg = h ? -1.0 : 1.0;
  if (rows) {
    const double sx = sg * wl.x, sy = sg * wl.y;
#pragma unroll
    for (int r = 0; r < Q; ++r) {
      const double2 own = v[0][r], oth = lane_swap(own);
      const double2 p = cadd(own, oth), d = csub(own, oth);
      v[0][r] = make_double2(mad(wl.y, d.x, mad(sx, p.y, p.x)), mad(sg, d.y, mad(sy, p.y, -wl.x * d.x)));
    }
  } else {                         // one row: C(kx) is F(kx), on both lanes
#pragma unroll
    for (int r = 0; r < Q; ++r) {
      const double2 oth = lane_swap(v[0][r]);
      if (h) v[0][r] = oth;
    }
  }
  if constexpr (SYM) {
    // the operation from the stored plane, at this lane's column (kx, ky)
    const int sx = sl.kx << 31, sy = (sl.l + h * nl) << 31;
#pragma unroll
    for (int r = 0; r < Q; ++r) {
      const int m = ((op[r] & 2) ? sx : 0) ^ ((op[r] & 4) ? sy : 0);
      v[0][r].x = sign_flip(v[0][r].x, m);
      v[0][r].y = sign_flip(v[0][r].y, m ^ (op[r] << 31));
      if constexpr (HALF) v[0][r] = cmul(v[0][r], wz[r]);
    }
  }
  double2 w[1][U][P];
  const auto eoff = [&](int, int i) { return i * (2 * ZW) + hc; };
  line_fwd<L, -1, 1, false>(v, w, E, eoff, tz, tw, act);
  double2* keep = ADJ ? t.keepK[kind == 0 ? job : 2] : nullptr;
  if (act) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (L::has(tz, u)) {
#pragma unroll
        for (int k2 = 0; k2 < P; ++k2) {
          if (ADJ && keep && (rows || !h))
            keep[sl.kx + N1H * (sl.l + h * nl + (long)N2 * L::at(tz, u, k2))] = cscale(w[0][u][k2], rows ? 0.5 : 1.0);
          w[0][u][k2] = cscale(w[0][u][k2], f[u][k2]);
        }
      }
  }
  line_inv<L, +1, 1, false>(w, v, E, eoff, tz, tw, act);
  // merge: C(kx,l) = E + i O on lane 0, C(-kx,-l) = conj(E - i O) on lane 1
  const double2 iw = cmul_si<+1>(cconj(wl));
#pragma unroll
  for (int r = 0; r < Q; ++r) {
    double2 a = v[0][r];
    if constexpr (HALF) a = cmul(a, cconj(wz[r]));
    if (rows) {
      const double2 oth = lane_swap(a);
      a = cfma(iw, csub(a, oth), cadd(a, oth));
    }
    a.y *= sg;
    if (act && !(h && sl.o[0] == sl.o[1]) && (!SYM || tz + P * r < np)) st16(arr, ob + P * r * pb, a);
  }
}

// ----------------------------------------------------------------------------
// A whole sweep of a grid with N3 = 1 (1D and 2D cells) in one launch: one
// workgroup per task keeps the contour field, the factors of the block and the
// spectra in registers and LDS, and writes each point to the slab.  Nothing
// passes between workgroups, where the step kernels take four launches per
// contour step.  Two teams of a plane's threads: in the first convolution team
// 0 does the full step and team 1 the first half step; in the second, team 1
// does the other half step, then the Richardson sum, and hands q to team 0.
// Reciprocal-space factor on packed rows (at StepPlane): with a = C(kx,l), m =
// C*(-kx,-l), w = exp(-2 pi i l / N2) and s, d the half sum and difference of
// the factors at ky = l and l + NL, split, product and merge are
//   C'(kx,l) = (s + d Im w) a + i d Re w m,
// two real numbers per packed column, held in registers while the block lasts.
// Bound by the latency of its chain of line transforms (four per step), LDS
// exchanges and nine barriers (1D: two).  density() + scf_stress() with 100
// steps, before (four launches per step) and now: 32 points 1260 -> 415 us,
// 48 x 48 1844 -> 1107 us.
// ----------------------------------------------------------------------------
template <int N1, int N2> struct SweepPlane {
  using SP = StepPlane<N1, N2, 160 * 1024, false, true>;
  static constexpr int NT = 2 * SP::NT;
  // both teams' buffers in one workgroup's LDS: edges to 64
  static constexpr bool OK = NT <= 1024 && !SP::ALIAS && 2 * SP::LDS <= 160 * 1024;
};

template <int N1, int N2>
__global__ void __launch_bounds__((SweepPlane<N1, N2>::NT))
k_sweep_plane(const StepTask* __restrict__ tasks, int last, const double2* __restrict__ tw1g,
              const double2* __restrict__ twlg, const double2* __restrict__ tw2g) {
  using SP = typename SweepPlane<N1, N2>::SP;
  using LX = typename SP::LX;
  using LY = typename SP::LY;
  constexpr int QX = SP::QX, QY = SP::QY, PY = SP::PY, UY = SP::UY, PX = SP::PX, UX = SP::UX, NL = SP::NL;
  constexpr int ZW = StepZ<1>::ZW;
  __shared__ double2 TWS[SP::TWN];
  __shared__ double2 EB[2][SP::EBUF];
  __shared__ double2 PB[2][SP::PBUF];
  const int team = threadIdx.x / SP::NT, tid = threadIdx.x % SP::NT;
  double2* const E = EB[team];
  double2* const PL = PB[team];
  const StepTask& t = tasks[blockIdx.x];
  const int jend = t.jend < last + t.jofs ? t.jend : last + t.jofs;   // launches 0 .. last
  if (t.skip || t.jbeg > jend) return;
  const typename SP::Roles R(tid);
  typename SP::Roles R1 = R;         // the second convolution: team 0 only meets the barriers
  if (team == 0) R1.xact = R1.yact = false;
  typename SP::Tw tw;
  tw.load(tw1g, twlg, TWS, R, tid);
  double2 q[QX], e1[QX], e2[QX];
#pragma unroll
  for (int r = 0; r < QX; ++r) q[r] = e1[r] = e2[r] = make_double2(0.0, 0.0);
  {
    const int s_in = task_in(t, t.jbeg);
    const int sl = t.slab ? task_slot(t, s_in) : -1;
    double* qin = sl >= 0 ? t.slab + (long)sl * t.fm : nullptr;
    if (R.xact) {
      if (t.init_one) {
#pragma unroll
        for (int r = 0; r < QX; ++r) q[r] = make_double2(1.0, SP::ROWS ? 1.0 : 0.0);
      } else {
        SP::get_all(t.start ? t.start : qin, R, q);
      }
      if (qin && team == 0 && (t.init_one || t.start)) {
#pragma unroll
        for (int r = 0; r < QX; ++r) SP::put(qin, R, r, q[r]);
      }
    }
  }
  SP::Tw::sync();
  // factors of the spectrum's points of this thread (2D: y role, layout B over
  // l; 1D: x role, layout B over kx), of the team's convolution
  double fa[SP::ROWS ? UY : UX][SP::ROWS ? PY : PX];
  double fb[SP::ROWS ? UY : 1][SP::ROWS ? PY : 1];
  const auto conv = [&](double2 (&a)[1][QX], const typename SP::Roles& W) {
    if constexpr (SP::ROWS) {
      double2 h[1][UY][PY], c[1][QY];
      SP::fwd(a, h, E, PL, tw, W);
      wave_sync();
      if (W.yact) {
#pragma unroll
        for (int u = 0; u < UY; ++u)
          if (LY::has(W.yt, u)) {
#pragma unroll
            for (int k2 = 0; k2 < PY; ++k2) E[W.ey(LY::at(W.yt, u, k2))] = h[0][u][k2];
          }
      }
      __syncthreads();
      if (W.yact) {
        const int other = (W.yk ? N1 - W.yk : 0) * SP::EYW;
#pragma unroll
        for (int u = 0; u < UY; ++u)
          if (LY::has(W.yt, u)) {
#pragma unroll
            for (int k2 = 0; k2 < PY; ++k2) {
              const int l = LY::at(W.yt, u, k2);
              const double2 o = E[other + (l ? NL - l : 0)], v = h[0][u][k2];
              h[0][u][k2] = make_double2(mad(fa[u][k2], v.x, fb[u][k2] * o.y),
                                         mad(fa[u][k2], v.y, fb[u][k2] * o.x));
            }
          }
      }
      __syncthreads();
      line_inv<LY, +1, 1>(h, c, E, [&](int, int i) { return W.ey(i); }, W.yt, tw.y, W.yact);
      if (W.yact) {
#pragma unroll
        for (int r = 0; r < QY; ++r) PL[(W.yt + PY * r) * SP::PLS + W.yk] = c[0][r];
      }
      __syncthreads();
      SP::inv_x(a, E, PL, tw, W);
    } else {
      double2 b[1][UX][PX];
      const auto ex = [&](int, int i) { return W.ex(i); };
      line_fwd<LX, -1, 1>(a, b, E, ex, W.xt, tw.x, W.xact);
#pragma unroll
      for (int u = 0; u < UX; ++u)
        if (W.xact && LX::has(W.xt, u)) {
#pragma unroll
          for (int k2 = 0; k2 < PX; ++k2) b[0][u][k2] = cscale(b[0][u][k2], fa[u][k2]);
        }
      line_inv<LX, +1, 1>(b, a, E, ex, W.xt, tw.x, W.xact);
    }
  };
  const double i3 = 1.0 / 3.0;
  double2* const X = PB[0] + R.xl * SP::PLS + R.xt;   // q1, then q: a thread's own words of its row
  int block = -1;
  for (int j = t.jbeg; j < jend; ++j) {
    const int b = task_block(t, j);
    const int so = t.slab ? task_slot(t, task_out(t, j)) : -1;
    if (b != block) {
      block = b;
      const double* kf = team ? task_k2(t, b) : task_k1(t, b);
      if (R.xact) {
        SP::get_all(task_e1(t, b), R, e1);
        SP::get_all(task_e2(t, b), R, e2);
      }
      if constexpr (SP::ROWS) {
        if (R.yact) {
#pragma unroll
          for (int u = 0; u < UY; ++u)
            if (LY::has(R.yt, u)) {
#pragma unroll
              for (int k2 = 0; k2 < PY; ++k2) {
                const int l = LY::at(R.yt, u, k2);
                const double f0 = kf[z_factor_at(R.yk, l, 0, N1, NL, ZW)];
                const double f1 = kf[z_factor_at(R.yk, l, 1, N1, NL, ZW)];
                const double2 w = tw2g[l];
                fa[u][k2] = 2.0 * mad(f0 - f1, w.y, f0 + f1);    // k_step_z's factor 4
                fb[u][k2] = 2.0 * (f0 - f1) * w.x;
              }
            }
        }
      } else if (R.xact) {
#pragma unroll
        for (int u = 0; u < UX; ++u)
          if (LX::has(R.xt, u)) {
#pragma unroll
            for (int k2 = 0; k2 < PX; ++k2)
              fa[u][k2] = kf[z_factor_at(LX::at(R.xt, u, k2), 0, 0, N1, 1, ZW)];
          }
      }
    }
    double2 a[1][QX];
#pragma unroll
    for (int r = 0; r < QX; ++r) {
      const double2 f = team ? e2[r] : e1[r];
      a[0][r] = make_double2(f.x * q[r].x, f.y * q[r].y);
    }
    conv(a, R);
#pragma unroll
    for (int r = 0; r < QX; ++r) a[0][r] = make_double2(e1[r].x * a[0][r].x, e1[r].y * a[0][r].y);
    if (team == 0 && R.xact) {
#pragma unroll
      for (int r = 0; r < QX; ++r) X[PX * r] = a[0][r];
    }
    if constexpr (!SP::ROWS) __syncthreads();
    conv(a, R1);
    if (R1.xact) {
#pragma unroll
      for (int r = 0; r < QX; ++r) {
        const double2 q1 = X[PX * r];
        const double2 q2 = make_double2(e2[r].x * a[0][r].x, e2[r].y * a[0][r].y);
        q[r] = make_double2(div_by(4.0 * q2.x - q1.x, 3.0, i3), div_by(4.0 * q2.y - q1.y, 3.0, i3));
        X[PX * r] = q[r];
      }
      if (so >= 0) {
        double* qo = t.slab + (long)so * t.fm;
#pragma unroll
        for (int r = 0; r < QX; ++r) SP::put(qo, R, r, q[r]);
      }
    }
    __syncthreads();
    if (team == 0 && R.xact) {
#pragma unroll
      for (int r = 0; r < QX; ++r) q[r] = X[PX * r];
    }
  }
}

// ----------------------------------------------------------------------------
// Split and forward z transform of scf_stress's contour-point spectra: `in`
// holds nin packed columns per plane (k_plane_r2c_cols), `out` the ncol
// half-spectrum columns that hold a star's representative wave, (z, column)
// at z ncol + c (arrays istride and ostride apart).  Column c, at
// cols[c] = (kx, ky), is split from the packed columns at positions
// src[c] = ((kx, l), (-kx, -l)), on the register lines of k_step_z.
// ----------------------------------------------------------------------------
template <int N3>
__global__ void __launch_bounds__(StepZ<N3>::NTC) k_zfwd_cols(int sym, const double2* __restrict__ in, long istride,
                                                          int nin, double2* __restrict__ out, long ostride,
                                                          int ncol, int N2, const int2* __restrict__ src,
                                                          const int2* __restrict__ cols,
                                                          const double2* __restrict__ tw2g,
                                                          const double2* __restrict__ tw3g) {
  using SZ = StepZ<N3>;
  using L = typename SZ::L;
  constexpr int P = SZ::P, Q = SZ::Q, U = SZ::U, ZW = SZ::ZW;
  __shared__ double2 E[N3 > 1 ? N3 * ZW : 1];
  __shared__ double2 TWS[SZ::TWN];
  const int tid = threadIdx.x, c = tid % ZW, tz = tid / ZW;
  const double2* arr = in + blockIdx.y * istride;
  double2* dst = out + blockIdx.y * ostride;
  const int col = blockIdx.x * ZW + c;
  const bool act = tz < P && col < ncol;
  double2 v[1][Q];
  if (act) {
    const int2 s = src[col];
    const double2 w = tw2g[cols[col].y];           // -w^l at ky = l + NL
#pragma unroll
    for (int r = 0; r < Q; ++r) {
      int u;
      const int op = sym_source(sym, N3, tz + P * r, u);
      const double2 a = arr[s.x + (long)u * nin];
      if (N2 > 1) {
        const double2 m = cconj(arr[s.y + (long)u * nin]);
        v[0][r] = cscale(cfma(w, cmul_si<-1>(csub(a, m)), cadd(a, m)), 0.5);
      } else {
        v[0][r] = a;
      }
      const int m = ((op & 2) ? cols[col].x << 31 : 0) ^ ((op & 4) ? cols[col].y << 31 : 0);
      v[0][r].x = sign_flip(v[0][r].x, m);
      v[0][r].y = sign_flip(v[0][r].y, m ^ (op << 31));
    }
  }
  typename SZ::Tw tw;
  SZ::template load_tw<SZ::NTC>(tw, tw3g, TWS, tz, tid);
  if constexpr (!SZ::TWREG) __syncthreads();
  double2 w[1][U][P];
  line_fwd<L, -1, 1, false>(v, w, E, [&](int, int i) { return i * ZW + c; }, tz, tw, act);
  if (act) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (L::has(tz, u)) {
#pragma unroll
        for (int k2 = 0; k2 < P; ++k2) dst[col + (long)L::at(tz, u, k2) * ncol] = w[0][u][k2];
      }
  }
}

// ----------------------------------------------------------------------------
// Adjoint gradient of one step for each (adjoint task, recomputed task) pair.
// With a the adjoint entering the step and q the field the step is applied
// to (both step inputs, read from their slabs), and U, V, W the kept
// pre-factor fields of the step on q (suffix q) and on a (suffix a):
//   d<a, T q>/d omega = -(ds/3) [ e2 (a Wq + q Wa) + 2 e1 Va Vq - (e1/2)(a Uq + q Ua) ]
// for T = (4 e2 C2 e1 C2 e2 - e1 C1 e1)/3 (src/step_mod.f90:156-174),
// accumulated into the omega gradient of the step's block.  The pairs of a
// chain share their block accumulators, so every thread applies all pairs to
// its points in turn (no two threads update one point).
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_adj_grad(const StepTask* __restrict__ tasks,
                                                  const int2* __restrict__ pairs, int npair, int jl,
                                                  long m) {
  for (int pr = 0; pr < npair; ++pr) {
    const StepTask& A = tasks[pairs[pr].x];
    const StepTask& Q = tasks[pairs[pr].y];
    const int j = jl + A.jofs, jq = jl + Q.jofs;
    if (A.skip || j < A.jbeg || j >= A.jend) continue;
    const int b = task_block(A, j);
    const double* a = A.keepA + (j & 1) * m;    // the adjoint entering step j (K_A(j) kept it)
    const double* q = Q.slab + (long)task_slot(Q, task_in(Q, jq)) * m;
    const double* e1 = task_e1(A, b);
    const double* e2 = task_e2(A, b);
    const double c = A.ds[b] / 3.0;
    double* grad = A.grad[b];
    for (long r = blockIdx.x * 256L + threadIdx.x; r < m; r += (long)gridDim.x * 256L) {
      const double av = a[r], qv = q[r];
      const double g = e2[r] * (av * Q.keepW[r] + qv * A.keepW[r]) +
                       2.0 * e1[r] * A.keepV[r] * Q.keepV[r] -
                       0.5 * e1[r] * (av * Q.keepU[r] + qv * A.keepU[r]);
      grad[r] -= c * g;
    }
  }
}

// ----------------------------------------------------------------------------
// Reciprocal-space part of the same step derivative.  With the unnormalised
// 3D spectra Aq = FFT[e1 q], Bq = FFT[e2 q], Cq = FFT[e1 Vq] (and likewise for
// a), and k1 = exp(-ds b^2 k^2/6), k2 = exp(-ds b^2 k^2/12):
//   d<a,Tq>/dk1(k) = -(1/3M) Re(Aq Aa*),  d<a,Tq>/dk2(k) = (4/3M) Re(Cq Ba* + Bq Ca*)
// so d<a,Tq>/d|k|^2 = (ds b^2/M) [ k1 Re(Aq Aa*)/18 - k2 Re(Cq Ba* + Bq Ca*)/9 ].
// A half-grid point with 0 < kx < N1/2 stands for k and -k and counts twice;
// at kx = 0 and N1/2 the spectra are kept at one of k and -k (z_slot), whose
// value both get.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_adj_kgrad(const StepTask* __restrict__ tasks,
                                                   const int2* __restrict__ pairs, int npair, int jl,
                                                   int n1, int n2, int n3, int zw) {
  const int n1h = n1 / 2 + 1, nl = n2 > 1 ? n2 / 2 : 1;
  for (int pr = 0; pr < npair; ++pr) {
    const StepTask& A = tasks[pairs[pr].x];
    const StepTask& Q = tasks[pairs[pr].y];
    const int j = jl + A.jofs;
    if (A.skip || j < A.jbeg || j >= A.jend) continue;
    const int b = task_block(A, j);
    const double* k1 = task_k1(A, b);
    const double* k2 = task_k2(A, b);
    const double c = A.ds[b] * A.bsq[b] * (n2 > 1 ? 2.0 : 1.0);   // 1/M is in k1 and k2
    double* kg = A.kgrad[b];
    // i runs over the factors' order
    for (long i = blockIdx.x * 256L + threadIdx.x; i < A.fk; i += (long)gridDim.x * 256L) {
      const long g = unpack_kindex(i, n1, n2, zw);
      if (g < 0 || (n2 == 1 && z_lane_h((int)(i % (2 * zw))))) continue;   // N2 = 1: both h alike
      const int kx = (int)(g % n1h), ky = (int)(g / n1h % n2), l = ky % nl;
      const bool edge = kx == 0 || 2 * kx == n1;
      const double2 aq = Q.keepK[0][g], aa = A.keepK[0][g];
      const double2 bq = Q.keepK[1][g], ba = A.keepK[1][g];
      const double2 cq = Q.keepK[2][g], ca = A.keepK[2][g];
      const double r1 = aq.x * aa.x + aq.y * aa.y;
      const double r2 = cq.x * ba.x + cq.y * ba.y + bq.x * ca.x + bq.y * ca.y;
      const double v = c * (k1[i] * r1 / 18.0 - k2[i] * r2 / 9.0);
      kg[g] += edge ? v : 2.0 * v;
      if (edge && l != 0 && 2 * l != nl) {
        const long kz = g / ((long)n1h * n2);
        kg[kx + n1h * ((n2 - ky) % n2 + n2 * ((n3 - kz) % n3))] += v;
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Standalone transform passes (batched over blockIdx.y arrays).
// ----------------------------------------------------------------------------

// real planes -> x,y forward transformed half planes; in[b*istride + ...].
// With `cols`, only the ncolp half-plane positions cols[c] are stored, at
// out[b*ostride + z*ncolp + c].
template <int N1, int N2>
__global__ void __launch_bounds__(plane_nt(N1, N2)) k_plane_r2c(const double* __restrict__ in, long istride,
                                                  double2* __restrict__ out, long ostride,
                                                  const double2* __restrict__ tw1g,
                                                  const double2* __restrict__ tw2g,
                                                  const int* __restrict__ cols, int ncolp) {
  constexpr int NT = plane_nt(N1, N2);
  using PL = Plane<N1, N2>;
  __shared__ double2 U[PL::USIZE];
  double2* const P = PL::Pbuf(U);
  double2* const H = PL::Hbuf(U);
  __shared__ double2 tw1[N1], tw2[N2];
  const int tid = threadIdx.x, z = blockIdx.x;
  stage<N1, NT>(tw1, tw1g, tid);
  stage<N2, NT>(tw2, tw2g, tid);
  const double* src = in + blockIdx.y * istride + (long)z * N1 * N2;
  for (int i = tid; i < PL::NP * N1; i += NT) {
    const int x = i % N1, y0 = 2 * (i / N1);
    P[PL::pidx(i)] = make_double2(src[y0 * N1 + x], (y0 + 1 < N2) ? src[(y0 + 1) * N1 + x] : 0.0);
  }
  __syncthreads();
  plane_forward<N1, N2, NT>(P, H, tw1, tw2, tid);
  if (cols) {
    double2* dst = out + blockIdx.y * ostride + (long)z * ncolp;
    for (int c = tid; c < ncolp; c += NT) dst[c] = H[cols[c]];
    return;
  }
  double2* dst = out + blockIdx.y * ostride + (long)z * PL::HSIZE;
  for (int i = tid; i < PL::HSIZE; i += NT) dst[i] = H[i];
}

// half planes -> x,y inverse transformed real planes, times `scale`
template <int N1, int N2>
__global__ void __launch_bounds__(plane_nt(N1, N2)) k_plane_c2r(const double2* __restrict__ in, long istride,
                                                  double* __restrict__ out, long ostride,
                                                  double scale, const double2* __restrict__ tw1g,
                                                  const double2* __restrict__ tw2g) {
  constexpr int NT = plane_nt(N1, N2);
  using PL = Plane<N1, N2>;
  __shared__ double2 U[PL::USIZE];
  double2* const P = PL::Pbuf(U);
  double2* const H = PL::Hbuf(U);
  __shared__ double2 tw1[N1], tw2[N2];
  const int tid = threadIdx.x, z = blockIdx.x;
  stage<N1, NT>(tw1, tw1g, tid);
  stage<N2, NT>(tw2, tw2g, tid);
  const double2* src = in + blockIdx.y * istride + (long)z * PL::HSIZE;
  for (int i = tid; i < PL::HSIZE; i += NT) H[i] = src[i];
  __syncthreads();
  plane_inverse<N1, N2, NT>(H, P, tw1, tw2, tid);
  double* dst = out + blockIdx.y * ostride + (long)z * N1 * N2;
  for (int i = tid; i < PL::NP * N1; i += NT) {
    const int x = i % N1, y0 = 2 * (i / N1);
    const double2 r = P[PL::pidx(i)];
    dst[y0 * N1 + x] = r.x * scale;
    if (y0 + 1 < N2) dst[(y0 + 1) * N1 + x] = r.y * scale;
  }
}

// in-place z transform of W-wide rows (W = N1/2+1 for half spectra, N1 for
// full complex grids), batched over blockIdx.y arrays
template <int W, int N3, int SIGN>
__global__ void __launch_bounds__(zcol_nt(W, N3)) k_zfft(double2* __restrict__ data, long stride, int N2,
                                             const double2* __restrict__ tw3g) {
  constexpr int NT = zcol_nt(W, N3);
  __shared__ double2 T[W * N3];
  __shared__ double2 tw3[N3];
  const int tid = threadIdx.x, ky = blockIdx.x;
  stage<N3, NT>(tw3, tw3g, tid);
  double2* arr = data + blockIdx.y * stride;
  const long rowstride = (long)W * N2;
  for (int i = tid; i < W * N3; i += NT) T[i] = arr[(i / W) * rowstride + (long)ky * W + i % W];
  __syncthreads();
  fft_lines<N3, SIGN, W, 1, W, false, NT>(T, tw3, tid);
  for (int i = tid; i < W * N3; i += NT) arr[(i / W) * rowstride + (long)ky * W + i % W] = T[i];
}

// full complex planes, in place, x then y (used by the c2c transform)
template <int N1, int N2, int SIGN>
__global__ void __launch_bounds__(c2c_nt(N1, N2)) k_plane_c2c(double2* __restrict__ data, long stride,
                                                  const double2* __restrict__ tw1g,
                                                  const double2* __restrict__ tw2g) {
  constexpr int NT = c2c_nt(N1, N2);
  __shared__ double2 T[N1 * N2];
  __shared__ double2 tw1[N1], tw2[N2];
  const int tid = threadIdx.x, z = blockIdx.x;
  stage<N1, NT>(tw1, tw1g, tid);
  stage<N2, NT>(tw2, tw2g, tid);
  double2* arr = data + blockIdx.y * stride + (long)z * N1 * N2;
  for (int i = tid; i < N1 * N2; i += NT) T[i] = arr[i];
  __syncthreads();
  fft_lines<N1, SIGN, N2, N1, 1, true, NT>(T, tw1, tid);
  fft_lines<N2, SIGN, N1, 1, N1, false, NT>(T, tw2, tid);
  for (int i = tid; i < N1 * N2; i += NT) arr[i] = T[i];
}

}  // namespace pscf
