// Pointwise, gather/scatter and reduction kernels of the SCFT inner loop.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_lds.hpp"
#include "geom.hpp"

namespace pscf {

constexpr int NTA = 256;

// ----------------------------------------------------------------------------
// Minimum-image wavevectors and |G|^2 on the half grid (GeomArgs and
// g_to_bz_vec: geom.hpp).  Outputs: ksq(kx,ky,kz) and, through the dense
// wave table wtab (index (G - gmin) over a box), the 1-based wave number
// (0 if the wave is not in the basis), as basis_to_kgrid looks it up.
// ----------------------------------------------------------------------------
// minimum image of half-grid point idx
__device__ __forceinline__ double g_to_bz_point(const GeomArgs& g, long idx, int best[3]) {
  const int n1h = g.n1 / 2 + 1;
  const int G[3] = {(int)(idx % n1h), (int)((idx / n1h) % g.n2), (int)(idx / ((long)n1h * g.n2))};
  return g_to_bz_vec(g, G, best);
}

__global__ void __launch_bounds__(NTA) k_g_to_bz(GeomArgs g, const int* __restrict__ wtab,
                                                 double* __restrict__ ksq, int* __restrict__ kwave) {
  const int n1h = g.n1 / 2 + 1;
  const long mk = (long)n1h * g.n2 * g.n3;
  for (long idx = blockIdx.x * (long)NTA + threadIdx.x; idx < mk; idx += (long)gridDim.x * NTA) {
    int best[3];
    const double bsq = g_to_bz_point(g, idx, best);
    ksq[idx] = bsq;
    int w = 0;
    bool inside = true;
    long off = 0, mul = 1;
    for (int d = 0; d < g.dim; ++d) {
      const int u = best[d] - g.gmin[d];
      if (u < 0 || u >= g.gext[d]) inside = false;
      off += (long)u * mul;
      mul *= g.gext[d];
    }
    if (inside) w = wtab[off];
    kwave[idx] = w;
  }
}

// ----------------------------------------------------------------------------
// Star basis -> half k grid (src/grid_basis_mod.f90:47-129), nf fields.
// kwave: 1-based wave per half-grid point (0 = none); coeff/star_of_wave/
// star_invert: basis_mod tables (src/basis_mod.f90:60-84).
// basis(nf, N_star) is the reference's omega(N_monomer, N_star) layout.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_basis_to_kgrid(const double* __restrict__ basis, int nf,
                                                        int nstar, const int* __restrict__ kwave,
                                                        const double2* __restrict__ coeff,
                                                        const int* __restrict__ star_of_wave,
                                                        const int* __restrict__ star_invert, long mk,
                                                        double2* __restrict__ out, int no_parity) {
  const double sq2 = 1.41421356237309514547;  // dsqrt(2.0_long)
  const long n = mk * nf;
  for (long gi = blockIdx.x * (long)NTA + threadIdx.x; gi < n; gi += (long)gridDim.x * NTA) {
    const int f = (int)(gi / mk);
    const long idx = gi % mk;
    const int w = kwave[idx];
    double2 z = make_double2(0.0, 0.0);
    if (w >= 1) {
      const double2 c = coeff[w - 1];
      const int s = star_of_wave[w - 1] - 1;
      const int inv = no_parity ? 0 : star_invert[s];
      if (inv == 0) {
        const double a = basis[(long)s * nf + f];
        z = make_double2(a * c.x, a * c.y);
      } else {
        double a, bb;
        if (inv == 1) { a = basis[(long)s * nf + f]; bb = -basis[(long)(s + 1) * nf + f]; }
        else          { a = basis[(long)(s - 1) * nf + f]; bb = basis[(long)s * nf + f]; }
        z = cmul(make_double2(a, bb), c);
        z = make_double2(z.x / sq2, z.y / sq2);
      }
    }
    out[gi] = z;
  }
}

// ----------------------------------------------------------------------------
// Half k grid -> star basis (src/grid_basis_mod.f90:146-200) for nf fields,
// then times `scale` (density() divides by M: src/scf_mod.fp.f90:224).
// sidx: half-grid index of the star's representative wave, sconj: 1 if the
// representative lies in kx > N1/2 and is read as conj of -k.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_kgrid_to_basis(const double2* __restrict__ kg, long mk,
                                                        int nf, int nstar,
                                                        const long* __restrict__ sidx,
                                                        const int* __restrict__ sconj,
                                                        const double2* __restrict__ scoef,
                                                        const int* __restrict__ star_invert,
                                                        double scale, double* __restrict__ basis,
                                                        int no_parity) {
  const double sq2 = 1.41421356237309514547;
  const long n = (long)nstar * nf;
  for (long gi = blockIdx.x * (long)NTA + threadIdx.x; gi < n; gi += (long)gridDim.x * NTA) {
    const int f = (int)(gi % nf);
    const int s = (int)(gi / nf);
    double2 z = kg[f * mk + sidx[s]];
    if (sconj[s] && !no_parity) z.y = -z.y;
    const double2 c = scoef[s];
    // z / c
    const double den = c.x * c.x + c.y * c.y;
    const double2 q = make_double2((z.x * c.x + z.y * c.y) / den, (z.y * c.x - z.x * c.y) / den);
    const int inv = no_parity ? 0 : star_invert[s];
    double v = inv == 0 ? q.x : (inv == 1 ? q.x * sq2 : q.y * sq2);
    basis[(long)s * nf + f] = v * scale;
  }
}

// ----------------------------------------------------------------------------
// make_propg (src/step_mod.f90:109-129) for one block: omega on the grid, the
// factors in the sweeps' packed orders (unpack_index, unpack_kindex; mk
// z_factors).
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_make_propg(double ds, double b, const double* __restrict__ ksq,
                                                    long mk, const double* __restrict__ omega, long m,
                                                    int n1, int n2, int zw, double rM, double* __restrict__ e1,
                                                    double* __restrict__ e2, double* __restrict__ k1,
                                                    double* __restrict__ k2) {
  const double lap = ds * (b * b) / 6.0;
  const double pot = ds / 2.0;
  const double norm = (n2 > 1 ? 2.0 : 1.0) * rM;    // see task_k1
  const long n = m > mk ? m : mk;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA) {
    if (i < mk) {
      const long g = unpack_kindex(i, n1, n2, zw);
      const double k = g < 0 ? 0.0 : ksq[g];
      k1[i] = exp(-(lap * k)) / norm;
      k2[i] = exp(-(lap / 2.0 * k)) / norm;
    }
    if (i < m) {
      const double w = omega[unpack_index(i, n1, n2)];
      e1[i] = exp(-(pot * w));
      e2[i] = exp(-(pot / 2.0 * w));
    }
  }
}

// nf fields between the grid order (mg points each) and the sweeps' packed order
// (m each)
__global__ void __launch_bounds__(NTA) k_unpack(const double* __restrict__ packed, long m, int nf, int n1,
                                                int n2, double* __restrict__ grid) {
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < m * nf; i += (long)gridDim.x * NTA)
    grid[i / m * m + unpack_index(i % m, n1, n2)] = packed[i];
}
__global__ void __launch_bounds__(NTA) k_pack(const double* __restrict__ grid, long mg, long m, int nf, int n1,
                                              int n2, double* __restrict__ packed) {
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < m * nf; i += (long)gridDim.x * NTA)
    packed[i] = grid[i / m * mg + unpack_index(i % m, n1, n2)];
}

// ----------------------------------------------------------------------------
// Block partial sums of x (n values); out[blockIdx.x]
// ----------------------------------------------------------------------------
// Sum of v over the NTA threads of a workgroup, returned to every thread: a
// butterfly of wavefront shuffles inside each 64-lane wavefront, then the
// wavefront sums (in wavefront order) through LDS -- one workgroup barrier.
// The summation order is fixed, so the result is reproducible bit for bit.
__device__ __forceinline__ double block_sum(double v, double* red) {
  constexpr int W = 64, NW = NTA / W;
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, W);
  const int tid = threadIdx.x;
  if (tid % W == 0) red[tid / W] = v;
  __syncthreads();
  double r = red[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) r += red[w];
  __syncthreads();
  return r;
}

// (a contour point's n values on planes of `plane` points each, weighted where
// a stored plane stands for several)
__global__ void __launch_bounds__(NTA) k_partial_sum(const double* __restrict__ x, long n, int sym, int n3,
                                                     long plane, double* __restrict__ part) {
  __shared__ double red[NTA];
  double acc = 0.0;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA)
    acc += sym ? x[i] * sym_weight(sym, n3, (int)(i / plane)) : x[i];
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// out[slot] = sum(part[0..np)) * scale
__global__ void __launch_bounds__(NTA) k_final_sum(const double* __restrict__ part, int np,
                                                   double scale, double* __restrict__ out) {
  __shared__ double red[NTA];
  double acc = 0.0;
  for (int i = threadIdx.x; i < np; i += NTA) acc += part[i];
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) out[0] = s * scale;
}

// solvent Boltzmann factor partial sums: sum exp(-size*w)
__global__ void __launch_bounds__(NTA) k_partial_sum_exp(const double* __restrict__ w, double size,
                                                         long n, double* __restrict__ part) {
  __shared__ double red[NTA];
  double acc = 0.0;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA)
    acc += exp((-size) * w[i]);
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ----------------------------------------------------------------------------
// Solvent density (src/scf_mod.fp.f90:251-295):
//   rho += phi_s exp(-size w)/Q_s, with phi_s = Q_s e^{mu_s} in the grand ensemble.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_solvent_rho(const double* __restrict__ w, double size,
                                                     const double* __restrict__ qs, int ensemble,
                                                     const double* __restrict__ phimu, long n,
                                                     double* __restrict__ rho) {
  const double Q = qs[0];
  const double ph = ensemble == 1 ? Q * exp(phimu[1]) : phimu[0];
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA)
    rho[i] = rho[i] + ph * exp((-size) * w[i]) / Q;
}

// ----------------------------------------------------------------------------
// Simpson contour integration of one chain (src/scf_mod.fp.f90:362-424, 212-218):
//   rho_b = ds_b/3 [qf qr(ibgn) + qf qr(iend) + 4 sum_odd + 2 sum_even]
//   rho_grid(monomer_b) += phi * rho_b / N / Q
// in the reference's summation order per point; q is packed (kernels.hpp), m
// stored points, rho_grid in grid order, mg points per monomer.  A small grid
// has few wavefronts, and waits for one contour point's values after the
// other: eight of them are requested at a time (32 launches at 32^3, nine
// stored planes each: 6652 -> 5783 us for the grouped call).
// ----------------------------------------------------------------------------
struct SimpsonArgs {
  int nblk;
  int bnd[17];           // 0-based contour index of block starts, bnd[nblk] = ns
  double ds[16];
  int monomer[16];       // 0-based
  double chain_length;
  int ensemble;
};

__global__ void __launch_bounds__(NTA) k_simpson(const double* __restrict__ qf,
                                                 const double* __restrict__ qr, long m, long mg,
                                                 SimpsonArgs a, const double* __restrict__ Qp,
                                                 const double* __restrict__ phimu, int n1, int n2,
                                                 double* __restrict__ rho_grid) {
  const double Q = Qp[0];
  const double phi = a.ensemble == 1 ? Q * exp(phimu[1]) : phimu[0];
  for (long r = blockIdx.x * (long)NTA + threadIdx.x; r < m; r += (long)gridDim.x * NTA) {
    const long g = unpack_index(r, n1, n2);
    for (int b = 0; b < a.nblk; ++b) {
      const int ibgn = a.bnd[b], iend = a.bnd[b + 1];
      double acc = qf[(long)ibgn * m + r] * qr[(long)ibgn * m + r];
      acc = acc + qf[(long)iend * m + r] * qr[(long)iend * m + r];
#pragma unroll 8
      for (int jj = ibgn + 1; jj <= iend - 1; jj += 2)
        acc = acc + qf[(long)jj * m + r] * qr[(long)jj * m + r] * 4.0;
#pragma unroll 8
      for (int jj = ibgn + 2; jj <= iend - 2; jj += 2)
        acc = acc + qf[(long)jj * m + r] * qr[(long)jj * m + r] * 2.0;
      acc = acc * a.ds[b] / 3.0;
      acc = acc / a.chain_length / Q;
      double* rg = rho_grid + (long)a.monomer[b] * mg;
      rg[g] = rg[g] + phi * acc;
    }
  }
}

// ----------------------------------------------------------------------------
// Stress (src/scf_mod.fp.f90:505-530): for each contour point p of a chunk,
// dot(p, beta) = sum_star qr_basis(star) * dGsq(star, beta) * qf_basis(star).
// qfb/qrb hold star coefficients as (ld, N_star) Fortran order (p fastest),
// the layout k_kgrid_to_basis writes (qf and qr of a chunk may share one such
// array, ld = 2 np); dgsq is (N_star, ncp).  One workgroup per point;
// out(p, beta) at out[p*ncp + beta].
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_stress_dots(const double* __restrict__ qfb,
                                                     const double* __restrict__ qrb, int ld,
                                                     int nstar, const double* __restrict__ dgsq,
                                                     int ncp, double* __restrict__ out) {
  __shared__ double red[NTA];
  const int p = blockIdx.x;
  for (int beta = 0; beta < ncp; ++beta) {
    double acc = 0.0;
    for (int s = threadIdx.x; s < nstar; s += NTA)
      acc += qrb[(long)s * ld + p] * dgsq[(long)beta * nstar + s] * qfb[(long)s * ld + p];
    const double v = block_sum(acc, red);
    if (threadIdx.x == 0) out[(long)p * ncp + beta] = v;
  }
}

// ----------------------------------------------------------------------------
// divide_energy head/tail terms (src/scf_mod.fp.f90:631-662): partial sums of
// sum_r [qf>0 & qr>0] qf qr log(q_sel) over one contour point.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_partial_qlogq(const double* __restrict__ qf,
                                                       const double* __restrict__ qr, int use_qf,
                                                       long n, int sym, int n3, long plane,
                                                       double* __restrict__ part) {
  __shared__ double red[NTA];
  double acc = 0.0;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA) {
    const double a = qf[i], b = qr[i];
    if (a > 0.0 && b > 0.0) {
      const double v = a * b * log(use_qf ? a : b);
      acc += sym ? v * sym_weight(sym, n3, (int)(i / plane)) : v;
    }
  }
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}


// ----------------------------------------------------------------------------
// Adjoint support.
// k_simpson_lam: per block b of a chain (blockIdx.y), workgroup partials of
//   T_b = ds_b/3 sum_r lam_mon(b)(r) [qf qr(ibgn) + qf qr(iend) + 4 sum_odd + 2 sum_even]
// i.e. the block's Simpson density weighted by lam (part[b*gridDim.x + x]);
// sym, n3, plane: as k_partial_sum.
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(NTA) k_simpson_lam(const double* __restrict__ qf,
                                                     const double* __restrict__ qr, long m,
                                                     SimpsonArgs a, const double* __restrict__ lam, int sym,
                                                     int n3, long plane, double* __restrict__ part) {
  __shared__ double red[NTA];
  const int b = blockIdx.y;
  const int ibgn = a.bnd[b], iend = a.bnd[b + 1];
  const double* lm = lam + (long)a.monomer[b] * m;    // packed order, as q
  double tot = 0.0;
  for (long r = blockIdx.x * (long)NTA + threadIdx.x; r < m; r += (long)gridDim.x * NTA) {
    double acc = qf[(long)ibgn * m + r] * qr[(long)ibgn * m + r];
    acc += qf[(long)iend * m + r] * qr[(long)iend * m + r];
    for (int jj = ibgn + 1; jj <= iend - 1; jj += 2) acc += 4.0 * qf[(long)jj * m + r] * qr[(long)jj * m + r];
    for (int jj = ibgn + 2; jj <= iend - 2; jj += 2) acc += 2.0 * qf[(long)jj * m + r] * qr[(long)jj * m + r];
    tot += sym ? lm[r] * acc * sym_weight(sym, n3, (int)(r / plane)) : lm[r] * acc;
  }
  const double s = block_sum(tot * a.ds[b] / 3.0, red);
  if (threadIdx.x == 0) part[(long)b * gridDim.x + blockIdx.x] = s;
}

// Checkpointed storage: Simpson integrals of one recomputed contour segment.
// For the points s of [lo, hi) (and hi itself when `last`), held at
// qf/qr + (s - lo)*M, every block b containing s gets
//   blk[b*M + r] += ds_b/3 * w_b(s) * qf(s, r) * qr(s, r)
// (w_b: 1 at the block's ends, 4 at odd and 2 at even interior offsets).
__global__ void __launch_bounds__(NTA) k_simpson_seg(const double* __restrict__ qf,
                                                     const double* __restrict__ qr, long m,
                                                     SimpsonArgs a, int lo, int hi, int last,
                                                     double* __restrict__ blk) {
  const int s_end = last ? hi : hi - 1;
  for (long r = blockIdx.x * (long)NTA + threadIdx.x; r < m; r += (long)gridDim.x * NTA) {
    for (int sp = lo; sp <= s_end; ++sp) {
      const double v = qf[(long)(sp - lo) * m + r] * qr[(long)(sp - lo) * m + r];
      for (int b = 0; b < a.nblk; ++b) {
        const int b0 = a.bnd[b], b1 = a.bnd[b + 1];
        if (sp < b0 || sp > b1) continue;
        const double w = (sp == b0 || sp == b1) ? 1.0 : (((sp - b0) & 1) ? 4.0 : 2.0);
        blk[(long)b * m + r] += a.ds[b] / 3.0 * w * v;
      }
    }
  }
}

// rho_grid(monomer_b) += phi / (N Q) * blk_b for every block of a chain
__global__ void __launch_bounds__(NTA) k_block_rho(const double* __restrict__ blk, long m, long mg,
                                                   SimpsonArgs a, const double* __restrict__ Qp,
                                                   const double* __restrict__ phimu, int n1, int n2,
                                                   double* __restrict__ rho_grid) {
  const double Q = Qp[0];
  const double phi = a.ensemble == 1 ? Q * exp(phimu[1]) : phimu[0];
  for (long r = blockIdx.x * (long)NTA + threadIdx.x; r < m; r += (long)gridDim.x * NTA) {
    const long g = unpack_index(r, n1, n2);
    for (int b = 0; b < a.nblk; ++b) {
      double* rg = rho_grid + (long)a.monomer[b] * mg;
      rg[g] = rg[g] + phi * (blk[(long)b * m + r] / a.chain_length / Q);
    }
  }
}

// workgroup partials of sum x*y (sym, n3, plane: as k_partial_sum)
__global__ void __launch_bounds__(NTA) k_partial_dot(const double* __restrict__ x,
                                                     const double* __restrict__ y, long n, int sym, int n3,
                                                     long plane, double* __restrict__ part) {
  __shared__ double red[NTA];
  double acc = 0.0;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA)
    acc += sym ? x[i] * y[i] * sym_weight(sym, n3, (int)(i / plane)) : x[i] * y[i];
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// y += x (n values), x in the sweeps' packed order, y in grid order
__global__ void __launch_bounds__(NTA) k_axpy1(const double* __restrict__ x, long n, int n1, int n2,
                                               double* __restrict__ y) {
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA)
    y[unpack_index(i, n1, n2)] += x[i];
}

// Cell derivative of a |k|^2 gradient: for each cell parameter p (blockIdx.y),
// workgroup partials of sum_k kg(k) * dksq_p(k), with dksq_p(k) = Gbz^T dGG_p Gbz
// at the minimum-image wavevector Gbz of k (the make_dGsq form,
// src/basis_mod.f90:1993-2014, on the grid).  dGG(dim, dim, ncp) Fortran order.
__global__ void __launch_bounds__(NTA) k_dksq_dot(GeomArgs g, const double* __restrict__ dgg,
                                                  const double* __restrict__ kg,
                                                  double* __restrict__ part) {
  __shared__ double red[NTA];
  const int p = blockIdx.y, dim = g.dim;
  const long mk = (long)(g.n1 / 2 + 1) * g.n2 * g.n3;
  const double* d = dgg + (long)p * dim * dim;
  double acc = 0.0;
  for (long idx = blockIdx.x * (long)NTA + threadIdx.x; idx < mk; idx += (long)gridDim.x * NTA) {
    int best[3];
    (void)g_to_bz_point(g, idx, best);
    double v = 0.0;
    for (int jj = 0; jj < dim; ++jj)
      for (int kk = 0; kk < dim; ++kk) v += (double)best[jj] * (double)best[kk] * d[jj + dim * kk];
    acc += kg[idx] * v;
  }
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) part[(long)p * gridDim.x + blockIdx.x] = s;
}

// nf grid fields whose stored planes (symmetric planes, kernels.hpp) are set:
// the others from them
__global__ void __launch_bounds__(NTA) k_sym_expand(double* __restrict__ f, int nf, int sym, int n1, int n2,
                                                    int n3) {
  const long m = (long)n1 * n2 * n3, m0 = (long)n1 * n2 * sym_planes(sym, n3);
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < (m - m0) * nf; i += (long)gridDim.x * NTA) {
    double* g = f + i / (m - m0) * m;
    const long p = m0 + i % (m - m0);
    g[p] = g[sym_point(sym, n1, n2, n3, p)];
  }
}
// one packed contour point on its stored planes -> the whole field, in packed
// (pack) or grid order
__global__ void __launch_bounds__(NTA) k_sym_point(const double* __restrict__ q, long qs, int sym, int n1, int n2,
                                                   int n3, int pack, double* __restrict__ out, long os) {
  const long m = (long)n1 * n2 * n3;
  q += blockIdx.y * qs;
  out += blockIdx.y * os;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < m; i += (long)gridDim.x * NTA) {
    const long g = pack ? unpack_index(i, n1, n2) : i;
    out[i] = q[pack_index(sym_point(sym, n1, n2, n3, g), n1, n2)];
  }
}
// flag[0] = epoch if a field has a value further than tol from that of its
// stored point: it is not symmetric
__global__ void __launch_bounds__(NTA) k_sym_check(const double* __restrict__ f, int nf, int sym, int n1, int n2,
                                                   int n3, double tol, double epoch, double* __restrict__ flag) {
  const long m = (long)n1 * n2 * n3, m0 = (long)n1 * n2 * sym_planes(sym, n3);
  bool bad = false;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < (m - m0) * nf; i += (long)gridDim.x * NTA) {
    const double* g = f + i / (m - m0) * m;
    const long p = m0 + i % (m - m0);
    bad = bad || !(fabs(g[p] - g[sym_point(sym, n1, n2, n3, p)]) <= tol);
  }
  if (bad) flag[0] = epoch;
}

// The check for fields given on the grid, which need not have the symmetry
// anywhere: every pair of sym_partner, against tol times the fields' largest
// modulus.  Workgroup maxima of |x|, then the check (part: np maxima).
__global__ void __launch_bounds__(NTA) k_partial_absmax(const double* __restrict__ x, long n,
                                                        double* __restrict__ part) {
  __shared__ double red[NTA];
  double v = 0.0;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA) v = fmax(v, fabs(x[i]));
  red[threadIdx.x] = v;
  __syncthreads();
  if (threadIdx.x) return;
  for (int i = 1; i < NTA; ++i) v = fmax(v, red[i]);
  part[blockIdx.x] = v;
}
__global__ void __launch_bounds__(NTA) k_sym_check_grid(const double* __restrict__ f, int nf, int sym, int n1,
                                                        int n2, int n3, const double* __restrict__ part, int np,
                                                        double tol, double epoch, double* __restrict__ flag) {
  const long m = (long)n1 * n2 * n3;
  double big = 0.0;
  for (int i = 0; i < np; ++i) big = fmax(big, part[i]);
  bool bad = false;
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < m * nf; i += (long)gridDim.x * NTA) {
    const double* g = f + i / m * m;
    bad = bad || !(fabs(g[i % m] - g[sym_partner(sym, n1, n2, n3, i % m)]) <= tol * big);
  }
  if (bad) flag[0] = epoch;
}

// constant fill
__global__ void __launch_bounds__(NTA) k_fill(double* __restrict__ x, long n, double v) {
  for (long i = blockIdx.x * (long)NTA + threadIdx.x; i < n; i += (long)gridDim.x * NTA) x[i] = v;
}

}  // namespace pscf
