// Host side of libpscf_hip: plans, system state and the C ABI of
// include/pscf_hip.h.  All compute runs in the gfx950 kernels of
// kernels.hpp / kernels_aux.hpp.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <cstdlib>
#include <exception>
#include <thread>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/pscf_hip.h"
#include "kernels.hpp"
#include "kernels_aux.hpp"

using namespace pscf;

namespace {

thread_local std::string g_err;

struct Fail {
  std::string msg;
};

#define HIPCHK(expr)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw Fail{std::string(#expr) + ": " + hipGetErrorString(e_)};                        \
  } while (0)

#define REQUIRE(cond, msg)                  \
  do {                                                                                      \
    if (!(cond)) throw Fail{msg};           \
  } while (0)

template <class F>
int guarded(F&& f) {
  try {
    g_err.clear();
    f();
    return 0;
  } catch (const Fail& e) {
    g_err = e.msg;
    return 1;
  } catch (const std::exception& e) {
    g_err = e.what();
    return 2;
  }
}

// ------------------------------------------------------------ device memory
template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void alloc(size_t count) {
    if (count == n && p) return;
    release();
    if (count == 0) return;
    HIPCHK(hipMalloc((void**)&p, count * sizeof(T)));
    n = count;
  }
  void upload(const T* h, size_t count, hipStream_t s) {
    alloc(count);
    HIPCHK(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
  }
};

// Page-locked host staging: copies between it and the device are truly
// asynchronous, so a stream's work can be queued for many systems before
// one synchronisation (a copy from pageable memory waits for the stream).
template <class T>
struct HostPin {
  T* p = nullptr;
  size_t n = 0;
  HostPin() = default;
  HostPin(const HostPin&) = delete;
  HostPin& operator=(const HostPin&) = delete;
  ~HostPin() {
    if (p) (void)hipHostFree(p);
  }
  void alloc(size_t count) {
    if (count <= n && p) return;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    n = 0;
    HIPCHK(hipHostMalloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T), 0));
    n = count;
  }
};

// --------------------------------------------------------------- twiddles
// tw[m] = exp(-2 pi i m / N), m < N, computed with the angle reduced to the
// first octant so that each entry is correctly rounded to ~1 ulp.
std::mutex g_tw_mutex;
std::map<int, double2*> g_tw;

void host_twiddles(int n, double2* h) {
  for (int m = 0; m < n; ++m) {
    // angle = 2 pi m / n; use symmetric reduction for accuracy
    long double a = 2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)n;
    h[m] = make_double2((double)cosl(a), (double)(-sinl(a)));
  }
}

const double2* twiddles(int n) {
  std::lock_guard<std::mutex> lk(g_tw_mutex);
  auto it = g_tw.find(n);
  if (it != g_tw.end()) return it->second;
  std::vector<double2> h(z_tables(n));      // of length n, then n/2
  host_twiddles(n, h.data());
  if (n > 1) host_twiddles(n / 2, h.data() + n);
  double2* d = nullptr;
  HIPCHK(hipMalloc((void**)&d, sizeof(double2) * h.size()));
  HIPCHK(hipMemcpy(d, h.data(), sizeof(double2) * h.size(), hipMemcpyHostToDevice));
  g_tw[n] = d;
  return d;
}

// ------------------------------------------------------- kernel dispatch
using StepPlaneFn = void (*)(const StepTask*, int, const double2*, const double2*);
using StepZFn = void (*)(const StepTask*, int, int, int, const double2*, const double2*);
using SweepFn = void (*)(const StepTask*, int, const double2*, const double2*, const double2*);
using R2CFn = void (*)(const double*, long, double2*, long, const double2*, const double2*,
                       const int*, int);
using C2RFn = void (*)(const double2*, long, double*, long, double, const double2*, const double2*);
using R2CColsFn = void (*)(const double*, const double*, long, double2*, long, const double2*,
                           const double2*, const int*, int);
using ZfftFn = void (*)(double2*, long, int, const double2*);
using ZColsFn = void (*)(int, const double2*, long, int, double2*, long, int, int, const int2*, const int2*,
                         const double2*, const double2*);
using C2CFn = void (*)(double2*, long, const double2*, const double2*);

struct PlaneSet {
  int nt = 0, nt_c2c = 0;     // workgroup sizes of the transform kernels (plane_nt, c2c_nt)
  int nt_step = 0;            // workgroup size of the step plane kernels
  int ajobs = 0;              // workgroups per plane of k_step_a (0: by occupancy)
  size_t lds_step = 0;        // LDS bytes of a step plane workgroup
  // [adjoint sweeps]: k_step_a with one and two workgroups per plane, k_step_c,
  // and k_step_c with shared exchange/plane LDS (wide launches)
  StepPlaneFn a1[2] = {}, a[2] = {}, c[2] = {}, c_wide[2] = {};
  SweepFn sweep = nullptr;    // whole sweeps of grids with N3 = 1, where compiled
  int nt_sweep = 0;
  R2CFn r2c = nullptr;
  R2CColsFn r2c_cols = nullptr;   // register-line XY pass of scf_stress's transforms
  C2RFn c2r = nullptr;
  C2CFn c2c_f = nullptr, c2c_i = nullptr;
};
struct ZSet {
  int nt_half = 0, nt_full = 0;   // workgroup sizes (zcol_nt for N1/2+1 and N1 wide rows)
  int nt_step = 0;                // workgroup size of the step z kernel
  int nt_cols = 0;                // of the stress transform's z kernel
  int zw = 1;                     // their column slots and columns per workgroup
  StepZFn z[4] = {};              // by the flags Z_ADJ, Z_SYM
  StepZFn z_half = nullptr;       // Z_HALF, where N3/2 has a line plan
  int nt_half_step = 0;
  ZfftFn half_f = nullptr, half_i = nullptr, full_f = nullptr, full_i = nullptr;
  ZColsFn cols_f = nullptr;       // register-line forward z pass of scf_stress's spectra
};

// complex words that fit one workgroup's LDS (160 KB on gfx950)
constexpr bool lds_fits(long words) { return words * 16 <= 160L * 1024; }

template <int A, int B>
PlaneSet make_plane() {
  PlaneSet s;
  s.nt = plane_nt(A, B);
  s.nt_c2c = c2c_nt(A, B);
  s.nt_step = StepPlane<A, B>::NT;
  s.ajobs = plan_ajobs(A);
  s.lds_step = StepPlane<A, B>::LDS;
  s.a[0] = k_step_a<A, B, false, false>;
  s.a[1] = k_step_a<A, B, false, true>;
  s.a1[0] = k_step_a<A, B, true, false>;
  s.a1[1] = k_step_a<A, B, true, true>;
  s.c[0] = k_step_c<A, B, false>;
  s.c[1] = k_step_c<A, B, true>;
  // at most 128 VGPRs where that costs no spills and frees a resident
  // workgroup (edges 48 to 64; lines of 40 points spill under the cap)
  constexpr int wpe = A >= 48 && A <= 64 && B >= 48 && B <= 64 ? 4 : 1;
  s.c_wide[0] = k_step_c<A, B, false, 40 * 1024, wpe>;
  s.c_wide[1] = k_step_c<A, B, true, 40 * 1024, wpe>;
  if constexpr (SweepPlane<A, B>::OK) {
    s.sweep = k_sweep_plane<A, B>;
    s.nt_sweep = SweepPlane<A, B>::NT;
  }
  s.r2c = k_plane_r2c<A, B>;
  s.r2c_cols = k_plane_r2c_cols<A, B>;
  s.c2r = k_plane_c2r<A, B>;
  if constexpr (lds_fits(A * B + A + B)) {    // a full complex plane in LDS
    s.c2c_f = k_plane_c2c<A, B, -1>;
    s.c2c_i = k_plane_c2c<A, B, +1>;
  }
  return s;
}
template <int A, int C>
ZSet make_z() {
  ZSet s;
  s.nt_half = zcol_nt(A / 2 + 1, C);
  s.nt_full = zcol_nt(A, C);
  s.nt_step = StepZ<C>::NT;
  s.nt_cols = StepZ<C>::NTC;
  s.zw = StepZ<C>::ZW;
  s.z[Z_PLAIN] = k_step_z<A, C, Z_PLAIN>;
  s.z[Z_ADJ] = k_step_z<A, C, Z_ADJ>;
  if constexpr (C > 1) {
    s.z[Z_SYM] = k_step_z<A, C, Z_SYM>;
    s.z[Z_ADJ | Z_SYM] = k_step_z<A, C, (Z_ADJ | Z_SYM)>;
    if constexpr (z_half_ok(C)) {
      s.z_half = k_step_z<A, C, (Z_SYM | Z_HALF)>;
      s.nt_half_step = StepZ<C, C / 2>::NT;
    }
  }
  s.half_f = k_zfft<A / 2 + 1, C, -1>;
  s.cols_f = k_zfwd_cols<C>;
  s.half_i = k_zfft<A / 2 + 1, C, +1>;
  if constexpr (lds_fits(A * C + C)) {        // full complex rows in LDS
    s.full_f = k_zfft<A, C, -1>;
    s.full_i = k_zfft<A, C, +1>;
  }
  return s;
}

// Grid edges with compiled kernels.  A grid N1 x N2 x N3 runs when its XY
// plane (N1, N2) and its XZ pair (N1, N3) both have kernels: edges from this
// list, equal (cubic, square; 1D/2D grids have unused dimensions 1) or
// within a factor 2 of each other (PSCF_GRID_PAIRS: tetragonal, hexagonal,
// orthorhombic and rectangular cells on anisotropic grids).
#ifdef PSCF_TUNE_BUILD
// tuning builds (pscf_amd/autotune.py): the timed cubic lengths only
#define PSCF_GRID_SIZES(X) X(32) X(48) X(56) X(64) X(96) X(128)
#define PSCF_GRID_PAIRS(X)
#else
#define PSCF_GRID_SIZES(X) X(8) X(12) X(16) X(20) X(24) X(28) X(32) X(40) X(48) X(56) X(64) X(96) \
   X(128)
#define PSCF_GRID_PAIRS(X) X(28, 56) X(56, 28) X(48, 56) X(56, 48) X(56, 64) X(64, 56) X(64, 128) \
   X(128, 64) X(8, 12) X(8, 16) X(12, 8) X(12, 16) X(12, 20) X(12, 24) X(16, 8) \
   X(16, 12) X(16, 20) X(16, 24) X(16, 32) X(20, 12) X(20, 16) X(20, 24) X(20, 32) X(20, 40) \
   X(24, 12) X(24, 16) X(24, 20) X(24, 32) X(24, 40) X(24, 48) X(32, 16) X(32, 20) X(32, 24) \
   X(32, 40) X(32, 48) X(32, 64) X(40, 20) X(40, 24) X(40, 32) X(40, 48) X(40, 64) X(48, 24) \
   X(48, 32) X(48, 40) X(48, 64) X(48, 96) X(64, 32) X(64, 40) X(64, 48) X(64, 96) X(96, 48) \
   X(96, 64)
#endif

const std::map<std::pair<int, int>, PlaneSet>& plane_table() {
  static const std::map<std::pair<int, int>, PlaneSet> t = [] {
    std::map<std::pair<int, int>, PlaneSet> m;
#define PSCF_PL(n)                          \
  m[{n, n}] = make_plane<n, n>();           \
  m[{n, 1}] = make_plane<n, 1>();
    PSCF_GRID_SIZES(PSCF_PL)
#undef PSCF_PL
#define PSCF_PL2(a, b) m[{a, b}] = make_plane<a, b>();
    PSCF_GRID_PAIRS(PSCF_PL2)
#undef PSCF_PL2
    return m;
  }();
  return t;
}
const std::map<std::pair<int, int>, ZSet>& z_table() {
  static const std::map<std::pair<int, int>, ZSet> t = [] {
    std::map<std::pair<int, int>, ZSet> m;
#define PSCF_Z(n)                 \
  m[{n, n}] = make_z<n, n>();     \
  m[{n, 1}] = make_z<n, 1>();
    PSCF_GRID_SIZES(PSCF_Z)
#undef PSCF_Z
#define PSCF_Z2(a, b) m[{a, b}] = make_z<a, b>();
    PSCF_GRID_PAIRS(PSCF_Z2)
#undef PSCF_Z2
    return m;
  }();
  return t;
}

int grid_blocks(long n) {
  long b = (n + NTA - 1) / NTA;
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (int)b;
}

// ------------------------------------------------------------- geometry
struct Grid {
  int n1 = 0, n2 = 0, n3 = 0, dim = 0, n1h = 0;
  int nl = 1;                 // packed rows per plane
  long m = 0, mk = 0;
  long mc = 0;                // complex words of a packed spectrum
  long mf = 0;                // reciprocal-space factors of a block (z_factors)
  // symmetric planes (kernels.hpp): the code (0: none), and what the sweeps
  // store: np planes, ms points of a real field (mc counts those planes too)
  int sym = 0, np = 0;
  long ms = 0;
  const PlaneSet* pl = nullptr;
  const ZSet* zs = nullptr;
  long cus = 0;               // compute units
  long plane_slots = 0;       // plane workgroups resident at once (CUs x LDS fit)
  const double2 *tw1 = nullptr, *tw2 = nullptr, *tw3 = nullptr, *twl = nullptr;

  // with_tw false: the twiddle tables are left to the caller (no device allocation)
  void init(const int ng[3], int d, bool with_tw = true) {
    n1 = ng[0];
    n2 = ng[1];
    n3 = ng[2];
    dim = d;
    REQUIRE(n1 >= 2 && n2 >= 1 && n3 >= 1, "invalid grid dimensions");
    REQUIRE(n1 % 2 == 0, "the first grid dimension must be even");
    n1h = n1 / 2 + 1;
    m = (long)n1 * n2 * n3;
    mk = (long)n1h * n2 * n3;
    nl = n2 > 1 ? n2 / 2 : 1;
    set_sym(0);
    auto ip = plane_table().find({n1, n2});
    auto iz = z_table().find({n1, n3});
    char buf[160];
    snprintf(buf, sizeof buf, "grid %dx%dx%d has no compiled gfx950 kernels", n1, n2, n3);
    REQUIRE(ip != plane_table().end() && iz != z_table().end(), buf);
    pl = &ip->second;
    zs = &iz->second;
    mf = z_factors(n1, n2, n3, zs->zw);
    int dev = 0, cus = 0, lds_cu = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHK(hipDeviceGetAttribute(&lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev));
    this->cus = cus;
    plane_slots = (long)cus * std::max<long>(1, (long)lds_cu / (long)pl->lds_step);
    if (with_tw) {
      tw1 = twiddles(n1);
      tw2 = twiddles(n2);
      tw3 = twiddles(n3);
      twl = twiddles(nl);
    }
  }

  void set_sym(int code) {
    sym = code;
    np = sym_planes(code, n3);
    ms = (long)n1 * n2 * np;
    mc = (long)plane_words(n1, nl) * np;
  }

  // step kernels over ntask sweep tasks at launch step j (run_sweeps' order:
  // step_a, step_z kind 0 (2 jobs), step_c (2 jobs), step_z kind 1)
  // With events (t0, t1), the launch records them at the start and the end of
  // the kernel's execution (hipExtLaunchKernelGGL: no launch gaps included).
  // adj: the tasks are adjoint or recomputed sweeps
  // half_z: every task's planes allow the half-length z lines (sym_half)
  void step_z(const StepTask* tasks, int ntask, int j, int kind, int jobs, bool adj, bool half_z, hipStream_t s,
              hipEvent_t t0 = nullptr, hipEvent_t t1 = nullptr) const {
    const dim3 grid(z_tiles(n1, nl, zs->zw), ntask, jobs);
    const bool half = !adj && half_z && zs->z_half;
    const StepZFn k = half ? zs->z_half : zs->z[(adj ? Z_ADJ : 0) | (sym ? Z_SYM : 0)];
    const dim3 nt(half ? zs->nt_half_step : zs->nt_step);
    if (t0)
      hipExtLaunchKernelGGL(k, grid, nt, 0, s, t0, t1, 0, tasks, j, n2, kind, tw2, tw3);
    else
      hipLaunchKernelGGL(k, grid, nt, 0, s, tasks, j, n2, kind, tw2, tw3);
  }
  // launches that need more than two rounds of resident workgroups take the
  // form whose smaller LDS footprint lets more of them reside on a CU at once
  void step_c(const StepTask* tasks, int ntask, int j, bool adj, hipStream_t s, hipEvent_t t0 = nullptr,
              hipEvent_t t1 = nullptr) const {
    const StepPlaneFn k = (long)np * ntask * 2 > 2 * plane_slots ? pl->c_wide[adj] : pl->c[adj];
    if (t0)
      hipExtLaunchKernelGGL(k, dim3(np, ntask, 2), dim3(pl->nt_step), 0, s, t0, t1, 0, tasks, j,
                            tw1, twl);
    else
      hipLaunchKernelGGL(k, dim3(np, ntask, 2), dim3(pl->nt_step), 0, s, tasks, j, tw1, twl);
  }
  // real (nb arrays, stride m) -> half spectra (stride mk)
  void r2c(const double* in, double2* out, int nb, hipStream_t s) const {
    hipLaunchKernelGGL(pl->r2c, dim3(n3, nb), dim3(pl->nt), 0, s, in, m, out, mk, tw1, tw2,
                       (const int*)nullptr, 0);
    if (n3 > 1)
      hipLaunchKernelGGL(zs->half_f, dim3(n2, nb), dim3(zs->nt_half), 0, s, out, mk, n2, tw3);
  }
  // contour points in packed order (nb arrays at `in` and, when in2 is given,
  // nb more at in2, outputs after the first nb) -> their half spectra on ncol
  // columns, out[b][z][c]; the XY pass keeps the nin packed columns (cpos:
  // packed-plane entry -> column or -1) that those are split from (src, cols:
  // k_zfwd_cols) in `work`.  Both passes run on the step kernels' lines.
  void r2c_cols(const double* in, const double* in2, double2* work, double2* out, int nb, const int* cpos,
                int nin, int ncol, const int2* src, const int2* cols, hipStream_t s) const {
    const int sets = in2 ? 2 : 1;
    hipLaunchKernelGGL(pl->r2c_cols, dim3(np, nb, sets), dim3(pl->nt_step), 0, s, in, in2, ms, work,
                       (long)np * nin, tw1, twl, cpos, nin);
    hipLaunchKernelGGL(zs->cols_f, dim3((unsigned)((ncol + zs->zw - 1) / zs->zw), nb * sets),
                       dim3(zs->nt_cols), 0, s, sym, work, (long)np * nin, nin, out, (long)n3 * ncol, ncol, n2,
                       src, cols, tw2, tw3);
  }
  // half spectra -> real, in place on `in` for the z pass
  void c2r(double2* in, double* out, int nb, double scale, hipStream_t s) const {
    if (n3 > 1)
      hipLaunchKernelGGL(zs->half_i, dim3(n2, nb), dim3(zs->nt_half), 0, s, in, mk, n2, tw3);
    hipLaunchKernelGGL(pl->c2r, dim3(n3, nb), dim3(pl->nt), 0, s, in, mk, out, m, scale, tw1, tw2);
  }
  void c2c(double2* data, int sign, hipStream_t s) const {
    REQUIRE(pl->c2c_f && (n3 == 1 || zs->full_f),
            "the complex FFT (fftc) is not compiled for this grid: its full complex planes "
            "exceed one workgroup's LDS");
    hipLaunchKernelGGL(sign < 0 ? pl->c2c_f : pl->c2c_i, dim3(n3, 1), dim3(pl->nt_c2c), 0, s, data,
                       m, tw1, tw2);
    if (n3 > 1)
      hipLaunchKernelGGL(sign < 0 ? zs->full_f : zs->full_i, dim3(n2, 1), dim3(zs->nt_full), 0, s,
                         data, m, n2, tw3);
  }
};

struct Stream {
  hipStream_t s = nullptr;
  Stream() { HIPCHK(hipStreamCreate(&s)); }
  ~Stream() {
    if (s) (void)hipStreamDestroy(s);
  }
  void sync() const { HIPCHK(hipStreamSynchronize(s)); }
};

// -------------------------------------------------- allocation-free step
// Device scratch of pscf_step_exp_noalloc (the step's propagator factors,
// spectra, full-step result, two contour points, task record and twiddle
// tables), 20 MiB: enough for a 64^3 grid.  Every device the library runs
// on holds its own copy until the process ends; calls on one device share
// it, so calls that overlap on one device race.
constexpr size_t kScratchDoubles = (size_t)20 * 1024 * 1024 / sizeof(double);
static __device__ __align__(256) double scratch[kScratchDoubles];

// Device address of `scratch` on each device, looked up once per device with
// that device current; host code uses it (the name `scratch` in host code is
// a host-side stand-in, not a device address).
std::mutex g_scratch_mutex;
std::map<int, double*> g_scratch_ptr;

double* scratch_on_current_device() {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_scratch_mutex);
  auto it = g_scratch_ptr.find(dev);
  if (it != g_scratch_ptr.end()) return it->second;
  double* ptr = nullptr;
  HIPCHK(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
  REQUIRE(ptr != nullptr, "no device address for the step scratch");
  g_scratch_ptr[dev] = ptr;
  return ptr;
}

// true when p is device memory of the current device (a host pointer handed
// to a kernel would fault the GPU)
bool is_device_pointer(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice;
}

// the single block of a one-step task with factors at f (pscf_step_*)
void one_step_blocks(StepTask& t, const Grid& g, const double* f) {
  t.nblk = 1;
  t.bnd[0] = 0;
  for (int b = 1; b <= MAXBLK; ++b) t.bnd[b] = 1;
  t.fac = f;
  t.fm = g.ms;
  t.fk = g.mf;
}

// ------------------------------------------------------------ fft plan
struct FftPlan {
  Grid g;
  Stream st;
  DevBuf<double> r;
  DevBuf<double2> k, c;
};

// -------------------------------------------------------- standalone step
struct StepState {
  Grid g;
  Stream st;
  DevBuf<double> fac;      // e1, e2 (m each), k1, k2 (mk each)
  DevBuf<double> slab;     // 2 points
  DevBuf<double> q1;
  DevBuf<double2> abc;     // A, B, C
  DevBuf<double> ksq, om;
  DevBuf<StepTask> task;
  bool have_propg = false;
};

// ---------------------------------------------------------------- system
struct ChainDev {
  int nblk = 0, ns = 0;
  int bnd[MAXBLK + 1] = {0};
  double ds[MAXBLK] = {0};
  int mon[MAXBLK] = {0};   // 0-based
  double length = 0;
  DevBuf<double> qf, qr;   // stored contour points: (ns+1) * m, or nslot * m when checkpointed
  DevBuf<double> fac;      // per block: e1, e2 (m), k1, k2 (mk)
  // checkpointed storage (system stride K > 0): slot of every stored point
  // (s % K == 0 or (ns - s) % K == 0), -1 for the others
  std::vector<int> slot;
  int nslot = 0;
  DevBuf<int> dslot;
  DevBuf<double> seg;      // recomputed segments: 4 x segpts points (f, r; two sides)
  int segpts = 0;          // points per segment buffer: min(K, ns) + 1
  DevBuf<double> blk;      // per block: Simpson integral of the last density() (m each)
  const double* point(int dir, int sp) const {    // stored contour point, or null
    const int sl = slot.empty() ? sp : slot[sp];
    return sl < 0 ? nullptr : (dir > 0 ? qf.p : qr.p) + (size_t)sl * m_;
  }
  long m_ = 0;
};

// Segment schedule of the checkpointed mode for stride K: round r recomputes,
// per chain, the "forward-side" segment R_r = [rK, min((r+1)K, ns)] and the
// "backward-side" segment F_r = [max(0, ns-(r+1)K), ns-rK] from checkpoints,
// into the chain's segment buffers; maps[(r*nchain + c)*2 + side] maps a
// contour point of the chain to its slot in that segment (-1 outside).
struct CkPlan {
  int nround = 0;
  std::vector<int> len;          // per round: longest segment over the chains
  DevBuf<int> maps;
  std::vector<size_t> map_off;   // per (round, chain, side) offset into maps
};

// Adjoint (reverse-mode) sweep state of a system: per chain four sweep tasks
// (adjoint of q, recomputed q, adjoint of q-dagger, recomputed q-dagger),
// their work and kept-field buffers, and the gradient accumulators.
struct AdjState {
  uint64_t id = 0;         // distinct for every AdjState made
  int ntask = 0, npair = 0;
  bool with_k = false;
  DevBuf<double> keep;     // per task: U, V, W (m each); adjoint tasks also 2 m of kept inputs
  DevBuf<double> lam;      // dL/drho_grid of the current call (m per monomer)
  DevBuf<double> scal;     // per chain: source coefficient, end term
  DevBuf<double2> keepk;   // per task: 3 spectra (mk each), with_k only
  DevBuf<double2> abc;     // per task: A, B, C (mk each)
  DevBuf<double> q1;       // per task (m)
  DevBuf<double> gblk;     // per chain and block: omega gradient (m)
  DevBuf<double> kblk;     // per chain and block: |k|^2 gradient (mk), with_k only
  DevBuf<StepTask> tasks;
  DevBuf<int2> pairs;
  DevBuf<double> part;     // reduction partials, and one result slot at the end
  // checkpointed storage: per round the recomputation tasks (4 per chain) and
  // the adjoint tasks re-pointed at that round's segments (4 per chain)
  DevBuf<StepTask> ck_rec, ck_adj;
  DevBuf<double2> rec_abc;
  DevBuf<double> rec_q1;
  std::vector<StepTask> h_tasks, h_ck_rec, h_ck_adj;
  std::vector<int2> h_pairs;
  std::vector<size_t> blk_off;   // per chain: first block in gblk/kblk
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~AdjState() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
};

struct Multi;

struct System {
  Grid g;
  Stream st;
  // basis
  int nstar = 0, nwave = 0;
  DevBuf<int> star_of_wave, star_invert, wtab, kwave, sconj;
  DevBuf<double2> coeff, scoef;
  DevBuf<long> sidx;
  // stress transforms keep only the ncol half-spectrum columns (kx, ky)
  // holding a star's representative wave, and the nin packed columns they are
  // split from; per star the index of its representative at (z, column)
  int ncol = 0, nin = 0;
  DevBuf<int> scpos;             // packed-plane entry -> its position among the nin, or -1
  DevBuf<int2> ssrc, scolk;      // per column: its two packed positions, its (kx, ky)
  DevBuf<long> sidx_c;
  std::vector<int> h_wave, h_wave_of_star, h_star_of_wave, h_star_invert;
  std::vector<int> h_wtab;   // dense which_wave table (1-based wave, 0: none) over gmin + [0, gext)
  std::vector<double2> h_coeff;
  int gmin[3] = {0, 0, 0}, gext[3] = {1, 1, 1};
  bool have_basis = false, have_cell = false;
  // geometry
  double gb[9] = {0};
  DevBuf<double> ksq;
  // chemistry
  int nmon = 0, nchain = 0, nsolv = 0, ensemble = 0;
  std::vector<double> kuhn, solv_size, chi;
  std::vector<int> solv_mon;
  std::vector<std::vector<std::pair<int, double>>> blocks;  // (monomer 0-based, length)
  // chain lengths N of the normalisations (chemistry_mod's chain_length:
  // the block-length sums when the chemistry is set, src/chemistry_mod.f90:
  // 272-276, 560-566; the driver may hand its own, which RESCALE leaves
  // unscaled, :1344-1361)
  std::vector<double> chain_length;
  std::vector<std::unique_ptr<ChainDev>> chains;
  bool have_chem = false, started = false;
  // work
  DevBuf<double> omega_in, rho_out, omega_grid, rho_grid, part, qdev, basis_tmp, chem_dev;
  DevBuf<double2> kwork;
  DevBuf<double2> abc;     // 3 * mk per task
  DevBuf<double> q1;       // m per task
  DevBuf<StepTask> tasks;
  std::vector<StepTask> h_tasks;
  std::vector<double> h_Q, h_Qs, h_chem;
  // staging of the per-call host inputs and outputs (see HostPin)
  HostPin<double> pin_in, pin_chem, pin_q, pin_rho, pin_dgsq, pin_dots;
  double* rho_dst = nullptr;     // where density_finish copies the rho stars
  bool have_density = false;
  // density() evaluations so far: the adjoint of a forward is valid only while
  // no later density() has overwritten the contour slabs it reads
  uint64_t density_gen = 0;
  // ensemble of the chain prefactors of the last density(): the reference
  // updates phi_chain = Q e^mu first only when qout is present
  // (src/scf_mod.fp.f90:202-205); otherwise rho uses the given phi_chain
  int chain_ens = 0;
  // generations of the basis and of the chain discretisation (density_many's
  // copies of the system are rebuilt when they change)
  uint64_t gen_basis = 0, gen_start = 0;
  std::unique_ptr<Multi> multi;
  // symmetric planes of the star basis (code, 0: none; found by detect_sym)
  // and, per star, a bound of its function's modulus
  int sym_code = 0;
  std::vector<double> star_bound;
  bool no_sym = false;           // store every plane whatever the basis
  bool sym_bad = false;          // an omega field of this basis was not symmetric
  double sym_epoch = 0.0;        // density() calls checked so far
  // the same system with every plane stored, for grid fields that do not have
  // the basis's symmetry (density on grids, reverse mode); made when needed.
  // last: it holds the results of the last density()
  std::unique_ptr<System> full;
  uint64_t full_basis = 0, full_start = 0;
  System* last = nullptr;
  ~System();
  // contour sweeps of one density() captured once as a HIP graph
  int ntask = 0, max_ns = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  bool use_graph = true;
  // optional timing (HIP events on the system stream): mode 1 brackets the
  // sweep graph (time per contour step); mode 2 launches the sweeps eagerly
  // with an event around every kernel (per-kernel durations)
  int profile = 0;
  std::vector<hipEvent_t> ev;
  double prof_ms[5] = {0, 0, 0, 0, 0};  // step A, Z0, C, Z1, whole sweep
  long prof_n[5] = {0, 0, 0, 0, 0};     // launches (kinds 0-3), contour steps (4)
  void drop_graph() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    graph_exec = nullptr;
    graph = nullptr;
  }
  std::unique_ptr<AdjState> adj;
  // checkpointed contour storage
  int ck_stride = 0;
  double chain_step = 0.0;
  CkPlan ck;
  DevBuf<StepTask> ck_tasks;     // Simpson recomputation tasks: per round 2 per chain
  hipGraph_t ck_graph = nullptr;
  hipGraphExec_t ck_exec = nullptr;
  void drop_ck_graph() {
    if (ck_exec) (void)hipGraphExecDestroy(ck_exec);
    if (ck_graph) (void)hipGraphDestroy(ck_graph);
    ck_exec = nullptr;
    ck_graph = nullptr;
  }
  // stress work
  DevBuf<double> sbuf;     // real chunk
  DevBuf<double2> skbuf;   // spectra chunk
  DevBuf<double> sbasis;   // star coefficients chunk
  DevBuf<double> dgsq, sdots;
};

template <class T>
T* from_handle(int64_t h, const char* what) {
  REQUIRE(h != 0, std::string("null ") + what + " handle");
  return reinterpret_cast<T*>(h);
}

// ----------------------------------------------------------- chain rule
// src/chain_mod.f90:141-156
void discretize(int nblk, const double* L, double ds0, int order, int* bgn, double* bds) {
  int bgns = 1;
  bgn[0] = bgns;
  for (int i = 0; i < nblk; ++i) {
    int iblk = (int)(L[i] / ds0 / 2.0 + 0.5);
    if (iblk == 0) {
      iblk = 1;
      bds[i] = L[i] / 2.0;
    } else {
      bds[i] = L[i] / (double)iblk / 2.0;
    }
    if (order >= 0) {
      bds[i] = bds[i] / std::pow(2.0, order);
      iblk = iblk * (1 << order);
    }
    bgns = bgns + iblk * 2;
    bgn[i + 1] = bgns;
  }
}

// ------------------------------------------------------------ reductions
// out_dev[0] = scale * sum of a contour point over the whole grid (async)
void dev_sum(const Grid& g, const double* x, double scale, double* part, double* out_dev, hipStream_t s) {
  const int nb = grid_blocks(g.ms) > 512 ? 512 : grid_blocks(g.ms);
  hipLaunchKernelGGL(k_partial_sum, dim3(nb), dim3(NTA), 0, s, x, g.ms, g.sym, g.n3, (long)g.n1 * g.n2, part);
  hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(NTA), 0, s, part, nb, scale, out_dev);
}

// k_step_a for ntask sweeps: two workgroups per plane (more parallelism)
// while one per plane would leave CUs idle and two all fit in one round of
// resident workgroups; else one (a quarter less work).  A plan may force either.
void launch_step_a(const Grid& g, const StepTask* tasks, int ntask, int j, bool adj, hipStream_t s,
                   hipEvent_t t0 = nullptr, hipEvent_t t1 = nullptr) {
  int aj = g.pl->ajobs;
  const long planes = (long)g.np * ntask;
  if (aj == 0) aj = (planes < g.cus && 2 * planes <= g.plane_slots) ? 2 : 1;
  StepPlaneFn k = aj == 1 ? g.pl->a1[adj] : g.pl->a[adj];
  const dim3 grid(g.np, ntask, aj);
  if (t0)
    hipExtLaunchKernelGGL(k, grid, dim3(g.pl->nt_step), 0, s, t0, t1, 0, tasks, j, g.tw1,
                          g.twl);
  else
    hipLaunchKernelGGL(k, grid, dim3(g.pl->nt_step), 0, s, tasks, j, g.tw1, g.twl);
}

// --------------------------------------------------- contour sweeps
// Advance the given sweep tasks through all their steps: one launch where the
// grid is one plane (k_sweep_plane), else 4 launches per step.
// With `ev` (2 (4 max_ns + 1) events) every launch records a pair of events at
// its kernel's start and end, for per-kernel timing.
// half_z: see step_z (the tasks of one launch may be of several systems)
void run_sweeps(const Grid& g, const StepTask* d_tasks, int ntask, int max_ns, bool half_z, hipStream_t s,
                hipEvent_t* ev = nullptr) {
  if (g.n3 == 1 && g.pl->sweep && !ev) {
    hipLaunchKernelGGL(g.pl->sweep, dim3(ntask), dim3(g.pl->nt_sweep), 0, s, d_tasks, max_ns, g.tw1, g.twl,
                       g.tw2);
    HIPCHK(hipGetLastError());
    return;
  }
  int e = 0;
  auto t0 = [&] { return ev ? ev[e] : nullptr; };
  auto t1 = [&] { return ev ? ev[e + 1] : nullptr; };
  auto next = [&] { if (ev) e += 2; };
  for (int j = 0; j <= max_ns; ++j) {
    launch_step_a(g, d_tasks, ntask, j, false, s, t0(), t1());
    next();
    if (j == max_ns) break;
    g.step_z(d_tasks, ntask, j, 0, 2, false, half_z, s, t0(), t1());
    next();
    g.step_c(d_tasks, ntask, j, false, s, t0(), t1());
    next();
    g.step_z(d_tasks, ntask, j, 1, 1, false, half_z, s, t0(), t1());
    next();
  }
  HIPCHK(hipGetLastError());
}

// accumulate the durations of the last profiled sweep
void collect_profile(System& S, int max_ns) {
  if (S.profile == 1) {
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, S.ev[0], S.ev[1]));
    S.prof_ms[4] += ms;
    S.prof_n[4] += max_ns;
    return;
  }
  const int nl = 4 * max_ns + 1;     // launches: A, Z0, C, Z1 per step, a final A
  for (int i = 0; i < nl; ++i) {
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, S.ev[2 * i], S.ev[2 * i + 1]));
    const int kind = i % 4;
    S.prof_ms[kind] += ms;
    S.prof_n[kind] += 1;
  }
  float ms = 0.0f;                   // the sweep from the first start to the last end
  HIPCHK(hipEventElapsedTime(&ms, S.ev[0], S.ev[2 * nl - 1]));
  S.prof_ms[4] += ms;
  S.prof_n[4] += max_ns;
}

void ensure_events(System& S, size_t n) {
  while (S.ev.size() < n) {
    hipEvent_t e;
    HIPCHK(hipEventCreate(&e));
    S.ev.push_back(e);
  }
}

// The code of the star basis's symmetric planes (kernels.hpp).  An operation
// r -> W r + t leaves every star function unchanged when the coefficients of
// its waves obey c(W^T G) = c(G) exp(i G t), W^T G in the same star.
// Translations z -> z + N3/2 are tried with a = +1 (centring) before a = -1
// (screw axis), reflections z -> -z with a = -1 (inversion) before +1, each
// with tau = 0 or half an edge.  Waves whose image lies outside the wave list
// (on the zone boundary) do not count; every field is checked besides
// (k_sym_check).
int detect_sym(const System& S) {
  const Grid& g = S.g;
  if (g.dim != 3 || g.n3 % 4 || g.n1 % 2 || g.n2 % 2 || S.no_sym) return 0;
  const long step = std::max(1, S.nwave / 8192);
  auto holds = [&](int sz, int a, int tx, int ty, int tz) {
    long seen = 0;
    for (long w = 0; w < S.nwave; w += w < 4096 ? 1 : step) {
      const int* G = &S.h_wave[(size_t)w * 3];
      const int Gp[3] = {a * G[0], a * G[1], sz * G[2]};
      long off = 0, mul = 1;
      bool in = true;
      for (int d = 0; d < 3; ++d) {
        const int u = Gp[d] - S.gmin[d];
        in = in && u >= 0 && u < S.gext[d];
        off += (long)u * mul;
        mul *= S.gext[d];
      }
      const int v = in ? S.h_wtab[off] : 0;
      if (v == 0) continue;
      const double2 c = S.h_coeff[w], cp = S.h_coeff[v - 1];
      const double sg = ((tx * G[0] + ty * G[1] + tz * G[2]) & 1) ? -1.0 : 1.0;
      if (S.h_star_of_wave[v - 1] != S.h_star_of_wave[w] || std::fabs(cp.x - sg * c.x) > 1e-10 ||
          std::fabs(cp.y - sg * c.y) > 1e-10)
        return false;
      ++seen;
    }
    return seen > 0;
  };
  int code = 0, t = 0, r = 0;
  for (int k = 0; k < 8 && !(code & SYM_T); ++k)
    if (holds(1, k < 4 ? 1 : -1, k & 1, k >> 1 & 1, 1)) {
      code |= SYM_T;
      t = (k < 4 ? 0 : 1) | (k & 1) << 1 | (k >> 1 & 1) << 2;
    }
  for (int k = 0; k < 8 && !(code & SYM_R); ++k)
    if (holds(-1, k < 4 ? -1 : 1, k & 1, k >> 1 & 1, 0)) {
      code |= SYM_R;
      r = (k < 4 ? 1 : 0) | (k & 1) << 1 | (k >> 1 & 1) << 2;
    }
  return code ? code | t << 2 | r << 5 | (t ^ r) << 8 : 0;
}

void build_basis_maps(System& S) {
  // dense which_wave table over the bounding box of the wave list
  const int dim = S.g.dim;
  int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  for (int d = 0; d < dim; ++d) {
    lo[d] = 1 << 30;
    hi[d] = -(1 << 30);
  }
  for (int w = 0; w < S.nwave; ++w)
    for (int d = 0; d < dim; ++d) {
      const int v = S.h_wave[(size_t)w * dim + d];
      lo[d] = std::min(lo[d], v);
      hi[d] = std::max(hi[d], v);
    }
  long tot = 1;
  for (int d = 0; d < 3; ++d) {
    S.gmin[d] = d < dim ? lo[d] : 0;
    S.gext[d] = d < dim ? hi[d] - lo[d] + 1 : 1;
    tot *= S.gext[d];
  }
  std::vector<int> wt(tot, 0);
  auto box = [&](const int* G) -> long {
    long off = 0, mul = 1;
    for (int d = 0; d < dim; ++d) {
      const int u = G[d] - S.gmin[d];
      if (u < 0 || u >= S.gext[d]) return -1;
      off += (long)u * mul;
      mul *= S.gext[d];
    }
    return off;
  };
  for (int w = 0; w < S.nwave; ++w) wt[box(&S.h_wave[(size_t)w * dim])] = w + 1;
  S.wtab.upload(wt.data(), wt.size(), S.st.s);
  S.h_wtab = wt;
  S.star_bound.assign(S.nstar, 0.0);
  for (int w = 0; w < S.nwave; ++w)
    S.star_bound[S.h_star_of_wave[w] - 1] += std::hypot(S.h_coeff[w].x, S.h_coeff[w].y);
  // per star: representative wave -> half-grid index (conj if kx > N1/2), coeff
  std::vector<long> sidx(S.nstar);
  std::vector<int> sconj(S.nstar);
  std::vector<double2> scoef(S.nstar);
  const int ng[3] = {S.g.n1, S.g.n2, S.g.n3};
  for (int s = 0; s < S.nstar; ++s) {
    int kbz[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) kbz[d] = S.h_wave_of_star[(size_t)s * dim + d];
    const long o = box(kbz);
    REQUIRE(o >= 0 && wt[o] > 0, "wave_of_star is not in the wave list");
    scoef[s] = S.h_coeff[wt[o] - 1];
    int kf[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) kf[d] = ((kbz[d] % ng[d]) + ng[d]) % ng[d];
    sconj[s] = 0;
    if (kf[0] > S.g.n1 / 2) {
      for (int d = 0; d < dim; ++d) kf[d] = (((-kbz[d]) % ng[d]) + ng[d]) % ng[d];
      sconj[s] = 1;
    }
    sidx[s] = kf[0] + (long)S.g.n1h * (kf[1] + (long)S.g.n2 * kf[2]);
  }
  S.sidx.upload(sidx.data(), sidx.size(), S.st.s);
  // half-spectrum columns (kx, ky) with a representative wave, and the packed
  // columns (kx, l), (-kx, -l) they are split from
  const long plane = (long)S.g.n1h * S.g.n2;
  const int nl = S.g.nl, n1 = S.g.n1;
  std::vector<int> cols;
  for (int s = 0; s < S.nstar; ++s) cols.push_back((int)(sidx[s] % plane));
  std::sort(cols.begin(), cols.end());
  cols.erase(std::unique(cols.begin(), cols.end()), cols.end());
  S.ncol = (int)cols.size();
  std::vector<long> sidx_c(S.nstar);
  for (int s = 0; s < S.nstar; ++s) {
    const int c = (int)(std::lower_bound(cols.begin(), cols.end(), (int)(sidx[s] % plane)) -
                        cols.begin());
    sidx_c[s] = c + (long)S.ncol * (sidx[s] / plane);
  }
  std::vector<int> cpos((size_t)n1 * nl, -1);
  std::vector<int2> src(S.ncol), colk(S.ncol);
  for (int c = 0; c < S.ncol; ++c) {
    const int kx = cols[c] % S.g.n1h, ky = cols[c] / S.g.n1h, l = ky % nl;
    colk[c] = make_int2(kx, ky);
    src[c] = make_int2(l * n1 + col_pos(kx, n1), (nl - l) % nl * n1 + col_pos((n1 - kx) % n1, n1));
    cpos[src[c].x] = cpos[src[c].y] = 0;
  }
  S.nin = 0;
  for (auto& p : cpos)
    if (p == 0) p = S.nin++;
  for (auto& p : src) p = make_int2(cpos[p.x], cpos[p.y]);
  S.scpos.upload(cpos.data(), cpos.size(), S.st.s);
  S.ssrc.upload(src.data(), src.size(), S.st.s);
  S.scolk.upload(colk.data(), colk.size(), S.st.s);
  S.sidx_c.upload(sidx_c.data(), sidx_c.size(), S.st.s);
  S.sconj.upload(sconj.data(), sconj.size(), S.st.s);
  S.scoef.upload(scoef.data(), scoef.size(), S.st.s);
  S.st.sync();
}

GeomArgs geom_args(const System& S) {
  GeomArgs a;
  a.n1 = S.g.n1;
  a.n2 = S.g.n2;
  a.n3 = S.g.n3;
  a.dim = S.g.dim;
  for (int i = 0; i < 9; ++i) a.gb[i] = S.gb[i];
  for (int d = 0; d < 3; ++d) {
    a.gmin[d] = S.gmin[d];
    a.gext[d] = S.gext[d];
  }
  return a;
}

void apply_cell(System& S) {
  const GeomArgs a = geom_args(S);
  S.ksq.alloc(S.g.mk);
  S.kwave.alloc(S.g.mk);
  hipLaunchKernelGGL(k_g_to_bz, dim3(grid_blocks(S.g.mk)), dim3(NTA), 0, S.st.s, a, S.wtab.p, S.ksq.p,
                     S.kwave.p);
  HIPCHK(hipGetLastError());
  S.have_cell = true;
}

// star coefficients (device, (nf, nstar)) -> real grids (nf arrays)
void basis_to_grid(System& S, const double* d_basis, int nf, double* d_grid, hipStream_t s) {
  const Grid& g = S.g;
  S.kwork.alloc((size_t)std::max(nf, 2) * g.mk);
  hipLaunchKernelGGL(k_basis_to_kgrid, dim3(grid_blocks(g.mk * nf)), dim3(NTA), 0, s, d_basis, nf,
                     S.nstar, S.kwave.p, S.coeff.p, S.star_of_wave.p, S.star_invert.p, g.mk,
                     S.kwork.p, 0);
  g.c2r(S.kwork.p, d_grid, nf, 1.0, s);
}

// real grids (nf arrays, stride m) -> star coefficients (nf, nstar) * scale
void grid_to_basis(System& S, const double* d_grid, int nf, double scale, double* d_basis,
                   hipStream_t s) {
  const Grid& g = S.g;
  S.kwork.alloc((size_t)std::max(nf, 2) * g.mk);
  g.r2c(d_grid, S.kwork.p, nf, s);
  hipLaunchKernelGGL(k_kgrid_to_basis, dim3(grid_blocks((long)S.nstar * nf)), dim3(NTA), 0, s,
                     S.kwork.p, g.mk, nf, S.nstar, S.sidx.p, S.sconj.p, S.scoef.p, S.star_invert.p,
                     scale, d_basis, 0);
}

// ---- full k grids (the RESPONSE command's karray_full / no_parity forms,
// src/grid_basis_mod.f90:47-200).  Host arithmetic: the response calculation
// calls these once per perturbation, outside the contour sweeps.
// 1-based wave number of the minimum-image wavevector kbz, 0 if absent
int host_wave_of(const System& S, const int kbz[3]) {
  long off = 0, mul = 1;
  for (int d = 0; d < S.g.dim; ++d) {
    const int u = kbz[d] - S.gmin[d];
    if (u < 0 || u >= S.gext[d]) return 0;
    off += (long)u * mul;
    mul *= S.gext[d];
  }
  return S.h_wtab[off];
}

// star coefficients -> every point of the full FFT grid (x fastest); with
// no_parity the coefficients multiply the star functions directly, without
// the star_invert +-1 pairing of real basis functions
void full_basis_to_kgrid(const System& S, const double* basis, double2* out, bool no_parity) {
  const GeomArgs ga = geom_args(S);
  const double sq2 = std::sqrt(2.0);
  long idx = 0;
  for (int i3 = 0; i3 < S.g.n3; ++i3)
    for (int i2 = 0; i2 < S.g.n2; ++i2)
      for (int i1 = 0; i1 < S.g.n1; ++i1, ++idx) {
        const int G[3] = {i1, i2, i3};
        int kbz[3] = {0, 0, 0};
        g_to_bz_vec(ga, G, kbz);
        const int w = host_wave_of(S, kbz);
        double2 z = make_double2(0.0, 0.0);
        if (w > 0) {
          const double2 c = S.h_coeff[w - 1];
          const int st = S.h_star_of_wave[w - 1] - 1;
          const int inv = no_parity ? 0 : S.h_star_invert[st];
          // the star's complex amplitude (a, b) times the wave's coefficient;
          // a +-1 pair shares (a - i b)/sqrt(2) and (a + i b)/sqrt(2)
          double a, b;
          if (inv == 0) a = basis[st], b = 0.0;
          else if (inv == 1) a = basis[st], b = -basis[st + 1];
          else a = basis[st - 1], b = basis[st];
          z = make_double2(a * c.x - b * c.y, a * c.y + b * c.x);
          if (inv != 0) z = make_double2(z.x / sq2, z.y / sq2);
        }
        out[idx] = z;
      }
}

// full FFT grid -> star coefficients: each star reads its representative
// wave (with no_parity at its own grid point; otherwise from the -k point,
// conjugated, when k lies in the upper half of the first dimension)
void full_kgrid_to_basis(const System& S, const double2* kg, double* basis, bool no_parity) {
  const int dim = S.g.dim;
  const int ng[3] = {S.g.n1, S.g.n2, S.g.n3};
  const double sq2 = std::sqrt(2.0);
  auto at = [&](const int* k, int sgn) {
    int kf[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) kf[d] = (((sgn * k[d]) % ng[d]) + ng[d]) % ng[d];
    return kg[kf[0] + (long)ng[0] * (kf[1] + (long)ng[1] * kf[2])];
  };
  for (int s = 0; s < S.nstar; ++s) {
    int kbz[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) kbz[d] = S.h_wave_of_star[(size_t)s * dim + d];
    const int w = host_wave_of(S, kbz);
    REQUIRE(w > 0, "wave_of_star is not in the wave list");
    const double2 c = S.h_coeff[w - 1];
    double2 z;
    if (no_parity) {
      z = at(kbz, 1);
    } else {
      const int k1 = ((kbz[0] % ng[0]) + ng[0]) % ng[0];
      if (k1 > ng[0] / 2) {
        z = at(kbz, -1);
        z.y = -z.y;
      } else {
        z = at(kbz, 1);
      }
    }
    const double cc = c.x * c.x + c.y * c.y;            // z / c
    const double re = (z.x * c.x + z.y * c.y) / cc, im = (z.y * c.x - z.x * c.y) / cc;
    const int inv = no_parity ? 0 : S.h_star_invert[s];
    basis[s] = inv == 0 ? re : (inv == 1 ? re * sq2 : im * sq2);
  }
}

// ---- checkpointed contour storage (stride K > 0)
// The sweeps of density() keep q_f and q_r only at checkpoints; the Simpson
// integrals and the adjoint recompute the points between them, one segment of
// K steps per chain and round, into the chain's segment buffers.

void build_ck_plan(System& S) {
  const int K = S.ck_stride;
  const int nc = S.nchain;
  CkPlan& P = S.ck;
  P.nround = (S.max_ns + K - 1) / K;
  P.len.assign(P.nround, 0);
  P.map_off.assign((size_t)P.nround * nc * 2, 0);
  std::vector<int> h;
  for (int r = 0; r < P.nround; ++r)
    for (int c = 0; c < nc; ++c) {
      const ChainDev& ch = *S.chains[c];
      for (int side = 0; side < 2; ++side) {
        int lo, hi;     // side 0: R_r, side 1: F_r
        if (side == 0) {
          lo = r * K;
          hi = std::min((r + 1) * K, ch.ns);
        } else {
          hi = ch.ns - r * K;
          lo = std::max(0, ch.ns - (r + 1) * K);
        }
        P.map_off[((size_t)r * nc + c) * 2 + side] = h.size();
        for (int sp = 0; sp <= ch.ns; ++sp) h.push_back(lo <= hi && sp >= lo && sp <= hi ? sp - lo : -1);
        if (lo < hi) P.len[r] = std::max(P.len[r], hi - lo);
      }
    }
  P.maps.upload(h.data(), h.size(), S.st.s);
  // forward Simpson tasks: per round, recompute R_r of every chain (q_f from
  // its checkpoint at lo, q_r from its checkpoint at hi) into segment buffers 0, 1
  std::vector<StepTask> ht((size_t)P.nround * 2 * nc);
  for (int r = 0; r < P.nround; ++r)
    for (int c = 0; c < nc; ++c) {
      const ChainDev& ch = *S.chains[c];
      const int lo = r * K, hi = std::min((r + 1) * K, ch.ns);
      for (int d = 0; d < 2; ++d) {
        StepTask t = S.h_tasks[2 * c + d];
        StepTask& o = ht[((size_t)r * nc + c) * 2 + d];
        t.init_one = 0;
        t.slab = ch.seg.p + (size_t)d * ch.segpts * S.g.ms;
        t.pmap = P.maps.p + P.map_off[((size_t)r * nc + c) * 2 + 0];
        if (lo >= hi) {
          t.skip = 1;
        } else if (d == 0) {          // q_f forward over [lo, hi]
          t.jbeg = t.jofs = lo;
          t.jend = hi;
          t.start = ch.point(+1, lo);
        } else {                      // q_r backward over [lo, hi]: steps ns-hi .. ns-lo-1
          t.jbeg = t.jofs = ch.ns - hi;
          t.jend = ch.ns - lo;
          t.start = ch.point(-1, hi);
        }
        o = t;
      }
    }
  S.ck_tasks.upload(ht.data(), ht.size(), S.st.s);
  S.st.sync();
}

// Simpson integrals of every block by segment recomputation (captured once)
void ck_simpson_rounds(System& S, hipStream_t s) {
  const Grid& g = S.g;
  const CkPlan& P = S.ck;
  const int nc = S.nchain, K = S.ck_stride;
  for (int c = 0; c < nc; ++c) {
    ChainDev& ch = *S.chains[c];
    hipLaunchKernelGGL(k_fill, dim3(grid_blocks((long)ch.nblk * g.ms)), dim3(NTA), 0, s, ch.blk.p,
                       (long)ch.nblk * g.ms, 0.0);
  }
  for (int r = 0; r < P.nround; ++r) {
    const StepTask* tk = S.ck_tasks.p + (size_t)r * 2 * nc;
    run_sweeps(g, tk, 2 * nc, P.len[r], sym_half(g.sym), s);
    for (int c = 0; c < nc; ++c) {
      ChainDev& ch = *S.chains[c];
      const int lo = r * K, hi = std::min((r + 1) * K, ch.ns);
      if (lo >= hi) continue;
      SimpsonArgs a;
      std::memset(&a, 0, sizeof a);
      a.nblk = ch.nblk;
      for (int b = 0; b <= ch.nblk; ++b) a.bnd[b] = ch.bnd[b];
      for (int b = 0; b < ch.nblk; ++b) a.ds[b] = ch.ds[b];
      hipLaunchKernelGGL(k_simpson_seg, dim3(grid_blocks(g.ms)), dim3(NTA), 0, s, ch.seg.p,
                         ch.seg.p + (size_t)ch.segpts * g.ms, g.ms, a, lo, hi, hi == ch.ns ? 1 : 0,
                         ch.blk.p);
    }
  }
  HIPCHK(hipGetLastError());
}

void startup(System& S, double chain_step) {
  REQUIRE(S.have_chem, "set_chemistry must precede startup");
  S.g.set_sym(S.no_sym ? 0 : S.sym_code);
  S.sym_bad = false;
  S.last = nullptr;
  S.full.reset();
  const Grid& g = S.g;
  S.chains.clear();
  for (int c = 0; c < S.nchain; ++c) {
    auto ch = std::make_unique<ChainDev>();
    const auto& bl = S.blocks[c];
    ch->nblk = (int)bl.size();
    REQUIRE(ch->nblk >= 1 && ch->nblk <= MAXBLK, "number of blocks per chain out of range");
    std::vector<double> L(ch->nblk);
    std::vector<int> bgn(ch->nblk + 1);
    for (int b = 0; b < ch->nblk; ++b) {
      L[b] = bl[b].second;
      ch->mon[b] = bl[b].first;
    }
    discretize(ch->nblk, L.data(), chain_step, -1, bgn.data(), ch->ds);
    for (int b = 0; b <= ch->nblk; ++b) ch->bnd[b] = bgn[b] - 1;
    ch->ns = ch->bnd[ch->nblk];
    ch->length = S.chain_length[c];
    ch->m_ = g.ms;
    if (S.ck_stride > 0) {
      const int K = S.ck_stride;
      ch->slot.assign(ch->ns + 1, -1);
      ch->nslot = 0;
      for (int sp = 0; sp <= ch->ns; ++sp)
        if (sp % K == 0 || (ch->ns - sp) % K == 0) ch->slot[sp] = ch->nslot++;
      ch->dslot.upload(ch->slot.data(), ch->slot.size(), S.st.s);
      ch->segpts = std::min(K, ch->ns) + 1;
      ch->seg.alloc((size_t)4 * ch->segpts * g.ms);
      ch->blk.alloc((size_t)ch->nblk * g.ms);
    } else {
      ch->nslot = ch->ns + 1;
    }
    ch->qf.alloc((size_t)ch->nslot * g.ms);
    ch->qr.alloc((size_t)ch->nslot * g.ms);
    ch->fac.alloc((size_t)ch->nblk * (2 * g.ms + 2 * g.mf));
    S.chains.push_back(std::move(ch));
  }
  S.chain_step = chain_step;
  const int ntask = 2 * S.nchain;
  S.abc.alloc((size_t)3 * g.mc * std::max(ntask, 1));
  S.q1.alloc((size_t)g.ms * std::max(ntask, 1));
  S.tasks.alloc(std::max(ntask, 1));
  S.omega_grid.alloc((size_t)S.nmon * g.m);
  S.rho_grid.alloc((size_t)S.nmon * g.m);
  S.part.alloc(1024);
  S.qdev.alloc(S.nchain + S.nsolv + 2);    // Q, a scratch value, the symmetry flag
  hipLaunchKernelGGL(k_fill, dim3(1), dim3(NTA), 0, S.st.s, S.qdev.p, (long)S.qdev.n, 0.0);
  S.chem_dev.alloc(2 * (S.nchain + S.nsolv) + 2);
  // sweep tasks: forward (qf) and backward (qr) sweep of every chain
  std::vector<StepTask> ht(ntask);
  int max_ns = 0;
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    max_ns = std::max(max_ns, ch.ns);
    for (int d = 0; d < 2; ++d) {
      StepTask& t = ht[2 * c + d];
      std::memset(&t, 0, sizeof t);
      t.slab = d == 0 ? ch.qf.p : ch.qr.p;
      t.pmap = S.ck_stride > 0 ? ch.dslot.p : nullptr;
      t.ns = ch.ns;
      t.jend = ch.ns;
      t.dir = d == 0 ? 1 : -1;
      t.init_one = 1;
      t.nblk = ch.nblk;
      for (int b = 0; b <= MAXBLK; ++b) t.bnd[b] = ch.bnd[std::min(b, ch.nblk)];
      t.fac = ch.fac.p;
      t.fm = g.ms;
      t.fk = g.mf;
      t.sym = g.sym;
      const int ti = 2 * c + d;
      t.A = S.abc.p + (size_t)(3 * ti) * g.mc;
      t.B = t.A + g.mc;
      t.C = t.B + g.mc;
      t.q1 = S.q1.p + (size_t)ti * g.ms;
    }
  }
  if (ntask > 0)
    HIPCHK(hipMemcpyAsync(S.tasks.p, ht.data(), sizeof(StepTask) * ntask, hipMemcpyHostToDevice,
                          S.st.s));
  S.st.sync();
  S.h_tasks = ht;
  S.ntask = ntask;
  S.max_ns = max_ns;
  S.drop_graph();
  S.drop_ck_graph();
  S.adj.reset();
  S.started = true;
  S.have_density = false;
  ++S.gen_start;
  if (S.ck_stride > 0) build_ck_plan(S);
}

// ---- density() in phases, each enqueued on stream s (src/scf_mod.fp.f90:144-229)

// The basis's symmetric planes hold for a cell: an operation with a s = -1
// besides (a = -1 with z -> z + c, a = +1 with z -> -z) also has to leave |k|
// unchanged, i.e. the third reciprocal vector normal to the other two.
bool sym_usable(const System& S) {
  if (!S.g.sym) return true;
  if (S.sym_bad || S.sym_code != S.g.sym) return false;
  if (!((S.g.sym & SYM_T) && (S.g.sym >> 2 & 1)) && !((S.g.sym & SYM_R) && !(S.g.sym >> 5 & 1))) return true;
  auto dot = [&](int i, int j) {
    return S.gb[i * 3] * S.gb[j * 3] + S.gb[i * 3 + 1] * S.gb[j * 3 + 1] + S.gb[i * 3 + 2] * S.gb[j * 3 + 2];
  };
  const double n3 = dot(2, 2);
  return std::fabs(dot(2, 0)) <= 1e-12 * std::sqrt(n3 * dot(0, 0)) &&
         std::fabs(dot(2, 1)) <= 1e-12 * std::sqrt(n3 * dot(1, 1));
}
// after the stream is synchronised: the omega of the last density_pre is not symmetric
bool sym_failed(System& S) {
  if (S.g.sym && S.pin_q.p[S.nchain + S.nsolv + 1] == S.sym_epoch) S.sym_bad = true;
  return S.sym_bad;
}

// Whether grid fields (one per monomer, device memory) have the symmetry of
// the stored planes, to tol of their largest value.  Waits for the answer.
// density() on grids and its reverse mode take the symmetric planes where it
// holds, every plane otherwise; the check and its wait cost about 25 us.
// Gradient of a gyroid at 64^3, 200 steps: 22.5 ms on every plane, 17.9 ms on
// 17 of 64; a checkpointed body-centred blend at 96^3: 189 and 92 ms.
// The tolerances are some tens of roundings, so that what the planes left out
// would have added is no larger than the transforms' own rounding.
bool grid_symmetric(System& S, const double* fields, double tol) {
  const Grid& g = S.g;
  hipStream_t s = S.st.s;
  const int nb = 64;
  double* flag = S.qdev.p + S.nchain + S.nsolv + 1;
  S.sym_epoch += 1.0;
  hipLaunchKernelGGL(k_partial_absmax, dim3(nb), dim3(NTA), 0, s, fields, (long)S.nmon * g.m, S.part.p);
  hipLaunchKernelGGL(k_sym_check_grid, dim3(grid_blocks(g.m * S.nmon)), dim3(NTA), 0, s, fields, S.nmon,
                     g.sym, g.n1, g.n2, g.n3, S.part.p, nb, tol, S.sym_epoch, flag);
  HIPCHK(hipGetLastError());
  S.pin_q.alloc(S.qdev.n);
  double* answer = S.pin_q.p + S.nchain + S.nsolv + 1;
  HIPCHK(hipMemcpyAsync(answer, flag, sizeof(double), hipMemcpyDeviceToHost, s));
  S.st.sync();
  return *answer != S.sym_epoch;
}

// omega stars -> grid (no 1/M, :182-185), propagator factors per block
// (make_propg), chemistry scalars for the device
// (grid_in: S.omega_grid already holds the omega grids, star input unused;
// chain_update false: density() without qout, whose chain densities take the
// given phi_chain in either ensemble)
void density_pre(System& S, const double* omega, const double* phi_c, const double* mu_c,
                 const double* phi_s, const double* mu_s, hipStream_t s, bool grid_in = false,
                 bool chain_update = true) {
  REQUIRE(S.started && S.have_basis && S.have_cell, "system not ready (basis, cell, startup)");
  const Grid& g = S.g;
  S.chain_ens = (S.ensemble == 1 && chain_update) ? 1 : 0;
  if (!grid_in) {
    const size_t nst = (size_t)S.nmon * S.nstar;
    S.pin_in.alloc(nst);
    std::memcpy(S.pin_in.p, omega, sizeof(double) * nst);
    S.omega_in.alloc(nst);
    HIPCHK(hipMemcpyAsync(S.omega_in.p, S.pin_in.p, sizeof(double) * nst, hipMemcpyHostToDevice, s));
    basis_to_grid(S, S.omega_in.p, S.nmon, S.omega_grid.p, s);
    if (g.sym) {
      // the planes left out have to hold what the stored ones say, to rounding
      // (against a bound of |omega|)
      double bound = 0.0;
      for (int a = 0; a < S.nmon; ++a) {
        double b = 0.0;
        for (int i = 0; i < S.nstar; ++i) b += std::fabs(omega[a + (size_t)S.nmon * i]) * S.star_bound[i];
        bound = std::max(bound, b);
      }
      S.sym_epoch += 1.0;
      hipLaunchKernelGGL(k_sym_check, dim3(grid_blocks((g.m - g.ms) * S.nmon)), dim3(NTA), 0, s,
                         S.omega_grid.p, S.nmon, g.sym, g.n1, g.n2, g.n3, 1e-12 * bound, S.sym_epoch,
                         S.qdev.p + S.nchain + S.nsolv + 1);
    }
  }
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    for (int b = 0; b < ch.nblk; ++b) {
      double* f = ch.fac.p + (size_t)b * (2 * g.ms + 2 * g.mf);
      hipLaunchKernelGGL(k_make_propg, dim3(grid_blocks(std::max(g.ms, g.mf))), dim3(NTA), 0, s, ch.ds[b],
                         S.kuhn[ch.mon[b]], S.ksq.p, g.mf, S.omega_grid.p + (size_t)ch.mon[b] * g.m,
                         g.ms, g.n1, g.n2, g.zs->zw, (double)g.m, f, f + g.ms, f + 2 * g.ms,
                         f + 2 * g.ms + g.mf);
    }
  }
  S.h_chem.assign(2 * (S.nchain + S.nsolv) + 2, 0.0);
  for (int c = 0; c < S.nchain; ++c) {
    S.h_chem[2 * c] = phi_c ? phi_c[c] : 0.0;
    S.h_chem[2 * c + 1] = mu_c ? mu_c[c] : 0.0;
  }
  for (int i = 0; i < S.nsolv; ++i) {
    S.h_chem[2 * (S.nchain + i)] = phi_s ? phi_s[i] : 0.0;
    S.h_chem[2 * (S.nchain + i) + 1] = mu_s ? mu_s[i] : 0.0;
  }
  S.pin_chem.alloc(S.h_chem.size());
  std::memcpy(S.pin_chem.p, S.h_chem.data(), sizeof(double) * S.h_chem.size());
  HIPCHK(hipMemcpyAsync(S.chem_dev.p, S.pin_chem.p, sizeof(double) * S.h_chem.size(),
                        hipMemcpyHostToDevice, s));
}

// both contour sweeps of every chain: 4 launches per contour step
void density_sweeps(System& S, hipStream_t s) {
  const Grid& g = S.g;
  const int max_ns = S.max_ns;
  ++S.density_gen;
  if (S.profile == 2) {
    ensure_events(S, (size_t)2 * (4 * max_ns + 1));
    run_sweeps(g, S.tasks.p, S.ntask, max_ns, sym_half(g.sym), s, S.ev.data());
    return;
  }
  if (S.profile == 1) {
    ensure_events(S, 2);
    HIPCHK(hipEventRecord(S.ev[0], s));
  }
  if (S.use_graph) {
    if (!S.graph_exec) {
      HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      run_sweeps(g, S.tasks.p, S.ntask, max_ns, sym_half(g.sym), s);
      HIPCHK(hipStreamEndCapture(s, &S.graph));
      HIPCHK(hipGraphInstantiate(&S.graph_exec, S.graph, nullptr, nullptr, 0));
    }
    HIPCHK(hipGraphLaunch(S.graph_exec, s));
  } else {
    run_sweeps(g, S.tasks.p, S.ntask, max_ns, sym_half(g.sym), s);
  }
  if (S.profile == 1) HIPCHK(hipEventRecord(S.ev[1], s));
}

// Q (:359-360), solvents (:193-200), Simpson rho (:362-424, 212-218),
// rho grid -> stars / M (:221-225); copies Q and rho stars to the host
void density_post(System& S, double* rho, hipStream_t s) {
  const Grid& g = S.g;
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    dev_sum(g, ch.point(+1, ch.ns), 1.0 / (double)g.m, S.part.p, S.qdev.p + c, s);
  }
  hipLaunchKernelGGL(k_fill, dim3(grid_blocks((long)S.nmon * g.m)), dim3(NTA), 0, s, S.rho_grid.p,
                     (long)S.nmon * g.m, 0.0);
  for (int i = 0; i < S.nsolv; ++i) {
    const double* w = S.omega_grid.p + (size_t)S.solv_mon[i] * g.m;
    const int nb = 512;
    hipLaunchKernelGGL(k_partial_sum_exp, dim3(nb), dim3(NTA), 0, s, w, S.solv_size[i], g.m, S.part.p);
    hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(NTA), 0, s, S.part.p, nb, 1.0 / (double)g.m,
                       S.qdev.p + S.nchain + i);
    hipLaunchKernelGGL(k_solvent_rho, dim3(grid_blocks(g.m)), dim3(NTA), 0, s, w, S.solv_size[i],
                       S.qdev.p + S.nchain + i, S.ensemble, S.chem_dev.p + 2 * (S.nchain + i), g.m,
                       S.rho_grid.p + (size_t)S.solv_mon[i] * g.m);
  }
  if (S.ck_stride > 0) {
    if (S.use_graph) {
      if (!S.ck_exec) {
        HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        ck_simpson_rounds(S, s);
        HIPCHK(hipStreamEndCapture(s, &S.ck_graph));
        HIPCHK(hipGraphInstantiate(&S.ck_exec, S.ck_graph, nullptr, nullptr, 0));
      }
      HIPCHK(hipGraphLaunch(S.ck_exec, s));
    } else {
      ck_simpson_rounds(S, s);
    }
  }
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    SimpsonArgs a;
    std::memset(&a, 0, sizeof a);
    a.nblk = ch.nblk;
    for (int b = 0; b <= ch.nblk; ++b) a.bnd[b] = ch.bnd[b];
    for (int b = 0; b < ch.nblk; ++b) {
      a.ds[b] = ch.ds[b];
      a.monomer[b] = ch.mon[b];
    }
    a.chain_length = ch.length;
    a.ensemble = S.chain_ens;
    if (S.ck_stride > 0)
      hipLaunchKernelGGL(k_block_rho, dim3(grid_blocks(g.ms)), dim3(NTA), 0, s, ch.blk.p, g.ms, g.m, a,
                         S.qdev.p + c, S.chem_dev.p + 2 * c, g.n1, g.n2, S.rho_grid.p);
    else
      hipLaunchKernelGGL(k_simpson, dim3(grid_blocks(g.ms)), dim3(NTA), 0, s, ch.qf.p, ch.qr.p, g.ms, g.m,
                         a, S.qdev.p + c, S.chem_dev.p + 2 * c, g.n1, g.n2, S.rho_grid.p);
  }
  if (g.sym)
    hipLaunchKernelGGL(k_sym_expand, dim3(grid_blocks((g.m - g.ms) * S.nmon)), dim3(NTA), 0, s, S.rho_grid.p,
                       S.nmon, g.sym, g.n1, g.n2, g.n3);
  const size_t nst = (size_t)S.nmon * S.nstar;
  if (rho) {
    S.rho_out.alloc(nst);
    grid_to_basis(S, S.rho_grid.p, S.nmon, 1.0 / (double)g.m, S.rho_out.p, s);
  }
  HIPCHK(hipGetLastError());
  S.pin_q.alloc(S.qdev.n);
  HIPCHK(hipMemcpyAsync(S.pin_q.p, S.qdev.p, sizeof(double) * S.qdev.n, hipMemcpyDeviceToHost, s));
  S.rho_dst = rho;
  if (rho) {
    S.pin_rho.alloc(nst);
    HIPCHK(hipMemcpyAsync(S.pin_rho.p, S.rho_out.p, sizeof(double) * nst, hipMemcpyDeviceToHost, s));
  }
}

// after the stream is synchronised: outputs and the grand-ensemble update (:202-209)
void density_finish(System& S, double* qout, double* qsolv, double* phi_c, double* mu_c,
                    double* phi_s, double* mu_s) {
  if (S.profile) collect_profile(S, S.max_ns);
  S.h_Q.assign(S.pin_q.p, S.pin_q.p + (S.nchain + S.nsolv));
  if (S.rho_dst)
    std::memcpy(S.rho_dst, S.pin_rho.p, sizeof(double) * (size_t)S.nmon * S.nstar);
  S.rho_dst = nullptr;
  for (int c = 0; c < S.nchain; ++c)
    if (qout) qout[c] = S.h_Q[c];
  for (int i = 0; i < S.nsolv; ++i)
    if (qsolv) qsolv[i] = S.h_Q[S.nchain + i];
  if (S.ensemble == 1) {
    for (int c = 0; c < S.nchain; ++c)
      if (phi_c && mu_c && S.chain_ens == 1) phi_c[c] = S.h_Q[c] * std::exp(mu_c[c]);
    for (int i = 0; i < S.nsolv; ++i)
      if (phi_s && mu_s) phi_s[i] = S.h_Q[S.nchain + i] * std::exp(mu_s[i]);
  }
  S.have_density = true;
}

System& full_of(System& S);

// density() by the system's companion that stores every plane
template <class F>
void on_full(System& S, F&& run) {
  System& D = full_of(S);
  D.profile = S.profile;
  run(D);
  for (int k = 0; k < 5; ++k) {
    S.prof_ms[k] += D.prof_ms[k];
    S.prof_n[k] += D.prof_n[k];
    D.prof_ms[k] = 0.0;
    D.prof_n[k] = 0;
  }
  S.h_Q = D.h_Q;
  S.have_density = true;
  ++S.density_gen;
  S.last = &D;
}

void density(System& S, const double* omega, double* rho, double* qout, double* qsolv, double* phi_c,
             double* mu_c, double* phi_s, double* mu_s) {
  if (sym_usable(S)) {
    hipStream_t s = S.st.s;
    density_pre(S, omega, phi_c, mu_c, phi_s, mu_s, s, false, qout != nullptr);
    density_sweeps(S, s);
    density_post(S, rho, s);
    S.st.sync();
    if (!sym_failed(S)) {
      density_finish(S, qout, qsolv, phi_c, mu_c, phi_s, mu_s);
      S.last = nullptr;
      return;
    }
  }
  on_full(S, [&](System& D) { density(D, omega, rho, qout, qsolv, phi_c, mu_c, phi_s, mu_s); });
}

// density() on real-space grids held in device memory: omega_grid (M, N_monomer)
// in, rho_grid (M, N_monomer) out, before any star projection.
void density_grid(System& S, const double* omega_grid, double* rho_grid, double* qout, double* qsolv,
                  double* phi_c, double* mu_c, double* phi_s, double* mu_s) {
  REQUIRE(S.started, "system not ready (startup)");
  // grid fields need not have the basis's symmetry
  if (S.g.sym && !(sym_usable(S) && grid_symmetric(S, omega_grid, 1e-14))) {
    on_full(S, [&](System& D) {
      density_grid(D, omega_grid, rho_grid, qout, qsolv, phi_c, mu_c, phi_s, mu_s);
    });
    return;
  }
  hipStream_t s = S.st.s;
  const size_t n = (size_t)S.nmon * S.g.m;
  HIPCHK(hipMemcpyAsync(S.omega_grid.p, omega_grid, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
  density_pre(S, nullptr, phi_c, mu_c, phi_s, mu_s, s, true, qout != nullptr);
  density_sweeps(S, s);
  density_post(S, nullptr, s);
  HIPCHK(hipMemcpyAsync(rho_grid, S.rho_grid.p, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
  S.st.sync();
  density_finish(S, qout, qsolv, phi_c, mu_c, phi_s, mu_s);
  S.last = nullptr;
}

// ---- many density() evaluations of one system in one launch set
//
// The finite-difference Jacobian of Newton-Raphson iteration
// (src/response_pd_mod.f90:91-147) evaluates density() at N_cut * N_monomer
// perturbed omega fields of one system.  density_many runs such a list
// through copies of the system (same grid, stars, cell, chemistry and
// contour discretisation) whose sweep tasks share one launch per contour step,
// captured once as a HIP graph; every copy runs the kernels of a lone
// density(), so each result equals the corresponding single call.

struct Multi {
  std::vector<std::unique_ptr<System>> cl;
  uint64_t gen_basis = 0, gen_start = 0;
  std::vector<StepTask> h_tasks;
  std::vector<int> owner;        // copy of every task
  DevBuf<StepTask> tasks;
  int max_ns = 0, nlive = -1;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~Multi() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
};

System::~System() {
  for (auto e : ev) (void)hipEventDestroy(e);
  drop_graph();
  drop_ck_graph();
}

// device bytes of one copy of S (contour storage, factors, step work)
size_t system_bytes(const System& S) {
  const Grid& g = S.g;
  size_t b = 0;
  for (const auto& ch : S.chains) {
    b += (size_t)2 * ch->nslot * g.ms * 8 + (size_t)ch->nblk * (2 * g.ms + 2 * g.mf) * 8;
    if (S.ck_stride > 0) b += (size_t)(4 * ch->segpts + ch->nblk) * g.ms * 8;
  }
  b += (size_t)2 * S.nchain * (3 * g.mc * 16 + g.ms * 8);
  b += (size_t)(2 * S.nmon + 4) * g.m * 8 + (size_t)2 * S.nmon * g.mk * 16;
  return b;
}

// a copy of S's grid, stars, cell, chemistry and discretisation
void copy_system(System& D, const System& S) {
  const int ng[3] = {S.g.n1, S.g.n2, S.g.n3};
  D.g.init(ng, S.g.dim);
  D.nwave = S.nwave;
  D.nstar = S.nstar;
  D.h_wave = S.h_wave;
  D.h_wave_of_star = S.h_wave_of_star;
  D.h_star_of_wave = S.h_star_of_wave;
  D.h_star_invert = S.h_star_invert;
  D.h_coeff = S.h_coeff;
  D.coeff.upload(D.h_coeff.data(), D.nwave, D.st.s);
  D.star_of_wave.upload(D.h_star_of_wave.data(), D.nwave, D.st.s);
  D.star_invert.upload(D.h_star_invert.data(), D.nstar, D.st.s);
  build_basis_maps(D);
  D.sym_code = S.sym_code;
  D.have_basis = true;
  for (int i = 0; i < 9; ++i) D.gb[i] = S.gb[i];
  apply_cell(D);
  D.nmon = S.nmon;
  D.nchain = S.nchain;
  D.nsolv = S.nsolv;
  D.ensemble = S.ensemble;
  D.kuhn = S.kuhn;
  D.blocks = S.blocks;
  D.chain_length = S.chain_length;
  D.solv_mon = S.solv_mon;
  D.solv_size = S.solv_size;
  D.chi = S.chi;
  D.have_chem = true;
  D.ck_stride = S.ck_stride;
  D.use_graph = S.use_graph;
  startup(D, S.chain_step);
}

void set_copy_cell(System& D, const System& S) {
  bool same = true;
  for (int i = 0; i < 9; ++i) same = same && D.gb[i] == S.gb[i];
  if (same) return;
  for (int i = 0; i < 9; ++i) D.gb[i] = S.gb[i];
  apply_cell(D);
  D.st.sync();
}

// S's companion that stores every plane, at S's current state
System& full_of(System& S) {
  if (S.full && (S.full_basis != S.gen_basis || S.full_start != S.gen_start)) {
    if (S.last) S.have_density = false;
    S.last = nullptr;
    S.full.reset();
  }
  if (!S.full) {
    auto D = std::make_unique<System>();
    D->no_sym = true;
    copy_system(*D, S);
    S.full_basis = S.gen_basis;
    S.full_start = S.gen_start;
    S.full = std::move(D);
  }
  System& D = *S.full;
  set_copy_cell(D, S);
  if (D.use_graph != S.use_graph) {
    D.use_graph = S.use_graph;
    D.drop_graph();
    D.drop_ck_graph();
  }
  D.chi = S.chi;
  return D;
}

// the system that holds the results of S's last density()
System& live(System& S) { return S.last ? *S.last : S; }

// at least P copies matching S's current state (cell refreshed on every call)
void ensure_multi(System& S, int P) {
  if (S.multi && (S.multi->gen_basis != S.gen_basis || S.multi->gen_start != S.gen_start ||
                  (int)S.multi->cl.size() < P))
    S.multi.reset();
  if (!S.multi) {
    auto M = std::make_unique<Multi>();
    M->gen_basis = S.gen_basis;
    M->gen_start = S.gen_start;
    for (int i = 0; i < P; ++i) {
      M->cl.push_back(std::make_unique<System>());
      copy_system(*M->cl.back(), S);
      const System& D = *M->cl.back();
      for (const auto& t : D.h_tasks) {
        M->h_tasks.push_back(t);
        M->owner.push_back(i);
      }
      M->max_ns = std::max(M->max_ns, D.max_ns);
    }
    M->tasks.alloc(std::max<size_t>(M->h_tasks.size(), 1));
    for (auto& D : M->cl) D->st.sync();
    S.multi = std::move(M);
  }
  for (auto& D : S.multi->cl) {
    set_copy_cell(*D, S);
    D->use_graph = S.use_graph;
  }
}

void stress(System& S, int ncp, const double* dgsq, const double* phi_c, const double* mu_c, double* out);
void stress_launch(System& S, int ncp, const double* dgsq, hipStream_t s);
void stress_finish(System& S, int ncp, const double* phi_c, const double* mu_c, double* out);

// omega (n consecutive (N_monomer, N_star) arrays) -> rho (same), qout
// (N_chain per evaluation) and q_solvent (N_solvent per evaluation), each as
// density(); phi/mu in and out as n density() calls in a row.  max_batch > 0
// caps the evaluations per launch set (default: 64 copies, within 32 GiB).
// With cells (n consecutive Fortran G_basis(dim,dim)), evaluation k runs at
// cell k instead of the system's; with stress_out, it is followed by
// scf_stress with its own dGsq (n consecutive (N_star, ncp) arrays) into
// stress_out (ncp per evaluation), as density(); scf_stress in a row.
void density_many(System& S, int n, const double* omega, double* rho, double* qout, double* qsolv,
                  double* phi_c, double* mu_c, double* phi_s, double* mu_s, int max_batch,
                  const double* cells = nullptr, int ncp = 0, const double* dgsq = nullptr,
                  double* stress_out = nullptr) {
  REQUIRE(S.started && S.have_basis && S.have_cell, "system not ready (basis, cell, startup)");
  REQUIRE(n >= 0 && max_batch >= 0, "negative count");
  if (n == 0) return;
  REQUIRE(omega && rho, "null omega or rho");
  REQUIRE(!stress_out || (dgsq && ncp > 0 && ncp <= 6), "stress needs dGsq and 1..6 cell parameters");
  int cap = max_batch;
  if (cap == 0) {
    const size_t per = std::max<size_t>(system_bytes(S), 1);
    cap = (int)std::min<size_t>(64, std::max<size_t>(1, ((size_t)32 << 30) / per));
  }
  const int P = std::min(n, cap);
  ensure_multi(S, P);
  Multi& Mu = *S.multi;
  const Grid& g = S.g;
  hipStream_t s = S.st.s;
  const size_t nst = (size_t)S.nmon * S.nstar;
  const bool upd = qout != nullptr;
  for (int k0 = 0; k0 < n; k0 += P) {
    const int cnt = std::min(P, n - k0);
    if (cnt != Mu.nlive) {         // copies past cnt sit out this launch set
      for (size_t t = 0; t < Mu.h_tasks.size(); ++t) Mu.h_tasks[t].skip = Mu.owner[t] < cnt ? 0 : 1;
      HIPCHK(hipMemcpyAsync(Mu.tasks.p, Mu.h_tasks.data(), sizeof(StepTask) * Mu.h_tasks.size(),
                            hipMemcpyHostToDevice, s));
      Mu.nlive = cnt;
    }
    if (cells) {                     // evaluation k's cell on copy i
      const int dim = S.g.dim;
      for (int i = 0; i < cnt; ++i) {
        System& D = *Mu.cl[i];
        const double* G = cells + (size_t)(k0 + i) * dim * dim;
        bool same = true;
        for (int a = 0; a < dim; ++a)
          for (int b = 0; b < dim; ++b) same = same && D.gb[a * 3 + b] == G[a + dim * b];
        if (!same) {
          for (int a = 0; a < dim; ++a)
            for (int b = 0; b < dim; ++b) D.gb[a * 3 + b] = G[a + dim * b];
          apply_cell(D);
          D.st.sync();
        }
      }
    }
    for (int i = 0; i < cnt; ++i)
      density_pre(*Mu.cl[i], omega + (size_t)(k0 + i) * nst, phi_c, mu_c, phi_s, mu_s, s, false, upd);
    const int nt = (int)Mu.h_tasks.size();
    if (nt > 0) {
      if (S.use_graph) {
        if (!Mu.exec) {
          HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
          run_sweeps(g, Mu.tasks.p, nt, Mu.max_ns, sym_half(g.sym), s);
          HIPCHK(hipStreamEndCapture(s, &Mu.graph));
          HIPCHK(hipGraphInstantiate(&Mu.exec, Mu.graph, nullptr, nullptr, 0));
        }
        HIPCHK(hipGraphLaunch(Mu.exec, s));
      } else {
        run_sweeps(g, Mu.tasks.p, nt, Mu.max_ns, sym_half(g.sym), s);
      }
    }
    for (int i = 0; i < cnt; ++i) density_post(*Mu.cl[i], rho + (size_t)(k0 + i) * nst, s);
    if (stress_out)                  // in stream order after each copy's density()
      for (int i = 0; i < cnt; ++i) {
        Mu.cl[i]->have_density = true;
        stress_launch(*Mu.cl[i], ncp, dgsq + (size_t)(k0 + i) * S.nstar * ncp, s);
      }
    S.st.sync();
    for (int i = 0; i < cnt; ++i) {
      System& D = *Mu.cl[i];
      if (!sym_usable(D) || sym_failed(D)) {     // this field or cell needs every plane
        density(D, omega + (size_t)(k0 + i) * nst, rho + (size_t)(k0 + i) * nst,
                qout ? qout + (size_t)(k0 + i) * S.nchain : nullptr,
                qsolv ? qsolv + (size_t)(k0 + i) * S.nsolv : nullptr, phi_c, mu_c, phi_s, mu_s);
        if (stress_out)
          stress(live(D), ncp, dgsq + (size_t)(k0 + i) * S.nstar * ncp, phi_c, mu_c,
                 stress_out + (size_t)(k0 + i) * ncp);
        D.sym_bad = false;                       // another field may be symmetric
        continue;
      }
      D.last = nullptr;
      density_finish(*Mu.cl[i], qout ? qout + (size_t)(k0 + i) * S.nchain : nullptr,
                     qsolv ? qsolv + (size_t)(k0 + i) * S.nsolv : nullptr, phi_c, mu_c, phi_s, mu_s);
      if (stress_out) stress_finish(*Mu.cl[i], ncp, phi_c, mu_c, stress_out + (size_t)(k0 + i) * ncp);
    }
  }
}

// ---- reverse mode of density()
//
// For a scalar L(rho_grid, Q) with lam = dL/drho_grid (M, N_monomer) and dL/dQ
// per chain, the adjoint fields of the two sweeps obey
//   a_f(s) = g_f(s) + T_s a_f(s+1),   a_f(Ns) = g_f(Ns)      (backward in s)
//   a_r(s) = g_r(s) + T_{s-1} a_r(s-1), a_r(0) = g_r(0)       (forward in s)
// with the sources g_f(s) = c sum_b w_b(s) lam_mon(b) q_r(s) [+ Gam/M at Ns],
// g_r(s) = c sum_b w_b(s) lam_mon(b) q_f(s) (w_b: Simpson weights times ds_b/3,
// c = phi/(N Q) or e^mu/N, src/scf_mod.fp.f90:362-424) and Gam = dL/dQ
// (canonical: minus sum lam rho_chain / Q, since rho ~ 1/Q).  The step
// operator T (src/step_mod.f90:146-176) is symmetric, so the adjoint sweeps use
// the forward step kernels.  Each adjoint sweep runs beside a recomputation of
// the forward sweep it pairs with (same launches, steps in reverse order,
// inputs re-read from the stored q slabs); every step keeps its convolution
// fields, and the gradient kernels combine the pair after each step.

constexpr int ADJ_NB = 512;   // workgroups of the adjoint reductions

void adjoint_setup(System& S, bool with_k) {
  if (S.adj && S.adj->with_k == with_k) return;
  S.adj.reset();
  auto A = std::make_unique<AdjState>();
  static std::atomic<uint64_t> next_id{1};
  A->id = next_id++;
  const Grid& g = S.g;
  A->with_k = with_k;
  A->ntask = 4 * S.nchain;
  A->npair = 2 * S.nchain;
  size_t nblk = 0;
  for (int c = 0; c < S.nchain; ++c) {
    A->blk_off.push_back(nblk);
    nblk += S.chains[c]->nblk;
  }
  A->keep.alloc((size_t)5 * g.ms * A->ntask);
  A->lam.alloc((size_t)S.nmon * g.ms);
  A->scal.alloc((size_t)2 * S.nchain);
  if (with_k) {
    A->keepk.alloc((size_t)3 * g.mk * A->ntask);
    A->kblk.alloc((size_t)g.mk * nblk);
  }
  A->abc.alloc((size_t)3 * g.mc * A->ntask);
  A->q1.alloc((size_t)g.ms * A->ntask);
  A->gblk.alloc((size_t)g.ms * nblk);
  A->tasks.alloc(A->ntask);
  A->pairs.alloc(A->npair);
  A->part.alloc((size_t)ADJ_NB * MAXBLK + 1);
  std::vector<StepTask> ht(A->ntask);
  std::vector<int2> hp(A->npair);
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    // task order per chain: a_f, q_f recomputed, a_r, q_r recomputed
    for (int k = 0; k < 4; ++k) {
      const int ti = 4 * c + k;
      StepTask t = S.h_tasks[2 * c + (k < 2 ? 0 : 1)];   // factors, blocks, ns of the chain
      t.init_one = 0;
      t.skip = 0;
      t.keepA = nullptr;
      t.oth = nullptr;
      t.scal = nullptr;
      t.src_end = -1;
      for (int b = 0; b < MAXBLK; ++b) t.lam[b] = nullptr;
      if (k == 0 || k == 2) {       // adjoint sweeps, opposite direction to their q; no slab
        t.dir = k == 0 ? -1 : 1;
        t.slab = nullptr;
        t.add_src = 1;
        t.nostore = 1;
        t.rev = t.reload = 0;
        t.oth = k == 0 ? ch.qr.p : ch.qf.p;        // g_f uses q_r, g_r uses q_f
        t.src_end = k == 0 ? ch.ns : -1;           // dL/dQ enters a_f at s = Ns
        t.scal = A->scal.p + 2 * c;
        for (int b = 0; b < ch.nblk; ++b) t.lam[b] = A->lam.p + (size_t)ch.mon[b] * g.ms;
        t.keepA = A->keep.p + ((size_t)5 * ti + 3) * g.ms;
      } else {                      // recomputed forward sweeps
        t.dir = k == 1 ? 1 : -1;
        t.slab = k == 1 ? ch.qf.p : ch.qr.p;
        t.add_src = 0;
        t.rev = t.reload = t.nostore = 1;
      }
      t.A = A->abc.p + (size_t)(3 * ti) * g.mc;
      t.B = t.A + g.mc;
      t.C = t.B + g.mc;
      t.q1 = A->q1.p + (size_t)ti * g.ms;
      t.keepU = A->keep.p + (size_t)(5 * ti) * g.ms;
      t.keepV = t.keepU + g.ms;
      t.keepW = t.keepV + g.ms;
      for (int q = 0; q < 3; ++q)
        t.keepK[q] = with_k ? A->keepk.p + (size_t)(3 * ti + q) * g.mk : nullptr;
      for (int b = 0; b < ch.nblk; ++b) {
        t.ds[b] = ch.ds[b];
        t.bsq[b] = S.kuhn[ch.mon[b]] * S.kuhn[ch.mon[b]];
        t.grad[b] = A->gblk.p + (A->blk_off[c] + b) * g.ms;
        t.kgrad[b] = with_k ? A->kblk.p + (A->blk_off[c] + b) * g.mk : nullptr;
      }
      ht[ti] = t;
    }
    hp[2 * c] = make_int2(4 * c, 4 * c + 1);
    hp[2 * c + 1] = make_int2(4 * c + 2, 4 * c + 3);
  }
  HIPCHK(hipMemcpyAsync(A->tasks.p, ht.data(), sizeof(StepTask) * A->ntask, hipMemcpyHostToDevice,
                        S.st.s));
  HIPCHK(hipMemcpyAsync(A->pairs.p, hp.data(), sizeof(int2) * A->npair, hipMemcpyHostToDevice,
                        S.st.s));
  if (S.ck_stride > 0) {
    // segment buffers of a chain: 0 q_f(R_r), 1 q_r(R_r), 2 q_f(F_r), 3 q_r(F_r)
    const int K = S.ck_stride, nc = S.nchain;
    const CkPlan& P = S.ck;
    A->rec_abc.alloc((size_t)3 * g.mc * 4 * nc);
    A->rec_q1.alloc((size_t)g.ms * 4 * nc);
    std::vector<StepTask> rec((size_t)P.nround * 4 * nc), adj((size_t)P.nround * 4 * nc);
    for (int r = 0; r < P.nround; ++r)
      for (int c = 0; c < nc; ++c) {
        ChainDev& ch = *S.chains[c];
        auto seg = [&](int i) { return ch.seg.p + (size_t)i * ch.segpts * g.ms; };
        const int* mapR = P.maps.p + P.map_off[((size_t)r * nc + c) * 2 + 0];
        const int* mapF = P.maps.p + P.map_off[((size_t)r * nc + c) * 2 + 1];
        // adjoint tasks of this round; a chain whose steps ended in an earlier
        // round (its last finishing step may fall here) keeps that round's segments
        const int rl = std::min(r, (ch.ns + K - 1) / K - 1);
        const int* amapR = P.maps.p + P.map_off[((size_t)rl * nc + c) * 2 + 0];
        const int* amapF = P.maps.p + P.map_off[((size_t)rl * nc + c) * 2 + 1];
        for (int k = 0; k < 4; ++k) {
          StepTask t = ht[4 * c + k];
          if (k == 0) { t.oth = seg(3); t.omap = amapF; }         // a_f: sources from q_r on F_r
          if (k == 1) { t.slab = seg(2); t.pmap = amapF; }        // q_f recomputed on F_r
          if (k == 2) { t.oth = seg(0); t.omap = amapR; }         // a_r: sources from q_f on R_r
          if (k == 3) { t.slab = seg(1); t.pmap = amapR; }        // q_r recomputed on R_r
          adj[((size_t)r * nc + c) * 4 + k] = t;
        }
        // recomputation tasks: q_f and q_r on R_r (buffers 0, 1) and on F_r (2, 3)
        for (int k = 0; k < 4; ++k) {
          const int side = k / 2, d = k % 2;         // d 0: q_f forward, 1: q_r backward
          int lo, hi;
          if (side == 0) { lo = r * K; hi = std::min((r + 1) * K, ch.ns); }
          else { hi = ch.ns - r * K; lo = std::max(0, ch.ns - (r + 1) * K); }
          StepTask t = S.h_tasks[2 * c + d];
          t.init_one = 0;
          t.slab = seg(2 * side + d);
          t.pmap = side == 0 ? mapR : mapF;
          const int ti = 4 * c + k;
          t.A = A->rec_abc.p + (size_t)(3 * ti) * g.mc;
          t.B = t.A + g.mc;
          t.C = t.B + g.mc;
          t.q1 = A->rec_q1.p + (size_t)ti * g.ms;
          if (lo >= hi) {
            t.skip = 1;
          } else if (d == 0) {
            t.jbeg = t.jofs = lo;
            t.jend = hi;
            t.start = ch.point(+1, lo);
          } else {
            t.jbeg = t.jofs = ch.ns - hi;
            t.jend = ch.ns - lo;
            t.start = ch.point(-1, hi);
          }
          rec[((size_t)r * nc + c) * 4 + k] = t;
        }
      }
    A->ck_rec.upload(rec.data(), rec.size(), S.st.s);
    A->ck_adj.upload(adj.data(), adj.size(), S.st.s);
    A->h_ck_rec = rec;
    A->h_ck_adj = adj;
  }
  S.st.sync();
  A->h_tasks = ht;
  A->h_pairs = hp;
  S.adj = std::move(A);
}

// the adjoint sweeps with their gradient kernels (launch order as run_sweeps).
// Checkpointed storage: step j runs with the tasks of round j / K, whose
// segments the recomputation sweeps fill just before the round's first step.
// One launch set of adjoint sweeps: the tasks and pairs of one or more
// systems on one grid, with the checkpoint rounds (K > 0) of all of them.
struct AdjSweeps {
  const StepTask* tasks = nullptr;
  int ntask = 0;
  const int2* pairs = nullptr;
  int npair = 0;
  int max_ns = 0;
  bool with_k = false;
  bool half_z = false;                   // every system's planes allow it (step_z)
  int K = 0, nround = 0;
  const int* len = nullptr;              // per round: longest segment
  const StepTask* ck_rec = nullptr;      // per round: ntask recomputation tasks
  const StepTask* ck_adj = nullptr;      // per round: ntask adjoint tasks
};

void run_adj_sweeps(const Grid& g, const AdjSweeps& W, hipStream_t s) {
  const int nt = W.ntask, max_ns = W.max_ns;
  const int gb = grid_blocks(g.ms), gk = grid_blocks(g.mk);
  const int K = W.K;
  const StepTask* tasks = W.tasks;
  for (int j = 0; j <= max_ns; ++j) {
    if (K > 0) {
      const int r = std::min(j / K, W.nround - 1);
      if (j % K == 0 && j / K < W.nround)
        run_sweeps(g, W.ck_rec + (size_t)r * nt, nt, W.len[r], W.half_z, s);
      tasks = W.ck_adj + (size_t)r * nt;
    }
    launch_step_a(g, tasks, nt, j, true, s);
    if (j >= 1)
      hipLaunchKernelGGL(k_adj_grad, dim3(gb), dim3(256), 0, s, tasks, W.pairs, W.npair, j - 1, g.ms);
    if (j == max_ns) break;
    g.step_z(tasks, nt, j, 0, 2, true, false, s);
    g.step_c(tasks, nt, j, true, s);
    g.step_z(tasks, nt, j, 1, 1, true, false, s);
    if (W.with_k)
      hipLaunchKernelGGL(k_adj_kgrad, dim3(gk), dim3(256), 0, s, tasks, W.pairs, W.npair, j, g.n1,
                         g.n2, g.n3, g.zs->zw);
  }
  HIPCHK(hipGetLastError());
}

// the adjoint sweeps of one system
void run_adj_sweeps(const System& S, hipStream_t s) {
  const AdjState& A = *S.adj;
  AdjSweeps W;
  W.tasks = A.tasks.p;
  W.ntask = A.ntask;
  W.pairs = A.pairs.p;
  W.npair = A.npair;
  W.max_ns = S.max_ns;
  W.with_k = A.with_k;
  W.half_z = sym_half(S.g.sym);
  W.K = S.ck_stride;
  if (W.K > 0) {
    W.nround = S.ck.nround;
    W.len = S.ck.len.data();
    W.ck_rec = A.ck_rec.p;
    W.ck_adj = A.ck_adj.p;
  }
  run_adj_sweeps(S.g, W, s);
}

// reduce np device partials to one host value (stream synchronised)
double host_sum(System& S, const double* part, int np) {
  double* slot = S.adj->part.p + S.adj->part.n - 1;
  hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(NTA), 0, S.st.s, part, np, 1.0, slot);
  double v = 0.0;
  HIPCHK(hipMemcpyAsync(&v, slot, sizeof(double), hipMemcpyDeviceToHost, S.st.s));
  S.st.sync();
  return v;
}

// lam (M, N_monomer) and dQ (N_chain, may be null) on input; out: grad
// (M, N_monomer, device) = dL/d omega_grid; with dgg (dim, dim, ncp) also
// dL/d cell_param (ncp); with dlen also dL/d block length per chain and block
// (block step count fixed; the chain length in the prefactor is the sum of
// the block lengths); with dphi dL/d phi_chain (canonical ensemble: rho of a
// chain is proportional to its phi; 0 in the grand ensemble).
// Host scalars of one adjoint call: the Simpson sums T_b and the density
// prefactor c of every chain.
struct AdjCall {
  std::vector<std::vector<double>> T;
  std::vector<double> coef;
};

// Before the sweeps: adjoint state (with |k|^2 gradients when with_k), the
// sums T_b = sum_r lam_b rho-integrand of every block (for Gam and d/d ds),
// the sources' coefficients, cleared gradient accumulators.
void adjoint_pre(System& S, const double* lam, const double* dQ, bool with_k, AdjCall& C) {
  REQUIRE(S.have_density, "the adjoint requires a previous density()");
  REQUIRE(S.nsolv == 0, "the adjoint does not support solvent species");
  adjoint_setup(S, with_k);
  AdjState& A = *S.adj;
  const Grid& g = S.g;
  hipStream_t s = S.st.s;
  const int nb = ADJ_NB;
  // lam in the sweeps' packed order
  hipLaunchKernelGGL(k_pack, dim3(grid_blocks(S.nmon * g.ms)), dim3(NTA), 0, s, lam, g.m, g.ms, S.nmon, g.n1,
                     g.n2, A.lam.p);
  const long plane = (long)g.n1 * g.n2;
  lam = A.lam.p;
  double* part = A.part.p;
  auto& T = C.T;
  auto& coef = C.coef;
  T.assign(S.nchain, {});
  coef.assign(S.nchain, 0.0);
  std::vector<double> gam(S.nchain);
  std::vector<SimpsonArgs> sa(S.nchain);
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    SimpsonArgs& a = sa[c];
    std::memset(&a, 0, sizeof a);
    a.nblk = ch.nblk;
    for (int b = 0; b <= ch.nblk; ++b) a.bnd[b] = ch.bnd[b];
    for (int b = 0; b < ch.nblk; ++b) {
      a.ds[b] = ch.ds[b];
      a.monomer[b] = ch.mon[b];
    }
    a.chain_length = ch.length;
    a.ensemble = S.chain_ens;
    T[c].resize(ch.nblk);
    if (S.ck_stride > 0) {      // the block integrals of the last density() are kept
      for (int b = 0; b < ch.nblk; ++b) {
        hipLaunchKernelGGL(k_partial_dot, dim3(nb), dim3(NTA), 0, s, ch.blk.p + (size_t)b * g.ms,
                           lam + (size_t)ch.mon[b] * g.ms, g.ms, g.sym, g.n3, plane, part);
        T[c][b] = host_sum(S, part, nb);
      }
    } else {
      hipLaunchKernelGGL(k_simpson_lam, dim3(nb, ch.nblk), dim3(NTA), 0, s, ch.qf.p, ch.qr.p, g.ms, a,
                         lam, g.sym, g.n3, plane, part);
      for (int b = 0; b < ch.nblk; ++b) T[c][b] = host_sum(S, part + (size_t)b * nb, nb);
    }
    const double Q = S.h_Q[c];
    coef[c] = S.chain_ens == 1 ? std::exp(S.h_chem[2 * c + 1]) / ch.length
                               : S.h_chem[2 * c] / (ch.length * Q);
    double tsum = 0.0;
    for (int b = 0; b < ch.nblk; ++b) tsum += T[c][b];
    gam[c] = (dQ ? dQ[c] : 0.0) - (S.chain_ens == 1 ? 0.0 : coef[c] * tsum / Q);
  }
  // sources: coefficient and end term per chain
  std::vector<double> hs(2 * S.nchain);
  for (int c = 0; c < S.nchain; ++c) {
    hs[2 * c] = coef[c];
    hs[2 * c + 1] = gam[c] / (double)g.m;
  }
  HIPCHK(hipMemcpyAsync(A.scal.p, hs.data(), sizeof(double) * hs.size(), hipMemcpyHostToDevice, s));
  size_t nblk = 0;
  for (int c = 0; c < S.nchain; ++c) nblk += S.chains[c]->nblk;
  hipLaunchKernelGGL(k_fill, dim3(grid_blocks((long)(nblk * g.ms))), dim3(NTA), 0, s, A.gblk.p,
                     (long)(nblk * g.ms), 0.0);
  if (with_k)
    hipLaunchKernelGGL(k_fill, dim3(grid_blocks((long)(nblk * g.mk))), dim3(NTA), 0, s, A.kblk.p,
                       (long)(nblk * g.mk), 0.0);
}

// After the sweeps: the gradients from the accumulators (see density_adjoint)
void adjoint_post(System& S, const AdjCall& C, double* grad, int ncp, const double* dgg,
                  double* dcell, double* dlen, double* dphi) {
  AdjState& A = *S.adj;
  const Grid& g = S.g;
  hipStream_t s = S.st.s;
  const int nb = ADJ_NB;
  double* part = A.part.p;
  const auto& T = C.T;
  const auto& coef = C.coef;
  size_t nblk = 0;
  for (int c = 0; c < S.nchain; ++c) nblk += S.chains[c]->nblk;
  // omega gradient per monomer: sum of its blocks
  hipLaunchKernelGGL(k_fill, dim3(grid_blocks((long)S.nmon * g.m)), dim3(NTA), 0, s, grad,
                     (long)S.nmon * g.m, 0.0);
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev& ch = *S.chains[c];
    for (int b = 0; b < ch.nblk; ++b)
      hipLaunchKernelGGL(k_axpy1, dim3(grid_blocks(g.ms)), dim3(NTA), 0, s,
                         A.gblk.p + (A.blk_off[c] + b) * g.ms, g.ms, g.n1, g.n2,
                         grad + (size_t)ch.mon[b] * g.m);
  }
  if (g.sym)
    hipLaunchKernelGGL(k_sym_expand, dim3(grid_blocks((g.m - g.ms) * S.nmon)), dim3(NTA), 0, s, grad, S.nmon,
                       g.sym, g.n1, g.n2, g.n3);
  HIPCHK(hipGetLastError());
  GeomArgs ga;
  ga.n1 = g.n1;
  ga.n2 = g.n2;
  ga.n3 = g.n3;
  ga.dim = g.dim;
  for (int i = 0; i < 9; ++i) ga.gb[i] = S.gb[i];
  for (int d = 0; d < 3; ++d) {
    ga.gmin[d] = S.gmin[d];
    ga.gext[d] = S.gext[d];
  }
  if (dgg && ncp > 0) {
    DevBuf<double> d_dgg;
    d_dgg.upload(dgg, (size_t)g.dim * g.dim * ncp, s);
    for (int p = 0; p < ncp; ++p) dcell[p] = 0.0;
    for (size_t k = 0; k < nblk; ++k) {
      hipLaunchKernelGGL(k_dksq_dot, dim3(nb, ncp), dim3(NTA), 0, s, ga, d_dgg.p,
                         A.kblk.p + k * g.mk, part);
      for (int p = 0; p < ncp; ++p) dcell[p] += host_sum(S, part + (size_t)p * nb, nb);
    }
  }
  if (dphi) {
    for (int c = 0; c < S.nchain; ++c) {
      double tsum = 0.0;
      for (double t : T[c]) tsum += t;
      const double phi = S.h_chem[2 * c];
      dphi[c] = (S.chain_ens == 0 && phi != 0.0) ? coef[c] * tsum / phi : 0.0;
    }
  }
  if (dlen) {
    // d/d ds_b = [sum_r omega grad_b + sum_k ksq kgrad_b + c T_b] / ds_b, and
    // ds_b = L_b / (2 iblk_b) at a fixed step count, so d/dL_b = d/d ds_b * ds_b / L_b;
    // plus the prefactor's 1/N, N = sum_b L_b: -c sum_b T_b / N
    size_t o = 0;
    for (int c = 0; c < S.nchain; ++c) {
      ChainDev& ch = *S.chains[c];
      double tsum = 0.0;
      for (int b = 0; b < ch.nblk; ++b) tsum += T[c][b];
      for (int b = 0; b < ch.nblk; ++b, ++o) {
        const double* gb_ = A.gblk.p + (A.blk_off[c] + b) * g.ms;
        // omega in packed order, into a buffer that is free after the sweeps
        hipLaunchKernelGGL(k_pack, dim3(grid_blocks(g.ms)), dim3(NTA), 0, s,
                           S.omega_grid.p + (size_t)ch.mon[b] * g.m, g.m, g.ms, 1, g.n1, g.n2, A.keep.p);
        hipLaunchKernelGGL(k_partial_dot, dim3(nb), dim3(NTA), 0, s, gb_, A.keep.p, g.ms, g.sym, g.n3,
                           (long)g.n1 * g.n2, part);
        const double t1 = host_sum(S, part, nb);
        hipLaunchKernelGGL(k_partial_dot, dim3(nb), dim3(NTA), 0, s, A.kblk.p + (A.blk_off[c] + b) * g.mk,
                           S.ksq.p, g.mk, 0, g.n3, 1L, part);
        const double t2 = host_sum(S, part, nb);
        const double dds = (t1 + t2 + coef[c] * T[c][b]) / ch.ds[b];
        const double L = S.blocks[c][b].second;
        dlen[o] = dds * ch.ds[b] / L - coef[c] * tsum / ch.length;
      }
    }
  }
  S.st.sync();
}

// Whether the reverse mode of S's last density() can run on symmetric planes:
// that density() did, and lam = dL/drho, given on the grid, is symmetric too
// (the gradient is linear in lam and its sources are lam times contour points).
bool adjoint_symmetric(System& S, const double* lam) {
  REQUIRE(S.have_density, "the adjoint requires a previous density()");
  System& L = live(S);
  return L.g.sym && grid_symmetric(L, lam, 1e-13);
}

// The system whose stored planes the reverse mode of S's last density() reads.
// sym: those of that density(); otherwise every plane, and after a density()
// on symmetric planes the companion takes over its fields and contour points.
System& adjoint_of(System& S, bool sym) {
  REQUIRE(S.have_density, "the adjoint requires a previous density()");
  System& L = live(S);
  if (sym || !L.g.sym) return L;
  System& D = full_of(S);
  const Grid& g = S.g;
  hipStream_t s = D.st.s;
  S.st.sync();
  const size_t n = sizeof(double) * (size_t)S.nmon * g.m;
  HIPCHK(hipMemcpyAsync(D.omega_grid.p, S.omega_grid.p, n, hipMemcpyDeviceToDevice, s));
  HIPCHK(hipMemcpyAsync(D.rho_grid.p, S.rho_grid.p, n, hipMemcpyDeviceToDevice, s));
  const double* hc = S.h_chem.data();
  std::vector<double> phi(S.nchain), mu(S.nchain), phis(S.nsolv), mus(S.nsolv);
  for (int c = 0; c < S.nchain; ++c) phi[c] = hc[2 * c], mu[c] = hc[2 * c + 1];
  for (int i = 0; i < S.nsolv; ++i) phis[i] = hc[2 * (S.nchain + i)], mus[i] = hc[2 * (S.nchain + i) + 1];
  density_pre(D, nullptr, phi.data(), mu.data(), phis.data(), mus.data(), s, true, S.chain_ens == 1);
  for (int c = 0; c < S.nchain; ++c) {
    ChainDev &a = *S.chains[c], &b = *D.chains[c];
    const auto expand = [&](const double* from, double* to, int np) {
      hipLaunchKernelGGL(k_sym_point, dim3(grid_blocks(g.m), np), dim3(NTA), 0, s, from, g.ms, g.sym, g.n1,
                         g.n2, g.n3, 1, to, g.m);
    };
    expand(a.qf.p, b.qf.p, a.nslot);
    expand(a.qr.p, b.qr.p, a.nslot);
    if (S.ck_stride > 0) expand(a.blk.p, b.blk.p, a.nblk);
  }
  HIPCHK(hipGetLastError());
  D.st.sync();
  D.h_Q = S.h_Q;
  D.chain_ens = S.chain_ens;
  D.have_density = true;
  S.last = &D;
  return D;
}

void density_adjoint(System& sys, const double* lam, const double* dQ, double* grad, int ncp,
                     const double* dgg, double* dcell, double* dlen, double* dphi) {
  System& S = adjoint_of(sys, adjoint_symmetric(sys, lam));
  REQUIRE(ncp <= 6, "at most 6 cell parameters");
  const bool with_k = dgg != nullptr || dlen != nullptr;
  AdjCall C;
  adjoint_pre(S, lam, dQ, with_k, C);
  AdjState& A = *S.adj;
  hipStream_t s = S.st.s;
  // the sweeps (captured once as a graph)
  if (S.use_graph) {
    if (!A.exec) {
      HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      run_adj_sweeps(S, s);
      HIPCHK(hipStreamEndCapture(s, &A.graph));
      HIPCHK(hipGraphInstantiate(&A.exec, A.graph, nullptr, nullptr, 0));
    }
    HIPCHK(hipGraphLaunch(A.exec, s));
  } else {
    run_adj_sweeps(S, s);
  }
  adjoint_post(S, C, grad, ncp, dgg, dcell, dlen, dphi);
}

// ---- reverse mode of several systems at once
//
// Systems on one grid (any chemistry, one checkpoint stride) run their
// adjoint sweeps, and the checkpoint rounds that recompute their segments,
// in one launch set per contour step, captured once as a HIP graph.  Each
// system's sources, reductions and gradients are its own (adjoint_pre/post);
// every system's tasks run the kernels of its lone adjoint, so the results
// equal the single calls'.
struct AdjGroup {
  std::vector<System*> members;  // as given
  std::vector<System*> sys;      // those whose planes their adjoints read (adjoint_of)
  std::vector<uint64_t> ids;     // AdjState ids the launch set was built from
  bool with_k = false;
  Stream st;
  DevBuf<StepTask> tasks, ck_rec, ck_adj;
  DevBuf<int2> pairs;
  std::vector<int> len;
  AdjSweeps W;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  void drop_graph() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    exec = nullptr;
    graph = nullptr;
  }
  ~AdjGroup() { drop_graph(); }
};

void build_adj_group(AdjGroup& G) {
  const System& S0 = *G.sys[0];
  const int K = S0.ck_stride;
  int ntot = 0, max_ns = 0, nround = 0;
  for (System* S : G.sys) {
    REQUIRE(S->g.n1 == S0.g.n1 && S->g.n2 == S0.g.n2 && S->g.n3 == S0.g.n3,
            "adjoint group: systems on different grids");
    REQUIRE(S->ck_stride == K, "adjoint group: systems with different checkpoint strides");
    ntot += S->adj->ntask;
    max_ns = std::max(max_ns, S->max_ns);
    if (K > 0) nround = std::max(nround, S->ck.nround);
  }
  std::vector<StepTask> ht;
  std::vector<int2> hp;
  std::vector<int> off;
  for (System* S : G.sys) {
    const AdjState& A = *S->adj;
    const int o = (int)ht.size();
    off.push_back(o);
    ht.insert(ht.end(), A.h_tasks.begin(), A.h_tasks.end());
    for (const int2& p : A.h_pairs) hp.push_back(make_int2(p.x + o, p.y + o));
  }
  G.tasks.upload(ht.data(), ht.size(), G.st.s);
  G.pairs.upload(hp.data(), hp.size(), G.st.s);
  G.W = AdjSweeps();
  G.W.tasks = G.tasks.p;
  G.W.ntask = ntot;
  G.W.pairs = G.pairs.p;
  G.W.npair = (int)hp.size();
  G.W.max_ns = max_ns;
  G.W.with_k = G.with_k;
  G.W.half_z = true;
  for (System* S : G.sys) G.W.half_z = G.W.half_z && sym_half(S->g.sym);
  G.W.K = K;
  if (K > 0) {
    // round r of a system past its own rounds: recomputation skipped, adjoint
    // tasks of its last round (whose windows end its sweeps)
    std::vector<StepTask> rec((size_t)nround * ntot), adj((size_t)nround * ntot);
    G.len.assign(nround, 0);
    for (int r = 0; r < nround; ++r)
      for (size_t i = 0; i < G.sys.size(); ++i) {
        const System& S = *G.sys[i];
        const AdjState& A = *S.adj;
        const int nt = A.ntask, ri = std::min(r, S.ck.nround - 1);
        for (int k = 0; k < nt; ++k) {
          StepTask tr = A.h_ck_rec[(size_t)ri * nt + k];
          if (r >= S.ck.nround) tr.skip = 1;
          rec[(size_t)r * ntot + off[i] + k] = tr;
          adj[(size_t)r * ntot + off[i] + k] = A.h_ck_adj[(size_t)ri * nt + k];
        }
        if (r < S.ck.nround) G.len[r] = std::max(G.len[r], S.ck.len[r]);
      }
    G.ck_rec.upload(rec.data(), rec.size(), G.st.s);
    G.ck_adj.upload(adj.data(), adj.size(), G.st.s);
    G.W.nround = nround;
    G.W.len = G.len.data();
    G.W.ck_rec = G.ck_rec.p;
    G.W.ck_adj = G.ck_adj.p;
  }
  G.st.sync();
  G.ids.clear();
  for (System* S : G.sys) G.ids.push_back(S->adj->id);
  G.drop_graph();
}

// per system i: lam[i], dQ[i] (may be null) in; grad[i] out; with dgg[i] the
// cell gradient, with dlen[i] the block-length gradient, with dphi[i] the
// phi_chain gradient, as density_adjoint (the pointer arrays may be null)
void adjoint_group(AdjGroup& G, const double* const* lam, const double* const* dQ,
                   double* const* grad, const int* ncp, const double* const* dgg,
                   double* const* dcell, double* const* dlen, double* const* dphi) {
  const size_t n = G.members.size();
  bool with_k = false;
  for (size_t i = 0; i < n; ++i) {
    REQUIRE(lam && lam[i] && grad && grad[i], "null grid pointer");
    const int nc = ncp ? ncp[i] : 0;
    REQUIRE(nc >= 0 && nc <= 6, "at most 6 cell parameters");
    REQUIRE(!(dgg && dgg[i]) || (dcell && dcell[i]), "dGG given without an output for the cell gradient");
    with_k = with_k || (dgg && dgg[i]) || (dlen && dlen[i]);
  }
  G.sys.clear();
  // on symmetric planes if every member can be, with as many of them
  bool sym = true;
  for (size_t i = 0; i < n; ++i)
    sym = sym && adjoint_symmetric(*G.members[i], lam[i]) && live(*G.members[i]).g.np == live(*G.members[0]).g.np;
  for (System* S : G.members) G.sys.push_back(&adjoint_of(*S, sym));
  std::vector<AdjCall> C(n);
  for (size_t i = 0; i < n; ++i)
    adjoint_pre(*G.sys[i], lam[i], dQ ? dQ[i] : nullptr, with_k, C[i]);
  for (System* S : G.sys) S->st.sync();
  bool same = G.ids.size() == n && G.with_k == with_k;
  for (size_t i = 0; same && i < n; ++i) same = G.sys[i]->adj->id == G.ids[i];
  if (!same) {
    G.with_k = with_k;
    build_adj_group(G);
  }
  hipStream_t s = G.st.s;
  if (G.sys[0]->use_graph) {
    if (!G.exec) {
      HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      run_adj_sweeps(G.sys[0]->g, G.W, s);
      HIPCHK(hipStreamEndCapture(s, &G.graph));
      HIPCHK(hipGraphInstantiate(&G.exec, G.graph, nullptr, nullptr, 0));
    }
    HIPCHK(hipGraphLaunch(G.exec, s));
  } else {
    run_adj_sweeps(G.sys[0]->g, G.W, s);
  }
  G.st.sync();
  for (size_t i = 0; i < n; ++i)
    adjoint_post(*G.sys[i], C[i], grad[i], ncp ? ncp[i] : 0, dgg ? dgg[i] : nullptr,
                 dcell ? dcell[i] : nullptr, dlen ? dlen[i] : nullptr, dphi ? dphi[i] : nullptr);
}

// ---- scf_stress (src/scf_mod.fp.f90:451-550)

// per contour point p of every chain: sum_star qr_basis * dGsq * qf_basis
// (:505-528) on the device, copied to the host (S.pin_dots)
void stress_launch(System& S, int ncp, const double* dgsq, hipStream_t s) {
  REQUIRE(S.have_density, "scf_stress requires a previous density()");
  REQUIRE(S.ck_stride == 0, "scf_stress needs every contour point (checkpointed storage is on)");
  const Grid& g = S.g;
  S.pin_dgsq.alloc((size_t)S.nstar * ncp);
  std::memcpy(S.pin_dgsq.p, dgsq, sizeof(double) * S.nstar * ncp);
  S.dgsq.alloc((size_t)S.nstar * ncp);
  HIPCHK(hipMemcpyAsync(S.dgsq.p, S.pin_dgsq.p, sizeof(double) * S.nstar * ncp,
                        hipMemcpyHostToDevice, s));
  const int chunk = 32;
  const long mkc = (long)g.n3 * S.ncol;       // one point's compact spectrum
  S.sbasis.alloc((size_t)2 * chunk * S.nstar);
  S.skbuf.alloc((size_t)2 * chunk * (mkc + (long)g.np * S.nin));
  double2* const work = S.skbuf.p + (size_t)2 * chunk * mkc;
  size_t npts = 0;
  for (int sp = 0; sp < S.nchain; ++sp) npts += (size_t)S.chains[sp]->ns + 1;
  S.sdots.alloc(npts * ncp);
  size_t off = 0;
  for (int sp = 0; sp < S.nchain; ++sp) {
    ChainDev& ch = *S.chains[sp];
    for (int p0 = 0; p0 <= ch.ns; p0 += chunk) {
      const int np = std::min(chunk, ch.ns + 1 - p0);
      // qf and qr of the chunk's points in one launch per pass: qr's spectra
      // after qf's, then star coefficients (2 np, N_star) with qr's at np + p
      g.r2c_cols(ch.qf.p + (size_t)p0 * g.ms, ch.qr.p + (size_t)p0 * g.ms, work, S.skbuf.p, np, S.scpos.p,
                 S.nin, S.ncol, S.ssrc.p, S.scolk.p, s);
      hipLaunchKernelGGL(k_kgrid_to_basis, dim3(grid_blocks((long)S.nstar * 2 * np)), dim3(NTA), 0,
                         s, S.skbuf.p, mkc, 2 * np, S.nstar, S.sidx_c.p, S.sconj.p, S.scoef.p,
                         S.star_invert.p, 1.0, S.sbasis.p, 0);
      hipLaunchKernelGGL(k_stress_dots, dim3(np), dim3(NTA), 0, s, S.sbasis.p, S.sbasis.p + np,
                         2 * np, S.nstar, S.dgsq.p, ncp, S.sdots.p + (off + p0) * ncp);
    }
    off += (size_t)ch.ns + 1;
  }
  HIPCHK(hipGetLastError());
  S.pin_dots.alloc(npts * ncp);
  HIPCHK(hipMemcpyAsync(S.pin_dots.p, S.sdots.p, sizeof(double) * npts * ncp,
                        hipMemcpyDeviceToHost, s));
}

// after synchronisation: Simpson weights and the sum over contour points in
// the reference's order (:497-544)
void stress_finish(System& S, int ncp, const double* phi_c, const double* mu_c, double* out) {
  const double rnodes = (double)S.g.m;
  const double normal = rnodes * rnodes * 3.0 * 6.0;        // :485-488
  for (int k = 0; k < ncp; ++k) out[k] = 0.0;
  size_t off = 0;
  for (int sp = 0; sp < S.nchain; ++sp) {
    ChainDev& ch = *S.chains[sp];
    std::vector<double> dQ(ncp, 0.0);
    for (int b = 0; b < ch.nblk; ++b) {
      const double bk = S.kuhn[ch.mon[b]];
      const double ds0 = ch.ds[b];
      const int ibgn = ch.bnd[b] + 1, iend = ch.bnd[b + 1] + 1;   // 1-based, as the reference
      for (int i = ibgn; i <= iend; ++i) {
        double ds = ds0;
        if (i != ibgn && i != iend) ds = (i % 2 == 0) ? 4.0 * ds : 2.0 * ds;
        for (int beta = 0; beta < ncp; ++beta) {
          double inc = S.pin_dots.p[(off + (size_t)(i - 1)) * ncp + beta];
          inc = inc * (bk * bk) * ds / normal;
          dQ[beta] = dQ[beta] - inc;
        }
      }
    }
    off += (size_t)ch.ns + 1;
    const double Q = S.h_Q[sp];
    for (int beta = 0; beta < ncp; ++beta) {
      if (S.ensemble == 0)
        out[beta] = out[beta] - (dQ[beta] / Q) * phi_c[sp] / ch.length;
      else
        out[beta] = out[beta] - (dQ[beta] / Q) * std::exp(mu_c[sp]) * Q / ch.length;
    }
  }
}

void stress(System& S, int ncp, const double* dgsq, const double* phi_c, const double* mu_c,
            double* out) {
  stress_launch(S, ncp, dgsq, S.st.s);
  S.st.sync();
  stress_finish(S, ncp, phi_c, mu_c, out);
}


// =========================================================== batched solves
// Many independent systems iterated together (iterate_AM's control flow,
// src/iterate_mod.fp.f90:1042-1490, per instance).  Systems with the same
// grid form a group whose contour sweeps run in one launch set per step
// (all instances' sweep tasks side by side), captured once as a HIP graph;
// converged instances stay in the graph with their tasks marked skip.

// free energy and pressure (src/scf_mod.fp.f90:834-886)
void thermo(const System& S, const double* rho, const double* omega, const double* phi_c,
            const double* mu_c, const double* phi_s, const double* mu_s, double* fo, double* po) {
  const int nm = S.nmon;
  double f = 0.0;
  for (int i = 0; i < S.nchain; ++i)
    if (phi_c[i] > 1.0e-8f) f = f + phi_c[i] * (mu_c[i] - 1.0) / S.chain_length[i];
  for (int i = 0; i < S.nsolv; ++i)
    if (phi_s[i] > 1.0e-8f) f = f + phi_s[i] * (mu_s[i] - 1.0) / S.solv_size[i];
  for (int i = 0; i < S.nstar; ++i)
    for (int a = 0; a < nm; ++a) {
      for (int b = a + 1; b < nm; ++b)
        f = f + rho[a + (size_t)nm * i] * S.chi[a + (size_t)nm * b] * rho[b + (size_t)nm * i];
      f = f - omega[a + (size_t)nm * i] * rho[a + (size_t)nm * i];
    }
  double p = -f;
  for (int i = 0; i < S.nchain; ++i)
    if (phi_c[i] > 1.0e-8f) p = p + mu_c[i] * phi_c[i] / S.chain_length[i];
  for (int i = 0; i < S.nsolv; ++i)
    if (phi_s[i] > 1.0e-8f) p = p + mu_s[i] * phi_s[i] / S.solv_size[i];
  *fo = f;
  *po = p;
}

struct BatchInst {
  System* S = nullptr;
  uint64_t gen_basis = 0;   // the system's basis generation at pscf_batch_add
  int64_t am = 0;
  std::string cs;
  int ncp = 0;
  std::vector<double> cell, omega, rho, dgsq, stress, phi_c, mu_c, phi_s, mu_s, q, qs;
  double f = 0.0, p = 0.0, err = 0.0;
  int itr = 0, status = -1;
  bool active = true;
};

struct Group {
  int n1 = 0, n2 = 0, n3 = 0, np = 0;
  bool half_z = true;            // every member's planes allow it (Grid::step_z)
  std::vector<int> members;
  // the members' chain-discretisation generations when the tasks were
  // copied: a restart (startup, set_checkpoint) frees the slabs the tasks
  // and the captured graph point at, so the group is rebuilt
  std::vector<uint64_t> gen_start;
  std::vector<StepTask> h_tasks;
  std::vector<int> task_owner;
  DevBuf<StepTask> tasks;
  int max_ns = 0;
  Stream st;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~Group() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
};

struct Batch {
  int nhist = 20, domain = 1, max_itr = 1000;
  double error_max = 1e-8;
  std::vector<BatchInst> inst;
  std::vector<std::unique_ptr<Group>> groups;
  int iterations = 0;
  ~Batch() {
    for (auto& b : inst)
      if (b.am) pscf_am_destroy(b.am);
  }
};

void dgsq_of(BatchInst& B) {
  System& S = *B.S;
  const int dim = S.g.dim;
  std::vector<double> dGG((size_t)dim * dim * 6);
  if (pscf_unit_cell(dim, B.cs.c_str(), B.ncp, B.cell.data(), nullptr, nullptr, dGG.data()))
    throw Fail{std::string("unit cell: ") + pscf_am_last_error()};
  B.dgsq.assign((size_t)S.nstar * B.ncp, 0.0);
  for (int k = 0; k < B.ncp; ++k)
    if (pscf_make_dgsq(dim, S.nstar, S.h_wave_of_star.data(), dGG.data() + (size_t)dim * dim * k,
                       B.dgsq.data() + (size_t)S.nstar * k))
      throw Fail{std::string("make_dGsq: ") + pscf_am_last_error()};
}

void build_groups(Batch& Bt) {
  Bt.groups.clear();
  for (int i = 0; i < (int)Bt.inst.size(); ++i) {
    System& S = *Bt.inst[i].S;
    Group* G = nullptr;
    for (auto& g : Bt.groups)
      if (g->n1 == S.g.n1 && g->n2 == S.g.n2 && g->n3 == S.g.n3 && g->np == S.g.np) G = g.get();
    if (!G) {
      Bt.groups.push_back(std::make_unique<Group>());
      G = Bt.groups.back().get();
      G->n1 = S.g.n1;
      G->n2 = S.g.n2;
      G->n3 = S.g.n3;
      G->np = S.g.np;
    }
    G->half_z = G->half_z && sym_half(S.g.sym);
    G->members.push_back(i);
    G->gen_start.push_back(S.gen_start);
    for (const auto& t : S.h_tasks) {
      G->h_tasks.push_back(t);
      G->task_owner.push_back(i);
    }
    G->max_ns = std::max(G->max_ns, S.max_ns);
  }
  for (auto& G : Bt.groups) G->tasks.alloc(G->h_tasks.size());
}

// one batched density() (+ scf_stress when domain) over the active instances
void batch_density(Batch& Bt, bool with_stress) {
  for (auto& Gp : Bt.groups) {
    Group& G = *Gp;
    hipStream_t s = G.st.s;
    for (size_t k = 0; k < G.h_tasks.size(); ++k) G.h_tasks[k].skip = Bt.inst[G.task_owner[k]].active ? 0 : 1;
    HIPCHK(hipMemcpyAsync(G.tasks.p, G.h_tasks.data(), sizeof(StepTask) * G.h_tasks.size(),
                          hipMemcpyHostToDevice, s));
    for (int i : G.members) {
      BatchInst& B = Bt.inst[i];
      if (!B.active) continue;
      density_pre(*B.S, B.omega.data(), B.phi_c.data(), B.mu_c.data(), B.phi_s.data(),
                  B.mu_s.data(), s);
    }
    const Grid& g = Bt.inst[G.members[0]].S->g;
    if (!G.exec) {
      HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      run_sweeps(g, G.tasks.p, (int)G.h_tasks.size(), G.max_ns, G.half_z, s);
      HIPCHK(hipStreamEndCapture(s, &G.graph));
      HIPCHK(hipGraphInstantiate(&G.exec, G.graph, nullptr, nullptr, 0));
    }
    HIPCHK(hipGraphLaunch(G.exec, s));
    for (int i : G.members) {
      BatchInst& B = Bt.inst[i];
      if (!B.active) continue;
      density_post(*B.S, B.rho.data(), s);
      B.S->have_density = true;
      ++B.S->density_gen;
      if (with_stress) stress_launch(*B.S, B.ncp, B.dgsq.data(), s);
    }
  }
  for (auto& Gp : Bt.groups) Gp->st.sync();
  for (auto& B : Bt.inst) {
    if (!B.active) continue;
    System& S = *B.S;
    if (!sym_usable(S) || sym_failed(S)) {       // this field or cell needs every plane
      density(S, B.omega.data(), B.rho.data(), B.q.data(), B.qs.data(), B.phi_c.data(), B.mu_c.data(),
              B.phi_s.data(), B.mu_s.data());
      if (with_stress)
        stress(live(S), B.ncp, B.dgsq.data(), B.phi_c.data(), B.mu_c.data(), B.stress.data());
      continue;
    }
    S.last = nullptr;
    density_finish(S, B.q.data(), B.qs.data(), B.phi_c.data(), B.mu_c.data(), B.phi_s.data(),
                   B.mu_s.data());
    if (with_stress) stress_finish(S, B.ncp, B.phi_c.data(), B.mu_c.data(), B.stress.data());
  }
}

void mu_phi(BatchInst& B) {
  System& S = *B.S;
  for (int i = 0; i < S.nchain; ++i) {
    if (S.ensemble == 0) B.mu_c[i] = std::log(B.phi_c[i] / B.q[i]);
    else B.phi_c[i] = B.q[i] * std::exp(B.mu_c[i]);
  }
  for (int i = 0; i < S.nsolv; ++i) {
    if (S.ensemble == 0) B.mu_s[i] = std::log(B.phi_s[i] / B.qs[i]);
    else B.phi_s[i] = B.qs[i] * std::exp(B.mu_s[i]);
  }
}

// Run f(0..n-1) on up to OMP_NUM_THREADS (default: 16, at most the hardware
// threads) host threads; the first exception is rethrown on the caller.
template <class F>
void parallel_for(size_t n, F&& f) {
  size_t T = std::min<size_t>(16, std::max(1u, std::thread::hardware_concurrency()));
  if (const char* e = std::getenv("OMP_NUM_THREADS")) {
    const long v = std::strtol(e, nullptr, 10);
    if (v >= 1) T = (size_t)v;
  }
  T = std::min(T, n);
  if (T <= 1) {
    for (size_t i = 0; i < n; ++i) f(i);
    return;
  }
  std::atomic<size_t> next{0};
  std::exception_ptr err;
  std::mutex m;
  std::vector<std::thread> th;
  for (size_t t = 0; t < T; ++t)
    th.emplace_back([&] {
      for (;;) {
        const size_t i = next++;
        if (i >= n) break;
        try {
          f(i);
        } catch (...) {
          std::lock_guard<std::mutex> lk(m);
          if (!err) err = std::current_exception();
        }
      }
    });
  for (auto& x : th) x.join();
  if (err) std::rethrow_exception(err);
}

// true when a member system was restarted since its group was built
bool groups_stale(const Batch& Bt) {
  for (const auto& G : Bt.groups)
    for (size_t k = 0; k < G->members.size(); ++k)
      if (Bt.inst[G->members[k]].S->gen_start != G->gen_start[k]) return true;
  return false;
}

void batch_solve(Batch& Bt) {
  REQUIRE(!Bt.inst.empty(), "empty batch");
  for (const auto& B : Bt.inst) {
    REQUIRE(B.S->started, "a batch member system is not started");
    REQUIRE(B.S->gen_basis == B.gen_basis,
            "a batch member's star basis changed after pscf_batch_add (its field arrays no longer fit)");
  }
  if (Bt.groups.empty() || groups_stale(Bt)) build_groups(Bt);
  for (auto& B : Bt.inst) {
    B.active = true;
    B.itr = 0;
    B.status = -1;
    if (B.am) pscf_am_destroy(B.am);
    if (pscf_am_create(B.S->nstar, B.S->nmon, B.ncp, Bt.nhist, Bt.domain, &B.am))
      throw Fail{std::string("am_create: ") + pscf_am_last_error()};
  }
  // initial density and mu (src/iterate_mod.fp.f90:1123-1128), dGsq, omega(:,1)
  batch_density(Bt, false);
  for (auto& B : Bt.inst) {
    mu_phi(B);
    dgsq_of(B);
    System& S = *B.S;
    if (S.ensemble == 0) {
      std::vector<double> phi_mon(S.nmon, 0.0);
      for (int i = 0; i < S.nchain; ++i)
        for (const auto& b : S.blocks[i])
          phi_mon[b.first] = phi_mon[b.first] + B.phi_c[i] * b.second / S.chain_length[i];
      for (int i = 0; i < S.nsolv; ++i) phi_mon[S.solv_mon[i]] = phi_mon[S.solv_mon[i]] + B.phi_s[i];
      for (int a = 0; a < S.nmon; ++a) {
        B.omega[a] = 0.0;
        for (int b = 0; b < S.nmon; ++b) B.omega[a] = B.omega[a] + S.chi[a + (size_t)S.nmon * b] * phi_mon[b];
      }
    }
    if (pscf_am_start(B.am, B.omega.data(), B.cell.data()))
      throw Fail{std::string("am_start: ") + pscf_am_last_error()};
  }
  Bt.iterations = 0;
  for (;;) {
    bool any = false;
    for (auto& B : Bt.inst) any = any || B.active;
    if (!any) break;
    ++Bt.iterations;
    batch_density(Bt, Bt.domain != 0);
    // the instances' host work (thermodynamics, Anderson step, new cell) is
    // independent: it runs on host threads, the device cell updates after
    std::vector<BatchInst*> act;
    for (auto& B : Bt.inst)
      if (B.active) act.push_back(&B);
    std::vector<std::vector<double>> Gnew(act.size());
    parallel_for(act.size(), [&](size_t k) {
      BatchInst& B = *act[k];
      System& S = *B.S;
      ++B.itr;
      mu_phi(B);
      thermo(S, B.rho.data(), B.omega.data(), B.phi_c.data(), B.mu_c.data(), B.phi_s.data(),
             B.mu_s.data(), &B.f, &B.p);
      int st = 0;
      if (pscf_am_iterate(B.am, B.omega.data(), B.rho.data(), S.chi.data(), B.stress.data(),
                          B.cell.data(), Bt.error_max, Bt.max_itr, &B.err, &st))
        throw Fail{std::string("am_iterate: ") + pscf_am_last_error()};
      if (st != 0) {
        B.status = st;
        B.active = false;
        return;
      }
      if (Bt.domain) {
        const int dim = S.g.dim;
        Gnew[k].assign((size_t)dim * dim, 0.0);
        if (pscf_unit_cell(dim, B.cs.c_str(), B.ncp, B.cell.data(), nullptr, Gnew[k].data(), nullptr))
          throw Fail{std::string("unit cell: ") + pscf_am_last_error()};
        dgsq_of(B);
      }
    });
    for (size_t k = 0; k < act.size(); ++k) {
      BatchInst& B = *act[k];
      if (!B.active || !Bt.domain) continue;
      System& S = *B.S;
      const int dim = S.g.dim;
      for (int i = 0; i < 9; ++i) S.gb[i] = 0.0;
      for (int i = 0; i < dim; ++i)
        for (int jj = 0; jj < dim; ++jj) S.gb[i * 3 + jj] = Gnew[k][i + dim * jj];
      apply_cell(S);
    }
    for (auto& B : Bt.inst) B.S->st.sync();   // cell updates run on each system's stream
  }
  // fixed cell: residual stress of the final fields (:1473)
  if (!Bt.domain) {
    for (auto& B : Bt.inst) {
      stress(live(*B.S), B.ncp, B.dgsq.data(), B.phi_c.data(), B.mu_c.data(), B.stress.data());
    }
  }
}

}  // namespace

// =====================================================================  C ABI
extern "C" {

const char* pscf_last_error(void) { return g_err.c_str(); }

int pscf_device_count(int* count) {
  return guarded([&] {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    *count = n;
  });
}

int pscf_chain_discretize(int nblk, const double* blk_length, double ds0, int order, int* block_bgn,
                          double* block_ds) {
  return guarded([&] { discretize(nblk, blk_length, ds0, order, block_bgn, block_ds); });
}

// ------------------------------------------------------------------ fft_mod
int pscf_fft_plan_create(const int ngrid[3], int64_t* plan) {
  return guarded([&] {
    auto* p = new FftPlan;
    try {
      int dim = ngrid[2] > 1 ? 3 : (ngrid[1] > 1 ? 2 : 1);
      p->g.init(ngrid, dim);
    } catch (...) {
      delete p;
      throw;
    }
    *plan = reinterpret_cast<int64_t>(p);
  });
}

int pscf_fft_plan_destroy(int64_t plan) {
  return guarded([&] { delete from_handle<FftPlan>(plan, "fft plan"); });
}

int pscf_fft_r2c(int64_t plan, const double* in, double* out) {
  return guarded([&] {
    FftPlan& P = *from_handle<FftPlan>(plan, "fft plan");
    P.r.upload(in, P.g.m, P.st.s);
    P.k.alloc(P.g.mk);
    P.g.r2c(P.r.p, P.k.p, 1, P.st.s);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, P.k.p, sizeof(double2) * P.g.mk, hipMemcpyDeviceToHost, P.st.s));
    P.st.sync();
  });
}

int pscf_fft_c2r(int64_t plan, const double* in, double* out) {
  return guarded([&] {
    FftPlan& P = *from_handle<FftPlan>(plan, "fft plan");
    P.k.upload(reinterpret_cast<const double2*>(in), P.g.mk, P.st.s);
    P.r.alloc(P.g.m);
    P.g.c2r(P.k.p, P.r.p, 1, 1.0, P.st.s);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, P.r.p, sizeof(double) * P.g.m, hipMemcpyDeviceToHost, P.st.s));
    P.st.sync();
  });
}

int pscf_fft_c2c(int64_t plan, int direction, const double* in, double* out) {
  return guarded([&] {
    FftPlan& P = *from_handle<FftPlan>(plan, "fft plan");
    P.c.upload(reinterpret_cast<const double2*>(in), P.g.m, P.st.s);
    P.g.c2c(P.c.p, direction == 1 ? -1 : +1, P.st.s);
    HIPCHK(hipGetLastError());
    std::vector<double2> h(P.g.m);
    HIPCHK(hipMemcpyAsync(h.data(), P.c.p, sizeof(double2) * P.g.m, hipMemcpyDeviceToHost, P.st.s));
    P.st.sync();
    const double rM = (double)P.g.m;
    for (long i = 0; i < P.g.m; ++i) {
      double2 v = h[i];
      if (direction == +1) v = make_double2(v.x / rM, v.y / rM);   // src/fft3_mod.f90:156
      out[2 * i] = v.x;
      out[2 * i + 1] = v.y;
    }
  });
}

int pscf_fft_r2c_dev(int64_t plan, const double* in, double* out, int nbatch) {
  return guarded([&] {
    FftPlan& P = *from_handle<FftPlan>(plan, "fft plan");
    P.g.r2c(in, reinterpret_cast<double2*>(out), nbatch, P.st.s);
    HIPCHK(hipGetLastError());
    P.st.sync();
  });
}

int pscf_fft_c2r_dev(int64_t plan, const double* in, double* out, int nbatch) {
  return guarded([&] {
    FftPlan& P = *from_handle<FftPlan>(plan, "fft plan");
    // the z pass works in place: copy the spectra first so `in` is preserved
    P.k.alloc((size_t)P.g.mk * nbatch);
    HIPCHK(hipMemcpyAsync(P.k.p, in, sizeof(double2) * P.g.mk * nbatch, hipMemcpyDeviceToDevice,
                          P.st.s));
    P.g.c2r(P.k.p, out, nbatch, 1.0, P.st.s);
    HIPCHK(hipGetLastError());
    P.st.sync();
  });
}

// ----------------------------------------------------------------- step_mod
int pscf_step_create(const int ngrid[3], int64_t* step) {
  return guarded([&] {
    auto* p = new StepState;
    try {
      int dim = ngrid[2] > 1 ? 3 : (ngrid[1] > 1 ? 2 : 1);
      p->g.init(ngrid, dim);
      const Grid& g = p->g;
      p->fac.alloc(2 * g.m + 2 * g.mf);
      p->slab.alloc(2 * g.m);
      p->q1.alloc(g.m);
      p->abc.alloc(3 * g.mc);
      p->task.alloc(1);
    } catch (...) {
      delete p;
      throw;
    }
    *step = reinterpret_cast<int64_t>(p);
  });
}

int pscf_step_destroy(int64_t step) {
  return guarded([&] { delete from_handle<StepState>(step, "step"); });
}

int pscf_step_make_propg(int64_t step, double ds, double b, const double* ksq, const double* omega) {
  return guarded([&] {
    StepState& S = *from_handle<StepState>(step, "step");
    const Grid& g = S.g;
    S.ksq.upload(ksq, g.mk, S.st.s);
    S.om.upload(omega, g.m, S.st.s);
    double* f = S.fac.p;
    hipLaunchKernelGGL(k_make_propg, dim3(grid_blocks(g.m)), dim3(NTA), 0, S.st.s, ds, b, S.ksq.p,
                       g.mf, S.om.p, g.m, g.n1, g.n2, g.zs->zw, (double)g.m, f, f + g.m, f + 2 * g.m, f + 2 * g.m + g.mf);
    HIPCHK(hipGetLastError());
    S.st.sync();
    S.have_propg = true;
  });
}

int pscf_step_exp(int64_t step, const double* q_in, double* q_out) {
  return guarded([&] {
    StepState& S = *from_handle<StepState>(step, "step");
    REQUIRE(S.have_propg, "step_exp requires make_propg");
    const Grid& g = S.g;
    // q1 holds the grid-order input, then output, while no kernel uses it
    HIPCHK(hipMemcpyAsync(S.q1.p, q_in, sizeof(double) * g.m, hipMemcpyHostToDevice, S.st.s));
    hipLaunchKernelGGL(k_pack, dim3(grid_blocks(g.m)), dim3(NTA), 0, S.st.s, S.q1.p, g.m, g.m, 1, g.n1, g.n2,
                       S.slab.p);
    StepTask t;
    std::memset(&t, 0, sizeof t);
    t.slab = S.slab.p;
    t.ns = 1;
    t.jend = 1;
    t.dir = 1;
    t.init_one = 0;
    one_step_blocks(t, g, S.fac.p);
    t.A = S.abc.p;
    t.B = S.abc.p + g.mc;
    t.C = S.abc.p + 2 * g.mc;
    t.q1 = S.q1.p;
    HIPCHK(hipMemcpyAsync(S.task.p, &t, sizeof t, hipMemcpyHostToDevice, S.st.s));
    run_sweeps(g, S.task.p, 1, 1, false, S.st.s);
    hipLaunchKernelGGL(k_unpack, dim3(grid_blocks(g.m)), dim3(NTA), 0, S.st.s, S.slab.p + g.m, g.m, 1,
                       g.n1, g.n2, S.q1.p);
    HIPCHK(hipMemcpyAsync(q_out, S.q1.p, sizeof(double) * g.m, hipMemcpyDeviceToHost, S.st.s));
    S.st.sync();
  });
}

int pscf_step_exp_noalloc(const int ngrid[3], double ds, double b, const double* ksq,
                          const double* omega, const double* q_in, double* q_out) {
  return guarded([&] {
    REQUIRE(ngrid && ksq && omega && q_in && q_out, "null argument");
    REQUIRE(is_device_pointer(ksq) && is_device_pointer(omega) && is_device_pointer(q_in) &&
                is_device_pointer(q_out),
            "pscf_step_exp_noalloc takes device pointers (ksq, omega, q_in, q_out)");
    const int dim = ngrid[2] > 1 ? 3 : (ngrid[1] > 1 ? 2 : 1);
    Grid g;
    g.init(ngrid, dim, false);
    // scratch layout in doubles, every part 256-byte aligned
    const auto up = [](size_t n) { return (n + 31) / 32 * 32; };
    const size_t o_tw = up((sizeof(StepTask) + sizeof(double) - 1) / sizeof(double));
    const size_t ntw = (size_t)g.n1 + g.n2 + g.n3 + g.nl;
    const size_t o_fac = o_tw + up(2 * ntw);
    const size_t o_abc = o_fac + up(2 * g.m + 2 * g.mf);
    const size_t o_q1 = o_abc + up(6 * g.mc);
    const size_t o_slab = o_q1 + up(g.m);
    const size_t need = o_slab + up(2 * g.m);
    char msg[200];
    snprintf(msg, sizeof msg,
             "grid %dx%dx%d needs %zu bytes of scratch; pscf_step_exp_noalloc has %zu (a 64^3 grid fits)",
             g.n1, g.n2, g.n3, need * sizeof(double), kScratchDoubles * sizeof(double));
    REQUIRE(need <= kScratchDoubles, msg);
    double* base = scratch_on_current_device();
    hipStream_t s = nullptr;                      // the default stream
    // twiddle tables of the three edges and the packed rows
    std::vector<double2> htw(ntw);
    host_twiddles(g.n1, htw.data());
    host_twiddles(g.n2, htw.data() + g.n1);
    host_twiddles(g.n3, htw.data() + g.n1 + g.n2);
    host_twiddles(g.nl, htw.data() + g.n1 + g.n2 + g.n3);
    double2* dtw = reinterpret_cast<double2*>(base + o_tw);
    HIPCHK(hipMemcpyAsync(dtw, htw.data(), sizeof(double2) * ntw, hipMemcpyHostToDevice, s));
    g.tw1 = dtw;
    g.tw2 = dtw + g.n1;
    g.tw3 = dtw + g.n1 + g.n2;
    g.twl = g.tw3 + g.n3;
    // make_propg (src/step_mod.f90:109-129)
    double* f = base + o_fac;
    hipLaunchKernelGGL(k_make_propg, dim3(grid_blocks(g.m)), dim3(NTA), 0, s, ds, b, ksq, g.mf, omega,
                       g.m, g.n1, g.n2, g.zs->zw, (double)g.m, f, f + g.m, f + 2 * g.m, f + 2 * g.m + g.mf);
    // one step (src/step_mod.f90:146-176): a one-step sweep from q_in
    StepTask t;
    std::memset(&t, 0, sizeof t);
    t.slab = base + o_slab;
    hipLaunchKernelGGL(k_pack, dim3(grid_blocks(g.m)), dim3(NTA), 0, s, q_in, g.m, g.m, 1, g.n1, g.n2, t.slab);
    t.ns = 1;
    t.jend = 1;
    t.dir = 1;
    one_step_blocks(t, g, f);
    t.A = reinterpret_cast<double2*>(base + o_abc);
    t.B = t.A + g.mc;
    t.C = t.B + g.mc;
    t.q1 = base + o_q1;
    StepTask* dtask = reinterpret_cast<StepTask*>(base);
    HIPCHK(hipMemcpyAsync(dtask, &t, sizeof t, hipMemcpyHostToDevice, s));
    run_sweeps(g, dtask, 1, 1, false, s);
    hipLaunchKernelGGL(k_unpack, dim3(grid_blocks(g.m)), dim3(NTA), 0, s, t.slab + g.m, g.m, 1, g.n1, g.n2,
                       q_out);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s));
  });
}

// ------------------------------------------------------------------ scf_mod
int pscf_system_create(const int ngrid[3], int dim, int64_t* sys) {
  return guarded([&] {
    auto* p = new System;
    try {
      p->g.init(ngrid, dim);
    } catch (...) {
      delete p;
      throw;
    }
    *sys = reinterpret_cast<int64_t>(p);
  });
}

int pscf_system_destroy(int64_t sys) {
  return guarded([&] {
    System* S = from_handle<System>(sys, "system");
    delete S;
  });
}

int pscf_profile_step_kernel(int64_t sys, int kind, int j, int reps, double* us) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_density, "profile_step_kernel requires a previous density()");
    REQUIRE(kind >= 0 && kind <= 3 && reps >= 1, "kind must be 0..3, reps >= 1");
    REQUIRE(j >= 1 && j < S.max_ns, "step index out of range");
    const Grid& g = S.g;
    hipStream_t s = S.st.s;
    ensure_events(S, 2);
    auto launch = [&] {
      if (kind == 0)
        launch_step_a(g, S.tasks.p, S.ntask, j, false, s);
      else if (kind == 2)
        g.step_c(S.tasks.p, S.ntask, j, false, s);
      else
        g.step_z(S.tasks.p, S.ntask, j, kind == 1 ? 0 : 1, kind == 1 ? 2 : 1, false, sym_half(g.sym), s);
    };
    launch();
    HIPCHK(hipEventRecord(S.ev[0], s));
    for (int r = 0; r < reps; ++r) launch();
    HIPCHK(hipEventRecord(S.ev[1], s));
    HIPCHK(hipGetLastError());
    S.st.sync();
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, S.ev[0], S.ev[1]));
    *us = (double)ms * 1e3 / reps;
    S.have_density = false;      // the z kernels transform their spectra in place
    ++S.density_gen;
  });
}

int pscf_profile_sweeps(int64_t sys, int mode, double* ms_sum, int64_t* count) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(mode >= 0 && mode <= 2, "profile mode must be 0, 1 or 2");
    for (int k = 0; k < 5; ++k) {
      if (ms_sum) ms_sum[k] = S.prof_ms[k];
      if (count) count[k] = S.prof_n[k];
      S.prof_ms[k] = 0.0;
      S.prof_n[k] = 0;
    }
    S.profile = mode;
  });
}

int pscf_system_set_checkpoint(int64_t sys, int stride) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(stride >= 0, "checkpoint stride must be >= 0");
    S.ck_stride = stride;
    if (S.started) startup(S, S.chain_step);
  });
}

int pscf_system_use_graph(int64_t sys, int enable) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    S.use_graph = enable != 0;
    if (!S.use_graph) {
      S.drop_graph();
      S.drop_ck_graph();
    }
  });
}

int pscf_system_set_basis(int64_t sys, int n_wave, int n_star, const int* wave, const double* coeff,
                          const int* star_of_wave, const int* star_invert, const int* wave_of_star) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(n_wave > 0 && n_star > 0, "empty basis");
    const int dim = S.g.dim;
    S.nwave = n_wave;
    S.nstar = n_star;
    S.h_wave.assign(wave, wave + (size_t)dim * n_wave);
    S.h_wave_of_star.assign(wave_of_star, wave_of_star + (size_t)dim * n_star);
    S.h_coeff.resize(n_wave);
    for (int i = 0; i < n_wave; ++i) S.h_coeff[i] = make_double2(coeff[2 * i], coeff[2 * i + 1]);
    for (int i = 0; i < n_star; ++i)
      REQUIRE(star_invert[i] >= -1 && star_invert[i] <= 1,
              "Illegal star_invert value in basis_to_kgrid.");
    for (int i = 0; i < n_star; ++i) {
      if (star_invert[i] == 1)
        REQUIRE(i + 1 < n_star && star_invert[i + 1] == -1, "star_invert(i)=1 without -1 partner");
      if (star_invert[i] == -1) REQUIRE(i > 0 && star_invert[i - 1] == 1, "star_invert(i)=-1 without +1 partner");
    }
    for (int i = 0; i < n_wave; ++i)
      REQUIRE(star_of_wave[i] >= 1 && star_of_wave[i] <= n_star, "star_of_wave out of range");
    S.h_star_of_wave.assign(star_of_wave, star_of_wave + n_wave);
    S.h_star_invert.assign(star_invert, star_invert + n_star);
    S.coeff.upload(S.h_coeff.data(), n_wave, S.st.s);
    S.star_of_wave.upload(star_of_wave, n_wave, S.st.s);
    S.star_invert.upload(star_invert, n_star, S.st.s);
    build_basis_maps(S);
    S.sym_code = detect_sym(S);
    S.sym_bad = false;
    S.have_basis = true;
    ++S.gen_basis;
    if (S.have_cell) {
      apply_cell(S);
      S.st.sync();
    }
  });
}

int pscf_system_set_cell(int64_t sys, const double* G_basis) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis, "set_basis must precede set_cell");
    const int dim = S.g.dim;
    for (int i = 0; i < 9; ++i) S.gb[i] = 0.0;
    // Fortran G_basis(dim,dim), element (i,j) at G_basis[i + dim*j]
    for (int i = 0; i < dim; ++i)
      for (int jj = 0; jj < dim; ++jj) S.gb[i * 3 + jj] = G_basis[i + dim * jj];
    apply_cell(S);
    S.st.sync();
    S.sym_bad = false;
  });
}

int pscf_system_get_ksq(int64_t sys, double* ksq) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_cell, "no cell");
    HIPCHK(hipMemcpy(ksq, S.ksq.p, sizeof(double) * S.g.mk, hipMemcpyDeviceToHost));
  });
}

int pscf_system_set_chemistry(int64_t sys, int n_monomer, const double* kuhn, int n_chain,
                              const int* n_block, int n_blk_max, const int* block_monomer,
                              const double* block_length, int n_solvent,
                              const int* solvent_monomer, const double* solvent_size,
                              int ensemble) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(n_monomer >= 1 && n_chain >= 0 && n_solvent >= 0, "invalid chemistry sizes");
    REQUIRE(ensemble == 0 || ensemble == 1, "Invalid ensemble");
    S.nmon = n_monomer;
    S.nchain = n_chain;
    S.nsolv = n_solvent;
    S.ensemble = ensemble;
    S.kuhn.assign(kuhn, kuhn + n_monomer);
    S.blocks.assign(n_chain, {});
    for (int c = 0; c < n_chain; ++c) {
      REQUIRE(n_block[c] >= 1 && n_block[c] <= n_blk_max && n_block[c] <= MAXBLK,
              "N_block out of range");
      for (int b = 0; b < n_block[c]; ++b) {
        const int mon = block_monomer[b + (size_t)n_blk_max * c];
        REQUIRE(mon >= 1 && mon <= n_monomer, "block_monomer out of range");
        S.blocks[c].push_back({mon - 1, block_length[b + (size_t)n_blk_max * c]});
      }
    }
    S.chain_length.assign(n_chain, 0.0);      // src/chemistry_mod.f90:272-276
    for (int c = 0; c < n_chain; ++c)
      for (const auto& b : S.blocks[c]) S.chain_length[c] = S.chain_length[c] + b.second;
    S.solv_mon.clear();
    S.solv_size.clear();
    for (int i = 0; i < n_solvent; ++i) {
      REQUIRE(solvent_monomer[i] >= 1 && solvent_monomer[i] <= n_monomer,
              "solvent_monomer out of range");
      S.solv_mon.push_back(solvent_monomer[i] - 1);
      S.solv_size.push_back(solvent_size[i]);
    }
    S.have_chem = true;
    S.started = false;
  });
}

int pscf_system_set_chain_length(int64_t sys, const double* chain_length) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_chem, "set_chemistry must precede set_chain_length");
    for (int c = 0; c < S.nchain; ++c) {
      REQUIRE(chain_length[c] > 0.0, "chain length must be positive");
      S.chain_length[c] = chain_length[c];
      if (c < (int)S.chains.size()) S.chains[c]->length = chain_length[c];
      if (S.full && c < (int)S.full->chains.size()) {
        S.full->chain_length[c] = chain_length[c];
        S.full->chains[c]->length = chain_length[c];
      }
    }
  });
}

int pscf_system_set_chi(int64_t sys, const double* chi) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_chem, "set_chemistry must precede set_chi");
    S.chi.assign(chi, chi + (size_t)S.nmon * S.nmon);
  });
}

// chain length N (chemistry_mod's chain_length)
static double chain_len(const System& S, int c) { return S.chain_length[c]; }

int pscf_mu_phi_chain(int64_t sys, double* mu, double* phi, const double* q) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    for (int i = 0; i < S.nchain; ++i) {
      if (S.ensemble == 0) mu[i] = std::log(phi[i] / q[i]);
      else phi[i] = q[i] * std::exp(mu[i]);
    }
  });
}

int pscf_mu_phi_solvent(int64_t sys, double* mu, double* phi, const double* q) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    for (int i = 0; i < S.nsolv; ++i) {
      if (S.ensemble == 0) mu[i] = std::log(phi[i] / q[i]);
      else phi[i] = q[i] * std::exp(mu[i]);
    }
  });
}

int pscf_free_energy(int64_t sys, const double* rho, const double* omega, const double* phi_chain,
                     const double* mu_chain, const double* phi_solvent, const double* mu_solvent,
                     double* f_helmholtz, double* pressure) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.chi.size() == (size_t)S.nmon * S.nmon, "chi not set");
    const int nm = S.nmon;
    double f = 0.0;
    for (int i = 0; i < S.nchain; ++i)
      if (phi_chain[i] > 1.0e-8f) f = f + phi_chain[i] * (mu_chain[i] - 1.0) / chain_len(S, i);
    for (int i = 0; i < S.nsolv; ++i)
      if (phi_solvent[i] > 1.0e-8f) f = f + phi_solvent[i] * (mu_solvent[i] - 1.0) / S.solv_size[i];
    for (int i = 0; i < S.nstar; ++i)
      for (int a = 0; a < nm; ++a) {
        for (int b = a + 1; b < nm; ++b)
          f = f + rho[a + (size_t)nm * i] * S.chi[a + (size_t)nm * b] * rho[b + (size_t)nm * i];
        f = f - omega[a + (size_t)nm * i] * rho[a + (size_t)nm * i];
      }
    *f_helmholtz = f;
    if (pressure) {
      double p = -f;
      for (int i = 0; i < S.nchain; ++i)
        if (phi_chain[i] > 1.0e-8f) p = p + mu_chain[i] * phi_chain[i] / chain_len(S, i);
      for (int i = 0; i < S.nsolv; ++i)
        if (phi_solvent[i] > 1.0e-8f) p = p + mu_solvent[i] * phi_solvent[i] / S.solv_size[i];
      *pressure = p;
    }
  });
}

int pscf_free_energy_fh(int64_t sys, const double* phi_chain, const double* phi_solvent, double* fo) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.chi.size() == (size_t)S.nmon * S.nmon, "chi not set");
    double f = 0.0;
    std::vector<double> rho(S.nmon, 0.0);
    for (int i = 0; i < S.nchain; ++i) {
      const double L = chain_len(S, i);
      if (phi_chain[i] > 1.0e-8f) f = f + (phi_chain[i] / L) * (std::log(phi_chain[i]) - 1);
      for (const auto& b : S.blocks[i]) rho[b.first] = rho[b.first] + phi_chain[i] * b.second / L;
    }
    if (phi_solvent)
      for (int i = 0; i < S.nsolv; ++i) {
        if (phi_solvent[i] > 1.0e-8f)
          f = f + (phi_solvent[i] / S.solv_size[i]) * (std::log(phi_solvent[i]) - 1);
        rho[S.solv_mon[i]] = rho[S.solv_mon[i]] + phi_solvent[i];
      }
    for (int i = 0; i < S.nmon - 1; ++i)
      for (int j = i + 1; j < S.nmon; ++j) f = f + S.chi[i + (size_t)S.nmon * j] * rho[i] * rho[j];
    *fo = f;
  });
}

int pscf_set_omega_uniform(int64_t sys, double* omega, const double* phi_chain,
                           const double* phi_solvent) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.chi.size() == (size_t)S.nmon * S.nmon, "chi not set");
    std::vector<double> phi_mon(S.nmon, 0.0);
    for (int i = 0; i < S.nchain; ++i) {
      const double L = chain_len(S, i);
      for (const auto& b : S.blocks[i])
        phi_mon[b.first] = phi_mon[b.first] + phi_chain[i] * b.second / L;
    }
    for (int i = 0; i < S.nsolv; ++i) phi_mon[S.solv_mon[i]] = phi_mon[S.solv_mon[i]] + phi_solvent[i];
    for (int a = 0; a < S.nmon; ++a) {
      omega[a] = 0.0;   // omega(alpha, 1): first star, column-major (N_monomer, N_star)
      for (int b = 0; b < S.nmon; ++b) omega[a] = omega[a] + S.chi[a + (size_t)S.nmon * b] * phi_mon[b];
    }
  });
}

int pscf_system_startup(int64_t sys, double chain_step) {
  return guarded([&] { startup(*from_handle<System>(sys, "system"), chain_step); });
}

int pscf_density(int64_t sys, const double* omega, double* rho, double* qout, double* q_solvent,
                 double* phi_chain, double* mu_chain, double* phi_solvent, double* mu_solvent) {
  return guarded([&] {
    density(*from_handle<System>(sys, "system"), omega, rho, qout, q_solvent, phi_chain, mu_chain,
            phi_solvent, mu_solvent);
  });
}

int pscf_density_many(int64_t sys, int n, const double* omega, double* rho, double* qout,
                      double* q_solvent, double* phi_chain, double* mu_chain, double* phi_solvent,
                      double* mu_solvent, int max_batch) {
  return guarded([&] {
    density_many(*from_handle<System>(sys, "system"), n, omega, rho, qout, q_solvent, phi_chain,
                 mu_chain, phi_solvent, mu_solvent, max_batch);
  });
}

int pscf_density_many_cells(int64_t sys, int n, const double* omega, const double* G_basis, int ncp,
                            const double* dGsq, double* rho, double* stress, double* phi_chain,
                            double* mu_chain, double* phi_solvent, double* mu_solvent) {
  return guarded([&] {
    REQUIRE(G_basis, "null G_basis");
    density_many(*from_handle<System>(sys, "system"), n, omega, rho, nullptr, nullptr, phi_chain,
                 mu_chain, phi_solvent, mu_solvent, 0, G_basis, ncp, dGsq, stress);
  });
}

int pscf_density_grid_dev(int64_t sys, const double* omega_grid, double* rho_grid, double* qout,
                          double* q_solvent, double* phi_chain, double* mu_chain,
                          double* phi_solvent, double* mu_solvent) {
  return guarded([&] {
    REQUIRE(omega_grid && rho_grid, "null grid pointer");
    density_grid(*from_handle<System>(sys, "system"), omega_grid, rho_grid, qout, q_solvent,
                 phi_chain, mu_chain, phi_solvent, mu_solvent);
  });
}

int pscf_density_adjoint_dev(int64_t sys, const double* lam_rho_grid, const double* dL_dQ,
                             double* grad_omega_grid, int n_cell_param, const double* dGG,
                             double* dL_dcell, double* dL_dlength, double* dL_dphi) {
  return guarded([&] {
    REQUIRE(lam_rho_grid && grad_omega_grid, "null grid pointer");
    REQUIRE(!dGG || dL_dcell, "dGG given without an output for the cell gradient");
    density_adjoint(*from_handle<System>(sys, "system"), lam_rho_grid, dL_dQ, grad_omega_grid,
                    n_cell_param, dGG, dL_dcell, dL_dlength, dL_dphi);
  });
}

int pscf_adjoint_group_create(int n, const int64_t* systems, int64_t* group) {
  return guarded([&] {
    REQUIRE(n >= 1 && systems && group, "invalid arguments");
    auto G = std::make_unique<AdjGroup>();
    for (int i = 0; i < n; ++i) {
      System* S = from_handle<System>(systems[i], "system");
      for (System* o : G->members) REQUIRE(o != S, "adjoint group: a system appears twice");
      G->members.push_back(S);
    }
    *group = reinterpret_cast<int64_t>(G.release());
  });
}

int pscf_adjoint_group_destroy(int64_t group) {
  return guarded([&] { delete from_handle<AdjGroup>(group, "adjoint group"); });
}

int pscf_adjoint_group_run(int64_t group, const double* const* lam_rho_grid,
                           const double* const* dL_dQ, double* const* grad_omega_grid,
                           const int* n_cell_param, const double* const* dGG,
                           double* const* dL_dcell, double* const* dL_dlength,
                           double* const* dL_dphi) {
  return guarded([&] {
    adjoint_group(*from_handle<AdjGroup>(group, "adjoint group"), lam_rho_grid, dL_dQ,
                  grad_omega_grid, n_cell_param, dGG, dL_dcell, dL_dlength, dL_dphi);
  });
}

int pscf_basis_to_grid_dev(int64_t sys, const double* basis, int nf, double* grid) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis && S.have_cell, "system not ready (basis, cell)");
    REQUIRE(nf >= 1 && basis && grid, "invalid arguments");
    basis_to_grid(S, basis, nf, grid, S.st.s);
    S.st.sync();
  });
}

int pscf_grid_to_basis_dev(int64_t sys, const double* grid, int nf, double scale, double* basis) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis && S.have_cell, "system not ready (basis, cell)");
    REQUIRE(nf >= 1 && basis && grid, "invalid arguments");
    grid_to_basis(S, grid, nf, scale, basis, S.st.s);
    S.st.sync();
  });
}

int pscf_scf_stress(int64_t sys, int ncp, const double* dGsq, const double* phi_chain,
                    const double* mu_chain, double* out) {
  return guarded([&] {
    stress(live(*from_handle<System>(sys, "system")), ncp, dGsq, phi_chain, mu_chain, out);
  });
}

int pscf_divide_energy_terms(int64_t sys, double* out) {
  return guarded([&] {
    System& S = live(*from_handle<System>(sys, "system"));
    REQUIRE(S.have_density, "divide_energy requires a previous density()");
    REQUIRE(S.ck_stride == 0, "divide_energy needs every contour point (checkpointed storage is on)");
    const Grid& g = S.g;
    for (int c = 0; c < S.nchain; ++c) {
      ChainDev& ch = *S.chains[c];
      const int nh = ch.bnd[1], nt = ch.bnd[ch.nblk - 1];
      for (int w = 0; w < 2; ++w) {
        const int pt = w == 0 ? nh : nt;
        const int nb = 512;
        hipLaunchKernelGGL(k_partial_qlogq, dim3(nb), dim3(NTA), 0, S.st.s, ch.qf.p + (size_t)pt * g.ms,
                           ch.qr.p + (size_t)pt * g.ms, w == 0 ? 1 : 0, g.ms, g.sym, g.n3,
                           (long)g.n1 * g.n2, S.part.p);
        hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(NTA), 0, S.st.s, S.part.p, nb,
                           1.0 / (S.h_Q[c] * (double)g.m), S.qdev.p + S.nchain + S.nsolv);
        double v = 0.0;
        HIPCHK(hipMemcpyAsync(&v, S.qdev.p + S.nchain + S.nsolv, sizeof(double),
                              hipMemcpyDeviceToHost, S.st.s));
        S.st.sync();
        out[2 * c + w] = v;
      }
    }
  });
}

int pscf_system_get_grids(int64_t sys, double* omega_grid, double* rho_grid) {
  return guarded([&] {
    System& S = live(*from_handle<System>(sys, "system"));
    REQUIRE(S.have_density, "no density computed yet");
    const size_t n = (size_t)S.nmon * S.g.m;
    if (omega_grid) HIPCHK(hipMemcpy(omega_grid, S.omega_grid.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    if (rho_grid) HIPCHK(hipMemcpy(rho_grid, S.rho_grid.p, sizeof(double) * n, hipMemcpyDeviceToHost));
  });
}

int pscf_system_density_generation(int64_t sys, int64_t* gen) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    *gen = (int64_t)S.density_gen;
  });
}

int pscf_system_get_q(int64_t sys, int chain, int dir, int s, double* q) {
  return guarded([&] {
    System& S = live(*from_handle<System>(sys, "system"));
    REQUIRE(S.have_density, "no density computed yet");
    REQUIRE(chain >= 0 && chain < S.nchain, "chain index out of range");
    ChainDev& ch = *S.chains[chain];
    REQUIRE(s >= 0 && s <= ch.ns, "contour index out of range");
    REQUIRE(S.ck_stride == 0 || ch.slot[s] >= 0, "contour point not stored (checkpointed storage)");
    const double* src = ch.point(dir > 0 ? 1 : -1, s);
    DevBuf<double> grid;
    grid.alloc(S.g.m);
    hipLaunchKernelGGL(k_sym_point, dim3(grid_blocks(S.g.m)), dim3(NTA), 0, S.st.s, src, 0L, S.g.sym, S.g.n1,
                       S.g.n2, S.g.n3, 0, grid.p, 0L);
    HIPCHK(hipMemcpyAsync(q, grid.p, sizeof(double) * S.g.m, hipMemcpyDeviceToHost, S.st.s));
    S.st.sync();
  });
}

// ----------------------------------------------------------- grid_basis_mod
int pscf_basis_to_kgrid(int64_t sys, const double* basis, double* kgrid, int no_parity) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis && S.have_cell, "basis/cell not set");
    S.basis_tmp.upload(basis, S.nstar, S.st.s);
    S.kwork.alloc((size_t)2 * S.g.mk);
    hipLaunchKernelGGL(k_basis_to_kgrid, dim3(grid_blocks(S.g.mk)), dim3(NTA), 0, S.st.s,
                       S.basis_tmp.p, 1, S.nstar, S.kwave.p, S.coeff.p, S.star_of_wave.p,
                       S.star_invert.p, S.g.mk, S.kwork.p, no_parity);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(kgrid, S.kwork.p, sizeof(double2) * S.g.mk, hipMemcpyDeviceToHost, S.st.s));
    S.st.sync();
  });
}

int pscf_kgrid_to_basis(int64_t sys, const double* kgrid, double* basis, int no_parity) {
  return guarded([&] {
    System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis, "basis not set");
    S.kwork.alloc((size_t)2 * S.g.mk);
    HIPCHK(hipMemcpyAsync(S.kwork.p, kgrid, sizeof(double2) * S.g.mk, hipMemcpyHostToDevice, S.st.s));
    S.basis_tmp.alloc(S.nstar);
    hipLaunchKernelGGL(k_kgrid_to_basis, dim3(grid_blocks(S.nstar)), dim3(NTA), 0, S.st.s, S.kwork.p,
                       S.g.mk, 1, S.nstar, S.sidx.p, S.sconj.p, S.scoef.p, S.star_invert.p, 1.0,
                       S.basis_tmp.p, no_parity);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(basis, S.basis_tmp.p, sizeof(double) * S.nstar, hipMemcpyDeviceToHost,
                          S.st.s));
    S.st.sync();
  });
}

int pscf_basis_to_kgrid_full(int64_t sys, const double* basis, double* kgrid, int no_parity) {
  return guarded([&] {
    const System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis && S.have_cell, "basis/cell not set");
    full_basis_to_kgrid(S, basis, reinterpret_cast<double2*>(kgrid), no_parity != 0);
  });
}

int pscf_kgrid_to_basis_full(int64_t sys, const double* kgrid, double* basis, int no_parity) {
  return guarded([&] {
    const System& S = *from_handle<System>(sys, "system");
    REQUIRE(S.have_basis, "basis not set");
    full_kgrid_to_basis(S, reinterpret_cast<const double2*>(kgrid), basis, no_parity != 0);
  });
}

// ------------------------------------------------------------ batched solves
int pscf_batch_create(int n_hist, int domain, double error_max, int max_itr, int64_t* batch) {
  return guarded([&] {
    auto* b = new Batch;
    b->nhist = n_hist;
    b->domain = domain;
    b->error_max = error_max;
    b->max_itr = max_itr;
    *batch = reinterpret_cast<int64_t>(b);
  });
}

int pscf_batch_destroy(int64_t batch) {
  return guarded([&] { delete from_handle<Batch>(batch, "batch"); });
}

int pscf_batch_add(int64_t batch, int64_t sys, const char* crystal_system, int n_cell_param,
                   const double* cell_param, const double* omega, const double* phi_chain,
                   const double* mu_chain, const double* phi_solvent, const double* mu_solvent,
                   int* index) {
  return guarded([&] {
    Batch& Bt = *from_handle<Batch>(batch, "batch");
    System* S = from_handle<System>(sys, "system");
    REQUIRE(S->started && S->have_basis && S->have_cell, "system not ready (basis, cell, startup)");
    REQUIRE(S->chi.size() == (size_t)S->nmon * S->nmon, "chi not set");
    for (const auto& o : Bt.inst)
      REQUIRE(o.S != S, "system already in this batch (instances need systems of their own)");
    BatchInst B;
    B.S = S;
    B.gen_basis = S->gen_basis;
    B.cs = crystal_system;
    B.ncp = n_cell_param;
    B.cell.assign(cell_param, cell_param + n_cell_param);
    B.omega.assign(omega, omega + (size_t)S->nmon * S->nstar);
    B.rho.assign((size_t)S->nmon * S->nstar, 0.0);
    B.stress.assign(n_cell_param, 0.0);
    B.phi_c.assign(phi_chain, phi_chain + S->nchain);
    B.mu_c.assign(S->nchain, 0.0);
    if (mu_chain) B.mu_c.assign(mu_chain, mu_chain + S->nchain);
    B.phi_s.assign(std::max(S->nsolv, 1), 0.0);
    B.mu_s.assign(std::max(S->nsolv, 1), 0.0);
    REQUIRE(S->nsolv == 0 || phi_solvent, "phi_solvent missing");
    REQUIRE(S->nsolv == 0 || S->ensemble == 0 || mu_solvent, "mu_solvent missing (grand ensemble)");
    for (int i = 0; i < S->nsolv; ++i) {
      B.phi_s[i] = phi_solvent[i];
      if (mu_solvent) B.mu_s[i] = mu_solvent[i];
    }
    B.q.assign(std::max(S->nchain, 1), 0.0);
    B.qs.assign(std::max(S->nsolv, 1), 0.0);
    Bt.inst.push_back(std::move(B));
    Bt.groups.clear();
    *index = (int)Bt.inst.size() - 1;
  });
}

int pscf_batch_solve(int64_t batch, int* iterations) {
  return guarded([&] {
    Batch& Bt = *from_handle<Batch>(batch, "batch");
    batch_solve(Bt);
    if (iterations) *iterations = Bt.iterations;
  });
}

int pscf_batch_result(int64_t batch, int index, double* omega, double* rho, double* cell_param,
                      double* stress, double* thermo_out, int* itr, int* status) {
  return guarded([&] {
    Batch& Bt = *from_handle<Batch>(batch, "batch");
    REQUIRE(index >= 0 && index < (int)Bt.inst.size(), "batch index out of range");
    const BatchInst& B = Bt.inst[index];
    if (omega) std::copy(B.omega.begin(), B.omega.end(), omega);
    if (rho) std::copy(B.rho.begin(), B.rho.end(), rho);
    if (cell_param) std::copy(B.cell.begin(), B.cell.end(), cell_param);
    if (stress) std::copy(B.stress.begin(), B.stress.end(), stress);
    if (thermo_out) {
      thermo_out[0] = B.f;
      thermo_out[1] = B.p;
      thermo_out[2] = B.err;
      thermo_out[3] = B.S->nchain > 0 ? B.mu_c[0] : 0.0;
    }
    if (itr) *itr = B.itr;
    if (status) *status = B.status;
  });
}

}  // extern "C"
