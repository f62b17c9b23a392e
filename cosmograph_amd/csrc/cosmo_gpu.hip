// cosmo_gpu.hip -- host runtime and C ABI for the MI355X BSSN hot path.
//
// Owns the device registers of one periodic grid, the FP64 FRW reference
// integrator (host side, scalar), and the launch sequence of the fused RK4
// stage kernels.  See include/cosmo_gpu.h for the reference method each
// entry point replaces.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/cosmo_gpu.h"
#include "bssn_stage.h"
#include "fftplan.h"
#include "runtime.h"
#include "stencil.h"

using namespace cg;

namespace {


const char* kFieldNames[NF] = {"DIFFgamma11", "DIFFgamma12", "DIFFgamma13", "DIFFgamma22", "DIFFgamma23",
                               "DIFFgamma33", "DIFFphi",     "A11",         "A12",         "A13",
                               "A22",         "A23",         "A33",         "DIFFK",       "Gamma1",
                               "Gamma2",      "Gamma3",      "DIFFalpha"};

// ------------------------------------------------- elementwise kernels --
// Register table: slot pointers of every field (DIFFphi always FP64).
struct MetScale {
  double s[7];
};

struct RegTable {
  void* r[NF][4];
  double ms[7], mi[7];  // fixed-point metric: scale 2^e and 2^-e per field
  unsigned* sat;        // ... and its count of saturated words
};

// the conformal metric (DIFFgamma_ij, DIFFphi) has its own storage type MT:
// FP64 in the drop-in and the split mode, FP32 in the all-FP32 mode, int
// (32-bit fixed point, scaled per field) in the fixed-point mode
__device__ __host__ inline bool is_metric(int f) { return f <= G33 || f == PHI; }

template <typename TS, typename MT>
__device__ __forceinline__ double ld(const RegTable& t, int f, int s, long x) {
  if (is_metric(f)) {
    if constexpr (std::is_same<MT, int>::value) return (double)((const int*)t.r[f][s])[x] * t.ms[f < 7 ? f : 0];
    return (double)((const MT*)t.r[f][s])[x];
  }
  return (double)((const TS*)t.r[f][s])[x];
}
template <typename TS, typename MT>
__device__ __forceinline__ void st(const RegTable& t, int f, int s, long x, double v) {
  if (is_metric(f)) {
    if constexpr (std::is_same<MT, int>::value) {
      if (fabs(v * t.mi[f < 7 ? f : 0]) > MQ_WMAX) atomicAdd(t.sat, 1u);
      ((int*)t.r[f][s])[x] = mq_word(v, t.mi[f < 7 ? f : 0]);
    }
    else ((MT*)t.r[f][s])[x] = (MT)v;
  } else {
    ((TS*)t.r[f][s])[x] = (TS)v;
  }
}

// det(gamma) = 1 and A_ij trace free at one point
__device__ __forceinline__ void normalise(double v[NF]) {
  // BSSN::set_DIFFgamma_Aij_norm (bssn.cc:61-119)
  double g11 = v[G11], g12 = v[G12], g13 = v[G13], g22 = v[G22], g23 = v[G23], g33 = v[G33];
  double omd = -1.0 * (g11 + g22 + g33 - g12 * g12 - g13 * g13 - g23 * g23 + g11 * g22 + g11 * g33 + g22 * g33 -
                       g23 * g23 * g11 - g13 * g13 * g22 - g12 * g12 * g33 + 2.0 * g12 * g13 * g23 + g11 * g22 * g33);
  double tn = -1.0 * expm1(log1p(-1.0 * omd) / 3.0);
  g11 = (g11 + tn) / (1.0 - tn); g22 = (g22 + tn) / (1.0 - tn); g33 = (g33 + tn) / (1.0 - tn);
  g12 = g12 / (1.0 - tn); g13 = g13 / (1.0 - tn); g23 = g23 / (1.0 - tn);
  v[G11] = g11; v[G12] = g12; v[G13] = g13; v[G22] = g22; v[G23] = g23; v[G33] = g33;
  double i11 = 1.0 + g22 + g33 - g23 * g23 + g22 * g33, i22 = 1.0 + g11 + g33 - g13 * g13 + g11 * g33;
  double i33 = 1.0 + g11 + g22 - g12 * g12 + g11 * g22, i12 = g13 * g23 - g12 * (1.0 + g33);
  double i13 = g12 * g23 - g13 * (1.0 + g22), i23 = g12 * g13 - g23 * (1.0 + g11);
  double trA = i11 * v[A11] + i22 * v[A22] + i33 * v[A33] + 2.0 * (i12 * v[A12] + i13 * v[A13] + i23 * v[A23]);
  v[A11] = (v[A11] - 1.0 / 3.0 * (1.0 + g11) * trA) / (1.0 - tn);
  v[A22] = (v[A22] - 1.0 / 3.0 * (1.0 + g22) * trA) / (1.0 - tn);
  v[A33] = (v[A33] - 1.0 / 3.0 * (1.0 + g33) * trA) / (1.0 - tn);
  v[A12] = (v[A12] - 1.0 / 3.0 * g12 * trA) / (1.0 - tn);
  v[A13] = (v[A13] - 1.0 / 3.0 * g13 * trA) / (1.0 - tn);
  v[A23] = (v[A23] - 1.0 / 3.0 * g23 * trA) / (1.0 - tn);
}

// Elementwise kernels run 256 threads per block; threads past the end keep
// going with point 0 and store nothing, so whole blocks reach the
// setExtraFieldData reduction (one partial row per block, see bssn_stage.h).
template <typename TS, typename MT>
__global__ void k_step_init(RegTable t, int rp, int ra, int rf, long n, int normalize, double* ext_part,
                            double phiF) {
  const long xg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = xg < n;
  const long x = valid ? xg : 0;
  // RK4Register::stepInit (RK4Register.h:118-127)
  double v[NF];
  for (int f = 0; f < NF; ++f) {
    v[f] = ld<TS, MT>(t, f, rp, x);
    if (valid && rf >= 0) st<TS, MT>(t, f, rf, x, 0.0);  // rf < 0: nothing reads _f after this call
  }
  // BSSN::stepInit calls setExtraFieldData before the normalisation, which
  // leaves DIFFphi and DIFFK alone (bssn.cc:219-226); DIFFr is not touched
  if (ext_part) block_ext_put(ext_part, blockIdx.x, valid, v[PHI], v[KK], 0.0, phiF);
  if (!valid) return;
  if (normalize) normalise(v);
  for (int f = 0; f < NF; ++f) st<TS, MT>(t, f, ra, x, v[f]);
}


// the normalised DIFFgamma_ij and A_ij of register rp into register rn, the
// only fields that differ from rp after stepInit
template <typename TS, typename MT>
__global__ void k_norm_copy(RegTable t, int rp, int rn, long n) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  double v[NF];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    v[G11 + q] = ld<TS, MT>(t, G11 + q, rp, x);
    v[A11 + q] = ld<TS, MT>(t, A11 + q, rp, x);
  }
  normalise(v);
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    st<TS, MT>(t, G11 + q, rn, x, v[G11 + q]);
    st<TS, MT>(t, A11 + q, rn, x, v[A11 + q]);
  }
}

template <typename TS>
__device__ __forceinline__ double diff_r(const SrcArgs& s, double dphi, long x) {
  if (s.rho) return s.rho[x];
  double r = 0.0;
  if (s.matter == MATTER_STATIC)
    r = exp(-6.0 * (dphi + s.phi_F)) * (double)((const TS*)s.DIFFD)[x] + s.rho_F * expm1(-6.0 * dphi);
  return r + s.lambda;
}

// RK4Register::K{n}Finalize (RK4Register.h:129-176) without the pointer swap,
// then setExtraFieldData (bssn.cc:267-305) of the new _a: ra is the _a of the
// finished stage, whose DIFFphi gives that stage's DIFFr
template <typename TS, typename MT>
__global__ void k_finalize(RegTable t, int rp, int rc, int rf, int ra, long n, int stage, double dt,
                           double* ext_part, SrcArgs src, double phiF_next) {
  const long xg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = xg < n;
  const long x = valid ? xg : 0;
  double phi_new = 0.0, K_new = 0.0;
  const double phi_old = ld<TS, MT>(t, PHI, ra, x);
  for (int f = 0; f < NF; ++f) {
    const double c = ld<TS, MT>(t, f, rc, x), p = ld<TS, MT>(t, f, rp, x), fo = ld<TS, MT>(t, f, rf, x);
    double fn, cn;
    if (stage == 1) { fn = fo + dt * c / 6.0; cn = p + dt * c / 2.0; }
    else if (stage == 2) { fn = fo + dt * c / 3.0; cn = p + dt * c / 2.0; }
    else if (stage == 3) { fn = fo + dt * c / 3.0; cn = p + dt * c; }
    else { fn = fo + (dt * c / 6.0 + p); cn = fn; }
    if (f == PHI) phi_new = (double)(MT)cn;
    if (f == KK) K_new = is_metric(f) ? cn : (double)(TS)cn;
    if (!valid) continue;
    st<TS, MT>(t, f, rf, x, fn);
    st<TS, MT>(t, f, rc, x, cn);
    if (stage == 4) st<TS, MT>(t, f, rp, x, fn);
  }
  if (ext_part) block_ext_put(ext_part, blockIdx.x, valid, phi_new, K_new, diff_r<TS>(src, phi_old, x), phiF_next);
}

// setExtraFieldData after a fused step's K4Finalize: the new _p, and the
// stage-4 input register for that stage's DIFFr
// (phi words times ms: 1 except for the fixed-point metric)
template <typename TS, typename MT>
__global__ void k_ext_post(const MT* __restrict__ phi, const TS* __restrict__ K,
                           const MT* __restrict__ phi_in, long n, double* ext_part, SrcArgs src, double phiF,
                           double ms) {
  const long xg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = xg < n;
  const long x = valid ? xg : 0;
  block_ext_put(ext_part, blockIdx.x, valid, (double)phi[x] * ms, (double)K[x],
                diff_r<TS>(src, (double)phi_in[x] * ms, x), phiF);
}

// setExtraFieldData over a register alone (DIFFr part left out): used when
// the averages are needed before any stage has produced them
template <typename TS, typename MT>
__global__ void k_ext_state(const MT* __restrict__ phi, const TS* __restrict__ K, long n, double* ext_part,
                            double phiF, double ms) {
  const long xg = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = xg < n;
  const long x = valid ? xg : 0;
  block_ext_put(ext_part, blockIdx.x, valid, (double)phi[x] * ms, (double)K[x], 0.0, phiF);
}

// Deterministic combine of partial rows: block b reduces the contiguous
// range [b*per, (b+1)*per) with a fixed per-thread stride and a fixed tree;
// with gridDim.x == 1 and ext != null it also forms the four averages of
// setExtraFieldData (math.h:1382-1415: sum/POINTS/vol, vol = sum w/POINTS).
constexpr int kExtThreads = 256;
constexpr int kExtMid = 64;  // first-level combine blocks
__global__ void k_ext_reduce(const double* __restrict__ in, long rows, double* __restrict__ out, double* ext,
                             double npts, int keep_rho) {
  __shared__ double sh[EXT_W][kExtThreads];
  const long per = (rows + gridDim.x - 1) / gridDim.x;
  const long lo = (long)blockIdx.x * per, hi = lo + per < rows ? lo + per : rows;
  double acc[EXT_W] = {0, 0, 0, 0, __builtin_huge_val()};
  for (long r = lo + threadIdx.x; r < hi; r += kExtThreads)
    for (int q = 0; q < EXT_W; ++q) {
      const double v = in[r * EXT_W + q];
      acc[q] = q == EXT_KMIN ? (v < acc[q] ? v : acc[q]) : acc[q] + v;
    }
  for (int q = 0; q < EXT_W; ++q) sh[q][threadIdx.x] = acc[q];
  __syncthreads();
  for (int w = kExtThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int q = 0; q < EXT_W; ++q) {
        const double o = sh[q][threadIdx.x + w];
        sh[q][threadIdx.x] = q == EXT_KMIN ? (o < sh[q][threadIdx.x] ? o : sh[q][threadIdx.x]) : sh[q][threadIdx.x] + o;
      }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int q = 0; q < EXT_W; ++q) out[(long)blockIdx.x * EXT_W + q] = sh[q][0];
    if (ext) {
      const double vol = sh[EXT_SW][0] / npts;
      ext[EXTV_KMIN] = sh[EXT_KMIN][0];
      ext[EXTV_KAVG] = sh[EXT_SWK][0] / npts / vol;
      ext[EXTV_AVGVOL] = exp(6.0 * (sh[EXT_SWPHI][0] / npts / vol));
      if (!keep_rho) ext[EXTV_RHOAVG] = sh[EXT_SWR][0] / npts / vol;
    }
  }
}

// ------------------------------------------------------------ dust fluid --
// Dust::populateDerivedFields, the flux part (dust.cc:109-131, 177-200): at
// every point of the stage input, v^i = e^{-10 phi} gamma~^{ij} S_j and the
// fluxes alpha D v^i, alpha S_j v^i (flux q*3 + i; q = 0 D, 1..3 S_j).  At
// stage 1 of a fused step the metric is normalised on the fly as the stage
// kernel does (bssn.cc:61-119).
// (MT: the metric's storage, FP64 or 32-bit fixed-point words times ms[f];
// either way field f, slot s at met + (f*4 + s)*rstride)
template <typename TS, typename MT>
__global__ void k_dust_flux(const MT* __restrict__ met, MetScale ms, const TS* __restrict__ alpha,
                            const TS* __restrict__ dreg, long rstride, int slot, int mslot, int normalize,
                            double phiF, TS* __restrict__ flux, long n) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  // DIFFgamma_ij at slot mslot (a normalised copy of slot's state, or slot)
  auto M = [&](int f) { return (double)met[((long)f * 4 + (f < PHI ? mslot : slot)) * rstride + x] * ms.s[f]; };
  double g11 = M(G11), g12 = M(G12), g13 = M(G13), g22 = M(G22), g23 = M(G23), g33 = M(G33);
  if (normalize) {
    const double omd = -1.0 * (g11 + g22 + g33 - g12 * g12 - g13 * g13 - g23 * g23 + g11 * g22 + g11 * g33 +
                               g22 * g33 - g23 * g23 * g11 - g13 * g13 * g22 - g12 * g12 * g33 +
                               2.0 * g12 * g13 * g23 + g11 * g22 * g33);
    const double tn = -1.0 * expm1(log1p(-1.0 * omd) / 3.0);
    g11 = (g11 + tn) / (1.0 - tn); g22 = (g22 + tn) / (1.0 - tn); g33 = (g33 + tn) / (1.0 - tn);
    g12 = g12 / (1.0 - tn); g13 = g13 / (1.0 - tn); g23 = g23 / (1.0 - tn);
  }
  // set_gammai_values (bssn.cc:447-455)
  const double i11 = 1.0 + g22 + g33 - g23 * g23 + g22 * g33, i22 = 1.0 + g11 + g33 - g13 * g13 + g11 * g33;
  const double i33 = 1.0 + g11 + g22 - g12 * g12 + g11 * g22, i12 = g13 * g23 - g12 * (1.0 + g33);
  const double i13 = g12 * g23 - g13 * (1.0 + g22), i23 = g12 * g13 - g23 * (1.0 + g11);
  const double phi = M(PHI) + phiF;
  const double al = (double)alpha[(long)slot * rstride + x] + 1.0;
  double q[4];
  for (int f = 0; f < NDUST; ++f) q[f] = (double)dreg[((long)f * 4 + slot) * rstride + x];
  const double S1 = q[1], S2 = q[2], S3 = q[3];
  const double em4phi = exp(-4.0 * phi), e6phi = exp(6.0 * phi);
  const double v[3] = {em4phi / e6phi * (i11 * S1 + i12 * S2 + i13 * S3),
                       em4phi / e6phi * (i12 * S1 + i22 * S2 + i23 * S3),
                       em4phi / e6phi * (i13 * S1 + i23 * S2 + i33 * S3)};
  for (int f = 0; f < NDUST; ++f)
    for (int d = 0; d < 3; ++d) flux[(long)(f * 3 + d) * rstride + x] = (TS)(al * q[f] * v[d]);
}

// RK4Register::stepInit of the dust registers (dust.cc:65-73)
template <typename TS>
__global__ void k_dust_reg_init(TS* __restrict__ dreg, long rstride, int rp, int ra, int rf, long n) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  for (int f = 0; f < NDUST; ++f) {
    TS* r = dreg + (long)f * 4 * rstride;
    r[(long)ra * rstride + x] = r[(long)rp * rstride + x];
    r[(long)rf * rstride + x] = TS(0);
  }
}

// Dust::K{n}Finalize (dust.cc:78-106): RK4Register::K{n}Finalize of D, S_j
template <typename TS>
__global__ void k_dust_finalize(TS* __restrict__ dreg, long rstride, int rp, int rc, int rf, long n, int stage,
                                double dt) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  for (int f = 0; f < NDUST; ++f) {
    TS* r = dreg + (long)f * 4 * rstride;
    const double c = (double)r[(long)rc * rstride + x], p = (double)r[(long)rp * rstride + x],
                 fo = (double)r[(long)rf * rstride + x];
    double fn, cn;
    if (stage == 1) { fn = fo + dt * c / 6.0; cn = p + dt * c / 2.0; }
    else if (stage == 2) { fn = fo + dt * c / 3.0; cn = p + dt * c / 2.0; }
    else if (stage == 3) { fn = fo + dt * c / 3.0; cn = p + dt * c; }
    else { fn = fo + (dt * c / 6.0 + p); cn = fn; }
    r[(long)rf * rstride + x] = (TS)fn;
    r[(long)rc * rstride + x] = (TS)cn;
    if (stage == 4) r[(long)rp * rstride + x] = (TS)fn;
  }
}

// Uploads and downloads of FP32 fields: the caller's FP64 values and the
// device's FP32 ones are converted here, through a device buffer of at most
// kIoValues.  Bound by the host link: a 256^3 field moves 134 MB instead of
// 67, but the conversion on the host (a 67 MB vector filled and read by one
// thread) cost more than both: 256^3 into pinned memory 20.3 -> 2.5 ms, into
// a new array 24.0 -> 13.0 ms, upload 18.7 -> 4.7 ms.
constexpr long kIoValues = 4l << 20;  // 32 MB
// Small pageable arrays stay with the host loop: the runtime's copy of twice
// the bytes out of pageable memory costs more than converting them (48^3
// download 0.066 ms against 0.045, 96^3 0.438 against 0.358, 128^3 equal);
// pinned ones go through the device at every size (48^3 0.038 ms against 0.041).
inline bool io_on_device(const void* host, size_t n) {
  if (n >= (2u << 20)) return true;
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, host) != hipSuccess) {
    (void)hipGetLastError();  // not an address the runtime knows: pageable
    return false;
  }
  return at.type == hipMemoryTypeHost;
}
inline unsigned io_blocks(size_t n) { return (unsigned)((n + 1023) / 1024); }
__global__ void __launch_bounds__(256) k_widen(const float* __restrict__ src, long n, double* __restrict__ dst) {
  const long b = (long)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (b + q * 256 < n) dst[b + q * 256] = (double)src[b + q * 256];
}
__global__ void __launch_bounds__(256) k_narrow(const double* __restrict__ src, long n, float* __restrict__ dst) {
  const long b = (long)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (b + q * 256 < n) dst[b + q * 256] = (float)src[b + q * 256];
}

// numNaNs (math.h:1524-1541): NaN test of the float-rounded value
template <typename TS>
__global__ void k_num_nans(const TS* __restrict__ f, long n, unsigned long long* count) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const float v = (float)f[x];
  if ((__float_as_uint(v) << 1) > 0xff000000u) atomicAdd(count, 1ull);
}

// ---------------------------------------------- constraint statistics --
// Deterministic FP64 reductions of the per-point constraint values: each
// block reduces a fixed chunk, a single block then combines the partials in
// block order.  Max uses `>` so that NaN values never win, like the
// reference's `if(fabs(C_val) > max_C)` (bssn_macros.h:581-585).
constexpr int kRedThreads = 256;
constexpr int kStats = 6;  // sum val, sum scale, sum scaled, sum val^2, max|val|, max|scaled|

__device__ __forceinline__ double red_max(double a, double b) { return b > a ? b : a; }

// Rows of the constraint kernel's one-pass mode (CONS_ROW_F columns per
// workgroup) into one row: column c of the output is the sum, or for 8q + 4,
// 8q + 5 the max, over the rows.  pass 1 combines only 8q + 6, 8q + 7: the
// workgroups' squared deviations move to the mean of all points, tot holding
// pass 0's totals:  sum (x - m)^2 = sum_b [ sum (x - m_b)^2 + n_b (m_b - m)^2 ].
// Thread (lane, r) of a block takes column lane of rows lo + r, lo + r + 16,
// ...; a fixed order, so the result is deterministic.
constexpr int kFinThreads = 1024, kFinBlocks = 128;
__global__ void __launch_bounds__(kFinThreads) k_cons_fin(const double* __restrict__ rows, long n, int pass,
                                                          const double* __restrict__ tot, double* __restrict__ out) {
  __shared__ double sh[kFinThreads / 64][64];
  const int col = threadIdx.x & 63, r = threadIdx.x >> 6;
  const long per = (n + gridDim.x - 1) / gridDim.x;
  const long lo = (long)blockIdx.x * per, hi = lo + per < n ? lo + per : n;
  const int c8 = col & 7;
  const bool dev = col < CONS_ROW_F - 1 && c8 >= 6, ismax = col < CONS_ROW_F - 1 && (c8 == 4 || c8 == 5);
  // the column of the sum a deviation column belongs to: 6 -> value, 7 -> scaled
  const int src = dev ? col - c8 + (c8 == 6 ? 0 : 2) : 0;
  const double mean = dev && pass == 1 && tot ? tot[src] / tot[CONS_ROW_F - 1] : 0.0;
  double acc = 0.0;
  if (col < CONS_ROW_F && (pass == 1) == dev)
    for (long x = lo + r; x < hi; x += kFinThreads / 64) {
      const double* row = rows + x * CONS_ROW_F;
      double v = row[col];
      if (dev && tot) {
        const double nb = row[CONS_ROW_F - 1], d = row[src] / nb - mean;
        v += nb * (d * d);
      }
      acc = ismax ? red_max(acc, v) : acc + v;
    }
  sh[r][col] = acc;
  __syncthreads();
  if (r == 0 && col < CONS_ROW_F && (pass == 1) == dev) {
    for (int k = 1; k < kFinThreads / 64; ++k) acc = ismax ? red_max(acc, sh[k][col]) : acc + sh[k][col];
    out[(long)blockIdx.x * CONS_ROW_F + col] = acc;
  }
}

// ------------------------------------- constraints without allocation --
// Scratch of cg_constraints_noalloc: the rows of one chunk of kNaRows tiles
// (one row per workgroup of the reduced constraint mode), then the running
// totals of pass 0 (CONS_ROW_W) and pass 1 (CONS_ROW_W1) and the 10 means.
// One copy per device, held until the process ends; host code reaches it
// only through the address hipGetSymbolAddress returned for that device.
constexpr int kNaRows = 4096;
constexpr long kNaTot = (long)kNaRows * CONS_ROW_W;
constexpr long kNaScratch = kNaTot + 64;  // doubles: 0.98 MB
static_assert(CONS_ROW_W == 5 * kStats && CONS_ROW_W + 2 * CONS_ROW_W1 <= 64, "scratch layout");
constexpr int kNaDevices = 64;
double* g_scratch_dev[kNaDevices];  // per device, set once at context creation
std::mutex g_scratch_mu;

constexpr int kFoldThreads = 256;
// acc[col] = (first ? 0 : acc[col]) (+ or max) the rows[r * stride + col],
// r < n, in a fixed order: thread t takes rows t, t + 256, ..., then a fixed
// tree.  Columns 6q + 4, 6q + 5 of pass 0 are maxima of non-negative values.
__global__ void __launch_bounds__(kFoldThreads) k_rows_fold(const double* __restrict__ rows, int n, int stride,
                                                           int width, int pass, int first, double* __restrict__ acc) {
  __shared__ double sh[kFoldThreads];
  for (int col = 0; col < width; ++col) {
    const bool ismax = pass == 0 && (col % 6) >= 4;
    double a = 0.0;
    for (int r = threadIdx.x; r < n; r += kFoldThreads) {
      const double v = rows[(long)r * stride + col];
      a = ismax ? red_max(a, v) : a + v;
    }
    sh[threadIdx.x] = a;
    __syncthreads();
    for (int w = kFoldThreads / 2; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w)
        sh[threadIdx.x] = ismax ? red_max(sh[threadIdx.x], sh[threadIdx.x + w]) : sh[threadIdx.x] + sh[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) acc[col] = first ? sh[0] : (ismax ? red_max(acc[col], sh[0]) : acc[col] + sh[0]);
    __syncthreads();
  }
}

// means of value and scaled per constraint for the second pass
__global__ void k_cons_means(const double* __restrict__ acc0, double n, double* __restrict__ means) {
  const int q = threadIdx.x;
  if (q < 5) {
    means[2 * q] = acc0[6 * q] / n;
    means[2 * q + 1] = acc0[6 * q + 2] / n;
  }
}

}  // namespace

// the scratch array itself (file scope; see kNaScratch above)
static __device__ __align__(256) double scratch[kNaScratch];

namespace cg {

void* reg_ptr(cg_ctx* c, int f, int slot) {
  // all-FP32 mode: one storage-type allocation of all 18 fields
  if (c->met32) return (char*)c->regs + ((long)f * c->fstride + (long)slot * c->rstride) * (long)c->ts;
  if (is_metric(f)) return c->met + ((long)f * 4 + slot) * c->rstride;  // f = 0..6
  return (char*)c->regs + ((long)(f - 7) * c->fstride + (long)slot * c->rstride) * (long)c->ts;  // f = 7..17
}

int halo_for(int order, double ko) {
  int R = order / 2;
  if (ko != 0.0 && order == 2) return 2;
  if (ko != 0.0 && order == 8) return 5;
  return R;
}

// the single conditional wrap in the halo loader needs n > tile + H - 2
bool variant_fits(const cg_ctx* c, const StageVariant& v) {
  const int t[3] = {v.ti, v.tj, v.tk}, n[3] = {c->p.nx, c->p.ny, c->p.nz};
  for (int d = 0; d < 3; ++d)
    if (n[d] < v.halo || n[d] <= t[d] + v.halo - 2) return false;
  return true;
}

// the LDS-DMA twin of v applies to this grid: compiled, rows of whole 16-byte
// groups, which then never straddle the periodic wrap (nz a multiple of 2 in
// FP64, of 4 where any field has 4 bytes; FP64 128x128x126, order 4: 0.288 ms a
// stage against 0.357 with register staging; the split kernels that move their
// FP32 fields in single words need a multiple of 2 and are for the grids that
// quads do not fit), and one wrap of the k halo (rounded up to 4) suffices; the
// 4-byte dust kernels address the three fluxes of a quantity from the first
// one, and the kernels with every field in 4 bytes Gamma^1 and Gamma^3 from K
// and Gamma^2, with a 32-bit byte offset; their halo offsets are formed with
// 24-bit multiplies (nx * ny < 2^24)
bool dma_fits(const cg_ctx* c, const StageVariant& v) {
  if (!v.launch_dma) return false;
  if ((long long)c->p.nx * c->p.ny >= (1ll << 24)) return false;
  const unsigned long long rs4 = 4ull * (unsigned long long)c->rstride;
  if (v.dust && v.prec != CG_FP64 && 3ull * rs4 > 0xFFFFFFFFull) return false;
  if ((v.prec == CG_FP32_ALL || v.prec == CG_FP32_FIX) && 5ull * rs4 > 0xFFFFFFFFull) return false;
  const int kh = (v.halo + 3) / 4 * 4;
  const int group = v.prec == CG_FP64 || v.dword ? 2 : 4;
  if (v.dword && c->p.nz % 4 == 0) return false;  // quads there
  return c->p.nz % group == 0 && c->p.nz >= kh && c->p.nz > v.tk + kh - 2;
}

long tile_count(const cg_ctx* c, const StageVariant& v) {
  auto up = [](int n, int t) { return (long)((n + t - 1) / t); };
  return up(c->p.nx, v.ti) * up(c->p.ny, v.tj) * up(c->p.nz, v.tk);
}

// Time of a stage over so many tiles, in units of variant_weight's points: the
// CUs take a tile each in turn, so on few tiles it goes by whole rounds of 256,
// and in the only round it is the time of one tile (us a stage):
//   40x40x39, order 8, live lapse: 125 8x8x8 tiles 46.7, 250 4x8x8 ones 31.3;
//     with KO 65.4 and 43.5; 24^3, 27 8x8x8 tiles by DMA 30.6, 4x4x16 16.6
//   43x47x52, FP64 order 4: 528 4x4x16 tiles (three rounds) 24.4, 462 4x8x8 18.1
// Beyond two rounds the tiles of a CU overlap and the last round counts half
// (59x51x56, split order 4: 780 4x4x16 tiles take 0.89 of the time of 735 4x8x8 ones);
// from 64^3 up it is the number of points, padding included.  Over 680 random
// grids of 20 to 111 points a side the default took 1.005 of the best
// variant's time in the mean, 1.21 at most; by points alone 1.015, 1.82.
double stage_estimate(const StageVariant& v, bool dma, double tiles) {
  const double r = tiles / 256.0, up = std::ceil(r);
  return variant_weight(v, dma) * (v.ti * v.tj * v.tk) * (r <= 2.0 ? up : 0.5 * (r + up));
}

// A wave of which no more than 8 lanes lie inside the grid takes 4 to 6 us
// longer than a full one, with either staging and at every order (why was not
// found): 20x22x20, order 4, corner waves of 2 rows of 4 points in the 4x4x16
// tile 16.1 us a stage, 4x8x8 9.8; 20x23x20 (3 rows of 4) 10.0 and 9.8.  It
// only shows where all tiles run at once.  In stage_estimate's units, a third
// of a 4x4x16 tile.
static double corner_wave(const cg_ctx* c, const StageVariant& v, double tiles) {
  const int rows = 64 / v.tk;  // of tk points along k, neighbours along j
  const int lanes = ((c->p.ny - 1) % rows + 1) * ((c->p.nz - 1) % v.tk + 1);
  return tiles <= 256.0 && lanes <= 8 ? 90.0 : 0.0;
}

// Relative time per tiled point, in units of the LDS-DMA 4x4x16 kernel of the
// same precision and order (of the DMA 8x8x8 one at halo 5, where that is the
// only one).  Ratios of the autotuner's mean stage time in tile order 5,
// frozen / live lapse, at 128^3 (orders 4, 6) and 96^3 (2, 8), where every
// tile divides the grid; register staging was measured there too and has the
// same ratios among its tiles on 127x128x125 and 95x96x97.
//   LDS-DMA                4x8x8          2x8x16         8x8x8
//     FP64 order 4, 6      1.13/1.08, 1.23/1.15   1.10/1.05, 1.12/1.12
//     FP64 order 8                                       1.13/1.14
//     split order 4, 6     1.21/1.22, 1.25/1.20   1.05/1.06, 1.23/1.06
//     split order 8                                      1.51/1.49
//     4-byte order 4, 6    1.27/1.40, 1.28/1.43
//   Register staging       4x4x16         4x8x8          2x8x16, 8x8x8
//     FP64 order 2         1.24/1.22      1.36/1.81 (1 wave)
//     FP64 order 4         1.31/1.26      1.46/1.39      1.37/1.46
//     FP64 order 6         1.40/1.46      1.49/1.48      1.45/1.62
//     FP64 order 8         1.45/1.49      1.59/1.53 (1)  1.25/1.29
//     FP64 halo 5                         1.84/1.49 (1)  1.48/1.34
//     split order 2        1.05/1.03      1.26/1.23 (1)
//     split order 4        1.18/1.07      1.41/1.28      1.23/1.11, 1.92/1.75
//     split order 6        1.34/1.15      1.50/1.32      1.60/1.39, 2.03/1.76
//     split order 8        2.20/2.22      1.49/1.49 (1)  1.73/1.72
//     split halo 5                        1.90/1.91 (1)  1.24/1.26
//     4-byte order 4       1.30/1.79      1.61/1.54      (1.23/1.69, 1.43/1.51 all-FP32)
//     4-byte order 6       1.58/1.52      1.75/1.69
// The live-lapse 4-byte kernel of order 4 spills 22 registers at the budget
// of four waves with register staging, and only there.  (1): compiled for one
// wave per SIMD; at orders 4 and 6 that budget costs the live FP64 kernels
// another 30% and is no faster anywhere.  4x8x8 at halo 5 stands at 2.05: a
// DMA tile of 8x8x8 takes less than two of its, also with the CU to itself
// (32^3: FP64 30 us against 38, split 29 against 34).  FP64 order 8 by
// registers: 4x4x16 stands beside 4x8x8, as their times do where either is
// taken (32x32x31: 25.7 and 25.5 us, live 28.3 and 28.0; 8x8x8 beyond that).
double variant_weight(const StageVariant& v, bool dma) {
  const bool f64 = v.prec == CG_FP64, split = v.prec == CG_FP32_SPLIT, wide = v.halo >= 4;
  const bool t4416 = v.ti == 4 && v.tj == 4, t2816 = v.ti == 2, t888 = v.ti == 8;  // else 4x8x8
  if (dma) {
    if (t4416) return 1.0;
    if (t2816) return 1.1;
    if (t888) return v.halo > 4 ? 1.0 : f64 ? 1.13 : 1.5;
    return f64 ? 1.15 : 1.25;
  }
  double w;
  if (wide) w = t888 ? (v.halo > 4 ? (f64 ? 1.4 : 1.25) : f64 ? 1.27 : 1.73)
                : t4416 ? (f64 ? 1.58 : 2.2)
                        : (v.halo > 4 ? 2.05 : f64 ? 1.56 : 1.49);
  else if (t4416) w = f64 ? 1.35 : split ? 1.2 : v.order == 4 ? (v.live_alpha ? 1.75 : 1.3) : 1.55;
  else if (t2816) w = 1.45;
  else if (t888) w = 1.9;
  else w = f64 ? 1.47 : split ? 1.4 : v.order == 4 ? 1.55 : 1.7;
  if (v.wpe == 1 && !wide) w *= f64 && v.live_alpha ? 1.3 : 1.02;
  return w;
}

// tile order 3 (Morton columns) needs power-of-two tile counts along i and j
bool morton_fits(int ntx, int nty) { return ntx > 0 && nty > 0 && !(ntx & (ntx - 1)) && !(nty & (nty - 1)); }

bool alpha_live(const cg_ctx* c) { return c->p.lapse != CG_LAPSE_STATIC || c->alpha_nonzero; }

}  // namespace cg

static RegTable reg_table(cg_ctx* c) {
  RegTable t;
  for (int f = 0; f < NF; ++f)
    for (int s = 0; s < 4; ++s) t.r[f][s] = reg_ptr(c, f, s);
  mq_scales(c, t.ms, t.mi);
  t.sat = c->mq_sat;
  return t;
}

static bool variant_matches(const cg_ctx* c, const StageVariant& v) {
  return v.prec == c->prec && v.order == c->p.stencil_order && v.halo == c->H && v.live_alpha == alpha_live(c) &&
         v.dust == (c->p.matter == CG_MATTER_DUST) && variant_fits(c, v);
}

// The variant without an autotuner run: among those that fit (and have the
// requested tile, if any), the one with the least estimated time of a stage.
static const StageVariant* pick_variant(const cg_ctx* c) {
  const StageVariant* best = nullptr;
  double least = 0.0;
  for (const auto& v : stage_variants()) {
    if (!variant_matches(c, v)) continue;
    if (c->req_ti && (v.ti != c->req_ti || v.tj != c->req_tj || v.tk != c->req_tk)) continue;
    const bool dma = c->dma_allowed && c->dma_pick && dma_fits(c, v);
    const double tiles = (double)tile_count(c, v);
    const double t = stage_estimate(v, dma, tiles) + corner_wave(c, v, tiles);
    if (!best || t < least) { best = &v; least = t; }
  }
  return best;
}

// The definitions below take C linkage from their declarations in cosmo_gpu.h.

const char* cg_last_error(const cg_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int cg_create(const cg_params* params, cg_ctx** out) {
  if (!params || !out) return CG_ERR_ARG;
  *out = nullptr;
  const cg_params& p = *params;
  if (p.nx <= 0 || p.ny <= 0 || p.nz <= 0) return CG_ERR_ARG;
  // The stage kernels address every array as a uniform base plus a 32-bit
  // byte offset (element offset * element size, unsigned), and the FP64
  // registers (the conformal metric in every precision) have 8-byte elements:
  // the largest element offset times 8 must stay below 2^32.
  if ((long long)p.nx * p.ny * p.nz > (1ll << 29)) return CG_ERR_ARG;
  if (p.stencil_order != 2 && p.stencil_order != 4 && p.stencil_order != 6 && p.stencil_order != 8) return CG_ERR_ARG;
  if (p.precision != CG_FP64 && p.precision != CG_FP32_SPLIT && p.precision != CG_FP32_ALL &&
      p.precision != CG_FP32_FIX)
    return CG_ERR_ARG;
  // all-FP32 and fixed-point storage: the shift-free gauges the stage kernel
  // forms by itself, on single grids; BSSN with static dust or vacuum (and,
  // with the fixed-point metric, the dust fluid)
  if ((p.precision == CG_FP32_ALL || p.precision == CG_FP32_FIX) &&
      (p.shift != CG_SHIFT_NONE || p.lapse == LAPSE_TEST_K_DRIVER))
    return CG_ERR_ARG;
  if (p.precision == CG_FP32_ALL && p.matter == CG_MATTER_DUST) return CG_ERR_ARG;
  if (p.matter != CG_MATTER_NONE && p.matter != CG_MATTER_STATIC && p.matter != CG_MATTER_DUST) return CG_ERR_ARG;
  if (p.lapse < 0 || p.lapse >= LAPSE_N) return CG_ERR_ARG;
  if (p.shift < 0 || p.shift >= SHIFT_N) return CG_ERR_ARG;
  if (p.shift != CG_SHIFT_NONE && p.matter == CG_MATTER_DUST) return CG_ERR_ARG;  // shift build: BSSN + static dust
  if (!(p.dx > 0) || !std::isfinite(p.dt)) return CG_ERR_ARG;
  cg_ctx* c = new cg_ctx();
  fft_pool_enter();
  c->p = p;
  c->prec = p.precision;
  c->ts = p.precision == CG_FP64 ? 8 : 4;
  c->met32 = p.precision == CG_FP32_ALL || p.precision == CG_FP32_FIX;
  c->mq = p.precision == CG_FP32_FIX;
  c->R = p.stencil_order / 2;
  c->H = halo_for(p.stencil_order, p.ko_coeff);
  c->lambda = p.lambda;
  if (p.tile_i > 0) { c->req_ti = p.tile_i; c->req_tj = p.tile_j; c->req_tk = p.tile_k; }
  c->npts = (long)p.nx * p.ny * p.nz;
  const long pad = ((c->npts + 63) / 64) * 64;  // 256/512-byte aligned registers
  c->rstride = pad;
  c->fstride = 4 * pad;
  *out = c;
  HIPCHK(c, hipSetDevice(p.device));
  if (p.device >= 0 && p.device < kNaDevices) {
    // the device address of this device's copy of `scratch`, once per device
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[p.device]) {
      void* ptr = nullptr;
      HIPCHK(c, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
      g_scratch_dev[p.device] = (double*)ptr;
    }
  }
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  const int nreg = c->met32 ? NF : NF - 7;  // storage-type fields
  HIPCHK(c, hipMalloc(&c->regs, (size_t)nreg * 4 * pad * c->ts));
  HIPCHK(c, hipMemsetAsync(c->regs, 0, (size_t)nreg * 4 * pad * c->ts, c->stream));
  if (!c->met32) {
    HIPCHK(c, hipMalloc((void**)&c->met, (size_t)7 * 4 * pad * sizeof(double)));
    HIPCHK(c, hipMemsetAsync(c->met, 0, (size_t)7 * 4 * pad * sizeof(double), c->stream));
  }
  // partial rows: one per tile of any compiled stage variant, or one per
  // 256-point block of the elementwise kernels
  long rows = (c->npts + 255) / 256;
  for (const auto& v : stage_variants()) {
    const long nt = (long)((p.nx + v.ti - 1) / v.ti) * ((p.ny + v.tj - 1) / v.tj) * ((p.nz + v.tk - 1) / v.tk);
    rows = nt > rows ? nt : rows;
  }
  c->ext_rows = rows;
  if (c->ts == 4) c->io_n = (size_t)std::min(c->npts, kIoValues);
  // the counters, scratch rows and staging of a context share one
  // allocation: what starts as zero first, each part on a 256-byte boundary
  size_t total = 0, zeroed = 0;
  auto part = [&](size_t bytes) {
    const size_t at = total;
    total += (bytes + 255) / 256 * 256;
    return at;
  };
  const size_t oD = part((size_t)pad * c->ts), oNan = part(sizeof(unsigned)), oSat = part(sizeof(unsigned)),
               oExt = part(4 * sizeof(double)), oCnt = part(sizeof(unsigned long long));
  zeroed = total;
  const size_t oMid = part((size_t)(kExtMid + 1) * EXT_W * sizeof(double)),
               oPart = part((size_t)rows * EXT_W * sizeof(double)), oIo = part(c->io_n * sizeof(double));
  HIPCHK(c, hipMalloc((void**)&c->arena, total));
  HIPCHK(c, hipMemsetAsync(c->arena, 0, zeroed, c->stream));
  c->DIFFD = c->arena + oD;
  c->nan_dev = (unsigned*)(c->arena + oNan);
  if (c->mq) c->mq_sat = (unsigned*)(c->arena + oSat);
  c->ext = (double*)(c->arena + oExt);
  c->nan_cnt = (unsigned long long*)(c->arena + oCnt);
  c->ext_mid = (double*)(c->arena + oMid);
  c->ext_part = (double*)(c->arena + oPart);
  if (c->io_n) c->io = (double*)(c->arena + oIo);
  c->nxf = n_xfields(p.shift);
  if (c->nxf) {
    HIPCHK(c, hipMalloc((void**)&c->xreg, (size_t)c->nxf * 4 * pad * sizeof(double)));
    HIPCHK(c, hipMemsetAsync(c->xreg, 0, (size_t)c->nxf * 4 * pad * sizeof(double), c->stream));
    HIPCHK(c, hipHostMalloc((void**)&c->nan_host, sizeof(unsigned long long)));
    HIPCHK(c, hipEventCreateWithFlags(&c->nan_ev, hipEventDisableTiming));
  }
  if (p.matter == CG_MATTER_DUST) {
    HIPCHK(c, hipMalloc(&c->dreg, (size_t)NDUST * 4 * pad * c->ts));
    HIPCHK(c, hipMemsetAsync(c->dreg, 0, (size_t)NDUST * 4 * pad * c->ts, c->stream));
    HIPCHK(c, hipMalloc(&c->flux, (size_t)NFLUX * pad * c->ts));
    HIPCHK(c, hipMalloc((void**)&c->rho_src, (size_t)pad * sizeof(double)));
    HIPCHK(c, hipMemsetAsync(c->rho_src, 0, (size_t)pad * sizeof(double), c->stream));
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CG_OK;
}

int cg_destroy(cg_ctx* c) {
  if (!c) return CG_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& e : c->ev) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
  if (c->regs) (void)hipFree(c->regs);
  if (c->met) (void)hipFree(c->met);
  if (c->cons) (void)hipFree(c->cons);
  if (c->cons_part) (void)hipFree(c->cons_part);
  if (c->obuf) (void)hipFree(c->obuf);
  if (c->dreg) (void)hipFree(c->dreg);
  if (c->flux) (void)hipFree(c->flux);
  if (c->rho_src) (void)hipFree(c->rho_src);
  if (c->xreg) (void)hipFree(c->xreg);
  if (c->nan_host) (void)hipHostFree(c->nan_host);
  if (c->nan_ev) (void)hipEventDestroy(c->nan_ev);
  if (c->arena) (void)hipFree(c->arena);
  mq_free(c);
  bardeen_free(c);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  fft_pool_leave();
  delete c;
  return CG_OK;
}

// a device pointer that is a register slot of a fixed-point metric field:
// its field and slot
static bool mq_register(const cg_ctx* c, const void* d, int* f, int* slot) {
  if (!c->mq || !d || d < c->regs) return false;
  const long off = ((const char*)d - (const char*)c->regs) / (long)c->ts;
  if (off >= 7 * c->fstride) return false;
  *f = (int)(off / c->fstride);
  *slot = (int)((off % c->fstride) / c->rstride);
  return true;
}

static int spare_slot(const cg_ctx* c) { return c->sC == 3 ? 2 : 3; }  // of the two stage registers

// After fused steps of the shift build: gives _a and _f registers of their own
// (copies of _p), as the method sequence leaves them.
int cg::unalias(cg_ctx* c) {
  if (!c->a_is_p || !c->a_raw) return CG_OK;
  if (int rc = ext_resolve(c)) return rc;  // it reads the slots written here
  // _f in slot 1 as everywhere, _a in the stage register that _c leaves
  c->sF = 1;
  c->sA = spare_slot(c);
  for (int s : {c->sA, c->sF}) {
    for (int f = 0; f < NF; ++f)
      HIPCHK(c, hipMemcpyAsync(reg_ptr(c, f, s), reg_ptr(c, f, c->sP), (size_t)c->npts * (f < 7 ? 8 : c->ts),
                               hipMemcpyDeviceToDevice, c->stream));
    for (int q = 0; q < c->nxf; ++q)
      HIPCHK(c, hipMemcpyAsync(c->xreg + ((long)q * 4 + s) * c->rstride, c->xreg + ((long)q * 4 + c->sP) * c->rstride,
                               (size_t)c->npts * 8, hipMemcpyDeviceToDevice, c->stream));
  }
  c->a_is_p = false;
  return CG_OK;
}

// resolve a reference field-map key to a device pointer and element size
static void* resolve(cg_ctx* c, const char* name, bool for_write, int* err, size_t* esz) {
  *err = 0;
  *esz = c->ts;
  std::string s(name ? name : "");
  if (s == "DIFFD_a") return c->DIFFD;
  if (s == "DIFFr_a" || s == "DIFFS_a") {  // sources (read only)
    if (for_write) { *err = 1; return nullptr; }
    *esz = 8;
    // dust: the source of the last stage, or of the state cg_constraints
    // evaluated (what initDustStep leaves in DIFFr_a, sims/dust.cc:53-63)
    if (s == "DIFFr_a" && c->rho_src) return c->rho_src;
    // otherwise the sources of the state cg_constraints evaluated
    // (initStaticStep's clearSrc + addBSSNSrc, sims/static.cc:74-82)
    if (!c->cons_valid) { *err = 3; return nullptr; }
    return c->cons + (long)(s == "DIFFr_a" ? CONS_RHO : CONS_SRCS) * c->rstride;
  }
  if (s.compare(0, 8, "Bardeen_") == 0) {  // Bardeen::Bardeen's field-map entries (bardeen.h:127-156)
    *esz = 8;
    int e4 = 0;
    const double* p = bardeen_field(c, s.substr(8), &e4);
    if (for_write) { *err = 1; return nullptr; }
    *err = e4;
    return (void*)p;
  }
  if (s == "ricci_a" || s == "AijAij_a") {
    if (for_write || !c->cons_valid) { *err = 3; return nullptr; }
    *esz = 8;
    return c->cons + (long)(s == "ricci_a" ? CONS_RICCI : CONS_AIJAIJ) * c->rstride;
  }
  if (s.size() < 3 || s[s.size() - 2] != '_') { *err = 1; return nullptr; }
  const std::string base = s.substr(0, s.size() - 2);
  const char r = s.back();
  if (for_write && r != 'c' && unalias(c)) { *err = 2; return nullptr; }
  auto slot_of = [&](char rr) {
    return rr == 'p' ? c->sP : rr == 'f' ? (c->a_is_p ? c->sP : c->sF) : rr == 'a' ? (c->a_is_p ? c->sP : c->sA)
           : rr == 'c' ? c->sC : -1;
  };
  static const char* kX[NXF] = {"beta1", "beta2", "beta3", "expN", "auxB1", "auxB2", "auxB3"};
  for (int q = 0; q < c->nxf; ++q) {
    if (base != kX[q]) continue;
    const int slot = slot_of(r);
    if (slot < 0) { *err = 1; return nullptr; }
    if (for_write && c->a_is_p && (r == 'a' || r == 'f')) { *err = 2; return nullptr; }
    *esz = 8;
    return c->xreg + ((long)q * 4 + slot) * c->rstride;
  }
  static const char* kDust[NDUST] = {"dust_D", "dust_S1", "dust_S2", "dust_S3"};
  for (int q = 0; q < NDUST && c->dreg; ++q) {
    if (base != kDust[q]) continue;
    const int slot = slot_of(r);
    if (slot < 0) { *err = 1; return nullptr; }
    if (for_write && c->a_is_p && (r == 'a' || r == 'f')) { *err = 2; return nullptr; }
    return (char*)c->dreg + ((long)q * 4 + slot) * c->rstride * (long)c->ts;
  }
  for (int f = 0; f < NF; ++f) {
    if (base != kFieldNames[f]) continue;
    int slot;
    if (r == 'p') slot = c->sP;
    else if (r == 'f') slot = c->a_is_p ? c->sP : c->sF;
    else if (r == 'a') slot = c->a_is_p ? c->sP : c->sA;
    else if (r == 'c') slot = c->sC;
    else { *err = 1; return nullptr; }
    if (for_write && c->a_is_p && (r == 'a' || r == 'f')) { *err = 2; return nullptr; }
    if (is_metric(f) && !c->met32) *esz = 8;
    return reg_ptr(c, f, slot);
  }
  *err = 1;
  return nullptr;
}

namespace cg {
const void* field_ptr(cg_ctx* c, const char* name, size_t* esz, int* err) {
  const void* d = resolve(c, name, false, err, esz);
  int f, s;
  if (mq_register(c, d, &f, &s)) {  // words, not values: read through cg_field_download
    *err = 5;
    return nullptr;
  }
  return d;
}
}  // namespace cg

int cg_field_upload(cg_ctx* c, const char* name, const double* host, size_t n) {
  if (!c || !host) return CG_ERR_ARG;
  if ((long)n != c->npts) return fail(c, CG_ERR_ARG, "size mismatch");
  int e;
  size_t esz;
  void* d = resolve(c, name, true, &e, &esz);
  if (!d) return fail(c, e == 2 ? CG_ERR_STATE : CG_ERR_ARG,
                      e == 2 ? "_a/_f alias _p after a fused step; write _p" : std::string("unknown field ") + name);
  if (int rc = ext_resolve(c)) return rc;  // the averages of the state before this write
  c->ext_fresh = false;
  if (!strncmp(name, "DIFFalpha_", 10))
    for (size_t x = 0; x < n; ++x)
      if (host[x] != 0.0) { c->alpha_nonzero = true; break; }
  int mf, ms;
  if (mq_register(c, d, &mf, &ms)) {
    // fixed-point metric: the FP64 values through the device, scaled there
    if (!c->mq_tmp) HIPCHK(c, hipMalloc((void**)&c->mq_tmp, (size_t)c->rstride * sizeof(double)));
    HIPCHK(c, hipMemcpyAsync(c->mq_tmp, host, n * 8, hipMemcpyHostToDevice, c->stream));
    return mq_store(c, mf, ms, c->mq_tmp);
  }
  if (esz == 8) {
    HIPCHK(c, hipMemcpyAsync(d, host, n * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  } else if (!io_on_device(host, n)) {
    std::vector<float> tmp(n);
    for (size_t x = 0; x < n; ++x) tmp[x] = (float)host[x];
    HIPCHK(c, hipMemcpyAsync(d, tmp.data(), n * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  } else {
    for (size_t at = 0; at < n; at += c->io_n) {
      const size_t m = n - at < c->io_n ? n - at : c->io_n;
      HIPCHK(c, hipMemcpyAsync(c->io, host + at, m * 8, hipMemcpyHostToDevice, c->stream));
      hipLaunchKernelGGL(k_narrow, dim3(io_blocks(m)), dim3(256), 0, c->stream, (const double*)c->io, (long)m,
                         (float*)d + at);
      HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  return CG_OK;
}

int cg_field_download(cg_ctx* c, const char* name, double* host, size_t n) {
  if (!c || !host) return CG_ERR_ARG;
  if ((long)n != c->npts) return fail(c, CG_ERR_ARG, "size mismatch");
  int e;
  size_t esz;
  void* d = resolve(c, name, false, &e, &esz);
  if (!d) return fail(c, e >= 3 ? CG_ERR_STATE : CG_ERR_ARG,
                      e == 3 ? std::string(name) + " is filled by cg_constraints"
                      : e == 4 ? std::string(name) + " is filled by cg_bardeen" : std::string("unknown field ") + name);
  int mf, ms;
  if (mq_register(c, d, &mf, &ms)) {
    if (!c->mq_tmp) HIPCHK(c, hipMalloc((void**)&c->mq_tmp, (size_t)c->rstride * sizeof(double)));
    if (int rc = mq_load(c, mf, ms, c->mq_tmp)) return rc;
    HIPCHK(c, hipMemcpyAsync(host, c->mq_tmp, n * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return CG_OK;
  }
  if (esz == 8) {
    HIPCHK(c, hipMemcpyAsync(host, d, n * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  } else if (!io_on_device(host, n)) {
    std::vector<float> tmp(n);
    HIPCHK(c, hipMemcpyAsync(tmp.data(), d, n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (size_t x = 0; x < n; ++x) host[x] = (double)tmp[x];
  } else {
    for (size_t at = 0; at < n; at += c->io_n) {
      const size_t m = n - at < c->io_n ? n - at : c->io_n;
      hipLaunchKernelGGL(k_widen, dim3(io_blocks(m)), dim3(256), 0, c->stream, (const float*)d + at, (long)m, c->io);
      HIPCHK(c, hipGetLastError());
      HIPCHK(c, hipMemcpyAsync(host + at, c->io, m * 8, hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  return CG_OK;
}

int cg_frw_set(cg_ctx* c, double phi, double K) {
  if (!c) return CG_ERR_ARG;
  c->frw.set(phi, K);
  c->ext_fresh = false;
  return CG_OK;
}
int cg_frw_add_fluid(cg_ctx* c, double rho, double w) {
  if (!c) return CG_ERR_ARG;
  c->frw.add_fluid(rho, w);
  return CG_OK;
}
int cg_frw_get(const cg_ctx* c, double out[4]) {
  if (!c || !out) return CG_ERR_ARG;
  out[0] = c->frw.g_phi; out[1] = c->frw.g_K; out[2] = c->frw.g_rho; out[3] = c->frw.g_S;
  return CG_OK;
}
int cg_set_lambda(cg_ctx* c, double lambda) {
  if (!c) return CG_ERR_ARG;
  c->lambda = lambda;
  return CG_OK;
}

int cg_set_dust_background(cg_ctx* c, int on) {
  if (!c) return CG_ERR_ARG;
  if (int rc = ext_resolve(c)) return rc;
  c->dust_bg = on != 0;
  return CG_OK;
}

int cg_set_tile_order(cg_ctx* c, int order) {
  if (!c || order < 0 || order > 5) return CG_ERR_ARG;
  c->tile_order = order;
  return CG_OK;
}

int cg_set_fused_accumulator(cg_ctx* c, int keep) {
  if (!c) return CG_ERR_ARG;
  c->keep_accumulator = keep != 0;
  return CG_OK;
}

int cg_set_dma(cg_ctx* c, int on) {
  if (!c) return CG_ERR_ARG;
  c->dma_allowed = on != 0;
  return CG_OK;
}

int cg_set_gauge_params(cg_ctx* c, double gd_c, double dw_mu_l, double dw_p) {
  if (!c) return CG_ERR_ARG;
  c->gd_c = gd_c; c->dw_mu_l = dw_mu_l; c->dw_p = dw_p;
  return CG_OK;
}

int cg_set_shift_params(cg_ctx* c, int gauge_wave_dir, double gd_eta, double dw_mu_s, double k_driver_coeff) {
  if (!c || gauge_wave_dir < 1 || gauge_wave_dir > 3) return CG_ERR_ARG;
  c->gauge_wave_dir = gauge_wave_dir;
  c->gd_eta = gd_eta; c->dw_mu_s = dw_mu_s; c->k_driver = k_driver_coeff;
  return CG_OK;
}

namespace cg {
StageArgs make_args(cg_ctx* c, int stage, int rin, int rp, int rf, int rout, int normalize) {
  StageArgs a{};
  a.met = c->met;
  // all-FP32 mode: regs points at field 7 so that the kernel's
  // regs + (f - 7)*4*rstride addresses the metric fields too
  a.regs = c->met32 ? (void*)((char*)c->regs + 7 * c->fstride * (long)c->ts) : c->regs;
  a.rstride = c->rstride;
  double msc[7], minv[7];
  mq_scales(c, msc, minv);
  a.mq_sat = c->mq_sat;
  a.s_in = rin; a.s_p = rp; a.s_f = rf; a.s_out = rout;
  a.s_in_norm = -1; a.s_norm_out = -1;
  a.incr = 0; a.s_a2 = -1;
  a.DIFFD = c->DIFFD;
  a.nx = c->p.nx; a.ny = c->p.ny; a.nz = c->p.nz;
  a.tile_order = c->tile_order;

  a.stage = stage;
  a.normalize = normalize;
  a.matter = c->p.matter;
  a.lapse = c->p.lapse;
  a.use_ko = c->p.ko_coeff != 0.0 && (c->p.stencil_order == 2 || c->p.stencil_order == 8);
  a.use_H = (c->p.a_adj_amp != 0.0 || c->p.k_damping_amp != 0.0);
  a.inv_dx = 1.0 / c->p.dx;
  a.inv_dx2 = 1.0 / (c->p.dx * c->p.dx);
  const int R = c->R;
  const double w1 = R == 1 ? c1<1>(1) : R == 2 ? c1<2>(1) : R == 3 ? c1<3>(1) : c1<4>(1);
  const double w2 = R == 1 ? c2<1>(1) : R == 2 ? c2<2>(1) : R == 3 ? c2<3>(1) : c2<4>(1);
  const double wm = R == 1 ? cm<1>(1) : R == 2 ? cm<2>(1) : R == 3 ? cm<3>(1) : cm<4>(1);
  for (int f = 0; f < 7; ++f) {
    a.mexp[f] = c->mq ? c->mq_exp[f] : 0;
    a.msd1[f] = (float)(msc[f] * a.inv_dx * w1);
    a.msd2[f] = (float)(msc[f] * a.inv_dx2 * w2 * (f == PHI ? 1.0 : -0.5));
    a.msdm[f] = (float)(msc[f] * a.inv_dx2 * wm * (f == PHI ? 1.0 : -1.0));
  }
  a.dt = c->p.dt;
  // RK4Register weights (RK4Register.h:129-176)
  const double dt = c->p.dt;
  a.cf = (stage == 1 || stage == 4) ? dt / 6.0 : dt / 3.0;
  a.ca = (stage == 3) ? dt : dt / 2.0;
  a.phi_F = c->frw.g_phi; a.K_F = c->frw.g_K; a.rho_F = c->frw.g_rho; a.S_F = c->frw.g_S;
  a.ext_in = c->ext;
  a.ext_part = lapse_needs_kavg(c->p.lapse) ? c->ext_part : nullptr;
  a.gd_c = c->gd_c; a.dw_mu_l = c->dw_mu_l; a.dw_p = c->dw_p;
  a.phi_F_next = c->frw.g_phi;
  a.lambda = c->lambda;
  a.dust_bg = c->dust_bg ? 1 : 0;
  a.dreg = c->dreg;
  a.flux = c->flux;
  a.s_lag = a.s_lag_met = rin;
  a.lag_mode = 0;
  a.phi_F_lag = c->frw.g_phi;
  a.rho_out = c->rho_src;
  const double dx = c->p.dx, ko = c->p.ko_coeff;
  // KO_dissipation_Q (math.h:36-72): ko*dx^3/64 * sum/dx^4 ; -ko*dx^9/1024 * sum/dx^10
  a.ko_pref = c->p.stencil_order == 2 ? ko / (64.0 * dx) : c->p.stencil_order == 8 ? -ko / (1024.0 * dx) : 0.0;
  a.a_adj = c->p.a_adj_amp;
  a.k_damp = c->p.k_damping_amp;
  a.H_frw = 2.0 / 3.0 * c->frw.g_K * c->frw.g_K - 16.0 * M_PI * c->frw.g_rho;
  a.nan_count = c->nan_dev;
  return a;
}
}  // namespace cg

// the stage kernel of the shift build's fused steps, or null where the grid,
// the order, the gauge or the tile the caller asked for has none (the method
// sequence then runs).  The autotuner's choice (req_ti) is among the other
// kernels and decides nothing here.
static const StageVariant* shift_variant(const cg_ctx* c) {
  if (!gauge_fusable(c)) return nullptr;
  for (const auto& v : shift_variants())
    if ((c->p.tile_i <= 0 || (v.ti == c->p.tile_i && v.tj == c->p.tile_j && v.tk == c->p.tile_k)) && v.prec == c->prec && v.order == c->p.stencil_order && v.halo == c->H && v.live_alpha == alpha_live(c) &&
        variant_fits(c, v) && dma_fits(c, v))
      return &v;
  return nullptr;
}

// var: the kernel to launch (null: the context's own choice)
static int launch(cg_ctx* c, StageArgs a, const StageVariant* var = nullptr) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (c->timing) {
    HIPCHK(c, hipEventCreate(&e0));
    HIPCHK(c, hipEventCreate(&e1));
    HIPCHK(c, hipEventRecord(e0, c->stream));
  }
  const bool fixed = var != nullptr;
  if (!fixed) {
    const bool live = alpha_live(c);
    if (!c->var || c->var->live_alpha != live) {
      c->var = pick_variant(c);
      if (!c->var) return fail(c, CG_ERR_ARG, "no stage kernel variant fits this grid/order");
    }
    var = c->var;
  }
  a.ntx = (c->p.nx + var->ti - 1) / var->ti;
  a.nty = (c->p.ny + var->tj - 1) / var->tj;
  a.ntz = (c->p.nz + var->tk - 1) / var->tk;
  if (a.tile_order == 3 && !morton_fits(a.ntx, a.nty)) a.tile_order = 0;
  a.per_xcd = (a.ntx * a.nty * a.ntz + 7) / 8;
  c->last_rows = (long)a.ntx * a.nty * a.ntz;
  if (c->last_rows > c->ext_rows) return fail(c, CG_ERR_STATE, "extra-field partial buffer too small");
  // stage-1 normalisation needs the register path (it transforms the metric on its way into LDS)
  const bool dma = fixed || (c->dma_allowed && c->dma_pick && !a.normalize && dma_fits(c, *var));
  if (a.s_norm_out >= 0 && !dma) return fail(c, CG_ERR_STATE, "normalised copy without DMA staging");
  int rc = (dma ? var->launch_dma : var->launch)(a, c->stream);
  if (rc != 0) return fail(c, CG_ERR_HIP, std::string("stage launch: ") + hipGetErrorString((hipError_t)rc));
  if (c->timing) {
    HIPCHK(c, hipEventRecord(e1, c->stream));
    c->ev.emplace_back(e0, e1);
  }
  return CG_OK;
}

// combine `rows` partial rows into c->ext (two deterministic passes)
static int ext_combine(cg_ctx* c, long rows, bool keep_rho) {
  const double n = (double)c->npts;
  hipLaunchKernelGGL(k_ext_reduce, dim3(kExtMid), dim3(kExtThreads), 0, c->stream, c->ext_part, rows, c->ext_mid,
                     (double*)nullptr, n, 0);
  hipLaunchKernelGGL(k_ext_reduce, dim3(1), dim3(kExtThreads), 0, c->stream, c->ext_mid, (long)kExtMid,
                     c->ext_mid + (long)kExtMid * EXT_W, c->ext, n, keep_rho ? 1 : 0);
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

// setExtraFieldData of _p alone (rho_avg kept), when no stage has produced it
static int ext_from_state(cg_ctx* c) {
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  const void* phi = reg_ptr(c, PHI, c->sP);
  double ms[7], mi[7];
  mq_scales(c, ms, mi);
  if (c->prec == CG_FP64)
    hipLaunchKernelGGL((k_ext_state<double, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)phi,
                       (const double*)reg_ptr(c, KK, c->sP), c->npts, c->ext_part, c->frw.g_phi, 1.0);
  else if (c->mq)
    hipLaunchKernelGGL((k_ext_state<float, int>), dim3(nb), dim3(bs), 0, c->stream, (const int*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), c->npts, c->ext_part, c->frw.g_phi, ms[PHI]);
  else if (c->met32)
    hipLaunchKernelGGL((k_ext_state<float, float>), dim3(nb), dim3(bs), 0, c->stream, (const float*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), c->npts, c->ext_part, c->frw.g_phi, 1.0);
  else
    hipLaunchKernelGGL((k_ext_state<float, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), c->npts, c->ext_part, c->frw.g_phi, 1.0);
  HIPCHK(c, hipGetLastError());
  int rc = ext_combine(c, nb, true);
  if (!rc) c->ext_fresh = true;
  return rc;
}

// form the pending K4Finalize averages of the last fused step
namespace cg {
int ext_resolve(cg_ctx* c) {
  if (!c->ext_lazy) return CG_OK;
  c->ext_lazy = false;
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  const void* phi = reg_ptr(c, PHI, c->sP);
  const void* phi_in = reg_ptr(c, PHI, c->ext_lazy_in);
  double ms[7], mi[7];
  mq_scales(c, ms, mi);
  if (c->prec == CG_FP64)
    hipLaunchKernelGGL((k_ext_post<double, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)phi,
                       (const double*)reg_ptr(c, KK, c->sP), (const double*)phi_in, c->npts, c->ext_part,
                       c->ext_lazy_src, c->ext_lazy_phiF, 1.0);
  else if (c->mq)
    hipLaunchKernelGGL((k_ext_post<float, int>), dim3(nb), dim3(bs), 0, c->stream, (const int*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), (const int*)phi_in, c->npts, c->ext_part,
                       c->ext_lazy_src, c->ext_lazy_phiF, ms[PHI]);
  else if (c->met32)
    hipLaunchKernelGGL((k_ext_post<float, float>), dim3(nb), dim3(bs), 0, c->stream, (const float*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), (const float*)phi_in, c->npts, c->ext_part,
                       c->ext_lazy_src, c->ext_lazy_phiF, 1.0);
  else
    hipLaunchKernelGGL((k_ext_post<float, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)phi,
                       (const float*)reg_ptr(c, KK, c->sP), (const double*)phi_in, c->npts, c->ext_part,
                       c->ext_lazy_src, c->ext_lazy_phiF, 1.0);
  HIPCHK(c, hipGetLastError());
  return ext_combine(c, nb, false);
}
}  // namespace cg

template <typename TS, typename MT>
static int step_init_t(cg_ctx* c) {
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  hipLaunchKernelGGL((k_step_init<TS, MT>), dim3(nb), dim3(bs), 0, c->stream, reg_table(c), c->sP, c->sA, c->sF, c->npts,
                     c->p.normalize_metric, c->ext_part, c->frw.g_phi);
  HIPCHK(c, hipGetLastError());
  int rc = ext_combine(c, nb, true);
  if (!rc) c->ext_fresh = true;
  return rc;
}

// DIFFgamma_ij and A_ij of slot rp, normalised, into slot rn
static int norm_copy(cg_ctx* c, int rp, int rn) {
  const int bs = 256;
  const long nbk = (c->npts + bs - 1) / bs;
  auto copy = [&](auto ts, auto mt) {
    hipLaunchKernelGGL((k_norm_copy<decltype(ts), decltype(mt)>), dim3(nbk), dim3(bs), 0, c->stream, reg_table(c), rp,
                       rn, c->npts);
  };
  if (c->prec == CG_FP64) copy(double(), double());
  else if (c->mq) copy(float(), int());
  else if (c->met32) copy(float(), float());
  else copy(float(), double());
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

// Dust::stepInit's register part (dust.cc:65-73) into slot ra
static int dust_reg_init(cg_ctx* c, int rp, int ra, int rf) {
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  if (c->prec == CG_FP64)
    hipLaunchKernelGGL(k_dust_reg_init<double>, dim3(nb), dim3(bs), 0, c->stream, (double*)c->dreg, c->rstride, rp,
                       ra, rf, c->npts);
  else
    hipLaunchKernelGGL(k_dust_reg_init<float>, dim3(nb), dim3(bs), 0, c->stream, (float*)c->dreg, c->rstride, rp,
                       ra, rf, c->npts);
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

// fluxes of the dust fluid at every point of register slot `slot`
static int dust_flux(cg_ctx* c, int slot, int normalize, int mslot = -1) {
  if (mslot < 0) mslot = slot;
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  MetScale ms, mi;
  for (int f = 0; f < 7; ++f) ms.s[f] = 1.0;
  if (c->mq) mq_scales(c, ms.s, mi.s);
  if (c->prec == CG_FP64)
    hipLaunchKernelGGL((k_dust_flux<double, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)c->met, ms,
                       (const double*)reg_ptr(c, ALPHA, 0), (const double*)c->dreg, c->rstride, slot, mslot, normalize,
                       c->frw.g_phi, (double*)c->flux, c->npts);
  else if (c->mq)
    hipLaunchKernelGGL((k_dust_flux<float, int>), dim3(nb), dim3(bs), 0, c->stream, (const int*)reg_ptr(c, 0, 0), ms,
                       (const float*)reg_ptr(c, ALPHA, 0), (const float*)c->dreg, c->rstride, slot, mslot, normalize,
                       c->frw.g_phi, (float*)c->flux, c->npts);
  else
    hipLaunchKernelGGL((k_dust_flux<float, double>), dim3(nb), dim3(bs), 0, c->stream, (const double*)c->met, ms,
                       (const float*)reg_ptr(c, ALPHA, 0), (const float*)c->dreg, c->rstride, slot, mslot, normalize,
                       c->frw.g_phi, (float*)c->flux, c->npts);
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

int cg_step_init(cg_ctx* c) {
  if (!c) return CG_ERR_ARG;
  c->ext_lazy = false;  // superseded by this stepInit's averages
  if (c->a_is_p) {
    // the shift build's _c (stage 4's input) stays where it is, as the method
    // sequence leaves it; other fused steps leave no register to keep
    c->sA = c->a_raw ? spare_slot(c) : 2;
    if (!c->a_raw) c->sC = 3;
    c->a_is_p = false;
  }
  if (c->dreg) {
    c->dust_rk = 0;
    if (int rc = dust_reg_init(c, c->sP, c->sA, c->sF)) return rc;
  }
  if (int rc = gauge_step_init(c)) return rc;
  return c->prec == CG_FP64 ? step_init_t<double, double>(c)
         : c->mq             ? step_init_t<float, int>(c)
         : c->met32          ? step_init_t<float, float>(c)
                             : step_init_t<float, double>(c);
}

int cg_rk_evolve(cg_ctx* c) {
  if (!c) return CG_ERR_ARG;
  if (int rc = unalias(c)) return rc;
  if (c->a_is_p) return fail(c, CG_ERR_STATE, "RKEvolve before stepInit");
  if (c->mq)
    return fail(c, CG_ERR_STATE, "the fixed-point metric holds states, not right-hand sides: step with cg_rk4_steps");
  StageArgs a = make_args(c, 0, c->sA, c->sP, c->sF, c->sC, 0);
  if (c->dreg) {
    // Dust::RKEvolve (dust.cc:160-174) with the sources addBSSNSrc formed
    // from the previous RKEvolve's derived fields: after swap_a_c that
    // stage's input sits in _c, read at each point before it is overwritten
    if (int rc = dust_flux(c, c->sA, 0)) return rc;
    if (c->dust_rk > 0) {
      a.lag_mode = 1;
      a.s_lag = a.s_lag_met = c->sC;
      a.phi_F_lag = c->dust_lag_phiF;
    }
    c->dust_lag_phiF = c->frw.g_phi;
    ++c->dust_rk;
  }
  if (int rc = launch(c, a)) return rc;
  // the shift build's terms (and the lapses that read other fields'
  // complete right-hand sides) on top of the stage kernel's _c
  return gauge_pass(c) ? gauge_rhs(c, c->sA, c->sC) : CG_OK;
}

namespace cg {
int rhs_at(cg_ctx* c, int rin, int rout) {
  StageArgs a = make_args(c, 0, rin, c->sP, c->sF, rout, 0);
  if (c->dreg && dust_flux(c, rin, 0)) return CG_ERR_HIP;  // sources from this state itself (lag_mode 0)
  if (int rc = launch(c, a)) return rc;
  return gauge_pass(c) ? gauge_rhs(c, rin, rout) : CG_OK;
}
}  // namespace cg

template <typename TS, typename MT>
static int finalize_t(cg_ctx* c, int n, const SrcArgs& src) {
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  hipLaunchKernelGGL((k_finalize<TS, MT>), dim3(nb), dim3(bs), 0, c->stream, reg_table(c), c->sP, c->sC, c->sF, c->sA,
                     c->npts, n, c->p.dt, c->ext_part, src, c->frw.g_phi);
  HIPCHK(c, hipGetLastError());
  return ext_combine(c, nb, false);
}

int cg_k_finalize(cg_ctx* c, int n) {
  if (!c || n < 1 || n > 4) return CG_ERR_ARG;
  if (int rc = unalias(c)) return rc;
  if (c->a_is_p) return fail(c, CG_ERR_STATE, "K-finalize before stepInit");
  if (c->mq)
    return fail(c, CG_ERR_STATE, "the fixed-point metric holds states, not right-hand sides: step with cg_rk4_steps");
  c->ext_lazy = false;
  // the finished stage's sources were formed with the FRW values before this step
  const SrcArgs src{c->DIFFD, c->p.matter, c->frw.g_phi, c->frw.g_rho, c->lambda, c->rho_src};
  c->frw.stage(n, c->p.dt);  // bssn.cc:269: FRW stage first
  if (c->dreg) {
    const int bs = 256;
    const long nb = (c->npts + bs - 1) / bs;
    if (c->prec == CG_FP64)
      hipLaunchKernelGGL(k_dust_finalize<double>, dim3(nb), dim3(bs), 0, c->stream, (double*)c->dreg, c->rstride,
                         c->sP, c->sC, c->sF, c->npts, n, c->p.dt);
    else
      hipLaunchKernelGGL(k_dust_finalize<float>, dim3(nb), dim3(bs), 0, c->stream, (float*)c->dreg, c->rstride,
                         c->sP, c->sC, c->sF, c->npts, n, c->p.dt);
    HIPCHK(c, hipGetLastError());
  }
  if (int rc = gauge_finalize(c, n)) return rc;
  int rc = c->prec == CG_FP64 ? finalize_t<double, double>(c, n, src)
           : c->met32          ? finalize_t<float, float>(c, n, src)
                               : finalize_t<float, double>(c, n, src);  // (not the fixed-point mode: rejected above)
  if (rc) return rc;
  std::swap(c->sA, c->sC);  // swap_a_c
  c->ext_fresh = (n == 4);
  return CG_OK;
}

constexpr int kMqCheck = 2;

// numNaNs (math.h:1524-1541) of a device array into c->nan_cnt
static int count_nans(cg_ctx* c, const void* d, size_t esz) {
  HIPCHK(c, hipMemsetAsync(c->nan_cnt, 0, sizeof(unsigned long long), c->stream));
  const int bs = 256;
  const long nb = (c->npts + bs - 1) / bs;
  if (esz == 8)
    hipLaunchKernelGGL(k_num_nans<double>, dim3(nb), dim3(bs), 0, c->stream, (const double*)d, c->npts, c->nan_cnt);
  else
    hipLaunchKernelGGL(k_num_nans<float>, dim3(nb), dim3(bs), 0, c->stream, (const float*)d, c->npts, c->nan_cnt);
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

int cg_rk4_steps(cg_ctx* c, int nsteps) {
  if (!c || nsteps < 0) return CG_ERR_ARG;
  c->svar = shift_variant(c);
  if (gauge_pass(c) && !c->svar) {
    // Without a fused form the shift build runs the reference's method sequence
    // (sims/static.cc:74-170): stepInit, the NaN guard, then RKEvolve (stage
    // kernel + gauge pass) and K{n}Finalize per stage.
    for (int s = 0; s < nsteps; ++s) {
      int rc;
      if ((rc = cg_step_init(c))) return rc;
      long long nn = 0;
      if ((rc = cg_num_nans(c, "DIFFphi_a", &nn))) return rc;
      if (nn) return fail(c, CG_ERR_NAN, "NAN detected in DIFFphi");
      for (int n = 1; n <= 4; ++n) {
        if ((rc = cg_rk_evolve(c))) return rc;
        if ((rc = cg_k_finalize(c, n))) return rc;
      }
    }
    return CG_OK;
  }
  // fixed physical slots for the fused path: P=0, F=1, X=2, Y=3.  No register
  // role and no pending average changes before the first step begins: a call
  // of no steps leaves the context as it was.
  const int X = 2, Y = 3;
  const bool ko_norm = ko_norm_path(c);
  // one fused stage: sources and RHS with the current FRW values, then the
  // FRW stage step (bssn.cc:269), whose phi weights the averages of the output
  const bool flrw = lapse_needs_kavg(c->p.lapse);  // averages needed inside the step
  SrcArgs src4{};
  // dust: the sources of stage n use W, detg, g_ij of stage n-1's input
  // (its DIFFgamma_ij from the normalised copy when that stage read one)
  int prev_in = 0, prev_met = 0, prev_norm = 0;
  double prev_phiF = 0.0;
  // Accumulator-free form (no _f sweeps)
  // (the shift build's four slots hold p, f, the stage's input and the gauge
  // pass's terms: the reference's accumulator)
  const bool shift = c->svar != nullptr;
  const bool incr = fused_incr(c) && c->incr_pick && !shift;
  auto stage = [&](int n, int rin, int rout, int normalize, int in_norm = -1, int norm_out = -1, int sf = 1,
                   int sa2 = -1) -> int {
    StageArgs a = make_args(c, n, rin, 0, sf, rout, normalize);
    a.s_in_norm = in_norm;
    a.s_norm_out = norm_out;
    a.incr = incr ? 1 : 0;
    a.s_a2 = sa2;
    if (c->dreg) {
      const int met_in = in_norm >= 0 ? in_norm : rin;
      if (int rc = dust_flux(c, rin, normalize, met_in)) return rc;
      if (n > 1) {
        a.lag_mode = prev_norm ? 2 : 1;
        a.s_lag = prev_in;
        a.s_lag_met = prev_met;
        a.phi_F_lag = prev_phiF;
      }
      prev_in = rin;
      prev_met = met_in;
      prev_norm = normalize;
      prev_phiF = c->frw.g_phi;
    }
    if (shift) {
      // the terms go to the slot the stage writes, at stage 4 (which writes
      // _p) to the dead one
      a.s_add = n == 4 ? Y : rout;
      a.auxB = c->p.shift == CG_SHIFT_GAMMA_DRIVER ? c->xreg + (long)XAUXB1 * 4 * c->rstride : nullptr;
      a.gd_eta = c->gd_eta;
      if (int rc = gauge_terms(c, a)) return rc;
    }
    src4 = SrcArgs{c->DIFFD, c->p.matter, c->frw.g_phi, c->frw.g_rho, c->lambda, c->rho_src};
    c->frw.stage(n, c->p.dt);
    a.phi_F_next = c->frw.g_phi;
    int rc = launch(c, a, c->svar);
    return (rc || !flrw) ? rc : ext_combine(c, c->last_rows, false);
  };
  // The method sequence's NaN guard in the shift build's fused steps: a step
  // does not change a state whose DIFFphi holds a NaN.  _p and the FRW values
  // are first written by stage 4, so the count of the state a step starts from
  // is waited for there, with the stages before it already queued: the guard
  // costs one small copy per step and no gap (waiting for it before stage 1
  // leaves the device idle while the host returns).
  auto guard_begin = [&](bool first) -> int {
    if (first) {
      if (int rc = count_nans(c, reg_ptr(c, PHI, 0), 8)) return rc;
      HIPCHK(c, hipMemcpyAsync(c->nan_host, c->nan_cnt, sizeof(*c->nan_host), hipMemcpyDeviceToHost, c->stream));
    } else {  // stage 4 of the step before counted them
      *c->nan_host = 0;
      HIPCHK(c, hipMemcpyAsync(c->nan_host, c->nan_dev, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(c, hipEventRecord(c->nan_ev, c->stream));
    return CG_OK;
  };
  auto guard_end = [&](bool first, const Frw& before) -> int {
    HIPCHK(c, hipEventSynchronize(c->nan_ev));
    const unsigned long long nn = *c->nan_host;
    if (nn == (first ? 0 : c->nan_seen)) return CG_OK;
    if (!first) c->nan_seen = (unsigned)nn;
    // the registers as the guard finds them, after stepInit
    c->frw = before;
    if (int rc = cg_step_init(c)) return rc;
    return fail(c, CG_ERR_NAN, "NAN detected in DIFFphi");
  };
  // With DMA staging, stage 4 also writes the normalised copy of the new
  // state (stepInit's _a) into the dead slot Y, so that the next step's
  // stage 1 runs the DMA kernel instead of normalising halos on the fly.
  bool have_norm = false;
  int norm_slot = Y;
  for (int s = 0; s < nsteps; ++s) {
    int rc;
    // fixed-point metric: exponents checked every kMqCheck steps (a field's
    // words stay below 2^MQ_BITS; twice that saturates)
    if (c->mq && s % kMqCheck == 0 && (rc = mq_check(c))) return rc;
    c->sP = 0; c->sF = 1;
    c->ext_lazy = false;  // this step writes the slots they are formed from
    const Frw frw0 = c->frw;
    if (shift && (rc = guard_begin(s == 0))) return rc;
    const bool pre = c->p.normalize_metric && s + 1 < nsteps &&
                     (shift || (c->var && c->dma_allowed && c->dma_pick && dma_fits(c, *c->var)));
    if ((ko_norm || (shift && c->p.normalize_metric)) && !have_norm) {
      // KO and the advection need normalised A_ij at halo points, which stage
      // 1 does not form on the fly: the copy is materialised where no stage 4
      // wrote one
      if ((rc = norm_copy(c, 0, Y))) return rc;
      have_norm = true;
      norm_slot = Y;
    }
    if (incr) {
      // a1, a2, a3 rotate over slots 1..3 so that the normalised copy of the
      // last stage 4 (written over a1) is the next stage 1's input
      if (flrw && !c->ext_fresh && (rc = ext_from_state(c))) return rc;
      int s1, s2, s3;
      incr_slots(have_norm ? norm_slot : 0, s1, s2, s3);
      if ((rc = have_norm ? stage(1, 0, s1, 0, norm_slot) : stage(1, 0, s1, c->p.normalize_metric))) return rc;
      if ((rc = stage(2, s1, s2, 0))) return rc;
      if ((rc = stage(3, s2, s3, 0))) return rc;
      if ((rc = stage(4, s3, 0, 0, -1, pre ? s1 : -1, s1, s2))) return rc;
      have_norm = pre;
      norm_slot = s1;
      c->sA = 0; c->sC = s3; c->a_is_p = true; c->a_raw = shift;
      c->ext_fresh = flrw;
      if (!flrw) {
        c->ext_lazy = true;
        c->ext_lazy_in = s3;
        c->ext_lazy_src = src4;
        c->ext_lazy_phiF = c->frw.g_phi;
      }
      continue;
    }
    // stepInit's setExtraFieldData equals the last K4Finalize's unless the
    // state changed in between; only the ConformalFLRW lapse reads it
    if (flrw && !c->ext_fresh && (rc = ext_from_state(c))) return rc;
    if ((rc = have_norm ? stage(1, 0, X, 0, Y) : stage(1, 0, X, c->p.normalize_metric))) return rc;
    if ((rc = stage(2, X, Y, 0))) return rc;
    if ((rc = stage(3, Y, X, 0))) return rc;
    if (shift && (rc = guard_end(s == 0, frw0))) return rc;
    if ((rc = stage(4, X, 0, 0, -1, pre ? Y : -1))) return rc;
    have_norm = pre;
    c->sA = 0; c->sC = X; c->a_is_p = true; c->a_raw = shift;
    c->ext_fresh = flrw;
    if (!flrw) {
      c->ext_lazy = true;
      c->ext_lazy_in = X;
      c->ext_lazy_src = src4;
      c->ext_lazy_phiF = c->frw.g_phi;
    }
  }
  unsigned nn = 0;
  HIPCHK(c, hipMemcpyAsync(&nn, c->nan_dev, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (nn != c->nan_seen) {
    c->nan_seen = nn;
    return fail(c, CG_ERR_NAN, "NAN detected in DIFFphi");
  }
  return CG_OK;
}

int cg_extra_field_data(cg_ctx* c, double out[4]) {
  if (!c || !out) return CG_ERR_ARG;
  if (int rc = ext_resolve(c)) return rc;
  HIPCHK(c, hipMemcpyAsync(out, c->ext, 4 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CG_OK;
}

int cg_num_nans(cg_ctx* c, const char* name, long long* count) {
  if (!c || !count) return CG_ERR_ARG;
  int e;
  size_t esz;
  void* d = resolve(c, name, false, &e, &esz);
  if (!d) return fail(c, CG_ERR_ARG, std::string("unknown field ") + (name ? name : ""));
  int mf, ms;
  if (mq_register(c, d, &mf, &ms)) {
    // fixed-point words hold no NaN: the stage kernels count a NaN DIFFphi
    // before rounding it (cg_rk4_steps reports it)
    *count = 0;
    return CG_OK;
  }
  if (int rc = count_nans(c, d, esz)) return rc;
  unsigned long long n = 0;
  HIPCHK(c, hipMemcpyAsync(&n, c->nan_cnt, sizeof n, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  *count = (long long)n;
  return CG_OK;
}

int cg_sync(cg_ctx* c) {
  if (!c) return CG_ERR_ARG;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CG_OK;
}

int cg_kernel_info(const cg_ctx* cc, int* vgprs, int* scratch, int* lds, int* ti, int* tj, int* tk) {
  cg_ctx* c = const_cast<cg_ctx*>(cc);
  if (!c) return CG_ERR_ARG;
  if (const StageVariant* v = shift_variant(c)) {
    const int rc = v->info_dma(vgprs, scratch, lds);
    *ti = v->ti; *tj = v->tj; *tk = v->tk;
    return rc ? CG_ERR_HIP : CG_OK;
  }
  if (!c->var || c->var->live_alpha != alpha_live(c)) c->var = pick_variant(c);
  if (!c->var) return fail(c, CG_ERR_ARG, "no stage kernel variant fits this grid/order");
  const bool dma = c->dma_allowed && c->dma_pick && dma_fits(c, *c->var);
  int rc = (dma ? c->var->info_dma : c->var->info)(vgprs, scratch, lds);
  *ti = c->var->ti; *tj = c->var->tj; *tk = c->var->tk;
  return rc ? CG_ERR_HIP : CG_OK;
}

// the constraint passes' own bounds on the grid (their 4x8x8 tile)
static int cons_fits(cg_ctx* c) {
  if (c->p.nx <= 4 + c->R - 2 || c->p.ny <= 8 + c->R - 2 || c->p.nz <= 8 + c->R - 2)
    return fail(c, CG_ERR_ARG, "grid too small for the constraint kernel tile");
  return CG_OK;
}

// The register the SVT pass reads: _a as the reference's output step
// sees it, after stepInit, i.e. the normalised _p when the last call was a
// fused step, materialised into the spare stage register.  Allocates nothing.
int cg::cons_input(cg_ctx* c, int* rin_out) {
  // the pending K4Finalize averages read the dust source this pass rewrites
  if (int rc = ext_resolve(c)) return rc;
  if (int rc = cons_fits(c)) return rc;
  int rin = c->a_is_p ? c->sP : c->sA;
  if (c->a_is_p && !c->a_raw) {
    rin = spare_slot(c);
    const int bs = 256;
    const long nbk = (c->npts + bs - 1) / bs;
    auto init = [&](auto ts, auto mt) {
      hipLaunchKernelGGL((k_step_init<decltype(ts), decltype(mt)>), dim3(nbk), dim3(bs), 0, c->stream, reg_table(c),
                         c->sP, rin, -1, c->npts, c->p.normalize_metric, (double*)nullptr, 0.0);
    };
    if (c->prec == CG_FP64) init(double(), double());
    else if (c->mq) init(float(), int());
    else if (c->met32) init(float(), float());
    else init(float(), double());
    HIPCHK(c, hipGetLastError());
    if (c->dreg && dust_reg_init(c, c->sP, rin, c->sF)) return CG_ERR_HIP;
  }
  *rin_out = rin;
  return CG_OK;
}

// Arguments of a constraint pass over the state the reference's output step
// sees (_a after stepInit).  The momentum constraint differentiates A_ij, so
// after a fused step the normalised DIFFgamma_ij and A_ij are materialised in
// the spare stage register and read from there, the other fields from _p.
// Dust: sources from this state itself (initDustStep's populate,
// sims/dust.cc:53-63).
static int cons_args(cg_ctx* c, StageArgs* out, bool* dma) {
  if (int rc = ext_resolve(c)) return rc;
  if (int rc = cons_fits(c)) return rc;
  StageArgs a = make_args(c, 0, c->a_is_p ? c->sP : c->sA, c->sP, c->sF, c->sC, 0);
  if (c->a_is_p && !c->a_raw && c->p.normalize_metric) {
    a.s_in_norm = spare_slot(c);
    if (int rc = norm_copy(c, c->sP, a.s_in_norm)) return rc;
  }
  // the DMA form's conditions are those of the stage kernels (dma_fits)
  StageVariant v{};
  v.prec = c->prec;
  v.halo = c->R;
  v.tk = CONS_DMA_TK;
  v.launch_dma = [](const StageArgs&, hipStream_t) { return 0; };
  *dma = c->prec == CG_FP64 && c->dma_allowed && dma_fits(c, v) && c->p.nx > CONS_DMA_TI + c->R - 2 &&
         c->p.ny > CONS_DMA_TJ + c->R - 2;
  const int ti = *dma ? CONS_DMA_TI : 4, tj = *dma ? CONS_DMA_TJ : 8, tk = *dma ? CONS_DMA_TK : 8;
  a.ntx = (c->p.nx + ti - 1) / ti;
  a.nty = (c->p.ny + tj - 1) / tj;
  a.ntz = (c->p.nz + tk - 1) / tk;
  if (a.tile_order == 3 && !morton_fits(a.ntx, a.nty)) a.tile_order = 0;
  a.per_xcd = (a.ntx * a.nty * a.ntz + 7) / 8;
  *out = a;
  return CG_OK;
}

// the constraint pass over every point (prepBSSNOutput's set_bd_values,
// sims/sim.cc:214-231, with the constraint values of setConstraintCalcs):
// every per-point array into c->cons, or with rows only the ones
// cg_field_download reads and one row per workgroup
static int cons_eval(cg_ctx* c, bool rows) {
  StageArgs a;
  bool dma;
  if (int rc = cons_args(c, &a, &dma)) return rc;
  const long pad = c->rstride, tiles = (long)a.ntx * a.nty * a.ntz;
  if (!c->cons) HIPCHK(c, hipMalloc((void**)&c->cons, (size_t)CONS_N * pad * sizeof(double)));
  if (rows && c->cons_tiles < tiles) {
    if (c->cons_part) (void)hipFree(c->cons_part);
    c->cons_part = nullptr;
    c->cons_tiles = 0;
    HIPCHK(c, hipMalloc((void**)&c->cons_part, (size_t)(tiles + kFinBlocks + 1) * CONS_ROW_F * sizeof(double)));
    c->cons_tiles = tiles;
  }
  a.cons = c->cons;
  a.cons_stride = pad;
  if (rows) {
    a.cons_rows = c->cons_part;
    a.cons_pass = 2;
  }
  int rc = launch_constraints(c->prec, c->p.stencil_order, alpha_live(c), c->dreg != nullptr, dma, a, c->stream);
  if (rc) return fail(c, CG_ERR_HIP, std::string("constraint launch: ") + hipGetErrorString((hipError_t)rc));
  c->cons_valid = true;
  c->cons_rows_last = tiles;
  if (!rows) return CG_OK;
  // totals, then the squared deviations from the means they give
  double* part = c->cons_part + tiles * CONS_ROW_F;
  double* fin = part + (long)kFinBlocks * CONS_ROW_F;
  for (int pass = 0; pass < 2; ++pass) {
    hipLaunchKernelGGL(k_cons_fin, dim3(kFinBlocks), dim3(kFinThreads), 0, c->stream, (const double*)c->cons_part, tiles,
                       pass, (const double*)(pass ? fin : nullptr), part);
    hipLaunchKernelGGL(k_cons_fin, dim3(1), dim3(kFinThreads), 0, c->stream, (const double*)part, (long)kFinBlocks, pass,
                       (const double*)nullptr, fin);
  }
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

// setConstraintCalcs' outputs from the totals: tot[6q + {0..5}] = sum val,
// sum scale, sum scaled, sum val^2, max|val|, max|scaled|; means[2q + {0, 1}]
// of val and scaled; var[2q + {0, 1}] their summed squared deviations
static void cons_stats(const cg_ctx* c, const double* tot, const double* means, const double* var, double* H,
                       double* M, double* G, double* A, double* S) {
  const double N = (double)c->npts;
  double* outs[5] = {H, M, G, A, S};
  const double dx3 = c->p.dx * c->p.dx * c->p.dx;
  for (int q = 0; q < 5; ++q) {
    double* o = outs[q];
    if (!o) continue;
    o[0] = means[2 * q];
    o[1] = sqrt(var[2 * q] / (N - 1.0));           // BSSN_NORMALIZE_STDEV
    o[2] = tot[q * kStats + 4];
    o[3] = tot[q * kStats + 1];                    // mean_scale is left as a sum
    o[4] = means[2 * q + 1];
    o[5] = sqrt(var[2 * q + 1] / (N - 1.0));
    o[6] = tot[q * kStats + 5];
    if (q < 2) o[7] = sqrt(tot[q * kStats + 3] * dx3);  // H_L2, M_L2 (bssn.cc:989, 994, 1067)
  }
}

int cg_constraints(cg_ctx* c, double H[8], double M[8], double G[7], double A[7], double S[7]) {
  if (!c) return CG_ERR_ARG;
  if (int rc = cons_eval(c, true)) return rc;
  double row[CONS_ROW_F];
  HIPCHK(c, hipMemcpyAsync(row, c->cons_part + (c->cons_rows_last + kFinBlocks) * CONS_ROW_F, sizeof row,
                           hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  const double N = (double)c->npts;
  double tot[5 * kStats], means[10], var[10];
  for (int q = 0; q < 5; ++q) {
    for (int k = 0; k < kStats; ++k) tot[q * kStats + k] = row[8 * q + k];
    means[2 * q] = tot[q * kStats + 0] / N;      // BSSN_NORMALIZE_MEAN
    means[2 * q + 1] = tot[q * kStats + 2] / N;
    var[2 * q] = row[8 * q + 6];
    var[2 * q + 1] = row[8 * q + 7];
  }
  cons_stats(c, tot, means, var, H, M, G, A, S);
  return CG_OK;
}

int cg_constraints_noalloc(cg_ctx* c, double H[8], double M[8], double G[7], double A[7], double S[7]) {
  if (!c) return CG_ERR_ARG;
  double* sc = (c->p.device >= 0 && c->p.device < kNaDevices) ? g_scratch_dev[c->p.device] : nullptr;
  if (!sc) return fail(c, CG_ERR_STATE, "no constraint scratch on this device (device ordinal >= 64)");
  StageArgs a;
  bool dma;
  if (int rc = cons_args(c, &a, &dma)) return rc;
  double* acc0 = sc + kNaTot;             // pass-0 totals [CONS_ROW_W]
  double* acc1 = acc0 + CONS_ROW_W;       // pass-1 totals [CONS_ROW_W1]
  double* dmeans = acc1 + CONS_ROW_W1;    // [10]
  a.cons = nullptr;
  a.cons_rows = sc;
  a.cons_means = dmeans;
  const int total = a.ntx * a.nty * a.ntz;
  for (int pass = 0; pass < 2; ++pass) {
    a.cons_pass = pass;
    for (int base = 0; base < total; base += kNaRows) {
      a.tile_base = base;
      a.tile_count = std::min(kNaRows, total - base);
      a.per_xcd = (a.tile_count + 7) / 8;
      int rc = launch_constraints(c->prec, c->p.stencil_order, alpha_live(c), c->dreg != nullptr, dma, a, c->stream);
      if (rc) return fail(c, CG_ERR_HIP, std::string("constraint launch: ") + hipGetErrorString((hipError_t)rc));
      hipLaunchKernelGGL(k_rows_fold, dim3(1), dim3(kFoldThreads), 0, c->stream, (const double*)sc, a.tile_count,
                         CONS_ROW_W, pass == 0 ? CONS_ROW_W : CONS_ROW_W1, pass, base == 0 ? 1 : 0,
                         pass == 0 ? acc0 : acc1);
      HIPCHK(c, hipGetLastError());
    }
    if (pass == 0) {
      hipLaunchKernelGGL(k_cons_means, dim3(1), dim3(64), 0, c->stream, (const double*)acc0, (double)c->npts, dmeans);
      HIPCHK(c, hipGetLastError());
    }
  }
  double res[CONS_ROW_W + 2 * CONS_ROW_W1];
  HIPCHK(c, hipMemcpyAsync(res, acc0, sizeof res, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  cons_stats(c, res, res + CONS_ROW_W + CONS_ROW_W1, res + CONS_ROW_W, H, M, G, A, S);
  return CG_OK;
}

// ------------------------------------------------ output-step readers --
// device staging of small results (strips, partial sums), grown on demand
static double* out_buf(cg_ctx* c, size_t n) {
  if (c->obuf_n < n) {
    if (c->obuf) {
      (void)hipStreamSynchronize(c->stream);
      (void)hipFree(c->obuf);
      c->obuf = nullptr;
      c->obuf_n = 0;
    }
    if (hipMalloc((void**)&c->obuf, n * sizeof(double)) != hipSuccess) {
      fail(c, CG_ERR_HIP, "out of device memory for output staging");
      return nullptr;
    }
    c->obuf_n = n;
  }
  return c->obuf;
}

static long wrap_index(long v, long n) { return ((v % n) + n) % n; }

// out[x] = f[base + (x mod wrap) * run], x < n
template <typename T>
__global__ void k_strip(const T* __restrict__ f, long base, long run, long wrap, long n, double* __restrict__ out) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x < n) out[x] = (double)f[base + (x % wrap) * run];
}

static int strip_gather(cg_ctx* c, const void* d, size_t esz, long base, long run, long wrap, long n, double* dev) {
  const int bs = 256;
  const long nb = (n + bs - 1) / bs;
  if (esz == 8)
    hipLaunchKernelGGL(k_strip<double>, dim3(nb), dim3(bs), 0, c->stream, (const double*)d, base, run, wrap, n, dev);
  else
    hipLaunchKernelGGL(k_strip<float>, dim3(nb), dim3(bs), 0, c->stream, (const float*)d, base, run, wrap, n, dev);
  HIPCHK(c, hipGetLastError());
  return CG_OK;
}

int cg_field_strip(cg_ctx* c, const char* name, int axis, long n1, long n2, double* out, size_t n) {
  if (!c || !out || axis < 1 || axis > 3) return CG_ERR_ARG;
  const long nx = c->p.nx, ny = c->p.ny, nz = c->p.nz;
  const long ext[3] = {nx, ny, nz};
  if ((long)n != ext[axis - 1]) return fail(c, CG_ERR_ARG, "a strip holds the grid's extent along its axis");
  int e;
  size_t esz;
  const void* d = field_ptr(c, name, &esz, &e);
  if (!d) return fail(c, e == 3 || e == 5 ? CG_ERR_STATE : CG_ERR_ARG,
                      e == 3   ? std::string(name) + " is filled by cg_constraints"
                      : e == 5 ? std::string(name) + " is stored in fixed point: read it with cg_field_download"
                               : std::string("unknown field ") + name);
  // field(i, n1, n2), field(n1, j, n2), field(n1, n2, k) with the offsets
  // wrapped as CosmoArray::idx wraps them (utils/Array.h:149-159)
  long base, run;
  if (axis == 1) { base = wrap_index(n1, ny) * nz + wrap_index(n2, nz); run = ny * nz; }
  else if (axis == 2) { base = wrap_index(n1, nx) * ny * nz + wrap_index(n2, nz); run = nz; }
  else { base = (wrap_index(n1, nx) * ny + wrap_index(n2, ny)) * nz; run = 1; }
  double* dev = out_buf(c, n);
  if (!dev) return CG_ERR_HIP;
  if (int rc = strip_gather(c, d, esz, base, run, (long)n, (long)n, dev)) return rc;
  HIPCHK(c, hipMemcpyAsync(out, dev, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CG_OK;
}

int cg_constraint_strip(cg_ctx* c, int axis, long n1, long n2, double* H, double* M, size_t n) {
  if (!c || !H || !M || axis < 1 || axis > 3) return CG_ERR_ARG;
  const long nx = c->p.nx, ny = c->p.ny, nz = c->p.nz;
  const long ext[3] = {nx, ny, nz};
  if ((long)n != ext[axis - 1]) return fail(c, CG_ERR_ARG, "a strip holds the grid's extent along its axis");
  if (int rc = cons_eval(c, false)) return rc;
  // set1DConstraintOutput passes the running index as i for every axis
  // (bssn.cc:918-934), so the points are (x, n1, n2) with x wrapped in i
  const long base = wrap_index(n1, ny) * nz + wrap_index(n2, nz), run = ny * nz;
  double* dev = out_buf(c, 2 * n);
  if (!dev) return CG_ERR_HIP;
  const double* cons = c->cons;
  if (int rc = strip_gather(c, cons + (long)CONS_H * c->rstride, 8, base, run, nx, (long)n, dev)) return rc;
  if (int rc = strip_gather(c, cons + (long)(CONS_MI + axis - 1) * c->rstride, 8, base, run, nx, (long)n, dev + n))
    return rc;
  HIPCHK(c, hipMemcpyAsync(H, dev, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(M, dev + n, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CG_OK;
}

// conformal_average / conformal_standard_deviation / volume_average partial
// sums (utils/math.h:1382-1415, 1458-1470): one row per block of
// sum w*f, sum w (pass 0) or sum w*(avg - f)^2 (pass 1), w = exp(6(DIFFphi + phi_FRW))
constexpr int kCwThreads = 256;
template <typename T>
__global__ void __launch_bounds__(kCwThreads) k_conformal_sums(const T* __restrict__ f, const double* __restrict__ dphi,
                                                             double phiF, long n, int pass, double avg,
                                                             double* __restrict__ part) {
  __shared__ double s0[kCwThreads], s1[kCwThreads];
  double a0 = 0.0, a1 = 0.0;
  for (long x = (long)blockIdx.x * kCwThreads + threadIdx.x; x < n; x += (long)gridDim.x * kCwThreads) {
    const double w = exp(6.0 * (dphi[x] + phiF));
    const double v = (double)f[x];
    if (pass == 0) {
      a0 += w * v;
      a1 += w;
    } else {
      const double d = avg - v;
      a0 += w * (d * d);
    }
  }
  s0[threadIdx.x] = a0;
  s1[threadIdx.x] = a1;
  __syncthreads();
  for (int h = kCwThreads / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      s0[threadIdx.x] += s0[threadIdx.x + h];
      s1[threadIdx.x] += s1[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s0[0];
    part[2 * blockIdx.x + 1] = s1[0];
  }
}

int cg_field_stats(cg_ctx* c, const char* name, double out[3]) {
  if (!c || !out) return CG_ERR_ARG;
  if (c->met32) return fail(c, CG_ERR_ARG, "conformal statistics read an FP64 DIFFphi (not in the all-FP32 mode)");
  int e;
  size_t esz, pesz;
  const void* d = resolve(c, name, false, &e, &esz);
  if (!d) return fail(c, e == 3 ? CG_ERR_STATE : CG_ERR_ARG,
                      e == 3 ? std::string(name) + " is filled by cg_constraints" : std::string("unknown field ") + name);
  const double* dphi = (const double*)resolve(c, "DIFFphi_a", false, &e, &pesz);
  const double phiF = c->frw.g_phi;
  const long n = c->npts;
  const int nb = (int)std::min<long>(1024, (n + kCwThreads - 1) / kCwThreads);
  double* dev = out_buf(c, 2 * (size_t)nb);
  if (!dev) return CG_ERR_HIP;
  std::vector<double> part(2 * (size_t)nb);
  auto pass = [&](int which, double avg) -> int {
    if (esz == 8)
      hipLaunchKernelGGL(k_conformal_sums<double>, dim3(nb), dim3(kCwThreads), 0, c->stream, (const double*)d, dphi,
                         phiF, n, which, avg, dev);
    else
      hipLaunchKernelGGL(k_conformal_sums<float>, dim3(nb), dim3(kCwThreads), 0, c->stream, (const float*)d, dphi,
                         phiF, n, which, avg, dev);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipMemcpyAsync(part.data(), dev, part.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return CG_OK;
  };
  if (int rc = pass(0, 0.0)) return rc;
  double swf = 0.0, sw = 0.0;
  for (int b = 0; b < nb; ++b) { swf += part[2 * b]; sw += part[2 * b + 1]; }  // block order: deterministic
  const double vol = sw / (double)n;
  const double avg = swf / (double)n / vol;
  if (int rc = pass(1, avg)) return rc;
  double sdev = 0.0;
  for (int b = 0; b < nb; ++b) sdev += part[2 * b];
  out[0] = avg;
  out[1] = sqrt(sdev / (double)(n - 1) / vol);
  out[2] = vol;
  return CG_OK;
}

int cg_autotune(cg_ctx* c, int reps, char* report, size_t report_len) {
  if (!c || reps < 1) return CG_ERR_ARG;
  if (!c->a_is_p || c->a_raw) return fail(c, CG_ERR_STATE, "autotune between method-level stages would clobber _a/_c");
  if (int rc = ext_resolve(c)) return rc;
  // Times stage-1, stage-2 and stage-4 shaped launches per candidate, in
  // each RK4 form the fused step may use, so the evolved state is untouched:
  // outputs into the spare slot 3, the NaN count into scratch, and dead
  // slots as the other inputs (stage 1: stencils of _p; stages 2 and 4:
  // stencils of slot 2, as their real input is not _p, whose point values
  // would otherwise come from cache; stage 4 reads its a2 from slot 3 just
  // before writing it).  The candidate's step
  // estimate is t1 + 2 t2 + t4 (stage 3 has stage 2's shape); the forms load
  // their stages differently, so the best form depends on the grid.
  std::string rep = "[";
  const StageVariant* best = nullptr;
  double best_ms = 1e30;
  // events and the per-launch timing switch are restored on every return
  struct Guard {
    cg_ctx* c;
    bool timing;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    ~Guard() {
      if (e0) (void)hipEventDestroy(e0);
      if (e1) (void)hipEventDestroy(e1);
      c->timing = timing;
    }
  } guard{c, c->timing};
  HIPCHK(c, hipEventCreate(&guard.e0));
  HIPCHK(c, hipEventCreate(&guard.e1));
  hipEvent_t e0 = guard.e0, e1 = guard.e1;
  c->timing = false;
  int best_order = 0;
  bool best_dma = false, best_incr = false;
  if (c->dreg) {  // dust: the fluxes of the state the timed launches read
    if (int rc = dust_flux(c, 0, 0)) return rc;
  }
  unsigned* nan_scratch = reinterpret_cast<unsigned*>(out_buf(c, 1));
  if (!nan_scratch) return CG_ERR_HIP;
  const bool can_incr = fused_incr(c);
  for (const auto& v : stage_variants()) {
    if (!variant_matches(c, v)) continue;
    c->var = &v;
    for (int d = 0; d < 2; ++d) {
      if (d == 1 && !(c->dma_allowed && dma_fits(c, v))) continue;
      if (d == 0 && v.dword) continue;  // the register-staged kernel of another entry
      c->dma_pick = d == 1;
      for (int order = 0; order < 6; ++order) {
        if (order == 3 && !morton_fits((c->p.nx + v.ti - 1) / v.ti, (c->p.ny + v.tj - 1) / v.tj)) continue;
        c->tile_order = order;
        for (int form = can_incr ? 1 : 0; form >= 0; --form) {
          double tq[3] = {0.0, 0.0, 0.0};
          for (int q = 0; q < 3; ++q) {
            const int st = q == 0 ? 1 : q == 1 ? 2 : 4;
            StageArgs a = make_args(c, st, st == 1 ? 0 : 2, 0, 1, 3, 0);
            if (st == 1 && c->p.normalize_metric) {
              // steady state of the fused step: the normalised copy with
              // DMA staging (slot 2 stands in), on the fly without
              if (d == 1 || ko_norm_path(c)) a.s_in_norm = 2;
              else a.normalize = 1;
            }
            a.rho_out = nullptr;  // dust: DIFFr_a keeps the last real stage's source
            a.incr = form;
            a.s_a2 = 3;
            a.nan_count = nan_scratch;
            if (c->mq) a.mq_sat = nan_scratch;  // timing launches count nothing real
            int rc = launch(c, a);
            if (rc) return rc;
            HIPCHK(c, hipEventRecord(e0, c->stream));
            for (int r = 0; r < reps; ++r)
              if ((rc = launch(c, a))) return rc;
            HIPCHK(c, hipEventRecord(e1, c->stream));
            HIPCHK(c, hipEventSynchronize(e1));
            float ms = 0;
            HIPCHK(c, hipEventElapsedTime(&ms, e0, e1));
            tq[q] = ms / reps;
          }
          const double avg = 0.25 * (tq[0] + 2.0 * tq[1] + tq[2]);  // mean stage of a step
          int vg = 0, sc = 0, ld = 0;
          (d ? v.info_dma : v.info)(&vg, &sc, &ld);
          char buf[320];
          snprintf(buf, sizeof buf,
                   "%s{\"tile\":[%d,%d,%d],\"wpe\":%d,\"dma\":%d,\"order\":%d,\"incr\":%d,\"ms\":%.4f,"
                   "\"ms1\":%.4f,\"ms2\":%.4f,\"ms4\":%.4f,\"vgprs\":%d,\"scratch\":%d}",
                   rep.size() > 1 ? "," : "", v.ti, v.tj, v.tk, v.wpe, d, order, form, avg, tq[0], tq[1], tq[2], vg,
                   sc);
          rep += buf;
          if (avg < best_ms) {
            best_ms = avg; best = &v; best_order = order; best_dma = d == 1; best_incr = form == 1;
          }
        }
      }
    }
  }
  c->tile_order = best_order;
  c->dma_pick = best_dma || !best;
  c->incr_pick = best_incr || !best;
  rep += "]";
  c->var = best;
  if (report && report_len) {
    strncpy(report, rep.c_str(), report_len - 1);
    report[report_len - 1] = 0;
  }
  if (!best) return fail(c, CG_ERR_ARG, "no stage kernel variant fits this grid/order");
  c->req_ti = best->ti; c->req_tj = best->tj; c->req_tk = best->tk;
  return CG_OK;
}

int cg_set_timing(cg_ctx* c, int on) {
  if (!c) return CG_ERR_ARG;
  c->timing = on != 0;
  return CG_OK;
}

int cg_stage_time_ms(cg_ctx* c, double* avg, int* count) {
  if (!c || !avg || !count) return CG_ERR_ARG;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  double tot = 0;
  int n = 0;
  for (auto& e : c->ev) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, e.first, e.second) == hipSuccess) { tot += ms; ++n; }
    (void)hipEventDestroy(e.first);
    (void)hipEventDestroy(e.second);
  }
  c->ev.clear();
  *avg = n ? tot / n : 0.0;
  *count = n;
  return CG_OK;
}

