// kernels_step.h — pointwise step kernels and FP64 statistics reductions.
#pragma once
#include "fft_device.h"
#include "kernels_fft.h"

namespace gnss {

template <typename T> struct CPtrs { cx<T>* p[MAXW]; };
template <typename T> struct RPtrs { T* p[MAXW]; };

// Grid geometry and the kept box of the 2/3 rule.
struct Geom {
  int nx, ny, nz, nzh, kzs;
  int keep_x, keep_y, keep_z;   // floor(n_i / 3): the largest |m_i| the mask can keep
  long long ax, ay, az, g2;     // mask: keep iff 9 * ((mx ax)^2 + (my ay)^2 + (mz az)^2) <= g2
};

// The dealiasing rule in integers: 9 * sum_i (m_i G / n_i)^2 <= G^2, G = lcm(nx, ny, nz).
// Follows deAliasKernel_mgpu (solver.cu:17-42) with the 2/3 filter (dnsparams.h:65).
__device__ __forceinline__ bool kept(const Geom& g, int mx, int my, int mz) {
  const long long a = mx * g.ax, b = my * g.ay, c = mz * g.az;
  return 9 * (a * a + b * b + c * c) <= g.g2;
}

// A box of spectral modes: outer kx (kept-mode map when kx_keep >= 0), ky likewise, kz < nkz.
struct Box {
  int bx, by, bz;       // extents
  int kx_keep, ky_keep; // -1 = all
};
__device__ __forceinline__ void box_index(const Geom& g, const Box& b, long long i, int& ix,
                                          int& iy, int& iz) {
  iz = (int)(i % b.bz);
  long long r = i / b.bz;
  const int oy = (int)(r % b.by);
  const int ox = (int)(r / b.by);
  ix = b.kx_keep < 0 ? ox : (ox <= b.kx_keep ? ox : g.nx - (2 * b.kx_keep + 1) + ox);
  iy = b.ky_keep < 0 ? oy : (oy <= b.ky_keep ? oy : g.ny - (2 * b.ky_keep + 1) + oy);
}

// i * k * f for real k: (-k f.y, k f.x)
template <typename V, typename T> __device__ __forceinline__ V ik(T k, V f) {
  V r;
  r.x = -k * f.y;
  r.y = k * f.x;
  return r;
}

// Spectral prologue of a substage: u, v, w, omega = i k x u^ (calcOmega*Kernel_mgpu,
// solver.cu:68-114) and grad phi = i k phi^ (gradientKernel_mgpu, solver.cu:233-256); with a
// colloid (the last scalar) also c^ itself and lap Z^ = -k^2 Z^ of its carrier Z = scalar 0
// (divergenceKernel_mgpu of the gradient, solver.cu:276-293, scalarAdvection solver.cu:423).
template <typename T>
__global__ void k_prologue(Geom g, Box b, CPtrs<T> q, CPtrs<T> ws, const T* __restrict__ kxv,
                           const T* __restrict__ kyv, const T* __restrict__ kzv, int S, int colloid,
                           long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int ix, iy, iz;
  box_index(g, b, i, ix, iy, iz);
  const long long o = ((long long)ix * g.ny + iy) * g.kzs + iz;
  const T kx = kxv[ix], ky = kyv[iy], kz = kzv[iz];
  const cx<T> u = q.p[0][o], v = q.p[1][o], w = q.p[2][o];
  ws.p[0][o] = u;
  ws.p[1][o] = v;
  ws.p[2][o] = w;
  ws.p[3][o] = csub(ik(ky, w), ik(kz, v));
  ws.p[4][o] = csub(ik(kz, u), ik(kx, w));
  ws.p[5][o] = csub(ik(kx, v), ik(ky, u));
  for (int s = 0; s < S; ++s) {
    const cx<T> ph = q.p[3 + s][o];
    ws.p[6 + 3 * s][o] = ik(kx, ph);
    ws.p[7 + 3 * s][o] = ik(ky, ph);
    ws.p[8 + 3 * s][o] = ik(kz, ph);
  }
  if (colloid) {
    const T k2 = kx * kx + ky * ky + kz * kz;
    const cx<T> zh = q.p[3][o];
    ws.p[6 + 3 * S][o] = q.p[2 + S][o];
    ws.p[7 + 3 * S][o] = mk<T>(-k2 * zh.x, -k2 * zh.y);
  }
}

// Physical products: u x w (crossProductKernel_mgpu, solver.cu:139-164, with the sign of
// computeRHSKernel_mgpu folded in), u . grad phi (dotKernel_mgpu, solver.cu:342-356) and, for a
// colloid c (the last scalar), u . grad c + alpha (lap Z c + grad Z . grad c)
// (colloidAdvectionKernel_mgpu, solver.cu:374-391).
template <typename T>
__global__ void k_products(RPtrs<T> p, RPtrs<T> nl, int S, int colloid, T alpha, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const T u = p.p[0][i], v = p.p[1][i], w = p.p[2][i];
  const T ox = p.p[3][i], oy = p.p[4][i], oz = p.p[5][i];
  nl.p[0][i] = v * oz - w * oy;
  nl.p[1][i] = w * ox - u * oz;
  nl.p[2][i] = u * oy - v * ox;
  for (int s = 0; s < S - colloid; ++s)
    nl.p[3 + s][i] = u * p.p[6 + 3 * s][i] + v * p.p[7 + 3 * s][i] + w * p.p[8 + 3 * s][i];
  if (colloid) {
    const int c0 = 6 + 3 * (S - 1);
    const T cx = p.p[c0][i], cy = p.p[c0 + 1][i], cz = p.p[c0 + 2][i];
    const T c = p.p[6 + 3 * S][i], lz = p.p[7 + 3 * S][i];
    nl.p[2 + S][i] = alpha * (lz * c + cx * p.p[6][i] + cy * p.p[7][i] + cz * p.p[8][i]) + (u * cx + v * cy + w * cz);
  }
}

// The integrating factor is applied as E x = x - eps x with eps = 1 - E = -expm1(-nu k^2 tau):
// for the slowly decaying modes E lies within 1e-4 of 1, and E rounded to the working precision
// would carry a relative error of up to half an ulp, the same in every substage, so that the
// state drifts by about (substages) x ulp/2 (~1e-5 after 100 FP32 steps).  eps is computed to
// its own relative precision, so 1 - eps is exact to far below an ulp.
template <typename T> __device__ __forceinline__ T dexpm1(T x);
template <> __device__ __forceinline__ double dexpm1<double>(double x) { return expm1(x); }
template <> __device__ __forceinline__ float dexpm1<float>(float x) { return expm1f(x); }
// x E for E = 1 - eps, one rounding: fma(-eps, x, x)
template <typename T> __device__ __forceinline__ T apply_if(T x, T eps) { return fma(-eps, x, x); }
// E (q + b d) = q + (b d - eps (q + b d)): the increment is formed at its own magnitude and added
// to the state once, so each substage rounds the state once.
template <typename T> __device__ __forceinline__ T if_update(T q, T b, T d, T eps) {
  const T s = fma(b, d, q);
  return q + fma(b, d, -eps * s);
}

struct RkCoef {
  double a, b, tau, dt;   // dq <- a dq + dt rhs;  q <- E (q + b dq);  dq <- E dq;  E = exp(-nu k^2 tau)
  int first, last;        // first: a = 0 (dq not read); last: dq not written
  double nu[MAXF];        // viscosity (velocity) and diffusivities (scalars)
  // batched contexts (k_rk): members nbox elements of the box apart in the launch, mstride
  // elements apart in memory, their viscosities/diffusivities in nu_m[member * MAXF + field]
  long long nbox, mstride;
  const double* nu_m;
};

// Projection + scalar sign (computeRHSKernel_mgpu, solver.cu:461-521), mask (solver.cu:17-42)
// and one low-storage RK3 substage with exact integrating factors (replaces solver.cu:547-657).
template <typename T>
__global__ void k_rk(Geom g, Box b, CPtrs<T> q, CPtrs<T> dq, CPtrs<T> nl, const T* __restrict__ kxv,
                     const T* __restrict__ kyv, const T* __restrict__ kzv, RkCoef c, int F,
                     long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int m = 0;
  if (c.nbox > 0) {
    m = (int)(i / c.nbox);
    i -= m * c.nbox;
  }
  int ix, iy, iz;
  box_index(g, b, i, ix, iy, iz);
  const long long o = m * c.mstride + ((long long)ix * g.ny + iy) * g.kzs + iz;
  const int mz = mode_of(iz, g.nz);
  // removed modes: the state holds zeros there (the step starts from a dealiased one)
  if (iz >= g.nzh || !kept(g, mode_of(ix, g.nx), mode_of(iy, g.ny), mz)) return;
  const T kx = kxv[ix], ky = kyv[iy], kz = kzv[iz];
  const T k2 = kx * kx + ky * ky + kz * kz;
  cx<T> rhs[MAXF];
  if (k2 == (T)0) {
#pragma unroll
    for (int f = 0; f < MAXF; ++f) rhs[f] = mk<T>(0, 0);
  } else {
    const cx<T> n0 = ld_s(&nl.p[0][o]), n1 = ld_s(&nl.p[1][o]), n2 = ld_s(&nl.p[2][o]);
    cx<T> kn;
    kn.x = (kx * n0.x + ky * n1.x + kz * n2.x) / k2;
    kn.y = (kx * n0.y + ky * n1.y + kz * n2.y) / k2;
    rhs[0] = csub(n0, cscale(kn, kx));
    rhs[1] = csub(n1, cscale(kn, ky));
    rhs[2] = csub(n2, cscale(kn, kz));
#pragma unroll
    for (int f = 3; f < MAXF; ++f) {
      const cx<T> v = f < F ? ld_s(&nl.p[f][o]) : mk<T>(0, 0);
      rhs[f] = mk<T>(-v.x, -v.y);
    }
  }
  const T a = (T)c.a, bb = (T)c.b, dt = (T)c.dt;
  // every field's loads before the first store (which the compiler cannot move them past)
  cx<T> oq[MAXF], od[MAXF];
#pragma unroll
  for (int f = 0; f < MAXF; ++f) {
    od[f] = (f < F && !c.first) ? ld_s(&dq.p[f][o]) : mk<T>(0, 0);
    oq[f] = f < F ? ld_s(&q.p[f][o]) : mk<T>(0, 0);
  }
#pragma unroll
  for (int f = 0; f < MAXF; ++f) {
    if (f >= F) break;
    const T eps = -dexpm1<T>(-(T)(c.nu_m ? c.nu_m[m * MAXF + f] : c.nu[f]) * k2 * (T)c.tau);
    cx<T> d = cscale(rhs[f], dt);
    if (!c.first) {
      d.x = a * od[f].x + d.x;
      d.y = a * od[f].y + d.y;
    }
    cx<T> qq = oq[f];
    qq.x = if_update(qq.x, bb, d.x, eps);
    qq.y = if_update(qq.y, bb, d.y, eps);
    st_s(&q.p[f][o], qq);
    if (!c.last) st_s(&dq.p[f][o], mk<T>(apply_if(d.x, eps), apply_if(d.y, eps)));
  }
}

// Zero every mode the 2/3 rule removes (and the kz padding): deAlias (solver.cu:44-66).
template <typename T>
__global__ void k_dealias(Geom g, CPtrs<T> q, int F, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int iz = (int)(i % g.kzs);
  const long long r = i / g.kzs;
  const int iy = (int)(r % g.ny), ix = (int)(r / g.ny);
  if (iz < g.nzh && kept(g, mode_of(ix, g.nx), mode_of(iy, g.ny), mode_of(iz, g.nz))) return;
  for (int f = 0; f < F; ++f) q.p[f][i] = mk<T>(0, 0);
}

// Mask in the ABI order [ky][kx][kz < nzh].
static __global__ void k_mask_abi(Geom g, unsigned char* __restrict__ out, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int iz = (int)(i % g.nzh);
  const long long r = i / g.nzh;
  const int ix = (int)(r % g.nx), iy = (int)(r / g.nx);
  out[i] = kept(g, mode_of(ix, g.nx), mode_of(iy, g.ny), mode_of(iz, g.nz)) ? 1 : 0;
}

// k_i = (2 pi / L_i) * m_i in FP64 (waveNumber_kernel, initialize.cu:678-691); `scale` is the
// host-computed 2 pi / L_i so the product is the same IEEE operation as on the host.
static __global__ void k_wavenumbers(double* __restrict__ k, int n, int len, double scale) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < len) k[i] = scale * (double)mode_of(i, n);
}

template <typename T>
__global__ void k_cast_wavenumbers(const double* __restrict__ in, T* __restrict__ out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (T)in[i];
}

struct IcEntry {
  long long index;  // device linear index [kx][ky][kz]
  int field;
  int pad;
  double re, im;
};

template <typename T>
__global__ void k_ic_scatter(const IcEntry* __restrict__ e, int n, CPtrs<T> q) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const IcEntry x = e[i];
  q.p[x.field][x.index] = mk<T>((T)x.re, (T)x.im);
}

// ---------------------------------------------------------------------------------------------
// Statistics: deterministic FP64 reductions (fixed per-thread order + fixed tree), one block per
// kx plane; the per-plane partials are summed in plane order.
// ---------------------------------------------------------------------------------------------
constexpr int STAT_THREADS = 256;

constexpr int SPEC_NQ = 4 + 2 * 4;

struct ShellArgs {
  int equal_box;        // 1: shell = nint(|m|) in integers
  double fx, fy, fz;    // else shell = nint(sqrt((mx fx)^2 + (my fy)^2 + (mz fz)^2))
};

__device__ __forceinline__ long long isqrt_ll(long long v) {
  long long r = (long long)sqrt((double)v);
  while (r * r > v) --r;
  while ((r + 1) * (r + 1) <= v) ++r;
  return r;
}
__device__ __forceinline__ int shell_of(const ShellArgs& a, int mx, int my, int mz) {
  if (a.equal_box) {
    const long long m2 = (long long)mx * mx + (long long)my * my + (long long)mz * mz;
    return (int)((isqrt_ll(4 * m2) + 1) / 2);
  }
  const double x = mx * a.fx, y = my * a.fy, z = mz * a.fz;
  return (int)floor(sqrt(x * x + y * y + z * z) + 0.5);
}

// Shell of the modes (mx, my, mz) with the integer rule's 4 |m|^2 in 32 bits (|m_i| <= 512, so
// 4 |m|^2 < 2^22 is exact in FP32): the hardware root is at most one off and put right in integers.
__device__ __forceinline__ int shell_small(int mx, int my, int mz) {
  const int v = 4 * (mx * mx + my * my + mz * mz);
  int r = (int)__fsqrt_rn((float)v);
  r -= r * r > v ? 1 : 0;
  r += (r + 1) * (r + 1) <= v ? 1 : 0;
  return (r + 1) / 2;
}

// Sums of one kx plane over ky and kz (calcVrms/Epsilon/IntegralLength/ScalarDissipation kernels,
// statistics.cu:1494-1845): [0] sum w|u|^2, [1] sum w k^2|u|^2, [2] sum w|u|^2/(2|k|),
// [3] sum w|k.u|^2, [4+2s] sum w k^2|phi|^2, [5+2s] sum_{k!=0} w|phi|^2 — all divided by NN^2; and,
// with BINS, the shell spectrum of the plane (the reference declares it but never computes it,
// statistics.cu:1847-1934) in the same read of the state.
// A wave takes whole ky rows, lane = kz.  Along a row the shell index does not decrease, so the modes
// of one shell are neighbouring lanes: a segmented scan over the wave leaves each shell's sum in its
// last lane, which adds it to the wave's own bins in LDS (no two lanes of a step share a shell); the
// bins of the waves are summed in wave order.  Every sum so has a fixed order.  Steps in which every
// mode is zero (those the 2/3 rule removed: 70 to 85 % of a dealiased state) are only read.
// Bound by the one read of the state: 512^3, one scalar, FP32 0.56 ms (3.8 TB/s), FP64 0.78 ms (5.5 TB/s);
// as two kernels (a thread per shell walking the rows for its modes, and a pass of its own for the
// sums) 5.5 and 5.9 ms.
constexpr int SPEC_THREADS = 1024;
template <typename T, bool BINS>
__global__ void __launch_bounds__(SPEC_THREADS)
k_spectral_stats(Geom g, CPtrs<T> q, const double* __restrict__ kxv, const double* __restrict__ kyv,
                 const double* __restrict__ kzv, int S, int nb, ShellArgs sa, double inn2,
                 double* __restrict__ part, double* __restrict__ spec) {
  extern __shared__ unsigned char smem_raw[];
  double* bins = reinterpret_cast<double*>(smem_raw);  // [wave][1 + S][nb]
  __shared__ double wsum[SPEC_THREADS / 64][SPEC_NQ];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int ix = blockIdx.x, mx = mode_of(ix, g.nx);
  const int per = (1 + S) * nb;
  double* mine = bins + (long long)wave * per;
  if (BINS) {
    for (int i = lane; i < per; i += 64) mine[i] = 0.0;
    lds_sync<true>();
  }
  double acc[SPEC_NQ];
#pragma unroll
  for (int qq = 0; qq < SPEC_NQ; ++qq) acc[qq] = 0.0;
  const double kx = kxv[ix];
  const int nch = (g.nzh + 63) / 64;
  for (int st = wave; st < g.ny * nch; st += nw) {
    const int iy = st / nch, iz = (st % nch) * 64 + lane;
    const bool on = iz < g.nzh;
    const long long o = ((long long)ix * g.ny + iy) * g.kzs + (on ? iz : 0);
    cx<T> f[MAXF];
#pragma unroll
    for (int i = 0; i < MAXF; ++i) f[i] = (on && i < 3 + S) ? ld_s(&q.p[i][o]) : mk<T>(0, 0);
    bool any = false;
#pragma unroll
    for (int i = 0; i < MAXF; ++i) any = any || f[i].x != (T)0 || f[i].y != (T)0;
    if (!__any(any)) continue;
    const double ky = kyv[iy], kz = on ? kzv[iz] : 0.0;
    const double k2 = kx * kx + ky * ky + kz * kz;
    const double w = (iz == 0 || 2 * iz == g.nz) ? 1.0 : 2.0;
    double e[1 + 4];
    {
      const double ux = f[0].x, uy = f[0].y, vx = f[1].x, vy = f[1].y, wx = f[2].x, wy = f[2].y;
      e[0] = (ux * ux + uy * uy + vx * vx + vy * vy + wx * wx + wy * wy) * inn2;
      const double dr = kx * ux + ky * vx + kz * wx, di = kx * uy + ky * vy + kz * wy;
      acc[0] += w * e[0];
      acc[1] += w * k2 * e[0];
      if (k2 > 0) acc[2] += w * e[0] / (2.0 * sqrt(k2));
      acc[3] += w * (dr * dr + di * di) * inn2;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double pr = f[3 + s].x, pi = f[3 + s].y;
      e[1 + s] = (pr * pr + pi * pi) * inn2;
      if (s < S) {
        acc[4 + 2 * s] += w * k2 * e[1 + s];
        if (k2 > 0) acc[5 + 2 * s] += w * e[1 + s];
      }
    }
    if constexpr (BINS) {
      const int my = mode_of(iy, g.ny), mz = iz < (g.nz >> 1) ? iz : -(g.nz >> 1);
      const int sh = !on ? 0x7FFFFFFF : (sa.equal_box ? shell_small(mx, my, mz) : shell_of(sa, mx, my, mz));
#pragma unroll
      for (int s = 0; s < 5; ++s) e[s] *= 0.5 * w;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const bool same = __shfl_up(sh, d) == sh && lane >= d;
        if (!__any(same)) break;
#pragma unroll
        for (int s = 0; s < 5; ++s) {
          if (s > S) break;
          const double up = __shfl_up(e[s], d);
          if (same) e[s] += up;
        }
      }
      const int next = __shfl_down(sh, 1);
      if (on && (lane == 63 || next != sh)) {
#pragma unroll
        for (int s = 0; s < 5; ++s) {
          if (s > S) break;
          mine[s * nb + sh] += e[s];
        }
      }
      lds_sync<true>();
    }
  }
#pragma unroll
  for (int qq = 0; qq < SPEC_NQ; ++qq) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) acc[qq] += __shfl_down(acc[qq], d);
    if (lane == 0) wsum[wave][qq] = acc[qq];
  }
  __syncthreads();
  if (threadIdx.x < SPEC_NQ) {
    double t = 0.0;
    for (int i = 0; i < nw; ++i) t += wsum[i][threadIdx.x];
    part[(long long)ix * SPEC_NQ + threadIdx.x] = t;
  }
  if constexpr (BINS) {
    for (int j = threadIdx.x; j < per; j += blockDim.x) {
      double t = 0.0;
      for (int i = 0; i < nw; ++i) t += bins[(long long)i * per + j];
      spec[(long long)ix * per + j] = t;
    }
  }
}

// The spectrum where a plane's bins do not fit the LDS (boxes with very unequal sides, whose shell
// count grows with the longest over the shortest): shells of one kx plane.
// Thread b owns shell b: for each ky it walks the kz interval of
// that shell (the shell index is non-decreasing in kz), so every sum has a fixed order.
template <typename T>
__global__ void __launch_bounds__(STAT_THREADS)
k_spectrum(Geom g, CPtrs<T> q, int S, int nb, ShellArgs sa, double inn2, double* __restrict__ spec) {
  const int ix = blockIdx.x;
  const int mx = mode_of(ix, g.nx);
  for (int b = threadIdx.x; b < nb; b += STAT_THREADS) {
    double acc[1 + 4];
    for (int s = 0; s <= S; ++s) acc[s] = 0.0;
    for (int iy = 0; iy < g.ny; ++iy) {
      const int my = mode_of(iy, g.ny);
      if (shell_of(sa, mx, my, 0) > b) continue;
      if (shell_of(sa, mx, my, g.nz / 2) < b) continue;
      // first kz with shell >= b, first kz with shell >= b + 1
      int lo = 0, hi = g.nzh;
      while (lo < hi) { int mid = (lo + hi) >> 1; if (shell_of(sa, mx, my, mid) >= b) hi = mid; else lo = mid + 1; }
      const int z0 = lo;
      hi = g.nzh;
      while (lo < hi) { int mid = (lo + hi) >> 1; if (shell_of(sa, mx, my, mid) >= b + 1) hi = mid; else lo = mid + 1; }
      const int z1 = lo;
      const long long base = ((long long)ix * g.ny + iy) * g.kzs;
      for (int iz = z0; iz < z1; ++iz) {
        const double w = (iz == 0 || 2 * iz == g.nz) ? 0.5 : 1.0;
        const cx<T> u = q.p[0][base + iz], v = q.p[1][base + iz], ww = q.p[2][base + iz];
        const double ux = u.x, uy = u.y, vx = v.x, vy = v.y, wx = ww.x, wy = ww.y;
        acc[0] += w * (ux * ux + uy * uy + vx * vx + vy * vy + wx * wx + wy * wy) * inn2;
        for (int s = 0; s < S; ++s) {
          const cx<T> ph = q.p[3 + s][base + iz];
          const double pr = ph.x, pi = ph.y;
          acc[1 + s] += w * (pr * pr + pi * pi) * inn2;
        }
      }
    }
    for (int s = 0; s <= S; ++s) spec[((long long)ix * (1 + S) + s) * nb + b] = acc[s];
  }
}

// x-z plane averages at one y (calcYprof_kernel_2D, statistics.cu:1936-1977): means, <u'u'>, <v'v'>,
// <w'w'>, <u'v'>, <phi'phi'>, <v'phi'>, plus the CFL and |u| maxima, in one read of the plane: sums
// of d = f - c and of their products, with c the mean of eight sample rows, so that |mean - c| lies
// within the fluctuations and <f'g'> = <d_f d_g> - <d_f><d_g> cancels nothing (all in FP64, fixed
// order).  16-byte loads (nz is a multiple of 8).  Bound by that read: 512^3, one scalar, FP32 0.38 ms
// (5.6 TB/s), FP64 0.79 ms; as two passes of scalar loads 3.1 and 3.3 ms.
constexpr int PLANE_THREADS = 1024;
constexpr int PLANE_NQ = MAXF + 4 + 2 * 4;
template <typename T>
__global__ void __launch_bounds__(PLANE_THREADS)
k_plane_stats(Geom g, RPtrs<T> ph, int S, double idx_, double idy_, double idz_,
              double* __restrict__ prof, double* __restrict__ cmax) {
  constexpr int V = 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(V)));
  __shared__ double wsum[PLANE_THREADS / 64][PLANE_NQ + 2];
  __shared__ double tot[PLANE_NQ + 2];
  const int y = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nv = g.nz / V, nt = blockDim.x;
  auto load = [&](int i, vec* f) {
    const int x = i / nv, z = i - x * nv;
    const long long o = ((long long)x * g.ny + y) * nv + z;
#pragma unroll
    for (int k = 0; k < MAXF; ++k)
      if (k < 3 + S) f[k] = reinterpret_cast<const vec*>(ph.p[k])[o];
  };
  // totals of the first n entries of acc over the block (every thread reads them in tot)
  auto reduce = [&](double* acc, int q) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) acc[0] += __shfl_down(acc[0], d);
    if (lane == 0) wsum[wave][q] = acc[0];
  };
  const int rows = g.nx < 8 ? g.nx : 8, xs = g.nx / rows;
  double c[MAXF];
#pragma unroll
  for (int k = 0; k < MAXF; ++k) c[k] = 0.0;
  for (int i = tid; i < rows * nv; i += nt) {
    vec f[MAXF];
    const int r = i / nv;
    load(r * xs * nv + (i - r * nv), f);
#pragma unroll
    for (int k = 0; k < MAXF; ++k)
      if (k < 3 + S)
#pragma unroll
        for (int j = 0; j < V; ++j) c[k] += (double)f[k][j];
  }
#pragma unroll
  for (int k = 0; k < MAXF; ++k) reduce(&c[k], k);
  __syncthreads();
  if (tid < MAXF) {
    double t = 0.0;
    for (int i = 0; i < nt / 64; ++i) t += wsum[i][tid];
    tot[tid] = t / ((double)rows * g.nz);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < MAXF; ++k) c[k] = tot[k];
  double acc[PLANE_NQ];
#pragma unroll
  for (int k = 0; k < PLANE_NQ; ++k) acc[k] = 0.0;
  double cm = 0.0, um = 0.0;
  const int n = g.nx * nv;
  for (int i = tid; i < n; i += nt) {
    vec f[MAXF];
    load(i, f);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const double u = f[0][j], v = f[1][j], w = f[2][j];
      const double du = u - c[0], dv = v - c[1], dw = w - c[2];
      acc[0] += du;
      acc[1] += dv;
      acc[2] += dw;
      acc[MAXF] += du * du;
      acc[MAXF + 1] += dv * dv;
      acc[MAXF + 2] += dw * dw;
      acc[MAXF + 3] += du * dv;
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s < S) {
          const double dp = (double)f[3 + s][j] - c[3 + s];
          acc[3 + s] += dp;
          acc[MAXF + 4 + 2 * s] += dp * dp;
          acc[MAXF + 5 + 2 * s] += dv * dp;
        }
      cm = fmax(cm, fabs(u) * idx_ + fabs(v) * idy_ + fabs(w) * idz_);
      um = fmax(um, fmax(fabs(u), fmax(fabs(v), fabs(w))));
    }
  }
#pragma unroll
  for (int k = 0; k < PLANE_NQ; ++k) reduce(&acc[k], k);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    cm = fmax(cm, __shfl_down(cm, d));
    um = fmax(um, __shfl_down(um, d));
  }
  if (lane == 0) {
    wsum[wave][PLANE_NQ] = cm;
    wsum[wave][PLANE_NQ + 1] = um;
  }
  __syncthreads();
  const double inv = 1.0 / ((double)g.nx * g.nz);
  if (tid < PLANE_NQ) {
    double t = 0.0;
    for (int i = 0; i < nt / 64; ++i) t += wsum[i][tid];
    tot[tid] = t * inv;
  } else if (tid < PLANE_NQ + 2) {
    double t = 0.0;
    for (int i = 0; i < nt / 64; ++i) t = fmax(t, wsum[i][tid]);
    tot[tid] = t;
  }
  __syncthreads();
  if (tid == 0) {
    const int ny = g.ny;
    const double* m = tot;          // <d_f>
    const double* p = tot + MAXF;   // <d_f d_g>
    prof[0 * ny + y] = c[0] + m[0];
    prof[1 * ny + y] = c[1] + m[1];
    prof[2 * ny + y] = c[2] + m[2];
    prof[3 * ny + y] = p[0] - m[0] * m[0];
    prof[4 * ny + y] = p[1] - m[1] * m[1];
    prof[5 * ny + y] = p[2] - m[2] * m[2];
    prof[6 * ny + y] = p[3] - m[0] * m[1];
    for (int s = 0; s < S; ++s) {
      prof[(7 + 3 * s) * ny + y] = tot[3 + s] + (s == 0 ? c[3] : s == 1 ? c[4] : s == 2 ? c[5] : c[6]);
      prof[(8 + 3 * s) * ny + y] = p[4 + 2 * s] - m[3 + s] * m[3 + s];
      prof[(9 + 3 * s) * ny + y] = p[5 + 2 * s] - m[1] * m[3 + s];
    }
    cmax[2 * y] = tot[PLANE_NQ];
    cmax[2 * y + 1] = tot[PLANE_NQ + 1];
  }
}

// Any non-finite value in the kz = 0 column of field blockIdx.y (cheap NaN/Inf watchdog after a step); the flag
// is in pinned host memory, which the host has cleared.
template <typename T>
__global__ void k_finite(Geom g, CPtrs<T> q, int* __restrict__ flag) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)g.nx * g.ny) return;
  const cx<T> v = q.p[blockIdx.y][i * g.kzs];
  if (!isfinite((double)v.x) || !isfinite((double)v.y)) flag[0] = 1;
}


// ---------------------------------------------------------------------------------------------
// x passes fused with the spectral ends of a substage.
// ---------------------------------------------------------------------------------------------

// Inverse x pass of the work fields of one field group, fed straight from the state.  Per
// (ky kept, kz chunk) tile it loads the group's state columns once (kept kx rows only), forms
// each work field in registers and transforms it:
//   GRP 0 (velocity): u, v, w -> u, v, w, omega = i k x u  (calcOmega*Kernel_mgpu, solver.cu:68-114)
//   GRP 1 (scalar):   phi_s   -> i k phi_s                 (gradientKernel_mgpu, solver.cu:233-256)
//   GRP 2 (colloid):  c, Z    -> i k c, c, -k^2 Z          (scalarAdvection, solver.cu:419-437)
// Replaces k_prologue and the separate inverse x passes of those work fields.
template <typename T, int L, int C, int GRP>
__global__ void __launch_bounds__(lb_threads(C * (L / Plan<L>::E)))
k_xinv_prologue(Geom g, CPtrs<T> q, CPtrs<T> ws, const T* __restrict__ kxv, const T* __restrict__ kyv,
                const T* __restrict__ kzv, const cx<T>* __restrict__ tw, int scalar, int nchunks, int G) {
  constexpr bool VEL = GRP == 0;
  constexpr int NIN = VEL ? 3 : (GRP == 2 ? 2 : 1);
  constexpr int NOUT = VEL ? 6 : (GRP == 2 ? 5 : 3);
  constexpr int E = Plan<L>::E;
  constexpr int TPC = L / E;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int c = tid % C;
  const int t = (tid / C) % TPC;
  const int gg = C * TPC >= 256 ? 0 : tid / (C * TPC);  // one group per block from 256 threads on
  const int chunk = blockIdx.x % nchunks;
  const int o = (blockIdx.x / nchunks) * G + gg;
  const int nouter = 2 * g.keep_y + 1;
  const bool active = o < nouter;
  const int iy = outer_index(active ? o : 0, g.keep_y, g.ny);
  const int iz = chunk * C + c;
  const long long col = (long long)iy * g.kzs + iz;
  const long long estride = (long long)g.ny * g.kzs;
  const T ky = kyv[iy], kz = kzv[iz];
  const int in0 = VEL ? 0 : 3 + scalar;
  const int out0 = VEL ? 0 : 6 + 3 * scalar;
  cx<T> qv[NIN][E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + e * TPC;
    const bool ld = active && row_kept(p, L, g.keep_x);
#pragma unroll
    for (int f = 0; f < NIN; ++f) {
      const int fi = f == 0 ? in0 : (GRP == 2 ? 3 : in0 + f);  // the colloid group also reads Z
      qv[f][e] = ld ? ld_s(&q.p[fi][col + p * estride]) : mk<T>(0, 0);
    }
  }
  const LdsCol idx{gg * L * C + c, C};
#pragma unroll 1
  for (int w = 0; w < NOUT; ++w) {
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const T kx = kxv[t + e * TPC];
      if (VEL) {
        const cx<T> u = qv[0][e], vv = qv[1][e], ww = qv[NIN - 1][e];
        if (w < 3) v[e] = w == 0 ? u : (w == 1 ? vv : ww);
        else if (w == 3) v[e] = csub(ik(ky, ww), ik(kz, vv));
        else if (w == 4) v[e] = csub(ik(kz, u), ik(kx, ww));
        else v[e] = csub(ik(kx, vv), ik(ky, u));
      } else if (GRP == 2 && w == 3) {
        v[e] = qv[0][e];
      } else if (GRP == 2 && w == 4) {
        const T k2 = kx * kx + ky * ky + kz * kz;
        v[e] = mk<T>(-k2 * qv[NIN - 1][e].x, -k2 * qv[NIN - 1][e].y);
      } else {
        v[e] = ik(w == 0 ? kx : (w == 1 ? ky : kz), qv[0][e]);
      }
    }
    __syncthreads();  // the previous field's last LDS reads are done
    fft<T, L, +1>(v, lds, t, idx, tw);
    if (active) {
#pragma unroll
      for (int e = 0; e < E; ++e) st_s(&ws.p[out0 + w][col + (long long)(t + e * TPC) * estride], v[e]);
    }
  }
}

// One work field of a substage formed from one or two state fields (the spectral prologue,
// calcOmega*Kernel_mgpu solver.cu:68-114, gradientKernel_mgpu solver.cu:233-256, the colloid's
// c and lap Z, solver.cu:419-437):  kind 0: A;  1: i k_da A;  2: i (k_da A - k_db B);  3: -k^2 A.
// Axis d picks kx (per row of the x column), ky (per tile) or kz (per lane).
struct XOp {
  int kind, da, db;
};
template <typename T> struct XOpList {
  cx<T>* out[MAXW];
  const cx<T>* A[MAXW];
  const cx<T>* B[MAXW];
  XOp op[MAXW];
};

// Inverse x passes of work fields with their prologue folded into the loads: persistent and
// software-pipelined like k_col_multi (the next tile's inputs are loaded before the current tile
// transforms); tile i is tile i % tpf of list entry i / tpf.  TWO: the two-input operation
// (kind 2); otherwise only A is read.  Inputs and output share the spectral layout, so a column of A (and B) sits at the
// output column's offset; only kept kx rows are read, every row is written.
template <typename T, int L, int C, bool TWO>
__global__ void __launch_bounds__(lb_threads(C * (L / Plan<L>::E)))
k_xinv_op_pipe(XOpList<T> li, const T* __restrict__ kxv, const T* __restrict__ kyv,
               const T* __restrict__ kzv, const cx<T>* __restrict__ tw, ColArgs a, int tpf, int ntiles) {
  constexpr int E = Plan<L>::E;
  constexpr int TPC = L / E;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int c = tid % C;
  const int t = (tid / C) % TPC;
  const int g = C * TPC >= 256 ? 0 : tid / (C * TPC);  // one group per block from 256 threads on
  auto offset_of = [&](int tile, TileRows& r, int& iy, int& iz) {
    const int lt = tile % tpf;
    const int chunk = lt % a.nchunks;
    const int o = (lt / a.nchunks) * a.G + g;
    const bool active = o < a.nouter;
    iy = outer_index(active ? o : 0, a.outer_keep, a.outer_n);
    iz = chunk * C + c;
    r = tile_rows(a.sph, iy, a.outer_n, chunk * C, a.in_keep);
    r.live = r.live && active;
    return (long long)iy * a.ostride + iz;
  };
  auto live_from = [&](int tile) {
    if (a.G == 1 && a.sph.axis == 0) {
      TileRows r;
      int iy, iz;
      for (; tile < ntiles; tile += gridDim.x) {
        (void)offset_of(tile, r, iy, iz);
        if (r.live) break;
      }
    }
    return tile;
  };
  // A is loaded one tile ahead; B (two-input operation) when the tile is formed, which keeps the
  // register footprint of a 16-column tile without spills
  auto load_col = [&](bool second, int tile, cx<T>* va) {
    const cx<T>* __restrict__ src = second ? li.B[tile / tpf] : li.A[tile / tpf];
    TileRows r;
    int iy, iz;
    const long long off = offset_of(tile, r, iy, iz);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = t + e * TPC;
      const bool ld = r.live && iz < a.cols && row_kept(p, L, r.keep);
      va[e] = ld ? ld_s(&src[off + (long long)p * a.estride]) : mk<T>(0, 0);
    }
  };
  auto form = [&](int tile, const cx<T>* va, cx<T>* v) {
    TileRows r;
    int iy, iz;
    (void)offset_of(tile, r, iy, iz);
    const T ky = kyv[iy], kz = kzv[iz];
    const XOp op = li.op[tile / tpf];
    cx<T> vb[TWO ? E : 1];
    if (TWO) load_col(true, tile, vb);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const T kx = kxv[t + e * TPC];
      const T ka = op.da == 0 ? kx : (op.da == 1 ? ky : kz);
      const T kb = op.db == 0 ? kx : (op.db == 1 ? ky : kz);
      if (TWO) v[e] = csub(ik(ka, va[e]), ik(kb, vb[TWO ? e : 0]));
      else if (op.kind == 0) v[e] = va[e];
      else if (op.kind == 1) v[e] = ik(ka, va[e]);
      else {
        const T k2 = kx * kx + ky * ky + kz * kz;
        v[e] = mk<T>(-k2 * va[e].x, -k2 * va[e].y);
      }
    }
  };
  int tile = live_from(blockIdx.x);
  if (tile >= ntiles) return;
  cx<T> va[E], v[E];
  load_col(false, tile, va);
  const LdsCol idx{g * L * C + c, C};
  while (true) {
    form(tile, va, v);
    const int next = live_from(tile + gridDim.x);
    const bool more = next < ntiles;
    if (more) load_col(false, next, va);
    fft<T, L, +1>(v, lds, t, idx, tw);
    TileRows r;
    int iy, iz;
    const long long off = offset_of(tile, r, iy, iz);
    if (r.live && iz < a.cols) {
      cx<T>* __restrict__ out = li.out[tile / tpf];
#pragma unroll
      for (int e = 0; e < E; ++e) st_s(&out[off + (long long)(t + e * TPC) * a.estride], v[e]);
    }
    if (!more) break;
    tile = next;
  }
}

// Inverse strided passes with the derivatives along the transformed axis applied on the way in
// (the late-derivative x mode): list entry i reads one or two input fields A, B and writes one to
// three transformed outputs out_j = (a_j + i b_j k) A + c_j B, or - d_j k^2 A + c_j B where d_j is not 0, with
// a_j .. d_j in {-1, 0, 1}, k the wavenumber of the element's mode along the axis.  The x pass reads the state
// once per field (u, v, w, phi) and writes it with its x-derivatives; the y pass adds the
// y-derivatives and omega_z = v_x - i k_y u; the fused z pass forms the remaining terms with
// i k_z (replaces the spectral prologue of the reference's computeRHS, solver.cu:419-437, and the
// curl/gradient kernels it calls).
struct PairOp {
  int nout;
  float a[3], b[3], c[3], d[3];
};
template <typename T> struct PairList {
  const cx<T>* A[MAXW];
  const cx<T>* B[MAXW];
  cx<T>* out[3][MAXW];
  PairOp op[MAXW];
};

// Bit e set: every row p of slab e (p in [e TPC, (e + 1) TPC), the rows a thread's element e takes
// in a length-L transform of TPC threads per column) has |mode| > L / 3, a row the 2/3 rule removes.
constexpr unsigned removed_slabs(int L, int TPC, int E) {
  unsigned m = 0;
  for (int e = 0; e < E; ++e) {
    bool all = true;
    for (int p = e * TPC; p < (e + 1) * TPC && all; ++p) {
      const int md = p < (L >> 1) ? p : p - L;
      all = (md < 0 ? -md : md) > L / 3;
    }
    if (all) m |= 1u << e;
  }
  return m;
}

// One block per tile, over the entries of a whole pass: tile i is tile i % tpf of list entry i / tpf, entries
// of one or two inputs and one to three outputs together (the branches are uniform over the block), so a pass is one
// launch.  The outputs go through the radix stages one after the other in one LDS region, each from a
// load of its own: the inputs stay in the L2, and a block keeps one set of values, which leaves room
// for two blocks per CU whose transforms and memory phases overlap.  (As one persistent block per CU
// that loaded the next tile ahead, its barriers put every wave into the same phase: 512^3 FP32 x 525 and
// y 998 us per substage, now 431 and 959; FP64 992 -> 741 and 2030 -> 1800; 256^3 FP64 163 -> 119 and
// 334 -> 276.)  Columns of removed modes end at once and only rows inside the ellipsoid are loaded.
// The twiddles and the axis' wavenumbers are read from copies in LDS, after the data regions.  An entry
// may write its outputs over its own inputs (the block that owns a tile writes output 0 last, over input
// A, and the last output, the only one to take B, over B); no entry may read a field another entry writes.
template <typename T, int L, int C>
__global__ void __launch_bounds__(lb_threads(C * (L / ColPlan<T, L>::E)), (col_waves<T, L, C>()))
k_inv_late(PairList<T> li, const T* __restrict__ kv, const cx<T>* __restrict__ tw, ColArgs a, int tpf) {
  using P = ColPlan<T, L>;
  constexpr int E = P::E;
  constexpr int TPC = L / E;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int c = tid % C;
  const int t = (tid / C) % TPC;
  const int g = C * TPC >= 256 ? 0 : tid / (C * TPC);  // one group per block from 256 threads on
  auto tile_off = [&](int tile, TileRows& r) {
    const int lt = tile % tpf;
    const int chunk = lt % a.nchunks;
    const int o = (lt / a.nchunks) * a.G + g;
    const bool active = o < a.nouter;
    int om = active ? o : 0;
    const long long mo = member_split(om, a.nouter_m, a.mstride);
    const int io = outer_index(om, a.outer_keep, a.outer_n);
    r = tile_rows(a.sph, io, a.outer_n, chunk * C, a.in_keep);
    r.live = r.live && active;
    return mo + (long long)io * a.ostride + chunk * C;
  };
  const unsigned lane_b = (unsigned)(c + (long long)t * a.estride) * (unsigned)sizeof(cx<T>);
  constexpr unsigned ZS = removed_slabs(L, TPC, E);
  const LdsCol idx{g * L * C + c, C};
  cx<T>* twl = lds + (long long)a.G * L * C;
  T* kl = reinterpret_cast<T*>(twl + L);
  const int ent = blockIdx.x / tpf;
  TileRows r;
  const long long off = tile_off(blockIdx.x, r);
  if (a.G == 1 && !r.live) return;
  r.live = r.live && (int)(blockIdx.x % tpf % a.nchunks) * C + c < a.cols;
  for (int i = tid; i < L; i += blockDim.x) {
    twl[i] = tw[i];
    kl[i] = kv[i];
  }
  auto load = [&](const cx<T>* __restrict__ src, cx<T>* v) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      v[e] = (!((ZS >> e) & 1u) && r.live && row_kept(t + e * TPC, L, r.keep))
                 ? ld_at(src + off + (long long)e * TPC * a.estride, lane_b)
                 : mk<T>(0, 0);
  };
  // the last output first: the first may be written over the inputs
#pragma unroll 1
  for (int j = li.op[ent].nout - 1; j >= 0; --j) {
    const PairOp* op = &li.op[ent];
    const T ra = (T)op->a[j], ba = (T)op->b[j], rb = (T)op->c[j], da = (T)op->d[j];
    cx<T> v[1][E];
    load(li.A[ent], v[0]);
    __syncthreads();  // the copies are there, and the LDS of the last transform is free
    if (da != (T)0) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const T k = kl[t + e * TPC], k2 = -da * k * k;
        v[0][e] = mk<T>(k2 * v[0][e].x, k2 * v[0][e].y);
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const T ka = ba * kl[t + e * TPC];
        v[0][e] = mk<T>(ra * v[0][e].x - ka * v[0][e].y, ra * v[0][e].y + ka * v[0][e].x);
      }
    }
    if (rb != (T)0) {
      cx<T> vb[E];
      load(li.B[ent], vb);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        v[0][e].x += rb * vb[e].x;
        v[0][e].y += rb * vb[e].y;
      }
    }
    fft_batch<T, L, +1, LdsCol, P, false, 1, L * C>(v, lds, t, idx, twl);
    if (r.live) {
      cx<T>* __restrict__ dst = li.out[j][ent];
#pragma unroll
      for (int e = 0; e < E; ++e) st_at(dst + off + (long long)e * TPC * a.estride, lane_b, v[0][e]);
    }
  }
}

// The velocity group of the fused forward x pass parks its projected right-hand sides in LDS
// (one slot per thread, field and element of a slab the 2/3 rule keeps) when they fit beside the
// twiddles and the x wavenumbers: its registers are then free to load the state of several
// elements before any store.
// Entries of that region for blocks of `threads` threads (0: the sides stay in registers).
template <typename T, int L, int C, bool VEL> __host__ __device__ constexpr long long xfwd_rhs_entries(int threads) {
  constexpr int E = Plan<L>::E, TPC = L / E;
  constexpr int NK = E - __builtin_popcount(removed_slabs(L, TPC, E));
  constexpr long long most = (long long)NK * 3 * lb_threads(C * TPC) * (long long)sizeof(cx<T>) +
                             L * (long long)(sizeof(cx<T>) + sizeof(T));
  return (VEL && most <= 160 * 1024) ? (long long)NK * 3 * threads : 0;
}

// Forward x pass of one field group's nonlinear terms fused with the projection (velocity),
// the sign of the scalar term (computeRHSKernel_mgpu solver.cu:461-521), the mask and the RK3-IF
// update of the state (replaces solver.cu:547-657): the transformed nonlinear terms never return
// to HBM.
template <typename T, int L, int C, bool VEL>
__global__ void __launch_bounds__(lb_threads(C * (L / Plan<L>::E)))
k_xfwd_rk(Geom g, CPtrs<T> q, CPtrs<T> dq, CPtrs<T> nl, const T* __restrict__ kxv,
          const T* __restrict__ kyv, const T* __restrict__ kzv, const cx<T>* __restrict__ tw, RkCoef rc,
          Sphere sph, int scalar, int nchunks, int G) {
  constexpr int NF = VEL ? 3 : 1;
  constexpr int E = Plan<L>::E;
  constexpr int TPC = L / E;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tid = threadIdx.x;
  const int c = tid % C;
  const int t = (tid / C) % TPC;
  const int gg = C * TPC >= 256 ? 0 : tid / (C * TPC);  // one group per block from 256 threads on
  const int chunk = blockIdx.x % nchunks;
  const int o = (blockIdx.x / nchunks) * G + gg;
  const int nouter = 2 * g.keep_y + 1;
  const int iy = outer_index(o < nouter ? o : 0, g.keep_y, g.ny);
  // a column of removed modes has no right-hand side, and its state is zero already
  const bool active = o < nouter && tile_rows(sph, iy, g.ny, chunk * C, g.keep_x).live;
  if (G == 1 && !active) return;
  const int iz = chunk * C + c;
  const long long estride = (long long)g.ny * g.kzs;
  // element (row p = t + e TPC, column c) at at(e) (wave-uniform with one group per block) plus the
  // lane's c + t estride, which the host keeps below 2^32 bytes
  const long long base = (long long)iy * g.kzs + chunk * C;
  auto at = [&](int e) { return base + (long long)e * TPC * estride; };
  const unsigned lane_b = (unsigned)(c + (long long)t * estride) * (unsigned)sizeof(cx<T>);
  const LdsCol idx{gg * L * C + c, C};
  const int f0 = VEL ? 0 : 3 + scalar;
  // every field's loads are issued before the first transform (the registers hold all NF fields
  // after the transforms anyway), so the later fields arrive while the earlier ones transform; the
  // twiddles are read from a copy in LDS after the G L C data entries (read from memory, each radix
  // stage would wait for all of those loads)
  cx<T> nv[NF][E];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int e = 0; e < E; ++e)
      nv[f][e] = active && iz <= g.keep_z ? ld_at(nl.p[f0 + f] + at(e), lane_b) : mk<T>(0, 0);
  // The x wavenumbers are read from a copy in LDS after the twiddles: loaded from memory per element
  // inside the projection and the update, each was one more wait, and after the first stores a wait
  // for every store in flight as well.
  const T ky = kyv[iy], kz = kzv[iz];
  const long long rhs_n = xfwd_rhs_entries<T, L, C, VEL>(blockDim.x);
  cx<T>* tws = lds + ((long long)G * L * C > rhs_n ? (long long)G * L * C : rhs_n);
  T* kxl = reinterpret_cast<T*>(tws + L);
  for (int i = tid; i < L; i += blockDim.x) {
    tws[i] = tw[i];
    kxl[i] = kxv[i];
  }
  __syncthreads();
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    if (f > 0) __syncthreads();
    fft<T, L, -1>(nv[f], lds, t, idx, (const cx<T>*)tws);
  }
  if (!active) return;
  const int my = mode_of(iy, g.ny), mz = mode_of(iz, g.nz);
  const T a = (T)rc.a, bb = (T)rc.b, dt = (T)rc.dt;
  const T nu = (T)rc.nu[f0];
  // right-hand side of element e: the projected nonlinear term (velocity) or its negative (scalar)
  auto rhs_of = [&](int e, cx<T>* rhs) {
    const T kx = kxl[t + e * TPC];
    const T k2 = kx * kx + ky * ky + kz * kz;
    if (k2 == (T)0) {
#pragma unroll
      for (int f = 0; f < NF; ++f) rhs[f] = mk<T>(0, 0);
    } else if (VEL) {
      const cx<T> n0 = nv[0][e], n1 = nv[NF > 1 ? 1 : 0][e], n2 = nv[NF - 1][e];
      cx<T> kn;
      kn.x = (kx * n0.x + ky * n1.x + kz * n2.x) / k2;
      kn.y = (kx * n0.y + ky * n1.y + kz * n2.y) / k2;
      rhs[0] = csub(n0, cscale(kn, kx));
      if (NF > 1) {
        rhs[NF > 1 ? 1 : 0] = csub(n1, cscale(kn, ky));
        rhs[NF - 1] = csub(n2, cscale(kn, kz));
      }
    } else {
      rhs[0] = mk<T>(-nv[0][e].x, -nv[0][e].y);
    }
  };
  // Slabs of rows the 2/3 rule removes are neither read nor written (the host checks keep_x = L / 3).
  constexpr unsigned ZS = removed_slabs(L, TPC, E);
  constexpr bool RL = xfwd_rhs_entries<T, L, C, VEL>(1) > 0;
  // slot of (kept slab e, field f) in the LDS region of the right-hand sides: thread-private, so no
  // barrier (every thread has read its last exchange of the transforms, which end in one)
  auto slot = [&](int e, int f) {
    const int ek = e - __builtin_popcount(ZS & ((1u << e) - 1u));
    return lds + ((long long)(ek * NF + f) * blockDim.x + tid);
  };
  if constexpr (RL) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if ((ZS >> e) & 1u) continue;
      cx<T> rhs[NF];
      rhs_of(e, rhs);
#pragma unroll
      for (int f = 0; f < NF; ++f) *slot(e, f) = rhs[f];
    }
  }
  // The state and RK-register values of EB elements are loaded before any of them is stored: the
  // stores may alias the loads as far as the compiler knows, so it keeps them in program order,
  // and loading per element and field would cost one HBM round trip each.  A velocity group whose
  // right-hand sides stay in registers has no room to load ahead (its loads go field by field).
  constexpr bool PRE = !VEL || RL;
  constexpr int EB = PRE ? (E / 2 < 4 ? E / 2 : 4) : 1;
  static_assert(E % EB == 0, "element batches must divide the elements of a thread");
#pragma unroll
  for (int e0 = 0; e0 < E; e0 += EB) {
    cx<T> oq[EB][NF], od[EB][NF];
#pragma unroll
    for (int j = 0; j < EB && PRE; ++j) {
      const int p = t + (e0 + j) * TPC;
      const long long o2 = at(e0 + j);
      const bool live = !((ZS >> (e0 + j)) & 1u) && iz < g.nzh && kept(g, mode_of(p, g.nx), my, mz);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        od[j][f] = (live && !rc.first) ? ld_at(dq.p[f0 + f] + o2, lane_b) : mk<T>(0, 0);
        oq[j][f] = live ? ld_at(q.p[f0 + f] + o2, lane_b) : mk<T>(0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int e = e0 + j;
      const int p = t + e * TPC;
      // removed modes: the state holds zeros there (the step starts from a dealiased one)
      if (((ZS >> e) & 1u) || iz >= g.nzh || !kept(g, mode_of(p, g.nx), my, mz)) continue;
      const long long o2 = at(e);
      const T kx = kxl[p];
      const T k2 = kx * kx + ky * ky + kz * kz;
      cx<T> rhs[NF];
      if constexpr (RL) {
#pragma unroll
        for (int f = 0; f < NF; ++f) rhs[f] = *slot(e, f);
      } else {
        rhs_of(e, rhs);
      }
      const T eps = -dexpm1<T>(-nu * k2 * (T)rc.tau);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        cx<T> d = cscale(rhs[f], dt);
        if (!rc.first) {
          const cx<T> old = PRE ? od[j][f] : ld_at(dq.p[f0 + f] + o2, lane_b);
          d.x = a * old.x + d.x;
          d.y = a * old.y + d.y;
        }
        cx<T> qq = PRE ? oq[j][f] : ld_at(q.p[f0 + f] + o2, lane_b);
        qq.x = if_update(qq.x, bb, d.x, eps);
        qq.y = if_update(qq.y, bb, d.y, eps);
        st_at(q.p[f0 + f] + o2, lane_b, qq);
        if (!rc.last) st_at(dq.p[f0 + f] + o2, lane_b, mk<T>(apply_if(d.x, eps), apply_if(d.y, eps)));
      }
    }
  }
}

// Sums of the per-plane partials in plane order, a thread per result: fin[q] = sum over x of
// part[x][q] (q < SPEC_NQ); fin[SPEC_NQ], fin[SPEC_NQ + 1] = max over y of the CFL sum and of max |u_i|;
// fin[SPEC_NQ + 2 + j] = sum over x of spec[x][j] (j < nspec shell entries).  Eight loads go out
// ahead of their additions (a serial chain of loads cost 1 us each).
static __global__ void __launch_bounds__(64)
k_stats_reduce(const double* __restrict__ part, const double* __restrict__ spec, const double* __restrict__ cmax,
               int nx, int ny, int nspec, double* __restrict__ fin) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= SPEC_NQ + 2 + nspec) return;
  const bool mx = t == SPEC_NQ || t == SPEC_NQ + 1;
  const double* src = t < SPEC_NQ ? part + t : (mx ? cmax + (t - SPEC_NQ) : spec + (t - SPEC_NQ - 2));
  const long long stride = t < SPEC_NQ ? SPEC_NQ : (mx ? 2 : nspec);
  const int n = mx ? ny : nx;  // multiples of 8
  double acc = 0.0;
  for (int i = 0; i < n; i += 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = src[(i + k) * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc = mx ? fmax(acc, v[k]) : acc + v[k];
  }
  fin[t] = acc;
}

// Rows of a spectral field from row r0 on, in the ABI's order (row ky nx + kx, kz < nzh), to or from
// host memory (pinned); unpacking also clears the kz padding.  Bound by the bus.
template <typename T>
__global__ void __launch_bounds__(256) k_spec_pack(const cx<T>* __restrict__ q, cx<T>* __restrict__ host, int nx, int ny,
                                                   int nzh, int kzs, long long r0, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const long long r = i / nzh;
    const int k = (int)(i - r * nzh), x = (int)((r0 + r) % nx), y = (int)((r0 + r) / nx);
    host[i] = q[((long long)x * ny + y) * kzs + k];
  }
}
template <typename T>
__global__ void __launch_bounds__(256) k_spec_unpack(const cx<T>* __restrict__ host, cx<T>* __restrict__ q, int nx,
                                                     int ny, int nzh, int kzs, long long r0, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const long long r = i / kzs;
    const int k = (int)(i - r * kzs), x = (int)((r0 + r) % nx), y = (int)((r0 + r) / nx);
    q[((long long)x * ny + y) * kzs + k] = k < nzh ? host[r * nzh + k] : mk<T>(0, 0);
  }
}
// Contiguous values to or from host memory, four per thread and step (nz is a multiple of 8).
template <typename T>
__global__ void __launch_bounds__(256) k_real_copy(const T* __restrict__ in, T* __restrict__ out, long long n4) {
  typedef T vec __attribute__((ext_vector_type(4)));
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x)
    reinterpret_cast<vec*>(out)[i] = reinterpret_cast<const vec*>(in)[i];
}

// Plain copy (bandwidth reference): block b copies the contiguous chunk [b chunk, (b + 1) chunk)
// of 16-byte elements with four nontemporal loads in flight per thread before the stores.  Of the
// copy forms measured on MI355X (grid-stride or chunked, 2-8 loads in flight, cached or
// nontemporal) this one moves the most bytes per second.
typedef float v4f __attribute__((ext_vector_type(4)));
static __global__ void __launch_bounds__(256) k_copy16(const v4f* __restrict__ in, v4f* __restrict__ out,
                                                       long long n, long long chunk) {
  const long long beg = (long long)blockIdx.x * chunk;
  const long long end = beg + chunk < n ? beg + chunk : n;
  long long i = beg + threadIdx.x;
  for (; i + 3 * 256 < end; i += 4 * 256) {
    v4f a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = __builtin_nontemporal_load(&in[i + u * 256]);
#pragma unroll
    for (int u = 0; u < 4; ++u) __builtin_nontemporal_store(a[u], &out[i + u * 256]);
  }
  for (; i < end; i += 256) __builtin_nontemporal_store(__builtin_nontemporal_load(&in[i]), &out[i]);
}

// ---------------------------------------------------------------------------------------------
// Diagnostics
// ---------------------------------------------------------------------------------------------

// omega^ = i k x u^ (calcOmega*Kernel_mgpu, solver.cu:68-114) over a box of modes: the whole array, whose
// kz padding is written as zero, or the kept box of a dealiased state.
template <typename T>
__global__ void k_vorticity(Geom g, Box b, CPtrs<T> q, CPtrs<T> w, const T* __restrict__ kxv,
                            const T* __restrict__ kyv, const T* __restrict__ kzv, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int ix, iy, iz;
  box_index(g, b, i, ix, iy, iz);
  const long long o = ((long long)ix * g.ny + iy) * g.kzs + iz;
  if (iz >= g.nzh) {
    for (int c = 0; c < 3; ++c) w.p[c][o] = mk<T>(0, 0);
    return;
  }
  const T kx = kxv[ix], ky = kyv[iy], kz = kzv[iz];
  const cx<T> u = q.p[0][o], v = q.p[1][o], ww = q.p[2][o];
  w.p[0][o] = csub(ik(ky, ww), ik(kz, v));
  w.p[1][o] = csub(ik(kz, u), ik(kx, ww));
  w.p[2][o] = csub(ik(kx, v), ik(ky, u));
}

// One physical plane of [x][y][z]: axis 2 (z = index) -> [x][y], axis 1 -> [x][z],
// axis 0 -> [y][z] (writexyfields / writexzfields / writeyzfields, iofuncs.cu:187-260).
template <typename T>
__global__ void k_plane(const T* __restrict__ a, T* __restrict__ out, int nx, int ny, int nz, int axis,
                        int index) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long src;
  if (axis == 2) {
    if (i >= (long long)nx * ny) return;
    src = i * nz + index;
  } else if (axis == 1) {
    if (i >= (long long)nx * nz) return;
    src = ((i / nz) * ny + index) * nz + i % nz;
  } else {
    if (i >= (long long)ny * nz) return;
    src = (long long)index * ny * nz + i;
  }
  out[i] = a[src];
}

// A plane of a field at one index of an axis is linear in the spectrum: summed over that axis' modes
// first, what is left to transform is a plane.  The sums are taken in FP64 (twiddles from the passes' tables)
// and read the state once, or its kept modes only (kept != 0: a dealiased state).

// z = index: h[kx][ky][0] = sum over kz, weighted so that the real part of the plane's transform is the field
// (2 for the modes whose conjugates the half spectrum leaves out); columns 1 to 7 are zeros (a column tile).  A
// row is summed by the 8 lanes that write its columns: 64 bytes a load in FP32, and the table index goes round by
// addition (a wave per row and a remainder per mode: 25 us at 256x384x192 FP32, now 12).
constexpr int PLANE_COLS = 8;
template <typename T>
__global__ void __launch_bounds__(256) k_sum_z(Geom g, const cx<T>* __restrict__ q, cx<T>* __restrict__ h,
                                               const cx<T>* __restrict__ tw, int index, int kept_only, int nkz) {
  const int lane = threadIdx.x % PLANE_COLS;
  const long long r = (long long)blockIdx.x * (256 / PLANE_COLS) + threadIdx.x / PLANE_COLS;
  if (r >= (long long)g.nx * g.ny) return;
  const int ix = (int)(r / g.ny), iy = (int)(r % g.ny);
  double re = 0.0, im = 0.0;
  if (!kept_only || kept(g, mode_of(ix, g.nx), mode_of(iy, g.ny), 0)) {
    const cx<T>* row = q + r * g.kzs;
    int at = (int)((unsigned)(lane * index) % (unsigned)g.nz);
    const int by = (int)((unsigned)(PLANE_COLS * index) % (unsigned)g.nz);
#pragma unroll 4
    for (int k = lane; k < nkz; k += PLANE_COLS) {
      const cx<T> f = row[k], w = tw[at];
      const double s = (k == 0 || 2 * k == g.nz) ? 1.0 : 2.0;
      re += s * ((double)f.x * w.x + (double)f.y * w.y);
      im += s * ((double)f.y * w.x - (double)f.x * w.y);
      at += by;
      at -= at >= g.nz ? g.nz : 0;
    }
#pragma unroll
    for (int d = PLANE_COLS / 2; d > 0; d >>= 1) {
      re += __shfl_xor(re, d, PLANE_COLS);
      im += __shfl_xor(im, d, PLANE_COLS);
    }
  }
  h[r * PLANE_COLS + lane] = lane == 0 ? mk<T>((T)re, (T)im) : mk<T>(0, 0);
}

// y = index (AXIS 1: a runs over kx, the sum over ky) or x = index (AXIS 0: a over ky, the sum over kx):
// h[a][kz], zeros from kz = nkz on.  A thread per (a, kz), keep: the sum's largest kept |mode|, or -1.
template <typename T, int AXIS>
__global__ void __launch_bounds__(256) k_sum_xy(Geom g, const cx<T>* __restrict__ q, cx<T>* __restrict__ h,
                                                const cx<T>* __restrict__ tw, int index, int keep, int nkz) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int na = AXIS ? g.nx : g.ny, n = AXIS ? g.ny : g.nx;
  if (i >= (long long)na * g.kzs) return;
  const int a = (int)(i / g.kzs), k = (int)(i % g.kzs);
  double re = 0.0, im = 0.0;
  if (k < nkz) {
    const int nm = keep < 0 ? n : 2 * keep + 1;
    // the modes in order from 0, or from -keep: the table index goes round by addition
    int m = keep < 0 ? 0 : n - keep, at = (int)((unsigned)(m * index) % (unsigned)n);
    if (keep == 0) m = 0;
#pragma unroll 4
    for (int o = 0; o < nm; ++o) {
      const long long row = AXIS ? (long long)a * g.ny + m : (long long)m * g.ny + a;
      const cx<T> f = q[row * g.kzs + k], w = tw[at];
      m = m + 1 == n ? 0 : m + 1;
      at += index;
      at -= at >= n ? n : 0;
      re += (double)f.x * w.x + (double)f.y * w.y;
      im += (double)f.y * w.x - (double)f.x * w.y;
    }
  }
  h[i] = mk<T>((T)re, (T)im);
}

// The real parts of column 0 of a z plane, from point i0 on, times `scale`, to (pinned host) memory.
template <typename T>
__global__ void __launch_bounds__(256) k_plane_out(const cx<T>* __restrict__ h, T* __restrict__ out, long long i0,
                                                   long long n, T scale) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = h[(i0 + i) * PLANE_COLS].x * scale;
}

// Iso-surface area by the indicator gradient (surfaceArea_kernel_mgpu, statistics.cu:1310-1460):
// per grid point -(grad F . grad chi) / |grad F| with chi = (F <= iso), central differences on the
// periodic grid; AREA_SPLIT blocks per x plane, each with every AREA_SPLIT-th group of rows, fixed per-thread
// order and tree -> part[x AREA_SPLIT + block] (FP64).  A thread takes 16 bytes of z; away from the surface
// the indicator has no gradient and nothing but the comparisons is computed.  Bound by reading F.
constexpr int AREA_SPLIT = 4;
constexpr int AREA_THREADS = 512;
template <typename T>
__global__ void __launch_bounds__(AREA_THREADS)
k_surface_area(Geom g, const T* __restrict__ F, double iso, double dx, double dy, double dz,
               double* __restrict__ part) {
  constexpr int V = 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(V)));
  __shared__ double sh[AREA_THREADS / 64];
  const int x = blockIdx.x;
  const int xm = x == 0 ? g.nx - 1 : x - 1, xp = x == g.nx - 1 ? 0 : x + 1;
  const int nv = g.nz / V, n = g.ny * nv;
  const vec* __restrict__ Fv = reinterpret_cast<const vec*>(F);
  double acc = 0.0;
  for (int i = blockIdx.y * AREA_THREADS + threadIdx.x; i < n; i += AREA_SPLIT * AREA_THREADS) {
    const int y = i / nv, zv = i - y * nv;
    const int ym = y == 0 ? g.ny - 1 : y - 1, yp = y == g.ny - 1 ? 0 : y + 1;
    auto at = [&](int a, int b) { return ((long long)a * g.ny + b) * nv + zv; };
    const vec c = Fv[at(x, y)], vxm = Fv[at(xm, y)], vxp = Fv[at(xp, y)], vym = Fv[at(x, ym)], vyp = Fv[at(x, yp)];
    const long long row = ((long long)x * g.ny + y) * g.nz;
    const T before = F[row + (zv == 0 ? g.nz - 1 : zv * V - 1)], after = F[row + (zv == nv - 1 ? 0 : zv * V + V)];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const double fxm = vxm[j], fxp = vxp[j], fym = vym[j], fyp = vyp[j];
      const double fzm = j == 0 ? (double)before : (double)c[j > 0 ? j - 1 : 0];
      const double fzp = j == V - 1 ? (double)after : (double)c[j < V - 1 ? j + 1 : 0];
      const int ix = (int)(fxp <= iso) - (int)(fxm <= iso), iy = (int)(fyp <= iso) - (int)(fym <= iso);
      const int iz = (int)(fzp <= iso) - (int)(fzm <= iso);
      if (ix == 0 && iy == 0 && iz == 0) continue;
      const double gx = (fxp - fxm) / (2.0 * dx), gy = (fyp - fym) / (2.0 * dy), gz = (fzp - fzm) / (2.0 * dz);
      if (gx == 0 && gy == 0 && gz == 0) continue;
      const double cxv = (double)ix / (2.0 * dx), cyv = (double)iy / (2.0 * dy), czv = (double)iz / (2.0 * dz);
      acc += -(gx * cxv + gy * cyv + gz * czv) / sqrt(gx * gx + gy * gy + gz * gz);
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) acc += __shfl_down(acc, d);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < AREA_THREADS / 64; ++w) t += sh[w];
    part[x * AREA_SPLIT + blockIdx.y] = t;
  }
}

}  // namespace gnss
