// clr_los.hip -- kappa_get_beam_properties (kappa.c:78-175) and
// isw_get_beam_properties (isw.c:78-147) on gfx950.
//
// One thread per HEALPix pixel (NEST order, so neighbouring lanes march
// neighbouring rays and their reads share cache lines), or several for small
// maps.  The march uses nr = N/2 radial steps of dr = r_max/nr
// (get_radial_params, common.c:333-337); at each step the NGP cell of
// (rm u + x_obs)/dx is read (interpolate_from_grid, beaming.c:120-268,
// periodic in x, y and z on one GPU).  kappa: transverse trace of the 19-point
// tidal tensor of phi (get_element, beaming.c:31-117) weighted by rm D (1+z)
// dr and rm^2 D (1+z) dr, cumulative over the source planes sorted by
// distance; ISW: phi weighted by 2 PD(rm) dr.  Accumulation in FP64.
// 1024^3, nside 512, three planes: kappa 8.87 ms (11.15 with FP64 cell
// indices, three loads per record and a block per row for the records), of
// which the records 4.4 (13.3 GB written) and the march 4.5 (bound by the
// records' fetch); ISW 2.11 ms (3.51), bound by its vector instructions.
#include "clr_internal.h"
#include <algorithm>
#include <limits.h>
#include <math.h>
#include <string.h>

using namespace clr;

namespace {

constexpr int kMaxPlanes = 100;   // NPLANES_MAX, common.h:133

struct LosArgs {
  const float *phi;
  const float2 *t6;       // k_records' tidal records, or null
  int N, ngx;
  double idx, dr, ox, oy, oz;
  int nr, nplanes, lg;    // 2^lg lanes per pixel
  int run;                // k_los_planes
  int mono;               // irmax does not decrease
  int irmax[kMaxPlanes];
  double inv_rmax[kMaxPlanes];
};

// The reference wraps once (beaming.c:129-133), which covers every cell the
// march and the source reads reach when r_max is below the box size; the
// full modulo keeps other inputs inside the grid.
__device__ inline int wrap1(int v, int N) {
  if (v >= N || v < 0) {
    v %= N;
    if (v < 0) v += N;
  }
  return v;
}

// The NGP cells of a march: step i reads cell (long)((rm u + x_obs) idx + 1/2)
// per axis, rm = (i + 1/2) dr, wrapped.  The position is kept in 32.32
// fixed point, base + i step, whose integer half is the cell; it is off by at
// most (i + 1) 2^-33 + 2^-40 of a cell, so where the fraction comes within
// 2^-20 of a cell edge (or the position is negative, where the reference
// truncates towards zero, or two boxes away) the FP64 expression decides: the same cells as it,
// for 2 + 2 integer operations per axis instead of 5 FP64 ones and 4 to wrap.
// Needs |x| < 2^30 cells and at most 2^12 steps.
struct Ray {
  double u[3];
  int64_t base[3], step[3];
};
__device__ inline void ray_setup(Ray &r, double dr, double idx, double ox, double oy, double oz) {
  const double o[3] = {ox, oy, oz};
#pragma unroll
  for (int ax = 0; ax < 3; ax++) {
    const double st = r.u[ax] * dr * idx;
    r.step[ax] = llrint(st * 4294967296.0);
    r.base[ax] = llrint((0.5 * st + o[ax] * idx + 0.5) * 4294967296.0);
  }
}
// The cell of step i, x = base + i step.
__device__ inline void ray_cell(const Ray &r, const int64_t x[3], int i, int N, double dr, double idx, double ox,
                                double oy, double oz, int c[3]) {
#pragma clang fp contract(off)
  constexpr uint32_t G = 1u << 12;   // 2^-20
  bool close = false;
#pragma unroll
  for (int ax = 0; ax < 3; ax++) {
    const uint32_t v = (uint32_t)(x[ax] >> 32);
    close = close || (uint32_t)x[ax] + G < 2 * G || v >= 2u * N;
    c[ax] = (int)min(v, v - N);
  }
  if (close) {
    const double rm = (i + 0.5) * dr;
    c[0] = wrap1((int)((rm * r.u[0] + ox) * idx + 0.5), N);
    c[1] = wrap1((int)((rm * r.u[1] + oy) * idx + 0.5), N);
    c[2] = wrap1((int)((rm * r.u[2] + oz) * idx + 0.5), N);
  }
}

// Second differences of phi at a cell (get_element, beaming.c:79-116), in FP32
// as the reference evaluates them on flouble values: xx, xy, xz, yy, yz, zz.
__device__ inline void tidal_at(const float *__restrict__ phi, int N, size_t ngx, size_t plane, const int c[3],
                                float t[6]) {
#pragma clang fp contract(off)
  const int xh = c[0] == N - 1 ? 0 : c[0] + 1, xl = c[0] == 0 ? N - 1 : c[0] - 1;
  const int yh = c[1] == N - 1 ? 0 : c[1] + 1, yl = c[1] == 0 ? N - 1 : c[1] - 1;
  const int zh = c[2] == N - 1 ? 0 : c[2] + 1, zl = c[2] == 0 ? N - 1 : c[2] - 1;
  const size_t Z0 = (size_t)c[2] * plane, ZH = (size_t)zh * plane, ZL = (size_t)zl * plane;
  const size_t Y0 = (size_t)c[1] * ngx, YH = (size_t)yh * ngx, YL = (size_t)yl * ngx;
  const int X0 = c[0];
  const float c0 = phi[X0 + Y0 + Z0];
  t[0] = phi[xh + Y0 + Z0] + phi[xl + Y0 + Z0] - 2 * c0;
  t[3] = phi[X0 + YH + Z0] + phi[X0 + YL + Z0] - 2 * c0;
  t[1] = 0.25f * (phi[xh + YH + Z0] + phi[xl + YL + Z0] - phi[xh + YL + Z0] - phi[xl + YH + Z0]);
  t[5] = phi[X0 + Y0 + ZH] + phi[X0 + Y0 + ZL] - 2 * c0;
  t[2] = 0.25f * (phi[xh + Y0 + ZH] + phi[xl + Y0 + ZL] - phi[xh + Y0 + ZL] - phi[xl + Y0 + ZH]);
  t[4] = 0.25f * (phi[X0 + YH + ZH] + phi[X0 + YL + ZL] - phi[X0 + YH + ZL] - phi[X0 + YL + ZH]);
}

template <int CTRL>
__device__ inline double dpp_get(double v) {
  const int l2 = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
  const int h2 = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(h2, l2);
}
// Sum over each group of 2^lg consecutive lanes (lg <= 4), in every one of them.
__device__ inline double lanes_add(double v, int lg) {
  if (lg > 0) v += dpp_get<0xB1>(v);    // quad_perm [1,0,3,2]
  if (lg > 1) v += dpp_get<0x4E>(v);    // quad_perm [2,3,0,1]
  if (lg > 2) v += dpp_get<0x141>(v);   // row_half_mirror
  if (lg > 3) v += dpp_get<0x140>(v);   // row_mirror
  return v;
}

// kappa (KAPPA) or ISW march: 2^lg consecutive lanes per pixel, each taking
// every 2^lg-th step (ONE: a lane per pixel, so that the step and its weights
// are the wavefront's), summed per source plane.  REC: the tidal records of
// k_records, one 24-byte read per step, instead of 19 stencil reads.
template <bool KAPPA, bool REC, bool ONE>
__global__ __launch_bounds__(256) void k_los(LosArgs a, const double *__restrict__ fac1,
                                             const double *__restrict__ fac2, int64_t nside, int64_t npix,
                                             float *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lg = ONE ? 0 : a.lg, sub = ONE ? 0 : (int)(t & ((1 << lg) - 1)), K = 1 << lg;
  const int64_t ip = t >> lg;
  if (ip >= npix) return;
  Ray ray;
  pix2vec_nest(nside, ip, ray.u);
  ray_setup(ray, a.dr, a.idx, a.ox, a.oy, a.oz);
  const int N = a.N;
  const size_t ngx = (size_t)a.ngx, plane = (size_t)N * ngx;
  const float *__restrict__ phi = a.phi;
  double rot[6];
  if (KAPPA) {
#pragma clang fp contract(off)
    double cth = ray.u[2];
    if (cth >= 1) cth = 1;
    if (cth <= -1) cth = -1;
    const double sth = sqrt((1 - cth) * (1 + cth));
    double cph = 1, sph = 0;
    if (sth != 0) { cph = ray.u[0] / sth; sph = ray.u[1] / sth; }
    const double pre = a.idx * a.idx;
    rot[0] = (cth * cth * cph * cph + sph * sph) * pre;
    rot[1] = (2 * cph * sph * (cth * cth - 1)) * pre;
    rot[2] = (-2 * cth * sth * cph) * pre;
    rot[3] = (cth * cth * sph * sph + cph * cph) * pre;
    rot[4] = (-2 * cth * sth * sph) * pre;
    rot[5] = (sth * sth) * pre;
  }
  double k1 = 0, k2 = 0;
  constexpr int U = KAPPA && !REC ? 1 : 4;   // steps in flight
  int i = sub;
  for (int pl = 0; pl < a.nplanes; pl++) {
    const int last = a.irmax[pl];
    int64_t x[3], kstep[3];
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
      x[ax] = ray.base[ax] + (int64_t)i * ray.step[ax];
      kstep[ax] = ray.step[ax] << lg;
    }
    for (; i <= last; i += U * K) {
      float tt[U][6];
#pragma unroll
      for (int u = 0; u < U; u++) {
        // (steps past the plane's last are read, not added)
        int c[3];
        ray_cell(ray, x, i + u * K, N, a.dr, a.idx, a.ox, a.oy, a.oz, c);
#pragma unroll
        for (int ax = 0; ax < 3; ax++) x[ax] += kstep[ax];
        if (!KAPPA) {
          tt[u][0] = phi[(size_t)c[2] * plane + (size_t)c[1] * ngx + c[0]];
        } else if (REC) {
          const float *r = (const float *)(a.t6 + (((size_t)c[2] * N + c[1]) * N + c[0]) * 3);
          __builtin_memcpy(tt[u], r, 16);
          __builtin_memcpy(tt[u] + 4, r + 4, 8);
        } else {
          tidal_at(phi, N, ngx, plane, c, tt[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int j = i + u * K;
        if (j > last) break;
        if (!KAPPA) {
          k1 = fma((double)tt[u][0], fac1[j], k1);
        } else {
          double dot = rot[0] * (double)tt[u][0];
#pragma unroll
          for (int q = 1; q < 6; q++) dot = fma(rot[q], (double)tt[u][q], dot);
          k1 = fma(dot, fac1[j], k1);
          k2 = fma(dot, fac2[j], k2);
        }
      }
    }
    // the next plane's first step of this lane
    if (i > last) i -= (i - last - 1) / K * K;
    double v = KAPPA ? k1 - a.inv_rmax[pl] * k2 : k1;
    for (int o = 1; o < K; o <<= 1) v += __shfl_xor(v, o);
    if (sub == 0) out[(size_t)pl * npix + ip] = (float)v;
  }
}

// The same march for many planes: the steps in flight run on across the planes'
// ends, and a plane's sum goes out when its last step has been added.  k_los
// starts anew at each plane, reading up to 4 rounds of steps past its end: with
// 100 planes ISW at 128^3, nside 64 took 175 us there and takes 26 here, kappa at
// 512^3, nside 64 505 and 423.  For few planes the plain loop is the faster one
// (kappa 371 and 409 us with one plane).
template <bool KAPPA, bool REC, bool ONE>
__global__ __launch_bounds__(256) void k_los_planes(LosArgs a, const double *__restrict__ fac1,
                                                    const double *__restrict__ fac2, int64_t nside, int64_t npix,
                                                    float *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lg = ONE ? 0 : a.lg, sub = ONE ? 0 : (int)(t & ((1 << lg) - 1)), K = 1 << lg;
  const int64_t ip = t >> lg;
  if (ip >= npix) return;
  Ray ray;
  pix2vec_nest(nside, ip, ray.u);
  ray_setup(ray, a.dr, a.idx, a.ox, a.oy, a.oz);
  const int N = a.N;
  const size_t ngx = (size_t)a.ngx, plane = (size_t)N * ngx;
  const float *__restrict__ phi = a.phi;
  double rot[6];
  if (KAPPA) {
#pragma clang fp contract(off)
    double cth = ray.u[2];
    if (cth >= 1) cth = 1;
    if (cth <= -1) cth = -1;
    const double sth = sqrt((1 - cth) * (1 + cth));
    double cph = 1, sph = 0;
    if (sth != 0) { cph = ray.u[0] / sth; sph = ray.u[1] / sth; }
    const double pre = a.idx * a.idx;
    rot[0] = (cth * cth * cph * cph + sph * sph) * pre;
    rot[1] = (2 * cph * sph * (cth * cth - 1)) * pre;
    rot[2] = (-2 * cth * sth * cph) * pre;
    rot[3] = (cth * cth * sph * sph + cph * cph) * pre;
    rot[4] = (-2 * cth * sth * sph) * pre;
    rot[5] = (sth * sth) * pre;
  }
  double k1 = 0, k2 = 0;
  constexpr int U = KAPPA && !REC ? 1 : 4;   // rounds of K steps in flight
  // the values of the U rounds from step i on (steps past the last are read, not added)
  auto read = [&](int i, int64_t x[3], const int64_t kstep[3], float tt[U][6]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      int c[3];
      ray_cell(ray, x, i + u * K, N, a.dr, a.idx, a.ox, a.oy, a.oz, c);
#pragma unroll
      for (int ax = 0; ax < 3; ax++) x[ax] += kstep[ax];
      if (!KAPPA) {
        tt[u][0] = phi[(size_t)c[2] * plane + (size_t)c[1] * ngx + c[0]];
      } else if (REC) {
        const float *r = (const float *)(a.t6 + (((size_t)c[2] * N + c[1]) * N + c[0]) * 3);
        __builtin_memcpy(tt[u], r, 16);
        __builtin_memcpy(tt[u] + 4, r + 4, 8);
      } else {
        tidal_at(phi, N, ngx, plane, c, tt[u]);
      }
    }
  };
  auto add = [&](const float t[6], int j, double &s1, double &s2) {
    if (!KAPPA) {
      s1 = fma((double)t[0], fac1[j], s1);
    } else {
      double dot = rot[0] * (double)t[0];
#pragma unroll
      for (int q = 1; q < 6; q++) dot = fma(rot[q], (double)t[q], dot);
      s1 = fma(dot, fac1[j], s1);
      s2 = fma(dot, fac2[j], s2);
    }
  };
  auto emit = [&](int pl, double s1, double s2) {
    double v = KAPPA ? s1 - a.inv_rmax[pl] * s2 : s1;
    if (!ONE) v = lanes_add(v, lg);
    if (sub == 0) out[(size_t)pl * npix + ip] = (float)v;
  };
  int pl = 0, first = 0, pend = a.irmax[0];   // the next plane, its first step and its last
  auto next = [&]() { if (++pl < a.nplanes) pend = a.irmax[pl]; };
  while (pl < a.nplanes) {
    if (pend < first) {   // no step of its own
      emit(pl, k1, k2);
      first = pend + 1;
      next();
      continue;
    }
    const int end = a.mono ? a.nplanes : pl + 1;   // these planes are one run of steps
    const int last = a.irmax[end - 1];
    int b = first >> lg << lg;   // the round's first step
    int64_t x[3], kstep[3];
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
      x[ax] = ray.base[ax] + (int64_t)(b + sub) * ray.step[ax];
      kstep[ax] = ray.step[ax] << lg;
    }
    for (; b <= last; b += U * K) {
      float tt[U][6];
      read(b + sub, x, kstep, tt);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int bu = b + u * K, j = bu + sub;
        if (bu > last) break;
        double n1 = k1, n2 = k2;   // the sums with step j
        if (ONE || (j >= first && j <= last)) add(tt[u], j, n1, n2);
        // planes that end before the next round: with the steps up to their last
        for (; pl < end && pend < bu + K; next()) {
          const bool in = j <= pend;
          emit(pl, in ? n1 : k1, in ? n2 : k2);
        }
        k1 = n1;
        k2 = n2;
      }
    }
    first = last + 1;
  }
}

// Per-cell records for the marches, for the cells within sqrt(r2lim) of the
// observer (no march reaches the others: the box corners are 42 % of the
// cube).  TID: the tidal records t6[cell][6], tidal_at's second differences;
// VEL: vrec[cell] = phi's unscaled central differences in FP32 (get_element,
// RETURN_VEL) and the density.  A block takes 64 x 4 cells and walks nzb
// planes of z: three planes of phi with their halo in LDS (the next one's
// loads in flight), so phi is read once (1.5 times with the halos; a block per
// row read it 7 times from L2), and the 24-byte records go through LDS so that
// consecutive lanes store consecutive float2.  Bound by the records' writes.
constexpr int kRecX = 64, kRecY = 4;
template <bool TID, bool VEL>
__global__ __launch_bounds__(256) void k_records(const float *__restrict__ phi, const float *__restrict__ dens, int N,
                                                 int ngx, int nzb, float dxf, float ox, float oy, float oz, float r2lim,
                                                 float2 *__restrict__ t6, float4 *__restrict__ vrec) {
#pragma clang fp contract(off)
  constexpr int LX = kRecX + 2, LY = kRecY + 2, LP = LX * LY;
  __shared__ float pl[3][LP];
  __shared__ float2 st[TID ? 256 * 3 : 1];
  __shared__ unsigned char ok[TID ? 256 : 1];
  const int x0 = blockIdx.x * kRecX, y0 = blockIdx.y * kRecY, zb = blockIdx.z * nzb;
  const int ze = min(zb + nzb, N);
  // the block's planes: those whose nearest cell is in reach (an interval)
  const float xa = x0 * dxf - ox, xb = (min(x0 + kRecX, N) - 1) * dxf - ox;
  const float ya = y0 * dxf - oy, yb = (y0 + kRecY - 1) * dxf - oy;
  // distances along an axis are periodic: a march or a CIC corner may wrap
  const float box = N * dxf;
  auto dist = [box](float x) { const float d = fabsf(x); return fminf(d, box - d); };
  auto nearest = [box](float lo, float hi) {
    return fmaxf(fminf(fmaxf(lo, -hi), box - fmaxf(-lo, hi)), 0.f);
  };
  const float xn = nearest(xa, xb), yn = nearest(ya, yb), rn = xn * xn + yn * yn;
  int z0 = zb, z1 = ze;
  auto far = [&](int z) { const float zc = dist(z * dxf - oz); return zc * zc + rn > r2lim; };
  while (z0 < z1 && far(z0)) z0++;
  while (z1 > z0 && far(z1 - 1)) z1--;
  if (z0 >= z1) return;
  const size_t plane = (size_t)N * ngx;
  // the thread's (up to two) places of a plane's LDS image and their rows
  size_t src[2];
  int dst[2];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int e = (int)threadIdx.x + 256 * k, cx = e % LX, cy = e / LX;
    int gx = x0 - 1 + cx, gy = y0 - 1 + cy;
    gx = gx < 0 ? gx + N : (gx >= N ? gx - N : gx);
    if (gx >= N) gx = 0;   // columns past a grid narrower than the tile: not used
    gy = gy < 0 ? gy + N : (gy >= N ? gy - N : gy);
    dst[k] = e < LP ? e : -1;
    src[k] = e < LP ? (size_t)gy * ngx + gx : 0;
  }
  auto fetch = [&](int z, float v[2]) {
    const int zw = z < 0 ? z + N : (z >= N ? z - N : z);
#pragma unroll
    for (int k = 0; k < 2; k++) v[k] = dst[k] >= 0 ? phi[(size_t)zw * plane + src[k]] : 0.f;
  };
  auto put = [&](int s, const float v[2]) {
#pragma unroll
    for (int k = 0; k < 2; k++)
      if (dst[k] >= 0) pl[s][dst[k]] = v[k];
  };
  float v[2];
  fetch(z0 - 1, v);
  put(0, v);
  fetch(z0, v);
  put(1, v);
  fetch(z0 + 1, v);
  const int lx = threadIdx.x % kRecX, ly = threadIdx.x / kRecX;
  const int ix = x0 + lx, iy = y0 + ly, o = (ly + 1) * LX + lx + 1;
  const float xc = dist(ix * dxf - ox), yc = dist(iy * dxf - oy), rho2 = xc * xc + yc * yc;
  for (int z = z0, s = 0; z < z1; z++, s = s == 2 ? 0 : s + 1) {
    // slots s, s+1, s+2 (mod 3) hold planes z-1, z, z+1
    const int s1 = s == 2 ? 0 : s + 1, s2 = s1 == 2 ? 0 : s1 + 1;
    put(s2, v);
    if (z + 1 < z1) fetch(z + 2, v);
    __syncthreads();
    const float zc = dist(z * dxf - oz);
    const bool in = ix < N && !(zc * zc + rho2 > r2lim);
    const size_t cell = ((size_t)z * N + iy) * N + ix;
    const float *L = pl[s] + o, *M = pl[s1] + o, *H = pl[s2] + o;
    if (in) {
      const float c0 = M[0], xl = M[-1], xh = M[1], yl = M[-LX], yh = M[LX], zl = L[0], zh = H[0];
      if (VEL) vrec[cell] = make_float4(xh - xl, yh - yl, zh - zl, dens[((size_t)z * N + iy) * ngx + ix]);
      if (TID) {
        const float txx = xh + xl - 2 * c0, tyy = yh + yl - 2 * c0, tzz = zh + zl - 2 * c0;
        const float txy = 0.25f * (M[1 + LX] + M[-1 - LX] - M[1 - LX] - M[-1 + LX]);
        const float txz = 0.25f * (H[1] + L[-1] - L[1] - H[-1]);
        const float tyz = 0.25f * (H[LX] + L[-LX] - L[LX] - H[-LX]);
        st[3 * threadIdx.x] = make_float2(txx, txy);
        st[3 * threadIdx.x + 1] = make_float2(txz, tyy);
        st[3 * threadIdx.x + 2] = make_float2(tyz, tzz);
      }
    }
    if (TID) ok[threadIdx.x] = in;
    __syncthreads();
    if (TID) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const int e = (int)threadIdx.x + 256 * k, row = e / (3 * kRecX), w = e % (3 * kRecX);
        if (ok[row * kRecX + w / 3])   // (streamed past the L2: 9.31 -> 8.87 ms for kappa at 1024^3)
          __builtin_nontemporal_store(*(const double *)&st[e],
                                      (double *)&t6[(((size_t)z * N + y0 + row) * N + x0) * 3 + w]);
      }
    }
  }
}

void launch_records(clr_ctx *c, bool tidal, bool vel, float rlim) {
  const int N = c->N;
  // 32 planes per block, fewer while that leaves less than 8 blocks per CU
  const int cols = (N + kRecX - 1) / kRecX * (N / kRecY);
  int nzb = 32;
  while (nzb > 4 && cols * ((N + nzb - 1) / nzb) < 2048) nzb /= 2;
  const dim3 g((N + kRecX - 1) / kRecX, N / kRecY, (N + nzb - 1) / nzb);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, g, dim3(256), 0, c->stream, c->npot, c->dens, N, c->ngx, nzb, (float)c->dx, (float)c->obs[0],
                       (float)c->obs[1], (float)c->obs[2], rlim * rlim, (float2 *)c->tidal, (float4 *)c->velrec);
  };
  if (tidal && vel) go(k_records<true, true>);
  else if (tidal) go(k_records<true, false>);
  else go(k_records<false, true>);
}

// Lanes per pixel of a march over nstep steps: as many as bring npix pixels to
// a quarter of a million threads (4 wavefronts on every SIMD), with 8 steps or
// more each, at most 16.  nside 32 on 512^3: ISW 194 -> 46 us, a custom map 287
// -> 49; nside 64 on 192^3: ISW 57 -> 24, custom map 85 -> 42.  Every plane adds
// its sum up over the lanes: where a march has its steps in flight, not more
// lanes than leave each a step for every second plane (100 planes at 64^3,
// nside 64: ISW 28 us with one lane, 40 with four).
int lanes_lg(int64_t npix, int nstep, int nplanes = 1) {
  int lg = 0;
  while (lg < 4 && (npix << lg) < (1 << 18) && (nstep >> lg) >= std::max(16, nplanes)) lg++;
  return lg;
}

template <bool KAPPA>
void launch_los(const LosArgs &a, const double *df, int nside, float *dout, hipStream_t s) {
  const int64_t npix = 12LL * nside * nside;
  const dim3 g((unsigned)(((npix << a.lg) + 255) / 256)), b(256);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, b, 0, s, a, df, df + a.nr, (int64_t)nside, npix, dout); };
  auto pick = [&](auto one, auto many) { go(a.lg == 0 ? one : many); };
  if constexpr (KAPPA) {
    if (a.t6) {
      if (a.run) pick(k_los_planes<true, true, true>, k_los_planes<true, true, false>);
      else pick(k_los<true, true, true>, k_los<true, true, false>);
      return;
    }
  }
  if (a.run) pick(k_los_planes<KAPPA, false, true>, k_los_planes<KAPPA, false, false>);
  else pick(k_los<KAPPA, false, true>, k_los<KAPPA, false, false>);
}

}  // namespace

// Host part of a kappa / ISW march: the kernel arguments (planes sorted as
// kappa_beams_preproc sorts them, their radial ranges) and the radial
// weights f1, f2 (FP64, from the host copies of the tables).
static int los_setup(clr_ctx *c, int which, int nside, int nplanes, const double *r_src, LosArgs &a,
                     std::vector<double> &f12) {
  if (nside < 1 || nside > 8192 || (nside & (nside - 1))) return clr_fail(c, CLR_ERR_ARG, "bad nside %d", nside);
  if (nplanes < 1 || nplanes > kMaxPlanes || !r_src)
    return clr_fail(c, CLR_ERR_ARG, "need 1..%d source planes", kMaxPlanes);
  const int N = c->N, na = c->na;
  const double r_max = c->r_max;
  if (!(r_max > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no r_max");
  if ((int)c->h_pd.size() != na) return clr_fail(c, CLR_ERR_STATE, "background tables missing");
  const int nr = N / 2;
  const double dr = r_max / nr, idr = 1. / dr;
  std::vector<double> rs(r_src, r_src + nplanes);
  std::vector<float> rsf(nplanes);
  for (int i = 0; i < nplanes; i++) rsf[i] = rs[i] == rs[i] ? (float)rs[i] : -INFINITY;   // ind_sort sorts flouble values
  std::vector<int> order(nplanes);
  for (int i = 0; i < nplanes; i++) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return rsf[x] < rsf[y]; });
  a = LosArgs{};
  a.phi = c->npot;
  a.N = N;
  a.ngx = c->ngx;
  a.idx = N / c->L;
  a.dr = dr;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.nr = nr;
  a.nplanes = nplanes;
  for (int i = 0; i < nplanes; i++) {
    // (a distance that is negative, NaN or no int of steps takes none: -1)
    const double st = rs[order[i]] * idr + 0.5;
    const int ih = st > -2147483648. && st < 2147483648. ? (int)st : INT_MIN;
    a.inv_rmax[i] = 1. / (ih * dr);
    a.irmax[i] = std::max(-1, std::min(ih, nr - 1));
  }
  // (plane i adds the steps after plane i-1's last; two distances that only
  // their float forms put in order may end at decreasing steps)
  a.mono = 1;
  for (int i = 1; i < nplanes; i++) a.mono = a.mono && a.irmax[i] >= a.irmax[i - 1];
  a.lg = lanes_lg(12LL * nside * nside, a.irmax[nplanes - 1] + 1);
  const double *rr = c->h_r.data(), *zz = c->h_z.data(), *dd = c->h_d1.data(), *pd = c->h_pd.data();
  f12.assign(2 * (size_t)nr, 0.0);
  for (int i = 0; i < nr; i++) {
    const double rm = (i + 0.5) * dr;
    if (which == 0) {
      const double pg = f_of_r(rr, dd, c->glob_idr, c->r_last, rm, 1.0, dd[na - 1]) *
                        (1 + f_of_r(rr, zz, c->glob_idr, c->r_last, rm, 0.0, zz[na - 1]));
      f12[i] = rm * pg * dr;
      f12[nr + i] = rm * rm * pg * dr;
    } else {
      const double pdg = f_of_r(rr, pd, c->glob_idr, c->r_last, rm, pd[0], pd[na - 1]);
      f12[i] = 2 * pdg * dr;
      f12[nr + i] = 0;
    }
  }
  return CLR_OK;
}

int clr_launch_los(clr_ctx *c, int which, int nside, int nplanes, const double *r_src, float *out) {
  if (!c->have_fields) return clr_fail(c, CLR_ERR_STATE, "clr_gaussian_fields must run first");
  if (!out) return clr_fail(c, CLR_ERR_ARG, "no output map");
  LosArgs a{};
  std::vector<double> f12;
  int rc = los_setup(c, which, nside, nplanes, r_src, a, f12);
  if (rc) return rc;
  {
    const int prc = clr_phi_ready(c, 0);   // phi's passes may still run on the second stream
    if (prc) return prc;
  }
  const int nr = a.nr;
  const int64_t npix = 12LL * nside * nside;
  const size_t need = 2 * (size_t)nr * sizeof(double) + (size_t)npix * nplanes * sizeof(float);
  rc = clr_ensure(c, &c->misc, &c->misc_n, need);
  if (rc) return rc;
  double *df = (double *)c->misc;
  float *dout = (float *)(df + 2 * nr);
  CLR_HIP(c, hipMemcpyAsync(df, f12.data(), 2 * nr * sizeof(double), hipMemcpyHostToDevice, c->stream));
  // kappa over precomputed tidal records (24 bytes per cell) when they fit in
  // a quarter of the free device memory and the march reads enough of them: a
  // record costs 8 ps per cell in reach, a step 3 ps with and 18 ps without them
  // (1024^3, nside 512), so the direct march is the faster one below about 0.4
  // steps per cell (0.96 -> 0.14 ms at 512^3, nside 32)
  const double steps = (double)npix * (a.irmax[nplanes - 1] + 1);
  const double reach = std::min(1.0, 4.18879 * pow(c->r_max / c->L, 3)) * pow((double)c->N, 3);
  const size_t t6_bytes = (size_t)c->N * c->N * c->N * 6 * sizeof(float);
  bool use_t6 = false;
  if (which == 0 && steps >= 0.4 * reach) {
    size_t fr = 0, tot = 0;
    if (c->tidal_n >= t6_bytes) use_t6 = true;
    else if (hipMemGetInfo(&fr, &tot) == hipSuccess && t6_bytes <= (fr + clr_idle_bytes(c)) / 4) use_t6 = true;
    else (void)hipGetLastError();
    if (use_t6) {
      rc = clr_ensure(c, &c->tidal, &c->tidal_n, t6_bytes);
      if (rc) return rc;
    }
  }
  // k_los_planes where planes end within the steps that k_los has in flight: 4
  // rounds of steps from records or phi alone (3 planes take the same time both
  // ways; 10 planes, nside 64: ISW 25 -> 12 us at 64^3, 116 -> 93 at 512^3),
  // one of the direct march's (30 planes: 65 -> 28 us at 64^3, nside 16 53 -> 26,
  // but 373 -> 412 at 512^3, nside 64, and 505 -> 423 with 100)
  const int nstep = a.irmax[nplanes - 1] + 1;
  if (which != 0 || use_t6) {
    a.lg = lanes_lg(npix, nstep, nplanes);
    a.run = nplanes > 3;
  } else {
    a.run = 8 * nplanes > nstep;
  }
  CLR_HIP(c, hipEventRecord(c->ev0, c->stream));
  if (use_t6) {
    launch_records(c, true, false, (float)(c->r_max + 2 * c->dx));
    a.t6 = (const float2 *)c->tidal;
  }
  if (which == 0) launch_los<true>(a, df, nside, dout, c->stream);
  else launch_los<false>(a, df, nside, dout, c->stream);
  CLR_HIP(c, hipGetLastError());
  CLR_HIP(c, hipEventRecord(c->ev1, c->stream));
  CLR_HIP(c, hipMemcpyAsync(out, dout, (size_t)npix * nplanes * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev0, c->ev1);
  c->stage_ms[which == 0 ? ST_KAPPA : ST_ISW] = ms;
  return CLR_OK;
}

// Graph-captured kappa (clr_ensemble.hip): the plan and its buffers first,
// then the march as one kernel launch into the context's map buffer.
int clr_prepare_kappa(clr_ctx *c, int nside, int nplanes, const double *r_src) {
  LosArgs a{};
  std::vector<double> f12;
  int rc = los_setup(c, 0, nside, nplanes, r_src, a, f12);
  if (rc) return rc;
  const int64_t npix = 12LL * nside * nside;
  const size_t need = 2 * (size_t)a.nr * sizeof(double) + (size_t)npix * nplanes * sizeof(float);
  if (c->los_buf_n < need) {
    if (c->los_buf) CLR_HIP(c, hipFree(c->los_buf));
    c->los_buf = nullptr;
    c->los_buf_n = 0;
    CLR_HIP(c, clr_malloc(c, &c->los_buf, need));
    c->los_buf_n = need;
  }
  CLR_HIP(c, hipMemcpy(c->los_buf, f12.data(), f12.size() * sizeof(double), hipMemcpyHostToDevice));
  c->los_plan.assign((const char *)&a, (const char *)&a + sizeof(LosArgs));
  c->los_nside = nside;
  c->los_nplanes = nplanes;
  return CLR_OK;
}

int clr_enqueue_kappa(clr_ctx *c, hipStream_t s) {
  if (c->los_plan.size() != sizeof(LosArgs) || !c->los_buf) return clr_fail(c, CLR_ERR_STATE, "kappa not prepared");
  LosArgs a;
  memcpy(&a, c->los_plan.data(), sizeof(LosArgs));
  a.phi = c->npot;
  a.t6 = nullptr;
  double *df = (double *)c->los_buf;
  launch_los<true>(a, df, c->los_nside, (float *)(df + 2 * a.nr), s);
  CLR_HIP(c, hipGetLastError());
  return CLR_OK;
}

// The last graph-captured kappa map (NEST), out[nplanes][npix].
int clr_fetch_kappa(clr_ctx *c, float *out) {
  if (c->los_plan.size() != sizeof(LosArgs) || !c->los_buf) return clr_fail(c, CLR_ERR_STATE, "kappa not prepared");
  LosArgs a;
  memcpy(&a, c->los_plan.data(), sizeof(LosArgs));
  const int64_t npix = 12LL * c->los_nside * c->los_nside;
  CLR_HIP(c, hipMemcpy(out, (double *)c->los_buf + 2 * a.nr, (size_t)npix * c->los_nplanes * sizeof(float),
                       hipMemcpyDeviceToHost));
  return CLR_OK;
}

// ---------------------------------------------------------------------------
// Sources' line-of-sight properties: srcs_beams_preproc_single
// (srcs.c:425-445), srcs_get_beam_properties_single (srcs.c:452-625, the
// build without _USE_FAST_LENSING) and srcs_beams_postproc_single
// (srcs.c:634-737) for one population.  2^lg lanes per source, sources in the
// order of their directions (k_dir_*), so that the rays of a wavefront, and of
// the wavefronts that run beside it on an XCD, cross the same cells.
// ---------------------------------------------------------------------------
namespace {

struct BeamArgs {
  const float *phi;
  int N, ngx, nr, na, lg;                 // 2^lg lanes per source
  double idx, dr, idr, ox, oy, oz, factor_vel;
  double glob_idr, r_last, z_last, v1_0, v1_last;
  const double *r_arr, *z_arr, *v1_arr;   // background r-tables
  const double *a2r;                      // r(a) at a = i/(na-1) (r_of_z, cosmo.c:101-112)
  const double *fac;                      // fac_r_0, fac_r_1, fac_r_2 (nr each)
  const float4 *vrec;                     // per cell (k_records): phi's central differences, delta
  const float2 *t6;                       // per cell (k_records): the tidal tensor's second differences
};

// get_element (beaming.c:31-117), RETURN_VEL: unscaled central differences,
// periodic in x, y and z on one GPU (fourier.c:412-413).
__device__ inline void vel_at(const float *__restrict__ phi, int N, size_t ngx, size_t plane, int ix, int iy,
                              int iz, double v[3]) {
  const int xh = ix == N - 1 ? 0 : ix + 1, xl = ix == 0 ? N - 1 : ix - 1;
  const int yh = iy == N - 1 ? 0 : iy + 1, yl = iy == 0 ? N - 1 : iy - 1;
  const int zh = iz == N - 1 ? 0 : iz + 1, zl = iz == 0 ? N - 1 : iz - 1;
  const size_t Z0 = (size_t)iz * plane, Y0 = (size_t)iy * ngx;
  v[0] = phi[xh + Y0 + Z0] - phi[xl + Y0 + Z0];   // FP32 differences, as get_element
  v[1] = phi[ix + (size_t)yh * ngx + Z0] - phi[ix + (size_t)yl * ngx + Z0];
  v[2] = phi[ix + Y0 + (size_t)zh * plane] - phi[ix + Y0 + (size_t)zl * plane];
}

// get_element, RETURN_VEL | RETURN_TID: velocity and the 19-point tidal
// tensor (xx, xy, xz, yy, yz, zz; mixed terms with 1/4).
__device__ inline void vel_tid_at(const float *__restrict__ phi, int N, size_t ngx, size_t plane, int ix, int iy,
                                  int iz, float v[3], float t[6]) {
#pragma clang fp contract(off)
  const int xh = ix == N - 1 ? 0 : ix + 1, xl = ix == 0 ? N - 1 : ix - 1;
  const int yh = iy == N - 1 ? 0 : iy + 1, yl = iy == 0 ? N - 1 : iy - 1;
  const int zh = iz == N - 1 ? 0 : iz + 1, zl = iz == 0 ? N - 1 : iz - 1;
  const size_t Z0 = (size_t)iz * plane, ZH = (size_t)zh * plane, ZL = (size_t)zl * plane;
  const size_t Y0 = (size_t)iy * ngx, YH = (size_t)yh * ngx, YL = (size_t)yl * ngx;
  // FP32 differences, as get_element evaluates them on flouble values
  const float c0 = phi[ix + Y0 + Z0];
  const float pxh = phi[xh + Y0 + Z0], pxl = phi[xl + Y0 + Z0];
  const float pyh = phi[ix + YH + Z0], pyl = phi[ix + YL + Z0];
  const float pzh = phi[ix + Y0 + ZH], pzl = phi[ix + Y0 + ZL];
  v[0] = pxh - pxl;
  v[1] = pyh - pyl;
  v[2] = pzh - pzl;
  t[0] = pxh + pxl - 2 * c0;
  t[3] = pyh + pyl - 2 * c0;
  t[5] = pzh + pzl - 2 * c0;
  t[1] = 0.25f * (phi[xh + YH + Z0] + phi[xl + YL + Z0] - phi[xh + YL + Z0] - phi[xl + YH + Z0]);
  t[2] = 0.25f * (phi[xh + Y0 + ZH] + phi[xl + Y0 + ZL] - phi[xh + Y0 + ZL] - phi[xl + Y0 + ZH]);
  t[4] = 0.25f * (phi[ix + YH + ZH] + phi[ix + YL + ZL] - phi[ix + YH + ZL] - phi[ix + YL + ZH]);
}

// A cell's velocity differences (and density) from its record or from phi.
template <bool REC>
__device__ inline void vel_cell(const float4 *__restrict__ vrec, const float *__restrict__ phi, int N, size_t ngx,
                                size_t plane, int ix, int iy, int iz, double v[3]) {
  if (REC) {
    const float4 q = vrec[((size_t)iz * N + iy) * N + ix];
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
  } else {
    vel_at(phi, N, ngx, plane, ix, iy, iz, v);
  }
}

// Order of the marches: sources by direction (cells of a G x G grid on each
// face of a cube around the observer, in Morton order), so that the lanes of a
// wavefront take nearly the same cells.  A counting sort: k_dir_count numbers the sources of a
// bin, k_dir_scan sums the bins, k_dir_place writes the permutation (its order
// within a bin is the atomics'; a source's result does not depend on it).
constexpr int kDirG = 64;
// The order pays where the records in reach (40 bytes per cell) are more than
// the 256 MB last-level cache holds: 950k sources at 512^3 3.57 -> 2.00 ms with
// the records' pass, 384^3 1.84 -> 1.10, 256^3 0.71 -> 0.61, but 192^3 0.38 ->
// 0.41 and 128^3 0.20 -> 0.28.  The line in sources: 24k in catalogue order and
// in order of direction 171 and 187 us at 256^3, 452 and 462 at 384^3, 1075 and
// 1083 at 512^3; 28k 179/184, 464/460, 1097/1089; 33k 188/186, 478/468,
// 1123/1102; 64k 216/212, 540/495, 1221/1155.  16 sources per bin (64: 2.07 ms;
// bins of 4 shells of distance in 4 times wider cells, 2.08).
constexpr int kDirMinN = 256;
// Skewers, whose every step of a source is a gather of its own, pay the order's
// 20 us back from fewer sources on: from 24576, where dir_grid's bins become
// finer (64 -> 16 sources in each).  At 256^3 20k sources took 65 us in
// catalogue order and 72 in order of direction, 24k 77/83, 28k 88/83, 64k
// 184/155; at 384^3 12k 92/94, 20k 137/132, 24k 157/149, 28k 179/149; at 512^3
// 4k 60/73, 12k 140/135, 24k 243/214, 28k 274/219; at 192^3 28k 56/61.
constexpr long long kDirMin = 32768, kDirMinSkw = 24576, kDirPer = 16;
constexpr size_t kBeamKeep = (size_t)1 << 30;

__device__ inline uint32_t spread(uint32_t v) {
  v = (v | (v << 4)) & 0x0f0fu;
  v = (v | (v << 2)) & 0x3333u;
  return (v | (v << 1)) & 0x5555u;
}

__device__ inline uint32_t dir_bin(const float4 p, int G) {
  const float ax = fabsf(p.x), ay = fabsf(p.y), az = fabsf(p.z);
  int face;
  float m, u, v;
  if (ax >= ay && ax >= az) { face = p.x < 0; m = ax; u = p.y; v = p.z; }
  else if (ay >= az) { face = 2 + (p.y < 0); m = ay; u = p.x; v = p.z; }
  else { face = 4 + (p.z < 0); m = az; u = p.x; v = p.y; }
  const float s = m > 0 ? __builtin_amdgcn_rcpf(m) : 0.f;
  const int iu = min(max((int)((u * s * 0.5f + 0.5f) * G), 0), G - 1);
  const int iv = min(max((int)((v * s * 0.5f + 0.5f) * G), 0), G - 1);
  return (uint32_t)(face * G * G) + (spread(iu) | spread(iv) << 1);
}

__global__ void k_dir_zero(uint32_t *__restrict__ cnt, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cnt[i] = 0;
}

__global__ __launch_bounds__(256) void k_dir_count(const float4 *__restrict__ pos, uint32_t n, int G,
                                                   uint32_t *__restrict__ cnt, uint2 *__restrict__ kr) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t k = dir_bin(pos[i], G);
  kr[i] = make_uint2(k, atomicAdd(&cnt[k], 1u));
}

// Exclusive sum of cnt[nb] in place, nb a multiple of 4: one block, all of a
// thread's loads in flight together (a run of bins per thread took 40 us).
__global__ __launch_bounds__(1024) void k_dir_scan(uint4 *__restrict__ cnt, int nb4) {
  constexpr int C = (6 * kDirG * kDirG + 4095) / 4096;
  __shared__ uint32_t ws[C][16];
  const int t = threadIdx.x, lane = t & 63;
  uint4 v[C];
  uint32_t inc[C];
#pragma unroll
  for (int k = 0; k < C; k++) v[k] = k * 1024 + t < nb4 ? cnt[k * 1024 + t] : make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < C; k++) {
    inc[k] = v[k].x + v[k].y + v[k].z + v[k].w;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t x = __shfl_up(inc[k], o);
      if (lane >= o) inc[k] += x;
    }
    if (lane == 63) ws[k][t >> 6] = inc[k];
  }
  __syncthreads();
  uint32_t base = 0;
#pragma unroll
  for (int k = 0; k < C; k++) {
    uint32_t run = base + inc[k] - (v[k].x + v[k].y + v[k].z + v[k].w);
    for (int w = 0; w < 16; w++) {
      const uint32_t x = ws[k][w];
      base += x;
      if (w < (t >> 6)) run += x;
    }
    const uint4 e = make_uint4(run, run + v[k].x, run + v[k].x + v[k].y, run + v[k].x + v[k].y + v[k].z);
    if (k * 1024 + t < nb4) cnt[k * 1024 + t] = e;
  }
}

__global__ __launch_bounds__(256) void k_dir_place(const uint2 *__restrict__ kr, uint32_t n,
                                                   const uint32_t *__restrict__ off, uint32_t *__restrict__ perm) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint2 e = kr[i];
  perm[off[e.x] + e.y] = i;
}

// Bins' grid for n sources, and the order itself: cnt[dir_bins(G)] and kr[n]
// are scratch, perm[n] the result.
inline int dir_grid(long long n) {
  int G = 1;
  while (G < kDirG && 24ll * G * G * kDirPer <= n) G *= 2;
  return G;
}
inline int dir_bins(int G) { return (6 * G * G + 3) / 4 * 4; }
void launch_order(const float4 *pos, long long n, int G, uint32_t *cnt, uint2 *kr, uint32_t *perm, hipStream_t s) {
  const int nb = dir_bins(G);
  const unsigned g = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(k_dir_zero, dim3((nb + 255) / 256), dim3(256), 0, s, cnt, nb);
  hipLaunchKernelGGL(k_dir_count, dim3(g), dim3(256), 0, s, pos, (uint32_t)n, G, cnt, kr);
  hipLaunchKernelGGL(k_dir_scan, dim3(1), dim3(1024), 0, s, (uint4 *)cnt, nb / 4);
  hipLaunchKernelGGL(k_dir_place, dim3(g), dim3(256), 0, s, kr, (uint32_t)n, cnt, perm);
}

// A thread takes every 2^lg-th step of a source.  The projections of the
// tidal tensor and of the gradient are constant along a ray, so the march
// sums the six and two or three components with their radial weights in FP64
// and projects the sums: 9 FP64 multiply-adds per step, where projecting at
// each step took 17 + 5 multiplies and as many adds.  Bound by the latency of
// the records' loads: 950k sources of 512^3 2.87 -> 0.96 ms (two steps in
// flight: the same), 48k of 256^3 0.34 -> 0.21 with the records' pass.  Blocks of neighbouring
// directions follow each other on one XCD (block b is logical block
// (b % 8) (gridDim.x / 8) + b / 8, gridDim.x a multiple of 8).
template <bool LENS, bool REC>
__global__ __launch_bounds__(256) void k_src_beams(BeamArgs a, const float4 *__restrict__ pos,
                                                   const uint32_t *__restrict__ perm, long long n,
                                                   float *__restrict__ dz, float *__restrict__ lens) {
#pragma clang fp contract(off)
  const unsigned blk = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int lg = LENS ? a.lg : 0, K = 1 << lg;
  const long long j = ((long long)blk * 256 + threadIdx.x) >> lg;
  const int sub = threadIdx.x & (K - 1);
  if (j >= n) return;
  const long long i = perm ? (long long)perm[j] : j;
  const float4 p = pos[i];
  const int N = a.N;
  const size_t ngx = (size_t)a.ngx, plane = (size_t)N * ngx;
  const float *__restrict__ phi = a.phi;
  const double px = p.x, py = p.y, pz = p.z;
  const double r = sqrt(px * px + py * py + pz * pz);
  const double ir = 1. / (r > 0.001 ? r : 0.001);
  const double u[3] = {px * ir, py * ir, pz * ir};
  const double xn[3] = {(px + a.ox) * a.idx, (py + a.oy) * a.idx, (pz + a.oz) * a.idx};

  // CIC velocity at the source (interpolate_from_grid with INTERP_TYPE_SKW,
  // beaming.c:193-266)
  int i0[3], i1[3];
  double h0[3], h1[3];
  for (int ax = 0; ax < 3; ax++) {
    const int c = (int)xn[ax];   // (long)x: truncation toward zero
    h0[ax] = xn[ax] - c;
    h1[ax] = 1 - h0[ax];
    i0[ax] = wrap1(c, N);
    i1[ax] = wrap1(c + 1, N);
  }
  double v[3] = {0, 0, 0};
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int bx = c & 1, by = (c >> 1) & 1, bz = c >> 2;
    const double w = (bz ? h0[2] : h1[2]) * (by ? h0[1] : h1[1]) * (bx ? h0[0] : h1[0]);
    double vc[3];
    vel_cell<REC>(a.vrec, phi, N, ngx, plane, bx ? i1[0] : i0[0], by ? i1[1] : i0[1], bz ? i1[2] : i0[2], vc);
    v[0] += vc[0] * w;
    v[1] += vc[1] * w;
    v[2] += vc[2] * w;
  }
  const float vr = (float)(0.5 * a.idx * (v[0] * u[0] + v[1] * u[1] + v[2] * u[2]));
  // postproc: dz_rsd *= V1(r_of_z(z0)) factor_vel, z0 the catalogue's float z(r)
  const float z0 = (float)f_of_r(a.r_arr, a.z_arr, a.glob_idr, a.r_last, r, 0.0, a.z_last);
  double rz;
  {
    const double aa = 1. / (1 + (double)z0);
    if (aa >= 1) rz = 0;
    else if (aa <= 0) rz = a.a2r[0];
    else {
      const int ia = (int)(aa * (a.na - 1));
      rz = a.a2r[ia] + (a.a2r[ia + 1] - a.a2r[ia]) * (aa - (double)ia / (a.na - 1)) * (a.na - 1.);
    }
  }
  const double vg = f_of_r(a.r_arr, a.v1_arr, a.glob_idr, a.r_last, rz, a.v1_0, a.v1_last);
  if (sub == 0) dz[i] = (float)((double)vr * (vg * a.factor_vel));
  if (!LENS) return;

  double cth = u[2];
  if (cth >= 1) cth = 1;
  if (cth <= -1) cth = -1;
  const double sth = sqrt((1 - cth) * (1 + cth));
  double cph = 1, sph = 0;
  if (sth != 0) { cph = u[0] / sth; sph = u[1] / sth; }
  const double pre = a.idx * a.idx * ir, prem = 0.5 * a.idx * ir;
  const double ux[3] = {cth * cph * prem, cth * sph * prem, -sth * prem};
  const double uy[2] = {-sph * prem, cph * prem};
  const double rk[6] = {(cth * cth * cph * cph + sph * sph) * pre, (2 * cph * sph * (cth * cth - 1)) * pre,
                        (-2 * cth * sth * cph) * pre,                (cth * cth * sph * sph + cph * cph) * pre,
                        (-2 * cth * sth * sph) * pre,                (sth * sth) * pre};
  const double re1[6] = {(cth * cth * cph * cph - sph * sph) * pre, (2 * cph * sph * (cth * cth + 1)) * pre,
                         (-2 * cth * sth * cph) * pre,                (cth * cth * sph * sph - cph * cph) * pre,
                         (-2 * cth * sth * sph) * pre,                (sth * sth) * pre};
  const double re2[5] = {(-2 * cth * cph * sph) * pre, (2 * cth * (cph * cph - sph * sph)) * pre,
                         (2 * sth * sph) * pre,        (2 * cth * sph * cph) * pre,
                         (-2 * sth * cph) * pre};
  const double *__restrict__ f0 = a.fac, *__restrict__ f1 = a.fac + a.nr, *__restrict__ f2 = a.fac + 2 * a.nr;
  double st[6] = {}, sv[3] = {};
  const int irmax = min((int)(r * a.idr + 0.5), a.nr - 1);
  Ray ray;
  int64_t x[3];
#pragma unroll
  for (int ax = 0; ax < 3; ax++) ray.u[ax] = u[ax];
  ray_setup(ray, a.dr, a.idx, a.ox, a.oy, a.oz);
#pragma unroll
  for (int ax = 0; ax < 3; ax++) x[ax] = ray.base[ax] + (int64_t)sub * ray.step[ax];
  for (int i_r = sub; i_r <= irmax; i_r += K) {
    int c[3];
    ray_cell(ray, x, i_r, N, a.dr, a.idx, a.ox, a.oy, a.oz, c);
#pragma unroll
    for (int ax = 0; ax < 3; ax++) x[ax] += ray.step[ax] << lg;
    float vp[4], tp[6];
    if (REC) {
      const size_t o = ((size_t)c[2] * N + c[1]) * N + c[0];
      const float *q = (const float *)(a.t6 + 3 * o);
      __builtin_memcpy(vp, &a.vrec[o], 16);
      __builtin_memcpy(tp, q, 16);
      __builtin_memcpy(tp + 4, q + 4, 8);
    } else {
      vel_tid_at(phi, N, ngx, plane, c[0], c[1], c[2], vp, tp);
    }
    const double fr = fma(f1[i_r], r, -f2[i_r]);
    const double frm = 2 * fma(f0[i_r], r, -f1[i_r]);
#pragma unroll
    for (int q = 0; q < 6; q++) st[q] = fma(fr, (double)tp[q], st[q]);
#pragma unroll
    for (int q = 0; q < 3; q++) sv[q] = fma(frm, (double)vp[q], sv[q]);
  }
  for (int o = 1; o < K; o <<= 1) {
#pragma unroll
    for (int q = 0; q < 6; q++) st[q] += __shfl_xor(st[q], o);
#pragma unroll
    for (int q = 0; q < 3; q++) sv[q] += __shfl_xor(sv[q], o);
  }
  if (sub != 0) return;
  double kp = 0, e1 = 0, e2 = 0;
#pragma unroll
  for (int q = 0; q < 6; q++) {
    e1 += re1[q] * st[q];
    if (q < 5) e2 += re2[q] * st[q];
    kp += rk[q] * st[q];
  }
  const double dtx = ux[0] * sv[0] + ux[1] * sv[1] + ux[2] * sv[2];
  const double dty = uy[0] * sv[0] + uy[1] * sv[1];
  const double RTOD = 57.2957795;
  float *o = lens + 5 * i;
  o[0] = (float)e1;
  o[1] = (float)e2;
  o[2] = (float)kp;
  o[3] = (float)(dty * RTOD);
  o[4] = (float)(dtx * RTOD);
}

}  // namespace

// Builds the per-cell records on the context's stream: velocity differences
// and density (16 bytes per cell), with `tidal` also the tidal tensor (24
// bytes per cell), when they fit in a quarter of the free device
// memory (buffers kept for later calls); false: the callers read phi directly.
bool clr_cell_records(clr_ctx *c, bool tidal) {
  const size_t cells = (size_t)c->N * c->N * c->N;
  const size_t vb = cells * sizeof(float4), tb = tidal ? cells * 6 * sizeof(float) : 0;
  size_t need = (c->velrec_n >= vb ? 0 : vb) + (c->tidal_n >= tb ? 0 : tb);
  if (need > 0) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    if (need > (fr + clr_idle_bytes(c)) / 4) return false;
  }
  if (clr_ensure(c, &c->velrec, &c->velrec_n, vb)) return false;
  if (tidal && clr_ensure(c, &c->tidal, &c->tidal_n, tb)) return false;
  // the marches stay within r_max, the sources within L/2 + 20 (their cells'
  // corners and the CIC neighbours within 2 cells of that)
  launch_records(c, tidal, true, (float)(std::max(c->r_max, 0.5 * c->L + 20.) + 3 * c->dx));
  return hipGetLastError() == hipSuccess;
}

int clr_launch_src_beams(clr_ctx *c, int ipop, const double *r_arr_a2r, float *dz, float *lens, long long n) {
  if (ipop < 0 || ipop >= c->n_tr[CLR_TRACER_SRCS]) return clr_fail(c, CLR_ERR_ARG, "no source population %d", ipop);
  if (!c->have_fields) return clr_fail(c, CLR_ERR_STATE, "clr_gaussian_fields must run first");
  const CatalogDev &C = c->cat[ipop];
  if (n != C.n) return clr_fail(c, CLR_ERR_ARG, "population %d holds %lld sources, not %lld", ipop, C.n, n);
  if (!r_arr_a2r || (n > 0 && !dz)) return clr_fail(c, CLR_ERR_ARG, "null r(a) table or output");
  const int N = c->N, na = c->na;
  const double r_max = c->r_max;
  if (!(r_max > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no r_max");
  if (!(c->hubble_0 > 0) || !(c->omega_m > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no H0 or Omega_M");
  if (n == 0) return CLR_OK;
  const int nr = N / 2;
  const double dr = r_max / nr;
  // fac_r_0/1/2 (srcs.c:470-480), FP64 on the host from the uploaded tables
  const double *rr = c->h_r.data(), *zz = c->h_z.data(), *dd = c->h_d1.data();
  std::vector<double> fac(3 * (size_t)nr);
  for (int i = 0; i < nr; i++) {
    const double rm = (i + 0.5) * dr;
    const double pg = f_of_r(rr, dd, c->glob_idr, c->r_last, rm, 1.0, dd[na - 1]) *
                      (1 + f_of_r(rr, zz, c->glob_idr, c->r_last, rm, 0.0, zz[na - 1]));
    fac[i] = pg * dr;
    fac[nr + i] = rm * pg * dr;
    fac[2 * nr + i] = rm * rm * pg * dr;
  }
  const size_t tab_bytes = (3 * (size_t)nr + na + 1) / 2 * 2 * sizeof(double);
  const int per = lens ? 6 : 1;
  // the tables, the order of the marches and the results: in a buffer that the
  // context keeps up to kBeamKeep bytes, else in one of this call
  bool order = lens && N >= kDirMinN && n >= kDirMin && n < (1ll << 31);
  const int G = dir_grid(n), nb = dir_bins(G);
  struct Own {
    void *p = nullptr;
    ~Own() {
      if (p) (void)hipFree(p);
    }
  } own;
  char *buf = nullptr;
  for (;;) {
    const size_t need =
        tab_bytes + (order ? (size_t)(n + 1) * 12 + (size_t)nb * 4 : 0) + (size_t)n * per * sizeof(float);
    int rc = CLR_OK;
    if (need <= kBeamKeep) {
      rc = clr_ensure(c, &c->beam_ws, &c->beam_ws_n, need);
      buf = (char *)c->beam_ws;
    } else if (clr_malloc(c, &own.p, need) != hipSuccess) {
      rc = clr_fail(c, CLR_ERR_HIP, "source beams: no device memory for %zu bytes", need);
    } else {
      buf = (char *)own.p;
    }
    if (rc == CLR_OK) break;
    if (!order) return rc;
    order = false;
  }
  const clr_ws_use use(c, own.p ? 0 : CLR_WS_BEAM);
  double *dfac = (double *)buf, *da2r = dfac + 3 * nr;
  uint32_t *cnt = (uint32_t *)(buf + tab_bytes), *perm = cnt + (order ? nb : 0);
  uint2 *kr = (uint2 *)(perm + (order ? (n + 1) / 2 * 2 : 0));
  float *tmp = (float *)(kr + (order ? n : 0));
  CLR_HIP(c, hipMemcpyAsync(dfac, fac.data(), 3 * (size_t)nr * sizeof(double), hipMemcpyHostToDevice, c->stream));
  CLR_HIP(c, hipMemcpyAsync(da2r, r_arr_a2r, na * sizeof(double), hipMemcpyHostToDevice, c->stream));
  BeamArgs a{};
  {
    const int prc = clr_phi_ready(c, 0);
    if (prc) return prc;
  }
  a.phi = c->npot;
  a.N = N;
  a.ngx = c->ngx;
  a.nr = nr;
  a.na = na;
  a.idx = N / c->L;
  a.dr = dr;
  a.idr = 1. / dr;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.factor_vel = -c->fgrowth_0 / (1.5 * c->hubble_0 * c->omega_m);
  a.glob_idr = c->glob_idr;
  a.r_last = c->r_last;
  a.z_last = c->h_bg_last[1];
  a.v1_0 = c->h_bg_first[3];
  a.v1_last = c->h_bg_last[3];
  a.r_arr = c->bg;
  a.z_arr = c->bg + na;
  a.v1_arr = c->bg + 3 * (size_t)na;
  a.a2r = da2r;
  a.fac = dfac;
  CLR_HIP(c, hipEventRecord(c->ev0, c->stream));
  const float4 *pos = (const float4 *)C.pos;
  a.lg = lens ? lanes_lg(n, nr) : 0;
  const unsigned nblk = (unsigned)((((n << a.lg) + 255) / 256 + 7) / 8 * 8);
  const dim3 grid(nblk);
  if (order) {
    launch_order(pos, n, G, cnt, kr, perm, c->stream);
  } else {
    perm = nullptr;
  }
  // per-cell records (velocity differences; with lensing also the tidal
  // tensor) when they fit in a quarter of the free device memory
  const bool rec = clr_cell_records(c, lens != nullptr);
  a.vrec = (const float4 *)c->velrec;
  a.t6 = (const float2 *)c->tidal;
  if (lens && rec)
    hipLaunchKernelGGL((k_src_beams<true, true>), grid, dim3(256), 0, c->stream, a, pos, perm, n, tmp, tmp + n);
  else if (lens)
    hipLaunchKernelGGL((k_src_beams<true, false>), grid, dim3(256), 0, c->stream, a, pos, perm, n, tmp, tmp + n);
  else if (rec)
    hipLaunchKernelGGL((k_src_beams<false, true>), grid, dim3(256), 0, c->stream, a, pos, perm, n, tmp,
                       (float *)nullptr);
  else
    hipLaunchKernelGGL((k_src_beams<false, false>), grid, dim3(256), 0, c->stream, a, pos, perm, n, tmp,
                       (float *)nullptr);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipEventRecord(c->ev1, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(dz, tmp, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess && lens)
    e = hipMemcpyAsync(lens, tmp + n, (size_t)n * 5 * sizeof(float), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return clr_fail(c, CLR_ERR_HIP, "source beams: %s", hipGetErrorString(e));
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev0, c->ev1);
  c->stage_ms[ST_BEAMS] = ms;
  return CLR_OK;
}

// ---------------------------------------------------------------------------
// Skewers (srcs.c:507-529) with their postproc scaling (srcs.c:725-733): one
// thread per (source, radial step), steps of a source in consecutive lanes,
// so a wavefront covers one or a few rays and writes whole rows.
// ---------------------------------------------------------------------------
namespace {

struct SkwArgs {
  const float *phi, *dens;
  const float4 *vrec;   // per cell (k_records), or null
  int N, ngx, nr, na, gaussian;
  double idx, dr, idr, ox, oy, oz, factor_vel, sigma2;
  double glob_idr, r_last, v1_0, v1_last, d1_last;
  float dxf;
  const double *r_arr, *d1_arr, *v1_arr;
};

// A block computes 16 steps of 16 consecutive sources (lane = step + 16 x
// source), in order of direction (perm) or of the catalogue: neighbouring
// sources lie in neighbouring directions or cells, so their lines of
// sight cross nearly the same cells at the same step and share the CIC
// corners' cache lines, where one thread per (source, step) in row order
// fetched ~170 bytes of HBM per value.  The blocks of one group of sources
// follow each other on one XCD (workgroups go to the 8 XCDs round-robin by
// linear id, each XCD with its own L2): logical block
// (b % 8) (gridDim.x / 8) + b / 8, gridDim.x a multiple of 8.  nr is a
// multiple of 16.
template <bool REC>
__global__ __launch_bounds__(256) void k_src_skewers(SkwArgs a, const float4 *__restrict__ pos,
                                                     const uint32_t *__restrict__ perm, long long n,
                                                     float *__restrict__ dg, float *__restrict__ vs) {
#pragma clang fp contract(off)
  const long long blk = (long long)(blockIdx.x % 8u) * (gridDim.x / 8u) + blockIdx.x / 8u;
  const int ntile = a.nr / 16;
  const long long j = (blk / ntile) * 16 + threadIdx.x / 16;
  const int i_r = (int)(blk % ntile) * 16 + (int)(threadIdx.x % 16);
  if (j >= n) return;
  const long long i = perm ? (long long)perm[j] : j;
  const long long t = i * a.nr + i_r;
  const float4 p = pos[i];
  const int N = a.N;
  const size_t ngx = (size_t)a.ngx, plane = (size_t)N * ngx;
  const double px = p.x, py = p.y, pz = p.z;
  const double r = sqrt(px * px + py * py + pz * pz);
  const double ir = 1. / (r > 0.001 ? r : 0.001);
  const double u[3] = {px * ir, py * ir, pz * ir};
  const int irmax = min((int)(r * a.idr + 0.5), a.nr - 1);
  if (i_r > irmax) {   // calloc'd rows (common.c:381-387)
    dg[t] = 0;
    vs[t] = 0;
    return;
  }
  const double rm = (i_r + 0.5) * a.dr;
  const double xn[3] = {(rm * u[0] + a.ox) * a.idx, (rm * u[1] + a.oy) * a.idx, (rm * u[2] + a.oz) * a.idx};
  int i0[3], i1[3];
  double h0[3], h1[3];
  for (int ax = 0; ax < 3; ax++) {
    const int c = (int)xn[ax];
    h0[ax] = xn[ax] - c;
    h1[ax] = 1 - h0[ax];
    i0[ax] = wrap1(c, N);
    i1[ax] = wrap1(c + 1, N);
  }
  double v[3] = {0, 0, 0}, d = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int bx = c & 1, by = (c >> 1) & 1, bz = c >> 2;
    const double w = (bz ? h0[2] : h1[2]) * (by ? h0[1] : h1[1]) * (bx ? h0[0] : h1[0]);
    const int cx = bx ? i1[0] : i0[0], cy = by ? i1[1] : i0[1], cz = bz ? i1[2] : i0[2];
    double vc[3];
    float dc;
    if (REC) {
      const float4 q = a.vrec[((size_t)cz * N + cy) * N + cx];
      vc[0] = q.x;
      vc[1] = q.y;
      vc[2] = q.z;
      dc = q.w;
    } else {
      vel_at(a.phi, N, ngx, plane, cx, cy, cz, vc);
      dc = a.dens[(size_t)cz * plane + (size_t)cy * ngx + cx];
    }
    v[0] += vc[0] * w;
    v[1] += vc[1] * w;
    v[2] += vc[2] * w;
    if (a.gaussian) {
      // get_element RETURN_GAUSS (beaming.c:46-57): the cell's offsets and
      // radius in float, D(r) from the FP64 table
      const float x0 = (float)((cx + 0.0) * a.dxf - a.ox), y0 = (float)((cy + 0.0) * a.dxf - a.oy);
      const float z0 = (float)((cz + 0.0) * a.dxf - a.oz);
      const double rc = sqrt((double)(x0 * x0 + y0 * y0 + z0 * z0));
      const double D = f_of_r(a.r_arr, a.d1_arr, a.glob_idr, a.r_last, rc, 1.0, a.d1_last);
      d += (log((double)(1.0f + dc)) / D + D * a.sigma2 * 0.5) * w;
    } else {
      d += (double)dc * w;
    }
  }
  const float vr = (float)(0.5 * a.idx * (v[0] * u[0] + v[1] * u[1] + v[2] * u[2]));
  const double vg = f_of_r(a.r_arr, a.v1_arr, a.glob_idr, a.r_last, rm, a.v1_0, a.v1_last);
  dg[t] = (float)d;
  vs[t] = (float)((double)vr * (vg * a.factor_vel));
}

}  // namespace

int clr_launch_src_skewers(clr_ctx *c, int ipop, int gaussian, double sigma2, float *dg, float *vs, long long n) {
  if (ipop < 0 || ipop >= c->n_tr[CLR_TRACER_SRCS]) return clr_fail(c, CLR_ERR_ARG, "no source population %d", ipop);
  if (!c->have_fields) return clr_fail(c, CLR_ERR_STATE, "clr_gaussian_fields must run first");
  if (!c->density_done) return clr_fail(c, CLR_ERR_STATE, "density field not computed");
  const CatalogDev &C = c->cat[ipop];
  if (n != C.n) return clr_fail(c, CLR_ERR_ARG, "population %d holds %lld sources, not %lld", ipop, C.n, n);
  if (n > 0 && (!dg || !vs)) return clr_fail(c, CLR_ERR_ARG, "null skewer output");
  if (gaussian && !(sigma2 >= 0)) return clr_fail(c, CLR_ERR_ARG, "bad sigma2 %g", sigma2);
  const int N = c->N, na = c->na;
  if (!(c->r_max > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no r_max");
  if (!(c->hubble_0 > 0) || !(c->omega_m > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no H0 or Omega_M");
  if (n == 0) return CLR_OK;
  {
    const int prc = clr_phi_ready(c, 0);
    if (prc) return prc;
  }
  SkwArgs a{};
  a.phi = c->npot;
  a.dens = c->dens;
  a.N = N;
  a.ngx = c->ngx;
  a.nr = N / 2;
  if (a.nr % 16) return clr_fail(c, CLR_ERR_ARG, "source skewers need N/2 a multiple of 16 (N = %d)", N);
  a.na = na;
  a.gaussian = gaussian ? 1 : 0;
  a.idx = N / c->L;
  a.dr = c->r_max / a.nr;
  a.idr = 1. / a.dr;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.factor_vel = -c->fgrowth_0 / (1.5 * c->hubble_0 * c->omega_m);
  a.sigma2 = sigma2;
  a.glob_idr = c->glob_idr;
  a.r_last = c->r_last;
  a.v1_0 = c->h_bg_first[3];
  a.v1_last = c->h_bg_last[3];
  a.d1_last = c->h_bg_last[2];
  a.dxf = (float)(c->L / N);
  a.r_arr = c->bg;
  a.d1_arr = c->bg + 2 * (size_t)na;
  a.v1_arr = c->bg + 3 * (size_t)na;
  a.vrec = clr_cell_records(c, false) ? (const float4 *)c->velrec : nullptr;
  // sources per launch: at most 2^26 skewer values (512 MiB of staging, kept in
  // the source passes' buffer: allocating and freeing it took as long as the kernel)
  const long long chunk = std::max(1LL, (1LL << 26) / a.nr);
  const long long cap = std::min(n, chunk);
  const bool order = N >= kDirMinN && cap >= kDirMinSkw;
  const int G = dir_grid(cap), nb = dir_bins(G);
  const size_t obytes = order ? ((size_t)nb * 4 + (size_t)cap * 12 + 15) / 16 * 16 : 0;
  const int wrc = clr_ensure(c, &c->beam_ws, &c->beam_ws_n, obytes + (size_t)cap * a.nr * 2 * sizeof(float));
  if (wrc) return wrc;
  const clr_ws_use use(c, CLR_WS_BEAM);
  uint32_t *cnt = (uint32_t *)c->beam_ws;
  uint2 *kr = (uint2 *)(cnt + nb);
  uint32_t *perm = order ? (uint32_t *)(kr + cap) : nullptr;
  float *tmp = (float *)((char *)c->beam_ws + obytes);
  hipError_t e = hipEventRecord(c->ev0, c->stream);
  float kms = 0;
  for (long long s0 = 0; s0 < n && e == hipSuccess; s0 += cap) {
    const long long m = std::min(cap, n - s0);
    const long long tot = m * a.nr;
    // 16 sources x 16 steps per block, the count rounded up to the 8 XCDs
    // (the extra blocks' sources are >= m and return)
    const unsigned nblk = (unsigned)(((m + 15) / 16 * (a.nr / 16) + 7) / 8 * 8);
    e = hipEventRecord(c->ev2, c->stream);
    if (e == hipSuccess) {
      if (order) launch_order((const float4 *)C.pos + s0, m, G, cnt, kr, perm, c->stream);
      if (a.vrec)
        hipLaunchKernelGGL(k_src_skewers<true>, dim3(nblk), dim3(256), 0, c->stream, a,
                           (const float4 *)C.pos + s0, perm, m, tmp, tmp + (size_t)cap * a.nr);
      else
        hipLaunchKernelGGL(k_src_skewers<false>, dim3(nblk), dim3(256), 0, c->stream, a,
                           (const float4 *)C.pos + s0, perm, m, tmp, tmp + (size_t)cap * a.nr);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(c->ev3, c->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(dg + (size_t)s0 * a.nr, tmp, (size_t)tot * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(vs + (size_t)s0 * a.nr, tmp + (size_t)cap * a.nr, (size_t)tot * sizeof(float),
                         hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    float cms = 0;
    if (e == hipSuccess && hipEventElapsedTime(&cms, c->ev2, c->ev3) == hipSuccess) kms += cms;
  }
  c->stage_ms[ST_SKW] = kms;
  if (e == hipSuccess) e = hipEventRecord(c->ev1, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return clr_fail(c, CLR_ERR_HIP, "source skewers: %s", hipGetErrorString(e));
  return CLR_OK;
}

// ---------------------------------------------------------------------------
// Custom projected maps: cstm_beams_preproc_single +
// cstm_get_beam_properties_single (cstm.c:39-150).  One thread per pixel
// centre (NEST order), the same radial march as kappa with a trilinear
// density read per step.
// ---------------------------------------------------------------------------
namespace {

struct CstmArgs {
  const float *dens;
  int N, ngx, ir_min, ir_max, model, lg;   // 2^lg lanes per pixel
  double idx, dr, ox, oy, oz;
};

// (1 + d)^b for d > -1 (the model-0 branch of bias_model_f64) as exp(b log1p):
// a few 1e-16 relative, and half of pow's instructions; the map is FP32.  Where
// that is NaN (0 x infinity: b = 0 and d infinite, ...) pow decides.
__device__ inline double bias_model_march(double d, double b, int model) {
  if (model == 0) {
    if (d <= -1) return 0.0;
    const double v = exp(b * log1p(d));
    if (v == v) return v;
  }
  return bias_model_f64(d, b, model);
}

// 2^lg consecutive lanes per pixel (lanes_lg), each taking every 2^lg-th step
// (ONE: a lane per pixel); the trilinear density as seven lerps.
template <bool ONE>
__global__ __launch_bounds__(256) void k_cstm(CstmArgs a, const double *__restrict__ kz,
                                              const double *__restrict__ bz, const double *__restrict__ nz,
                                              int64_t nside, int64_t npix, float *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lg = ONE ? 0 : a.lg, sub = ONE ? 0 : (int)(t & ((1 << lg) - 1)), K = 1 << lg;
  const int64_t ip = t >> lg;
  if (ip >= npix) return;
  double u[3];
  pix2vec_nest(nside, ip, u);
  const int N = a.N;
  const size_t ngx = (size_t)a.ngx, plane = (size_t)N * ngx;
  double cval = 0;
  constexpr int U = 2;   // steps in flight
  for (int irr = a.ir_min + sub; irr <= a.ir_max; irr += U * K) {
    float f[U][8];
    double h[U][3];
#pragma unroll
    for (int s = 0; s < U; s++) {
      const double rm = (min(irr + s * K, a.ir_max) + 0.5) * a.dr;
      const double o[3] = {a.ox, a.oy, a.oz};
      int i0[3], i1[3];
#pragma unroll
      for (int ax = 0; ax < 3; ax++) {
        const double xn = (rm * u[ax] + o[ax]) * a.idx;
        const int c = (int)xn;
        h[s][ax] = xn - c;
        i0[ax] = wrap1(c, N);
        i1[ax] = wrap1(c + 1, N);
      }
#pragma unroll
      for (int c = 0; c < 8; c++)
        f[s][c] = a.dens[(size_t)(c & 4 ? i1[2] : i0[2]) * plane + (size_t)(c & 2 ? i1[1] : i0[1]) * ngx +
                         (c & 1 ? i1[0] : i0[0])];
    }
#pragma unroll
    for (int s = 0; s < U; s++) {
      const int j = irr + s * K;
      if (j > a.ir_max) break;
      double e[4];
#pragma unroll
      for (int c = 0; c < 4; c++) e[c] = fma(h[s][0], (double)f[s][2 * c + 1] - (double)f[s][2 * c], (double)f[s][2 * c]);
      const double e0 = fma(h[s][1], e[1] - e[0], e[0]), e1 = fma(h[s][1], e[3] - e[2], e[2]);
      double d = fma(h[s][2], e1 - e0, e0);
      if (d != d) {
        // a corner that is not finite: by the corners' weights, as the reference
        d = 0;
#pragma unroll
        for (int c = 0; c < 8; c++)
          d += (double)f[s][c] * ((c & 4 ? h[s][2] : 1 - h[s][2]) * (c & 2 ? h[s][1] : 1 - h[s][1]) *
                                  (c & 1 ? h[s][0] : 1 - h[s][0]));
      }
      // the reference holds d as flouble before bias_model
      cval += kz[j] * (bias_model_march((double)(float)d, bz[j], a.model) * nz[j] - 1);
    }
  }
  for (int o = 1; o < K; o <<= 1) cval += __shfl_xor(cval, o);
  if (sub == 0) out[ip] = (float)(cval * a.dr);
}

}  // namespace

int clr_launch_cstm(clr_ctx *c, int ipop, int nside, float *out) {
  if (ipop < 0 || ipop >= c->n_tr[CLR_TRACER_CSTM]) return clr_fail(c, CLR_ERR_ARG, "no custom map %d", ipop);
  if (!c->density_done) return clr_fail(c, CLR_ERR_STATE, "density field not computed");
  if (nside < 1 || nside > 8192 || (nside & (nside - 1))) return clr_fail(c, CLR_ERR_ARG, "bad nside %d", nside);
  if (!out) return clr_fail(c, CLR_ERR_ARG, "null output");
  const TracerDev &T = c->tr[CLR_TRACER_CSTM][ipop];
  if (!T.set || !T.norm_set) return clr_fail(c, CLR_ERR_STATE, "custom map %d has no norm table", ipop);
  const int N = c->N, na = c->na;
  if (!(c->r_max > 0)) return clr_fail(c, CLR_ERR_STATE, "tables carry no r_max");
  const int nr = N / 2;
  const double dr = c->r_max / nr;
  // kernel K/IH, bias and norm at each step (cstm.c:87-99), FP64 on the host
  std::vector<double> rr(na), ih(na), kt(na), bt(na), nt(na);
  CLR_HIP(c, hipMemcpy(rr.data(), c->bg, na * sizeof(double), hipMemcpyDeviceToHost));
  CLR_HIP(c, hipMemcpy(ih.data(), c->bg + 5 * (size_t)na, na * sizeof(double), hipMemcpyDeviceToHost));
  CLR_HIP(c, hipMemcpy(kt.data(), T.amp, na * sizeof(double), hipMemcpyDeviceToHost));
  CLR_HIP(c, hipMemcpy(bt.data(), T.bz, na * sizeof(double), hipMemcpyDeviceToHost));
  CLR_HIP(c, hipMemcpy(nt.data(), T.norm, na * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<double> tab(3 * (size_t)nr);
  double kmax = -1e100;
  for (int ir = 0; ir < nr; ir++) {
    const double rm = (ir + 0.5) * dr;
    tab[ir] = f_of_r(rr.data(), kt.data(), c->glob_idr, c->r_last, rm, 0.0, 0.0) /
              f_of_r(rr.data(), ih.data(), c->glob_idr, c->r_last, rm, ih[0], ih[na - 1]);
    tab[nr + ir] = f_of_r(rr.data(), bt.data(), c->glob_idr, c->r_last, rm, bt[0], 1.0);
    tab[2 * nr + ir] = f_of_r(rr.data(), nt.data(), c->glob_idr, c->r_last, rm, T.norm0, T.normf);
    kmax = std::max(kmax, fabs(tab[ir]));
  }
  int ir_min = 0, ir_max = nr - 1;
  for (int ir = 0; ir < nr; ir++)
    if (fabs(tab[ir]) > 1e-4 * kmax) { ir_min = ir; break; }
  for (int ir = nr - 1; ir >= 0; ir--)
    if (fabs(tab[ir]) > 1e-4 * kmax) { ir_max = ir; break; }
  if (ir_max < ir_min) return clr_fail(c, CLR_ERR_ARG, "Custom kernel has no suppport");
  const int64_t npix = 12LL * nside * nside;
  const size_t need = 3 * (size_t)nr * sizeof(double) + (size_t)npix * sizeof(float);
  int rc = clr_ensure(c, &c->misc, &c->misc_n, need);
  if (rc) return rc;
  double *dt = (double *)c->misc;
  float *dout = (float *)(dt + 3 * nr);
  CLR_HIP(c, hipMemcpyAsync(dt, tab.data(), 3 * (size_t)nr * sizeof(double), hipMemcpyHostToDevice, c->stream));
  CstmArgs a{};
  a.dens = c->dens;
  a.N = N;
  a.ngx = c->ngx;
  a.ir_min = ir_min;
  a.ir_max = ir_max;
  a.model = T.model;
  a.lg = lanes_lg(npix, ir_max - ir_min + 1);
  a.idx = N / c->L;
  a.dr = dr;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  CLR_HIP(c, hipEventRecord(c->ev0, c->stream));
  const dim3 g((unsigned)(((npix << a.lg) + 255) / 256));
  if (a.lg == 0)
    hipLaunchKernelGGL(k_cstm<true>, g, dim3(256), 0, c->stream, a, dt, dt + nr, dt + 2 * nr, (int64_t)nside, npix,
                       dout);
  else
    hipLaunchKernelGGL(k_cstm<false>, g, dim3(256), 0, c->stream, a, dt, dt + nr, dt + 2 * nr, (int64_t)nside, npix,
                       dout);
  CLR_HIP(c, hipGetLastError());
  CLR_HIP(c, hipEventRecord(c->ev1, c->stream));
  CLR_HIP(c, hipMemcpyAsync(out, dout, (size_t)npix * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev0, c->ev1);
  c->stage_ms[ST_CSTM] = ms;
  return CLR_OK;
}
