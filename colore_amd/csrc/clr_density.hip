// clr_density.hip -- physical density (density.c:1034-1126) and the per-shell
// bias normalisation (density.c:1128-1393) on gfx950.
//
// k_transform : lognormalize / densclip in place.
// k_shells    : one pass over the grid.  Each wavefront walks tiles of 64-cell
//               rows; per cell the radius, then from packed FP32 tables D(r),
//               z(r) and every b_t(r); the shell index s = (int)(z*idz)+1 is
//               taken from the FP32 z where that is more than 5e-4 of a shell
//               away from a shell edge, otherwise from the reference's FP64
//               expressions (so the counts match bit for bit); then count, z
//               and bias_model(delta, b_t(r)) for every tracer, into FP64
//               registers per shell of the tile, combined once per tile in a
//               fixed order: the sums are bitwise repeatable.  With `fused`
//               the lognormal transform is applied in the same pass (one read
//               and one write of the grid for both stages).
//               Bound by VALU issue: 76 instructions per row of 64 cells (155
//               before) at 4 to 5 wavefronts per SIMD, 65 % of the issue
//               slots.  At 1024^3, three tracers, fused: 3.53 ms (4.85 ms with one
//               current-shell accumulator per lane, flushed by DPP sums at
//               every second change of shell, which also took 0.52 ms at 64^3,
//               now 13 us; 192^3 0.41 -> 0.078, 256^3 0.23 -> 0.078, 512^3
//               0.64 -> 0.41 ms).
// k_shell_final / k_norm_table : fixed-order reduction of the per-block
//               partials, norm = count/sum, edge fill and linear
//               interpolation in z onto the NA r-grid (density.c:1272-1355),
//               all on the device.
#include "clr_internal.h"
#include <math.h>
#include <algorithm>
#include <vector>

using namespace clr;

namespace {

constexpr int kShellBlocks = 8192;
constexpr int kShellThreads = 256;
constexpr int kWaves = kShellThreads / 64;
constexpr int kMaxTr = 8;
constexpr int kRegWin = 4;   // shells of a tile's window (FP64 registers)

struct ShellArgs {
  float *g;
  int N, ngx, nz, ntr, fused, na;
  double dx, ox, oy, oz, idr, r_last, z_last, sigma2, idz;
  const double *r_arr, *zt;
  const double *sigma2_dev;   // when set, sigma^2 is read here instead of `sigma2`
  const float2 *tab;   // [2 + ntr][na]: (value, slope) per bin (k_pack_shell_table)
  float d1_last_f, z_last_f, idr_f, idz_f;
  float bz0[kMaxTr];
  int model[kMaxTr];
  int nbin;              // shell_plan: staged table bins per tile
  int mono;              // z(r) never decreases
};

// FP32 tables of one shell pass as (f_i, f_{i+1} - f_i) per bin i, one row of
// na bins per quantity: 0 = D(r), 1 = z(r), 2 + t = b_t(r); f_i + slope * t is
// the same FP32 value as f_i + (f_{i+1} - f_i) * t.
struct ShellTabSrc {
  const float *d1f;
  const double *zt;
  const float *bzf[kMaxTr];
};
__global__ void k_pack_shell_table(ShellTabSrc src, int na, float2 *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, q = blockIdx.y;
  if (i >= na) return;
  const int j = i + 1 < na ? i + 1 : i;
  float f0, f1;
  if (q == 1) {
    f0 = (float)src.zt[i];
    f1 = (float)src.zt[j];
  } else {
    const float *f = q == 0 ? src.d1f : src.bzf[q - 2];
    f0 = f[i];
    f1 = f[j];
  }
  out[(size_t)q * na + i] = make_float2(f0, f1 - f0);
}

template <int CTRL>
__device__ inline double dpp_get(double v) {
  const int l2 = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
  const int h2 = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(h2, l2);
}

// Sum over each group of G consecutive lanes, in every lane of the group.
template <int G>
__device__ inline double lanes_sum(double x) {
  if (G >= 2) x += dpp_get<0xB1>(x);     // quad_perm [1,0,3,2]
  if (G >= 4) x += dpp_get<0x4E>(x);     // quad_perm [2,3,0,1]
  if (G >= 8) x += dpp_get<0x141>(x);    // row_half_mirror
  if (G >= 16) x += dpp_get<0x140>(x);   // row_mirror
  if (G >= 32) x += __shfl_xor(x, 16);
  if (G >= 64) x += __shfl_xor(x, 32);
  return x;
}

__global__ __launch_bounds__(256) void k_transform(float *__restrict__ g, int N, int ngx, double dx,
                                                   double ox, double oy, double oz,
                                                   const double *__restrict__ r_arr,
                                                   const double *__restrict__ d1, double idr,
                                                   double r_last, double d1_last, double sigma2,
                                                   int dens_type) {
#pragma clang fp contract(off)
  const double obs[3] = {ox, oy, oz};
  const size_t row = blockIdx.x;
  const int iz = (int)(row / N), iy = (int)(row % N);
  float *p = g + row * (size_t)ngx;
  for (int ix = threadIdx.x; ix < N; ix += blockDim.x) {
    double x0, y0, z0;
    const double r = cell_radius(ix, iy, iz, dx, obs, &x0, &y0, &z0);
    const double dg = f_of_r(r_arr, d1, idr, r_last, r, 1.0, d1_last);
    const double delta = p[ix];
    if (dens_type == CLR_DENS_CLIP) {
      p[ix] = (float)(fmax(1 + dg * delta, 0.0) - 1);
    } else {
      const float a = (float)(dg * (delta - 0.5 * dg * sigma2));
      p[ix] = expf(a) - 1.f;
    }
  }
}

// bias_model (common.h:414-431) for the shell sums, on the raw hardware
// exp2/log2 and a fast reciprocal (a few ulp: the sums are of FP32 terms):
//   0: (1+d)^b = exp2(b l2),            l2 = log2(1+d)
//   1: d < 0: exp(b d/(1+d)) = exp2(b q), q = log2(e) d/(1+d); else 1 + b d
//   2: max(1 + b d, 0)
// d <= -1 (or NaN) gives 0.
template <int MODEL>
__device__ inline float bias_sum_term(float d, float l2, float b) {
  float v;
  if (MODEL == 0) {
    v = __builtin_amdgcn_exp2f(b * l2);
  } else {
    v = fmaxf(__builtin_fmaf(b, d, 1.f), 0.f);
    if (MODEL == 1) {
      const float q = 1.44269504f * d * __builtin_amdgcn_rcpf(1.f + d);
      const float e = __builtin_amdgcn_exp2f(b * q);
      v = d < 0.f ? e : v;
    }
  }
  return d > -1.f ? v : 0.f;
}

// z(r) of cell (ix,iy,iz) by the reference's FP64 expressions (density.c:
// 1084-1094, f_of_r_linear).
__device__ inline double cell_z_f64(const ShellArgs &a, int ix, int iy, int iz) {
#pragma clang fp contract(off)
  const double obs[3] = {a.ox, a.oy, a.oz};
  double x0, y0, z0;
  const double r = cell_radius(ix, iy, iz, a.dx, obs, &x0, &y0, &z0);
  return f_of_r(a.r_arr, a.zt, a.idr, a.r_last, r, 0.0, a.z_last);
}

// M0: every tracer uses bias model 0 (no other model's code in the loop).
// A tile is ROWS rows along y of TX x TZ (x, z) cells, TX TZ = 64 (TX = 4:
// one row of 4 x 4 x 4 cells); STAGE: its part of the r-tables is staged in
// LDS (see shell_plan).
//
// A lane adds its cells, in the program's order, to FP64 registers, one set
// per shell of the tile's window (kRegWin shells), and at the end of a tile
// the 64 lanes of a (shell, quantity) are added up through LDS in a fixed
// order: the sums repeat bit for bit, and the loop has no test for a change of
// shell.  A tile that spans more shells takes further passes; one outside the
// last shell (48 % of a box) only gets its lognormal transform.
template <int NT, bool M0, int TX, int ROWS, bool STAGE>
__global__ __launch_bounds__(kShellThreads) __attribute__((amdgpu_waves_per_eu(NT <= 2 ? 5 : (NT <= 4 ? 4 : 2)))) void
k_shells(ShellArgs a, double *__restrict__ partial) {
  constexpr int NQ = 2 + NT, NF = 1 + NT;
  constexpr bool CUBE = TX == 4;
  constexpr int TY = CUBE ? 4 : 1, TZ = 64 / (TX * TY);
  constexpr int U = ROWS > 1 ? 2 : 1;   // rows worked together
  extern __shared__ double acc[];
  const int nz = a.nz, N = a.N, nbin = a.nbin;
  const int nwaves = blockDim.x / 64, lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  double *myacc = acc + (size_t)wave * nz * NQ;
  // the wavefront's LDS: one shell's [NF][64] sums and the tile's part of the
  // tables, [NQ][nbin] (value, slope)
  double *wsum = acc + (size_t)nwaves * nz * NQ + (size_t)wave * (NF * 64 + nbin * NQ);
  float2 *seg = (float2 *)(wsum + NF * 64);
  for (int i = threadIdx.x; i < nwaves * nz * NQ; i += blockDim.x) acc[i] = 0;
  __syncthreads();
  const float ox = (float)a.ox, oy = (float)a.oy, oz = (float)a.oz, dxf = (float)a.dx;
  const float s2f = (float)(a.sigma2_dev ? *a.sigma2_dev : a.sigma2);
  const int ntx = N / TX, nty = N / (TY * ROWS), ntz = N / TZ;
  const int ntiles = ntx * nty * ntz;
  const int nw = (int)gridDim.x * nwaves;
  for (int tile = (int)blockIdx.x * nwaves + wave; tile < ntiles; tile += nw) {
    const int tx = tile % ntx, rest = tile / ntx;
    const int ty = rest % nty, tz = rest / nty;
    const int ix = tx * TX + lane % TX, iy0 = ty * TY * ROWS + (lane / TX) % TY, iz = tz * TZ + lane / (TX * TY);
    float *const tb = a.g + ((size_t)iz * N + iy0) * a.ngx + ix;
    const int ystep = TY * a.ngx;
    // densities of U rows, and of the U after them (two groups ahead in the
    // loops below)
    float d[U], dn[U];
    auto load = [&](int r, float *v) {
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = tb[(r + u) * ystep];
    };
    load(0, d);
    if (ROWS > U) load(U, dn);
    auto next = [&](int r) {   // after the rows r .. r+U-1
#pragma unroll
      for (int u = 0; u < U; u++) d[u] = dn[u];
      if (r + 2 * U < ROWS) load(r + 2 * U, dn);
    };
    // table bins and shells that the tile's radii can fall in: its nearest
    // and farthest point, 1e-5 of the radius and 0.01 shell further out
    int s_lo, s_hi, b_lo, nb;
    bool edge;
    {
      const float xa = coord_f32(tx * TX, dxf, ox), xb = coord_f32(tx * TX + TX - 1, dxf, ox);
      const float ya = coord_f32(ty * TY * ROWS, dxf, oy), yb = coord_f32((ty + 1) * TY * ROWS - 1, dxf, oy);
      const float za = coord_f32(tz * TZ, dxf, oz), zb = coord_f32(tz * TZ + TZ - 1, dxf, oz);
      const float xn = fmaxf(fmaxf(xa, -xb), 0.f), yn = fmaxf(fmaxf(ya, -yb), 0.f), zn = fmaxf(fmaxf(za, -zb), 0.f);
      const float xf = fmaxf(-xa, xb), yf = fmaxf(-ya, yb), zf = fmaxf(-za, zb);
      const float rlo = radius_f32(xn, yn, zn) * (1.f - 1e-5f), rhi = radius_f32(xf, yf, zf) * (1.f + 1e-5f);
      const TabPos plo = tab_pos_f32(rlo, a.idr_f, a.na), phi = tab_pos_f32(rhi, a.idr_f, a.na);
      edge = plo.e0 || phi.e1;
      const int i_lo = plo.e1 ? a.na - 1 : plo.i0, i_hi = phi.e1 ? a.na - 1 : phi.i0;
      if (a.mono) {
        const float2 tl = a.tab[a.na + plo.i0], th = a.tab[a.na + phi.i0];
        const float zl = plo.e0 ? 0.f : (plo.e1 ? a.z_last_f : tl.x + tl.y * plo.tq);
        const float zh = phi.e0 ? 0.f : (phi.e1 ? a.z_last_f : th.x + th.y * phi.tq);
        s_lo = (int)(zl * a.idz_f - 0.01f) + 1;
        s_hi = (int)(zh * a.idz_f + 0.01f) + 1;
      } else {
        s_lo = 0;
        s_hi = nz - 1;
      }
      s_lo = __builtin_amdgcn_readfirstlane(max(s_lo, 0));
      s_hi = __builtin_amdgcn_readfirstlane(min(s_hi, nz - 1));
      b_lo = __builtin_amdgcn_readfirstlane(i_lo);
      nb = __builtin_amdgcn_readfirstlane(i_hi - i_lo + 1);
      edge = __builtin_amdgcn_readfirstlane((int)edge) != 0;
    }
    const bool inside = s_lo < nz;
    if (!inside && !a.fused) continue;
    if (STAGE) {
      nb = min(nb, nbin);
      for (int q = 0; q < (inside ? NQ : 1); q++)
        for (int i = lane; i < nb; i += 64) seg[q * nbin + i] = a.tab[q * a.na + b_lo + i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    // (value, slope) of quantity q at a cell's bin; an entry past the tile's
    // bins is only looked up for cells at the table's ends, which take the
    // edge values
    auto entry = [&](const TabPos &p, int q) {
      if (!STAGE) return a.tab[q * a.na + p.i0];
      return seg[q * nbin + (int)min((unsigned)(p.i0 - b_lo), (unsigned)(nb - 1))];
    };
    const float x32 = coord_f32(ix, dxf, ox), z32 = coord_f32(iz, dxf, oz), z2 = z32 * z32;
    // the lane's cell in row r: x, z fixed, y = iy0 + TY r.  With TY = 1 the
    // row's y is the wavefront's: lane r holds row r's y
    const float yl = CUBE ? 0.f : coord_f32(iy0 + lane, dxf, oy);
    auto radius_at = [&](int r) {
      const float y32 = CUBE ? coord_f32(iy0 + TY * r, dxf, oy)
                             : __int_as_float(__builtin_amdgcn_readlane(__float_as_int(yl), r));
      return __builtin_amdgcn_sqrtf(__builtin_fmaf(x32, x32, __builtin_fmaf(y32, y32, z2)));
    };
    // table position in row r (TY rows of a cube's row share ty)
    auto pos_at = [&](int r) { return cell_tab_pos_f32(radius_at(r), a.idr_f, a.na, ty * TY * ROWS + r); };
    if (!inside) {
      // no shell in reach: the transform alone
#pragma unroll 1
      for (int r = 0; r < ROWS; r += U) {
        float o[U];
#pragma unroll
        for (int u = 0; u < U; u++) o[u] = d[u];
        next(r);
#pragma unroll
        for (int u = 0; u < U; u++) {
          const TabPos p = pos_at(r + u);
          const float2 e = entry(p, 0);
          o[u] = lognormal_f32(o[u], growth_at(p, e.x, e.y, a.d1_last_f), s2f);
        }
#pragma unroll
        for (int u = 0; u < U; u++) tb[(r + u) * ystep] = o[u];
      }
      continue;
    }
    // the tile's shells, kRegWin at a time (later passes use the transformed
    // cells)
    for (int wb = s_lo; wb <= s_hi; wb += kRegWin) {
      const int wn = min(kRegWin, nz - wb);
      const bool fuse = a.fused && wb == s_lo;
      double ra[kRegWin][NF];
      uint32_t rc[kRegWin];
#pragma unroll
      for (int k = 0; k < kRegWin; k++) {
        rc[k] = 0u;
#pragma unroll
        for (int q = 0; q < NF; q++) ra[k][q] = 0;
      }
      if (wb != s_lo) {   // a later pass: the rows once more
        load(0, d);
        if (ROWS > U) load(U, dn);
      }
      {
#pragma unroll 1
        for (int g = 0; g < ROWS; g += U) {
          TabPos tp[U];
          float2 C[U][NQ];
#pragma unroll
          for (int u = 0; u < U; u++) {
            tp[u] = pos_at(g + u);
#pragma unroll
            for (int q = 0; q < NQ; q++) C[u][q] = entry(tp[u], q);
          }
          // the U rows step by step, so that their dependent chains interleave
          float comp[U][NQ], dl[U];
          bool ends[U];   // at the table's ends: the reference's edge values
#pragma unroll
          for (int u = 0; u < U; u++) {
#pragma unroll
            for (int q = 0; q < NQ; q++) comp[u][q] = __builtin_fmaf(C[u][q].y, tp[u].tq, C[u][q].x);
            dl[u] = d[u];
            ends[u] = false;
          }
          next(g);
          if (edge) {
#pragma unroll
            for (int u = 0; u < U; u++) {
              ends[u] = tp[u].e0 || tp[u].e1;
              comp[u][0] = tp[u].e0 ? 1.f : (tp[u].e1 ? a.d1_last_f : comp[u][0]);
              comp[u][1] = tp[u].e0 ? 0.f : (tp[u].e1 ? a.z_last_f : comp[u][1]);
#pragma unroll
              for (int t = 0; t < NT; t++) comp[u][2 + t] = tp[u].e0 ? a.bz0[t] : (tp[u].e1 ? 1.f : comp[u][2 + t]);
            }
          }
          if (fuse) {
            // the same float as lognormal_f32 of the fused count pass
#pragma unroll
            for (int u = 0; u < U; u++) dl[u] = lognormal_f32(dl[u], comp[u][0], s2f);
#pragma unroll
            for (int u = 0; u < U; u++) tb[(g + u) * ystep] = dl[u];
          }
          // shell index: FP32 z (error < 5e-5 shell) unless within 5e-4
          // shell of an edge (or at the table ends), where the reference's
          // FP64 radius and z decide
          double zz[U];
          int ind[U];
          bool near[U], any = false;
#pragma unroll
          for (int u = 0; u < U; u++) {
            zz[u] = (double)comp[u][1];
            const float sf = comp[u][1] * a.idz_f;
            ind[u] = (int)sf + 1;
            near[u] = ends[u] || !(fabsf(__builtin_amdgcn_fractf(sf) - 0.5f) < 0.5f - 5e-4f);
            any = any || near[u];
          }
          if (any) {
#pragma unroll
            for (int u = 0; u < U; u++)
              if (near[u]) {
                zz[u] = cell_z_f64(a, ix, iy0 + TY * (g + u), iz);
                ind[u] = (int)(zz[u] * a.idz) + 1;
              }
          }
          float term[U][NT > 0 ? NT : 1], l2[U];
#pragma unroll
          for (int u = 0; u < U; u++) l2[u] = __builtin_amdgcn_logf(1.f + dl[u]);
#pragma unroll
          for (int t = 0; t < NT; t++) {
            if (M0 || a.model[t] == 0) {
#pragma unroll
              for (int u = 0; u < U; u++) term[u][t] = bias_sum_term<0>(dl[u], l2[u], comp[u][2 + t]);
            } else if (a.model[t] == 1) {
#pragma unroll
              for (int u = 0; u < U; u++) term[u][t] = bias_sum_term<1>(dl[u], l2[u], comp[u][2 + t]);
            } else {
#pragma unroll
              for (int u = 0; u < U; u++) term[u][t] = bias_sum_term<2>(dl[u], l2[u], comp[u][2 + t]);
            }
          }
#pragma unroll
          for (int u = 0; u < U; u++) {
            const unsigned slot = (unsigned)(ind[u] - wb);
#pragma unroll
            for (int k = 0; k < kRegWin; k++)
              if (slot == (unsigned)k) {
                rc[k]++;
                ra[k][0] += zz[u];
#pragma unroll
                for (int t = 0; t < NT; t++) ra[k][1 + t] += (double)term[u][t];
              }
          }
        }
      }
      // the window's rows into the wavefront's accumulators
      constexpr int P = NF > 8 ? 16 : (NF > 4 ? 8 : (NF > 2 ? 4 : NF)), G = 64 / P;   // G lanes per quantity
      const int q = lane / G, part = lane % G;
#pragma unroll
      for (int k = 0; k < kRegWin; k++) {
        if (k >= wn || __ballot(rc[k] != 0u) == 0ull) continue;
#pragma unroll
        for (int f = 0; f < NF; f++) wsum[f * 64 + lane] = ra[k][f];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        double v = 0;
        if (q < NF)
#pragma unroll
          for (int j = 0; j < P; j++) v += wsum[q * 64 + G * j + part];
        v = lanes_sum<G>(v);
        int n = (int)rc[k];
        for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
        if (part == 0 && q < NF) myacc[(wb + k) * NQ + 1 + q] += v;
        if (lane == 0) myacc[(wb + k) * NQ] += (double)n;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  __syncthreads();
  double *out = partial + (size_t)blockIdx.x * nz * NQ;
  for (int i = threadIdx.x; i < nz * NQ; i += blockDim.x) {
    double v = 0;
    for (int w = 0; w < nwaves; w++) v += acc[(size_t)w * nz * NQ + i];
    out[i] = v;
  }
}

// ---------------------------------------------------------------------------
// k_shell_moments: the surrogate's read-only pass over the Gaussian grid.
// A work item is 256 consecutive x cells of one y row (4 per lane, one float4
// load) walked over zrun consecutive z planes: the wavefront reads 1 KB
// contiguous per plane (kMomPre planes in flight; 8 cells per lane, 2 KB,
// measured the same) and a lane's radius changes slowly,
// so it sums its current shell in FP32 registers and, when the shell
// changes, adds those sums to the wavefront's FP64 accumulators in LDS with
// atomics (lanes cross shell edges at different planes, so few collide).
// A lane's D(r) over its item is the quadratic through the FP64 table's
// values at its nearest, middle and farthest radius; the item's z length is
// chosen so that a lane spans at most ~160 Mpc/h, over which the quadratic
// is within ~1e-6 of the table (these are inputs of an approximation).  Per
// block the wavefronts' sums go to partial[block][nz][kMomQ], reduced in
// fixed order by k_shell_final.
// ---------------------------------------------------------------------------
constexpr int kMomQ = 6;            // count, G, G^2, G^3, G^4, D^2
constexpr int kMomBlocks = 4096;
constexpr int kMomMaxShells = 256;
constexpr int kMomZMax = 32;        // z planes per item, at most
constexpr int kMomPre = 8;          // planes loaded ahead (the item length is a multiple)
constexpr int kMomCPL = 4;          // x cells per lane (float4 loads)
constexpr int kMomXW = 64 * kMomCPL;  // x cells per item

struct MomArgs {
  const float *g;
  const double *r_arr, *d1;   // FP64 tables (f_of_r)
  const float *edge;          // nz FP32 edge radii
  int N, ngx, nz, zrun;
  double idr, r_last, d_last;
  float dxf, ox, oy, oz;
};

// largest s in [1, nz] with edge[s-1] <= r (s = nz: past the last shell)
__device__ inline int mom_shell(const float *edge, int nz, float r) {
  int lo = 1, hi = nz;
  while (hi > lo) {
    const int m = (lo + hi + 1) / 2;
    if (edge[m - 1] <= r) lo = m; else hi = m - 1;
  }
  return lo;
}

template <bool FULL>
__global__ __launch_bounds__(kShellThreads) void k_shell_moments(MomArgs a, double *__restrict__ partial) {
  extern __shared__ double macc[];   // [wave][nz][kMomQ] FP64, then nz FP32 edges
  const int nz = a.nz, N = a.N;
  float *ledge = (float *)(macc + (size_t)kWaves * nz * kMomQ);
  for (int i = threadIdx.x; i < kWaves * nz * kMomQ; i += blockDim.x) macc[i] = 0;
  for (int i = threadIdx.x; i < nz; i += blockDim.x) ledge[i] = a.edge[i];
  __syncthreads();
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  double *myacc = macc + (size_t)wave * nz * kMomQ;
  const int zrun = a.zrun;
  const int nxc = (N + kMomXW - 1) / kMomXW, nzc = (N + zrun - 1) / zrun;
  const long nwork = (long)nxc * N * nzc;
  const long nw = (long)gridDim.x * kWaves;
  const size_t plane = (size_t)N * a.ngx;
  for (long w = (long)blockIdx.x * kWaves + wave; w < nwork; w += nw) {
    const int xc = (int)(w % nxc);
    const long rest = w / nxc;
    const int iy = (int)(rest % N), zc = (int)(rest / N);
    const int ix = xc * kMomXW + lane * kMomCPL, iz0 = zc * zrun;   // the lane's cells: ix .. ix+kMomCPL-1
    const int nzi = FULL ? zrun : min(zrun, N - iz0);
    const bool valid = FULL || ix < N;   // N is a multiple of kMomCPL
    // D(r) on the lane's cells: quadratic through the table at its radius
    // range
    double c0, c1, c2;
    {
      const double xa = (valid ? ix : 0) * (double)a.dxf - a.ox, xb = xa + (kMomCPL - 1) * (double)a.dxf;
      const double yy = iy * (double)a.dxf - a.oy;
      const double za = iz0 * (double)a.dxf - a.oz, zb = (iz0 + nzi - 1) * (double)a.dxf - a.oz;
      const double dxn = xa > 0 ? xa : (xb < 0 ? -xb : 0), dzn = za > 0 ? za : (zb < 0 ? -zb : 0);
      const double r0 = sqrt(dxn * dxn + yy * yy + dzn * dzn);
      const double r2 = sqrt(fmax(xa * xa, xb * xb) + yy * yy + fmax(za * za, zb * zb));
      const double r1 = 0.5 * (r0 + r2);
      const double f0 = f_of_r(a.r_arr, a.d1, a.idr, a.r_last, r0, 1.0, a.d_last);
      const double f1 = f_of_r(a.r_arr, a.d1, a.idr, a.r_last, r1, 1.0, a.d_last);
      const double f2 = f_of_r(a.r_arr, a.d1, a.idr, a.r_last, r2, 1.0, a.d_last);
      const double h = r1 - r0;
      if (h > 1e-3) {
        // D(r) = f0 + (r - r0) (d01 + (r - r1) d012)
        const double d01 = (f1 - f0) / h, d012 = ((f2 - f1) / h - d01) / (2 * h);
        c2 = d012;
        c1 = d01 - d012 * (r0 + r1);
        c0 = f0 - r0 * d01 + d012 * r0 * r1;
      } else {
        c0 = f0; c1 = 0; c2 = 0;
      }
    }
    const float q0 = (float)c0, q1 = (float)c1, q2 = (float)c2;
    const float y = coord_f32(iy, a.dxf, a.oy);
    float rho2[kMomCPL];
#pragma unroll
    for (int k = 0; k < kMomCPL; k++) {
      const float x = coord_f32(valid ? ix + k : 0, a.dxf, a.ox);
      rho2[k] = __builtin_fmaf(x, x, y * y);
    }
    constexpr int V = kMomCPL / 4;   // float4 per lane and plane
    const float4 *col = (const float4 *)(a.g + ((size_t)iz0 * N + iy) * a.ngx + (valid ? ix : 0));
    const size_t plane4 = plane / 4;
    int key = -1;
    float e_lo = 0.f, e_hi = 0.f;
    float acc[kMomQ];
#pragma unroll
    for (int q = 0; q < kMomQ; q++) acc[q] = 0.f;
    float4 vq[kMomPre][V];
#pragma unroll
    for (int j = 0; j < kMomPre; j++)
#pragma unroll
      for (int v = 0; v < V; v++)
        vq[j][v] = (valid && (FULL || j < nzi)) ? col[(size_t)j * plane4 + v] : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j0 = 0; j0 < nzi; j0 += kMomPre) {
#pragma unroll
      for (int u = 0; u < kMomPre; u++) {
        const int j = j0 + u;
        float dls[kMomCPL];
#pragma unroll
        for (int v = 0; v < V; v++) {
          dls[4 * v] = vq[u][v].x;
          dls[4 * v + 1] = vq[u][v].y;
          dls[4 * v + 2] = vq[u][v].z;
          dls[4 * v + 3] = vq[u][v].w;
        }
        if (valid && (FULL ? j0 + kMomPre < zrun : j + kMomPre < nzi)) {
#pragma unroll
          for (int v = 0; v < V; v++) vq[u][v] = col[(size_t)(j + kMomPre) * plane4 + v];
        }
        if (FULL || (j < nzi && valid)) {
          const float zc2 = coord_f32(iz0 + j, a.dxf, a.oz);
#pragma unroll
          for (int k = 0; k < kMomCPL; k++) {
            const float r = __builtin_amdgcn_sqrtf(__builtin_fmaf(zc2, zc2, rho2[k]));
            if (!(r >= e_lo && r < e_hi)) {
              if (key >= 1 && key < nz) {
#pragma unroll
                for (int q = 0; q < kMomQ; q++) atomicAdd(&myacc[key * kMomQ + q], (double)acc[q]);
              }
#pragma unroll
              for (int q = 0; q < kMomQ; q++) acc[q] = 0.f;
              key = mom_shell(ledge, nz, r);
              e_lo = ledge[key - 1];
              e_hi = key < nz ? ledge[key] : 3.0e38f;
            }
            if (key < nz) {
              const float D = __builtin_fmaf(r, __builtin_fmaf(r, q2, q1), q0);
              const float G = D * dls[k], G2 = G * G;
              acc[0] += 1.f;
              acc[1] += G;
              acc[2] += G2;
              acc[3] = __builtin_fmaf(G2, G, acc[3]);
              acc[4] = __builtin_fmaf(G2, G2, acc[4]);
              acc[5] = __builtin_fmaf(D, D, acc[5]);
            }
          }
        }
      }
    }
    if (key >= 1 && key < nz) {
#pragma unroll
      for (int q = 0; q < kMomQ; q++) atomicAdd(&myacc[key * kMomQ + q], (double)acc[q]);
    }
  }
  __syncthreads();
  double *out = partial + (size_t)blockIdx.x * nz * kMomQ;
  for (int i = threadIdx.x; i < nz * kMomQ; i += blockDim.x) {
    double t = 0;
    for (int w2 = 0; w2 < kWaves; w2++) t += macc[(size_t)w2 * nz * kMomQ + i];
    out[i] = t;
  }
}

// out[i] = sum over blocks of partial[b][i], one 256-thread block per value,
// fixed-order tree: deterministic.
__global__ __launch_bounds__(256) void k_shell_final(const double *__restrict__ partial, int nblocks, int nvals,
                                                     double *__restrict__ out) {
  __shared__ double s[256];
  const int i = blockIdx.x;
  double v = 0;
  for (int b = threadIdx.x; b < nblocks; b += 256) v += partial[(size_t)b * nvals + i];
  s[threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[i] = s[0];
}

// Per tracer t: norm table on the NA r-grid.  sums = [nz][nq] from
// k_shell_final.
constexpr int kNormMaxShells = 1024;
struct NormOuts {
  double *p[3 * CLR_NPOP_MAX];
  double *e[3 * CLR_NPOP_MAX];   // optional per-tracer copies of (norm0, normf)
};

// Every tracer's norm table in one launch: blockIdx.y is the tracer, the x
// blocks split the NA entries; each block rebuilds the tracer's (z, norm)
// nodes in LDS from the FP64 shell sums.
__global__ __launch_bounds__(256) void k_norm_table(const double *__restrict__ sums, int nz, int nq, double zmax,
                                                   const double *__restrict__ r_arr, const double *__restrict__ zt,
                                                   double idr, double r_last, double z_last, int na, NormOuts outs,
                                                   double *__restrict__ edges) {
#pragma clang fp contract(off)
  __shared__ double zarr[kNormMaxShells], nrm[kNormMaxShells];
  const int t = blockIdx.y;
  for (int iz = threadIdx.x; iz < nz; iz += blockDim.x) {
    const double n = sums[iz * nq + 0];
    zarr[iz] = sums[iz * nq + 1];
    nrm[iz] = sums[iz * nq + 2 + t];
    if (n > 0) {
      zarr[iz] /= n;
      nrm[iz] = n / nrm[iz];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    zarr[0] = 0;
    zarr[nz - 1] = zmax;
    nrm[0] = nrm[1];
    nrm[nz - 1] = nrm[nz - 2];
    if (blockIdx.x == 0) {
      edges[2 * t] = nrm[0];
      edges[2 * t + 1] = nrm[nz - 1];
      if (outs.e[t]) {
        outs.e[t][0] = nrm[0];
        outs.e[t][1] = nrm[nz - 1];
      }
    }
  }
  __syncthreads();
  const double z0 = zarr[0], zf = zarr[nz - 1];
  const double n0 = nrm[0], nf = nrm[nz - 1];
  double *__restrict__ norm_out = outs.p[t];
  const int ii = blockIdx.x * blockDim.x + threadIdx.x;
  if (ii >= na) return;
  {
    const double z = f_of_r(r_arr, zt, idr, r_last, r_arr[ii], 0.0, z_last);
    double nm;
    if (z < z0) nm = n0;
    else if (z >= zf) nm = nf;
    else {
      int lo = 0, hi = nz - 1;
      while (hi > lo + 1) {
        const int i = (hi + lo) / 2;
        if (zarr[i] > z) hi = i; else lo = i;
      }
      const double xl = zarr[lo], xh = zarr[lo + 1];
      const double dxz = xh - xl;
      nm = dxz > 0.0 ? nrm[lo] + (z - xl) / dxz * (nrm[lo + 1] - nrm[lo]) : 0.0;
    }
    norm_out[ii] = nm;
  }
}

// The tiling of a shell pass: the largest tile that spans at most kRegWin
// shells (from its diagonal and the narrowest shell), since a tile's fixed
// costs -- its bounds, the staging, the sums at its end -- are of the order of
// two rows' work.  16 x 16 x 4 and 16 x 8 x 4 cells with their table bins in
// LDS while a wavefront's LDS stays within 10 KB (16 wavefronts per CU); then
// 8 x 4 x 8 cells, too few for the staging to pay; then 4 x 4 x 4, which span
// the fewest shells (64^3 .. 192^3 of a deep box, where further passes may be
// needed all the same).
struct ShellPlan {
  int kind, nbin, waves, blocks;
  size_t lds;
};
constexpr int kShellTile[4][4] = {{4, 4, 4, 0}, {8, 4, 8, 0}, {16, 8, 4, 1}, {16, 16, 4, 1}};   // cells in x, y, z; staged
// Shells x tracers are limited to what four wavefronts' accumulators and one
// logged shell per lane (a sum per quantity and an index) fit the LDS with.
int shell_plan(clr_ctx *c, int nz, int NT, ShellPlan &p) {
  if (kWaves * ((size_t)(nz + 64) * (2 + NT) * sizeof(double) + 64 * sizeof(int)) > 160 * 1024) return CLR_ERR_ARG;
  if (c->shell_dr <= 0) {
    // narrowest shell below r(L/2), and whether z(r) never decreases
    const std::vector<double> &zz = c->h_z, &rr = c->h_r;
    const double dz = c->zmax_half_box / (nz - 2);
    double last = 0, narrow = 1e300;
    int k = 1;
    c->shell_mono = 1;
    for (int i = 1; i < c->na; i++) {
      if (!(zz[i] >= zz[i - 1])) c->shell_mono = 0;
      while (k < nz - 1 && zz[i] >= k * dz) {
        narrow = std::min(narrow, rr[i] - last);
        last = rr[i];
        k++;
      }
    }
    c->shell_dr = std::max(std::min(narrow, c->L), 1e-3 * c->dx);
  }
  size_t winb = 0;
  int cells = 64;
  for (p.kind = 3; p.kind >= 0; p.kind--) {
    const int *t = kShellTile[p.kind];
    const double d = c->dx * sqrt((t[0] - 1.) * (t[0] - 1.) + (t[1] - 1.) * (t[1] - 1.) + (t[2] - 1.) * (t[2] - 1.));
    p.nbin = t[3] ? (int)std::min((double)c->na, ceil((d + 4e-5 * c->L) * c->glob_idr) + 3) : 0;
    winb = (size_t)(1 + NT) * 64 * sizeof(double) + (size_t)p.nbin * (2 + NT) * sizeof(float2);
    cells = t[0] * t[1] * t[2];
    if (p.kind == 0 || (ceil(d / c->shell_dr) + 1 <= kRegWin && winb <= 10 * 1024)) break;
  }
  const size_t accb = (size_t)nz * (2 + NT) * sizeof(double);
  for (p.waves = kWaves; p.waves > 1 && p.waves * (accb + winb) > 160 * 1024;) p.waves /= 2;
  p.lds = p.waves * (accb + winb);
  const long tiles = (long)c->N * c->N * c->N / cells;
  p.blocks = (int)std::min<long>(kShellBlocks, (tiles + p.waves - 1) / p.waves);
  return p.lds <= 160 * 1024 ? CLR_OK : CLR_ERR_ARG;
}

template <int NT, bool M0, int TX, int ROWS, bool STAGE>
void launch_shells(const ShellPlan &p, hipStream_t s, const ShellArgs &a, double *partial) {
  if (p.lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void *)k_shells<NT, M0, TX, ROWS, STAGE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
  hipLaunchKernelGGL((k_shells<NT, M0, TX, ROWS, STAGE>), dim3(p.blocks), dim3(64 * p.waves), p.lds, s, a, partial);
}
using ShellFn = void (*)(const ShellPlan &, hipStream_t, const ShellArgs &, double *);
#define CLR_SHELL_FNS(...)                                                                                  \
  {launch_shells<0, __VA_ARGS__>, launch_shells<1, __VA_ARGS__>, launch_shells<2, __VA_ARGS__>,             \
   launch_shells<3, __VA_ARGS__>, launch_shells<4, __VA_ARGS__>, launch_shells<5, __VA_ARGS__>,             \
   launch_shells<6, __VA_ARGS__>, launch_shells<7, __VA_ARGS__>, launch_shells<8, __VA_ARGS__>}
const ShellFn kShellFns[2][4][kMaxTr + 1] = {
    {CLR_SHELL_FNS(false, 4, 1, false), CLR_SHELL_FNS(false, 8, 4, false), CLR_SHELL_FNS(false, 16, 8, true),
     CLR_SHELL_FNS(false, 16, 16, true)},
    {CLR_SHELL_FNS(true, 4, 1, false), CLR_SHELL_FNS(true, 8, 4, false), CLR_SHELL_FNS(true, 16, 8, true),
     CLR_SHELL_FNS(true, 16, 16, true)}};
#undef CLR_SHELL_FNS

// Runs the shell pass and its fixed-order reduction (fin[nz][2 + ntr]).
int run_shells(clr_ctx *c, hipStream_t s, ShellArgs &a, bool all0, double *partial, double *fin, hipEvent_t after) {
  ShellPlan p;
  const int rc = shell_plan(c, a.nz, a.ntr, p);
  if (rc) return clr_fail(c, rc, "too many shells x tracers (%d x %d)", a.nz, a.ntr);
  a.nbin = p.nbin;
  a.mono = c->shell_mono;
  kShellFns[all0 ? 1 : 0][p.kind][a.ntr](p, s, a, partial);
  CLR_HIP(c, hipGetLastError());
  if (after) CLR_HIP(c, hipEventRecord(after, s));
  const int nvals = a.nz * (2 + a.ntr);
  hipLaunchKernelGGL(k_shell_final, dim3((unsigned)nvals), dim3(256), 0, s, partial, p.blocks, nvals, fin);
  CLR_HIP(c, hipGetLastError());
  return CLR_OK;
}

}  // namespace

int clr_launch_density(clr_ctx *c, int dens_type, double sigma2) {
  if (!c->have_fields) return clr_fail(c, CLR_ERR_STATE, "clr_gaussian_fields must run first");
  if (dens_type != CLR_DENS_LOGNORMAL && dens_type != CLR_DENS_CLIP)
    return clr_fail(c, CLR_ERR_ARG, "Density type %d not supported", dens_type);
  const int N = c->N;
  const double *r = c->bg, *d1 = c->bg + 2 * c->na;
  CLR_HIP(c, hipEventRecord(c->ev0, c->stream));
  hipLaunchKernelGGL(k_transform, dim3((unsigned)((size_t)N * N)), dim3(N >= 256 ? 256 : N), 0, c->stream,
                     c->dens, N, c->ngx, c->dx, c->obs[0], c->obs[1], c->obs[2], r, d1, c->glob_idr,
                     c->r_last, c->h_bg_last[2], sigma2, dens_type);
  CLR_HIP(c, hipGetLastError());
  CLR_HIP(c, hipEventRecord(c->ev1, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev0, c->ev1);
  c->stage_ms[ST_DENS] = ms;
  c->density_done = 1;
  c->norms_done = 0;
  return CLR_OK;
}

// ---------------------------------------------------------------------------
// Static scratch of the no-allocation variant (clr_shell_norms_noalloc):
// the per-block FP64 partials of k_shells, the final sums, k_norm_table's
// edge values and the packed FP32 table, for nz (2 + ntr) <= kNoAllocVals.
// One copy per GPU for the life of the process; host code reaches it only
// through the address hipGetSymbolAddress returns on that device.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocVals = 320;
constexpr size_t kNoAllocTabFloat4 = (size_t)CLR_NA * (2 + kMaxTr) / 2;
constexpr size_t kNoAllocDoubles = (size_t)kShellBlocks * kNoAllocVals + kNoAllocVals + 2 * (size_t)kMaxTr;
constexpr size_t kNoAllocBytes = (kNoAllocDoubles * sizeof(double) + 255) / 256 * 256 + kNoAllocTabFloat4 * 16;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

size_t clr_noalloc_scratch_bytes() { return kNoAllocBytes; }

int clr_noalloc_scratch_lookup(void **ptr) {
  return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch)) == hipSuccess ? 0 : -1;
}

int clr_launch_norms(clr_ctx *c, int lognormal_fused, double sigma2, int cap, int *nz_out,
                     unsigned long long *counts, double *zsum, double *sums, void *scratch_base) {
  if (!c->have_fields) return clr_fail(c, CLR_ERR_STATE, "clr_gaussian_fields must run first");
  if (lognormal_fused && c->density_done)
    return clr_fail(c, CLR_ERR_STATE, "density already transformed; call with lognormal_fused=0");
  if (!lognormal_fused && !c->density_done)
    return clr_fail(c, CLR_ERR_STATE, "clr_density must run first (or use lognormal_fused)");
  const int N = c->N, na = c->na;
  const double *r = c->bg, *zt = c->bg + na;
  const double z_last = c->h_bg_last[1];

  // shells: zmax = z(L/2), nz = (int)(zmax/DZ_SIGMA)+2, idz = (nz-2)/zmax
  const double zmax = c->zmax_half_box;
  const int nz = (int)(zmax / 0.05) + 2;
  if (nz > kNormMaxShells) return clr_fail(c, CLR_ERR_ARG, "%d redshift shells (at most %d)", nz, kNormMaxShells);
  const double idz = (nz - 2) / zmax;

  ShellArgs a{};
  ShellTabSrc tsrc{};
  int tk[3 * CLR_NPOP_MAX], tp[3 * CLR_NPOP_MAX];
  int ntr = 0;
  for (int k = 0; k < 3; k++)
    for (int i = 0; i < c->n_tr[k]; i++) {
      if (!c->tr[k][i].set) return clr_fail(c, CLR_ERR_STATE, "tracer %d/%d has no tables", k, i);
      if (ntr >= kMaxTr) return clr_fail(c, CLR_ERR_ARG, "at most %d tracers per normalisation pass", kMaxTr);
      tsrc.bzf[ntr] = c->tr[k][i].bzf;
      a.bz0[ntr] = (float)c->tr[k][i].bz0;
      a.model[ntr] = c->tr[k][i].model;
      tk[ntr] = k;
      tp[ntr] = i;
      ntr++;
    }
  for (int t = 0; t < ntr; t++)
    if (!tsrc.bzf[t] || !c->tr[tk[t]][tp[t]].norm) return clr_fail(c, CLR_ERR_STATE, "tracer tables missing");
  if (!c->d1f || !c->bg) return clr_fail(c, CLR_ERR_STATE, "background tables missing");
  a.g = c->dens;
  a.N = N;
  a.ngx = c->ngx;
  a.nz = nz;
  a.ntr = ntr;
  a.fused = lognormal_fused ? 1 : 0;
  a.na = na;
  a.dx = c->dx;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.idr = c->glob_idr;
  a.r_last = c->r_last;
  a.z_last = z_last;
  a.sigma2 = sigma2;
  a.idz = idz;
  a.r_arr = r;
  a.zt = zt;
  tsrc.d1f = c->d1f;
  tsrc.zt = zt;
  a.z_last_f = (float)z_last;
  a.idz_f = (float)idz;
  a.d1_last_f = (float)c->h_bg_last[2];
  a.idr_f = (float)c->glob_idr;
  const int nq = 2 + ntr;
  {
    ShellPlan plan;
    if (shell_plan(c, nz, ntr, plan)) return clr_fail(c, CLR_ERR_ARG, "too many shells x tracers (%d x %d)", nz, ntr);
  }
  bool all0 = true;
  for (int t = 0; t < ntr; t++) all0 = all0 && a.model[t] == CLR_BIAS_EXPONENTIAL;
  const size_t nvals = (size_t)nz * nq;
  double *partial, *fin;   // (the tracers' edge values follow the sums)
  float2 *tab;
  if (scratch_base) {
    // no allocation: everything in the device's static scratch
    if (nvals > kNoAllocVals)
      return clr_fail(c, CLR_ERR_ARG, "%d shells x (2 + %d tracers) = %zu values exceed the %zu of the static scratch",
                      nz, ntr, nvals, kNoAllocVals);
    if ((size_t)na * nq > 2 * kNoAllocTabFloat4)
      return clr_fail(c, CLR_ERR_ARG, "r-tables of %d entries exceed the static scratch", na);
    partial = (double *)scratch_base;
    fin = partial + (size_t)kShellBlocks * nvals;
    tab = (float2 *)((char *)scratch_base + (kNoAllocDoubles * sizeof(double) + 255) / 256 * 256);
  } else {
    const size_t need = (size_t)kShellBlocks * nvals + nvals + 2 * ntr;
    int rc = clr_ensure(c, (void **)&c->red, &c->red_n, need * sizeof(double));
    if (rc) return rc;
    partial = c->red;
    fin = c->red + (size_t)kShellBlocks * nvals;
    rc = clr_ensure(c, &c->misc, &c->misc_n, (size_t)na * nq * sizeof(float2));
    if (rc) return rc;
    tab = (float2 *)c->misc;
  }
  a.tab = tab;

  CLR_HIP(c, hipEventRecord(c->ev0, c->stream));
  hipLaunchKernelGGL(k_pack_shell_table, dim3((na + 255) / 256, nq), dim3(256), 0, c->stream, tsrc, na, tab);
  CLR_HIP(c, hipGetLastError());
  CLR_HIP(c, hipEventRecord(c->ev2, c->stream));
  {
    const int rc = run_shells(c, c->stream, a, all0, partial, fin, c->ev3);
    if (rc) return rc;
  }
  if (ntr > 0) {
    NormOuts outs{};
    for (int t = 0; t < ntr; t++) {
      outs.p[t] = c->tr[tk[t]][tp[t]].norm;
      outs.e[t] = c->tr[tk[t]][tp[t]].edge;
    }
    hipLaunchKernelGGL(k_norm_table, dim3((unsigned)((na + 255) / 256), (unsigned)ntr), dim3(256), 0, c->stream,
                       fin, nz, nq, zmax, r, zt, c->glob_idr, c->r_last, z_last, na, outs, fin + nvals);
    CLR_HIP(c, hipGetLastError());
  }
  CLR_HIP(c, hipEventRecord(c->ev1, c->stream));
  // host copies of the sums and edge values (a fixed array when they fit, so
  // that the no-allocation variant allocates nothing on the host either)
  double hfix[kNoAllocVals + 2 * kMaxTr];
  std::vector<double> hv;
  double *h = hfix;
  if (nvals > kNoAllocVals) {
    hv.resize(nvals + 2 * ntr);
    h = hv.data();
  }
  CLR_HIP(c, hipMemcpyAsync(h, fin, (nvals + 2 * ntr) * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  for (int t = 0; t < ntr; t++) {
    TracerDev &T = c->tr[tk[t]][tp[t]];
    T.norm0 = h[nvals + 2 * t];
    T.normf = h[nvals + 2 * t + 1];
    T.norm_set = 1;
  }
  float ms = 0;
  hipEventElapsedTime(&ms, c->ev0, c->ev1);
  c->stage_ms[ST_NORM] = ms;
  hipEventElapsedTime(&ms, c->ev2, c->ev3);
  c->stage_ms[ST_SHELLS] = ms;
  if (nz_out) *nz_out = nz;
  if ((counts || zsum || sums) && cap < nz)
    return clr_fail(c, CLR_ERR_ARG, "output capacity %d < nz=%d", cap, nz);
  for (int iz = 0; iz < nz; iz++) {
    if (counts) counts[iz] = (unsigned long long)h[(size_t)iz * nq + 0];
    if (zsum) zsum[iz] = h[(size_t)iz * nq + 1];
    if (sums)
      for (int t = 0; t < ntr; t++) sums[(size_t)t * nz + iz] = h[(size_t)iz * nq + 2 + t];
  }
  if (lognormal_fused) c->density_done = 1;
  c->norms_done = 1;
  return CLR_OK;
}

namespace {

// Arguments of a shell pass over the geometry only (no tracer columns): the
// shell binning of compute_density_normalization (density.c:1128-1211).
int shell_geo_args(clr_ctx *c, ShellArgs &a, ShellTabSrc &tsrc, int &nz) {
  if (!c->tables_set || !c->d1f) return clr_fail(c, CLR_ERR_STATE, "clr_upload_tables must be called first");
  const int na = c->na;
  const double zmax = c->zmax_half_box;
  nz = (int)(zmax / 0.05) + 2;
  if (nz > kNormMaxShells) return clr_fail(c, CLR_ERR_ARG, "%d redshift shells (at most %d)", nz, kNormMaxShells);
  a = ShellArgs{};
  tsrc = ShellTabSrc{};
  a.g = c->dens;
  a.N = c->N;
  a.ngx = c->ngx;
  a.nz = nz;
  a.ntr = 0;
  a.fused = 0;
  a.na = na;
  a.dx = c->dx;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.idr = c->glob_idr;
  a.r_last = c->r_last;
  a.z_last = c->h_bg_last[1];
  a.idz = (nz - 2) / zmax;
  a.r_arr = c->bg;
  a.zt = c->bg + na;
  tsrc.d1f = c->d1f;
  tsrc.zt = c->bg + na;
  a.z_last_f = (float)c->h_bg_last[1];
  a.idz_f = (float)a.idz;
  a.d1_last_f = (float)c->h_bg_last[2];
  a.idr_f = (float)c->glob_idr;
  return CLR_OK;
}

// One geometry-type shell pass with ntr table columns, reduced to
// fin[nz][2 + ntr] on the host.
template <int NT>
int shell_pass_to_host(clr_ctx *c, ShellArgs &a, const ShellTabSrc &tsrc, int nz, std::vector<double> &h) {
  const int na = c->na, nq = 2 + NT;
  const size_t nvals = (size_t)nz * nq;
  int rc = clr_ensure(c, (void **)&c->red, &c->red_n, ((size_t)kShellBlocks * nvals + nvals) * sizeof(double));
  if (rc) return rc;
  double *partial = c->red, *fin = c->red + (size_t)kShellBlocks * nvals;
  rc = clr_ensure(c, &c->misc, &c->misc_n, (size_t)na * nq * sizeof(float2));
  if (rc) return rc;
  a.tab = (const float2 *)c->misc;
  hipLaunchKernelGGL(k_pack_shell_table, dim3((na + 255) / 256, nq), dim3(256), 0, c->stream, tsrc, na,
                     (float2 *)c->misc);
  rc = run_shells(c, c->stream, a, true, partial, fin, nullptr);
  if (rc) return rc;
  h.resize(nvals);
  CLR_HIP(c, hipMemcpyAsync(h.data(), fin, nvals * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  return CLR_OK;
}

}  // namespace

// Cells and z sums per normalisation shell (the count and zsum columns of
// collect_density_normalization_from_grid, density.c:1128-1211): the shell
// pass without tracers; they depend only on the grid geometry and tables.
int clr_launch_shell_geometry(clr_ctx *c) {
  if (c->geo_nz > 0) return CLR_OK;
  ShellArgs a;
  ShellTabSrc tsrc;
  int nz = 0;
  int rc = shell_geo_args(c, a, tsrc, nz);
  if (rc) return rc;
  std::vector<double> h;
  rc = shell_pass_to_host<0>(c, a, tsrc, nz, h);
  if (rc) return rc;
  c->geo_cnt.resize(nz);
  c->geo_zsum.resize(nz);
  for (int iz = 0; iz < nz; iz++) {
    c->geo_cnt[iz] = h[(size_t)iz * 2];
    c->geo_zsum[iz] = h[(size_t)iz * 2 + 1];
  }
  c->geo_zmax = c->zmax_half_box;
  c->geo_nz = nz;
  return CLR_OK;
}

// Gaussian moments per normalisation shell of the current (untransformed)
// grid, for the surrogate: with G = D(r) delta_G per cell, out[nz][6] = the
// cell count and the sums of G, G^2, G^3, G^4 and D^2 (k_shell_moments).
// The shell of a cell is the one its FP32 radius falls in between the FP32
// radii of the z edges (nz shells of compute_density_normalization,
// density.c:1233-1244); D(r) from the FP32 growth table.
int clr_launch_shell_moments(clr_ctx *c, std::vector<double> &out) {
  if (!c->have_fields || c->density_done)
    return clr_fail(c, CLR_ERR_STATE, "the shell moments need the Gaussian field (fields done, density not transformed)");
  if (!c->tables_set || !c->d1f) return clr_fail(c, CLR_ERR_STATE, "clr_upload_tables must be called first");
  const int na = c->na;
  const double zmax = c->zmax_half_box;
  const int nz = (int)(zmax / 0.05) + 2;
  if (nz > kMomMaxShells) return clr_fail(c, CLR_ERR_ARG, "%d redshift shells (the moments pass takes %d)", nz, kMomMaxShells);
  const double idz = (nz - 2) / zmax;
  // E[k] = r(z = k / idz), k = 0 .. nz-1: shell s holds E[s-1] <= r < E[s]
  std::vector<float> hedge(nz);
  const std::vector<double> &zz = c->h_z, &rr = c->h_r;
  for (int k = 0; k < nz; k++) {
    const double z = k / idz;
    double r;
    if (z <= zz[0]) r = rr[0];
    else if (z >= zz[na - 1]) r = rr[na - 1] * 4;   // past the table: no cell reaches it
    else {
      int lo = 0, hi = na - 1;
      while (hi > lo + 1) {
        const int m = (lo + hi) / 2;
        if (zz[m] > z) hi = m; else lo = m;
      }
      r = rr[lo] + (z - zz[lo]) / (zz[hi] - zz[lo]) * (rr[hi] - rr[lo]);
    }
    hedge[k] = (float)r;
  }
  hedge[0] = 0.f;
  const size_t nvals = (size_t)nz * kMomQ;
  int rc = clr_ensure(c, (void **)&c->red, &c->red_n, ((size_t)kMomBlocks * nvals + nvals) * sizeof(double));
  if (rc) return rc;
  double *partial = c->red, *fin = c->red + (size_t)kMomBlocks * nvals;
  rc = clr_ensure(c, &c->misc, &c->misc_n, (size_t)nz * sizeof(float));
  if (rc) return rc;
  float *dedge = (float *)c->misc;
  CLR_HIP(c, hipMemcpyAsync(dedge, hedge.data(), nz * sizeof(float), hipMemcpyHostToDevice, c->stream));
  MomArgs a{};
  a.g = c->dens;
  a.r_arr = c->bg;
  a.d1 = c->bg + 2 * (size_t)na;
  a.edge = dedge;
  a.N = c->N;
  a.ngx = c->ngx;
  a.nz = nz;
  a.idr = c->glob_idr;
  a.r_last = c->r_last;
  a.d_last = c->h_bg_last[2];
  a.dxf = (float)c->dx;
  a.ox = (float)c->obs[0];
  a.oy = (float)c->obs[1];
  a.oz = (float)c->obs[2];
  // items of zrun planes: a multiple of kMomPre, at most kMomZMax, spanning
  // at most ~160 Mpc/h
  a.zrun = std::max(kMomPre, std::min(kMomZMax, (int)(160.0 / c->dx) / kMomPre * kMomPre));
  const size_t lds = (size_t)kWaves * nz * kMomQ * sizeof(double) + (size_t)nz * sizeof(float);
  if (c->N % kMomCPL) return clr_fail(c, CLR_ERR_ARG, "the shell moments need N divisible by %d", kMomCPL);
  if (c->N % kMomXW == 0 && c->N % a.zrun == 0)
    hipLaunchKernelGGL(k_shell_moments<true>, dim3(kMomBlocks), dim3(kShellThreads), lds, c->stream, a, partial);
  else
    hipLaunchKernelGGL(k_shell_moments<false>, dim3(kMomBlocks), dim3(kShellThreads), lds, c->stream, a, partial);
  hipLaunchKernelGGL(k_shell_final, dim3((unsigned)nvals), dim3(256), 0, c->stream, partial, kMomBlocks, (int)nvals,
                     fin);
  CLR_HIP(c, hipGetLastError());
  out.resize(nvals);
  CLR_HIP(c, hipMemcpyAsync(out.data(), fin, nvals * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  return CLR_OK;
}

// Norm tables of the given tracers from per-shell norms norm_s[t][nz] on the
// cached geometry: the sums are count/norm, and k_norm_table then applies the
// reference's edge fill and interpolation in z (density.c:1272-1355).
int clr_launch_norm_tables_given(clr_ctx *c, int ntr, const int *kinds, const int *ipops, const double *norm_s) {
  if (c->geo_nz <= 0) return clr_fail(c, CLR_ERR_STATE, "no shell geometry");
  if (ntr < 1 || ntr > 3 * CLR_NPOP_MAX) return clr_fail(c, CLR_ERR_ARG, "bad tracer count %d", ntr);
  const int nz = c->geo_nz, na = c->na, nq = 2 + ntr;
  std::vector<double> fin((size_t)nz * nq + 2 * (size_t)ntr, 0.0);
  for (int iz = 0; iz < nz; iz++) {
    const double n = c->geo_cnt[iz];
    fin[(size_t)iz * nq] = n;
    fin[(size_t)iz * nq + 1] = c->geo_zsum[iz];
    for (int t = 0; t < ntr; t++) {
      const double nm = norm_s[(size_t)t * nz + iz];
      fin[(size_t)iz * nq + 2 + t] = n > 0 ? n / nm : 0.0;
    }
  }
  const size_t bytes = fin.size() * sizeof(double);
  int rc = clr_ensure(c, (void **)&c->red, &c->red_n, bytes);
  if (rc) return rc;
  double *dfin = c->red, *edges = c->red + (size_t)nz * nq;
  CLR_HIP(c, hipMemcpyAsync(dfin, fin.data(), (size_t)nz * nq * sizeof(double), hipMemcpyHostToDevice, c->stream));
  NormOuts outs{};
  for (int t = 0; t < ntr; t++) {
    TracerDev &T = c->tr[kinds[t]][ipops[t]];
    if (!T.set || !T.norm) return clr_fail(c, CLR_ERR_STATE, "tracer %d/%d has no tables", kinds[t], ipops[t]);
    outs.p[t] = T.norm;
    outs.e[t] = T.edge;
  }
  hipLaunchKernelGGL(k_norm_table, dim3((unsigned)((na + 255) / 256), (unsigned)ntr), dim3(256), 0, c->stream,
                     dfin, nz, nq, c->geo_zmax, c->bg, c->bg + na, c->glob_idr, c->r_last, c->h_bg_last[1], na,
                     outs, edges);
  CLR_HIP(c, hipGetLastError());
  std::vector<double> e(2 * (size_t)ntr);
  CLR_HIP(c, hipMemcpyAsync(e.data(), edges, 2 * ntr * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  CLR_HIP(c, hipStreamSynchronize(c->stream));
  for (int t = 0; t < ntr; t++) {
    TracerDev &T = c->tr[kinds[t]][ipops[t]];
    T.norm0 = e[2 * t];
    T.normf = e[2 * t + 1];
    T.norm_set = 1;
  }
  return CLR_OK;
}

// ---------------------------------------------------------------------------
// The shell-sum stage for graph capture: buffers first (clr_prepare_norms),
// then kernel launches only (clr_enqueue_norms): the packed table, the shell
// pass with the fused lognormal (sigma^2 read from the device), the final
// sums and every tracer's norm table, its edge values left in each tracer's
// device copy.  The same kernels and order as clr_launch_norms.
// ---------------------------------------------------------------------------
static int norms_tracers(clr_ctx *c, int *tk, int *tp) {
  int ntr = 0;
  for (int k = 0; k < 3; k++)
    for (int i = 0; i < c->n_tr[k]; i++) {
      tk[ntr] = k;
      tp[ntr] = i;
      ntr++;
    }
  return ntr;
}

int clr_prepare_norms(clr_ctx *c) {
  int tk[3 * CLR_NPOP_MAX], tp[3 * CLR_NPOP_MAX];
  const int ntr = norms_tracers(c, tk, tp);
  if (ntr < 1 || ntr > kMaxTr) return clr_fail(c, CLR_ERR_ARG, "%d tracers (1 .. %d)", ntr, kMaxTr);
  const int nz = (int)(c->zmax_half_box / 0.05) + 2;
  if (nz > kNormMaxShells) return clr_fail(c, CLR_ERR_ARG, "%d redshift shells (at most %d)", nz, kNormMaxShells);
  const size_t nvals = (size_t)nz * (2 + ntr);
  int rc = clr_ensure(c, (void **)&c->red, &c->red_n,
                      ((size_t)kShellBlocks * nvals + nvals + 2 * nz + 2 * ntr) * sizeof(double));
  if (rc) return rc;
  rc = clr_ensure(c, &c->misc, &c->misc_n, (size_t)c->na * (2 + ntr) * sizeof(float2));
  if (rc) return rc;
  for (int t = 0; t < ntr; t++) {
    TracerDev &T = c->tr[tk[t]][tp[t]];
    if (!T.edge) CLR_HIP(c, hipMalloc((void **)&T.edge, 2 * sizeof(double)));
  }
  return CLR_OK;
}

int clr_enqueue_norms(clr_ctx *c, hipStream_t st, const double *sigma2_dev) {
  int tk[3 * CLR_NPOP_MAX], tp[3 * CLR_NPOP_MAX];
  const int ntr = norms_tracers(c, tk, tp);
  const int N = c->N, na = c->na;
  const double zmax = c->zmax_half_box;
  const int nz = (int)(zmax / 0.05) + 2;
  const int nq = 2 + ntr;
  const size_t nvals = (size_t)nz * nq;
  if (ntr < 1 || ntr > kMaxTr || c->red_n < ((size_t)kShellBlocks * nvals + nvals + 2 * nz + 2 * ntr) * sizeof(double))
    return clr_fail(c, CLR_ERR_STATE, "normalisation buffers not prepared");
  ShellArgs a{};
  ShellTabSrc tsrc{};
  bool all0 = true;
  NormOuts outs{};
  for (int t = 0; t < ntr; t++) {
    TracerDev &T = c->tr[tk[t]][tp[t]];
    if (!T.set || !T.bzf || !T.norm || !T.edge) return clr_fail(c, CLR_ERR_STATE, "tracer tables missing");
    tsrc.bzf[t] = T.bzf;
    a.bz0[t] = (float)T.bz0;
    a.model[t] = T.model;
    all0 = all0 && T.model == CLR_BIAS_EXPONENTIAL;
    outs.p[t] = T.norm;
    outs.e[t] = T.edge;
  }
  a.g = c->dens;
  a.N = N;
  a.ngx = c->ngx;
  a.nz = nz;
  a.ntr = ntr;
  a.fused = 1;
  a.na = na;
  a.dx = c->dx;
  a.ox = c->obs[0];
  a.oy = c->obs[1];
  a.oz = c->obs[2];
  a.idr = c->glob_idr;
  a.r_last = c->r_last;
  a.z_last = c->h_bg_last[1];
  a.sigma2 = 0;
  a.sigma2_dev = sigma2_dev;
  a.idz = (nz - 2) / zmax;
  a.r_arr = c->bg;
  a.zt = c->bg + na;
  tsrc.d1f = c->d1f;
  tsrc.zt = c->bg + na;
  a.z_last_f = (float)c->h_bg_last[1];
  a.idz_f = (float)a.idz;
  a.d1_last_f = (float)c->h_bg_last[2];
  a.idr_f = (float)c->glob_idr;
  a.tab = (const float2 *)c->misc;
  double *partial = c->red, *fin = c->red + (size_t)kShellBlocks * nvals, *work = fin + nvals;
  hipLaunchKernelGGL(k_pack_shell_table, dim3((na + 255) / 256, nq), dim3(256), 0, st, tsrc, na, (float2 *)c->misc);
  {
    const int rc = run_shells(c, st, a, all0, partial, fin, nullptr);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(k_norm_table, dim3((unsigned)((na + 255) / 256), (unsigned)ntr), dim3(256), 0, st, fin, nz, nq,
                     zmax, c->bg, c->bg + na, c->glob_idr, c->r_last, c->h_bg_last[1], na, outs, work + 2 * nz);
  CLR_HIP(c, hipGetLastError());
  return CLR_OK;
}

