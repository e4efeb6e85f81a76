// Neutrino fluid: the dispersive sum of three isothermal-start fluids at the
// Gauss-Laguerre velocities (hydrodf.f90), each a finite-volume fluid
// (hydrogr.f90) updated by dimensionally split MUSCL-minmod/HLL sweeps
// (hydro1d.f90:113-225, hydro3d.f90:33-108), coupled to the PM meshes
// through its density (pm.f90:55-74, 198-242) and the PM forces
// (pm.f90:157-171, 374-422).
//
// One box, so every fluid is a periodic nc^3 array with no halo cells: the
// reference's halo shells (ncb >= 2 cells) only carry periodic copies for
// the stencil, and a periodic line sweep gives the same physical cells.
// Fields are structure-of-arrays [5][nc^3] (rho, mx, my, mz, E), x fastest.
//
// Gravity: the reference adds each fine cell's impulse to the eight fluid
// cells around it one after another, the energy term using the momentum
// already kicked.  With x_k = dV_k a_k summed over all contributions k of a
// fluid cell, that sequence equals, for any order,
//   m += rho J,   E += m0.J + rho/2 (|J|^2 + Q),
//   J = sum dV_k a_k,   Q = sum dV_k (1 - dV_k) |a_k|^2,
// so each fluid cell gathers J and Q from its stencil and is updated once:
// no atomics and the same result on every run.
#include "cube_internal.hpp"
#include <math.h>
#include <string.h>
#include <algorithm>
#include <vector>

#define FL_NT 256
#define FL_W 4       // fewest lines per workgroup in a sweep
#define FL_SNT 512   // threads of a sweep workgroup
#define FL_SPER 4    // cells per thread in a sweep: 2048 per workgroup
#define H_CFL 0.71f
#define H_LIM 1.5f

// ------------------------------------------------------------- 1-D pieces
__device__ __forceinline__ float sgn1(float a) { return copysignf(1.0f, a); }
__device__ __forceinline__ float minmod(float a, float b, float c) {
  const float m = fminf(fminf(fabsf(a), fabsf(b)), fabsf(c));
  return 0.25f * fabsf(sgn1(a) + sgn1(b)) * (sgn1(a) + sgn1(c)) * m;
}
__device__ __forceinline__ float kin(float r, float m1, float m2, float m3) {
  return 0.5f * ((m1 * m1 + m2 * m2) + m3 * m3) / r;
}
__device__ __forceinline__ float press(float r, float m1, float m2, float m3, float e, float g) {
  const float p = (e - kin(r, m1, m2, m3)) * (g - 1.0f);
  return p > 0.0f ? p : 0.0f;
}

// Several quotients by one denominator b: with y the correctly rounded 1/b,
// the estimate x*y corrected by its exact remainder is the correctly rounded
// x/b (Markstein 1990), in three operations instead of some eleven.  That
// needs a remainder above the smallest denormal and a quotient that is neither
// denormal nor beyond the largest float (an infinite estimate leaves a NaN, and
// a denormal one may be a unit off).  The caller checks with div_safe that all
// numerators lie between 1e-30 and 1e30 in magnitude and b between 1e-7 and
// 1e7; otherwise it divides.
__device__ __forceinline__ float div_by(float x, float b, float y) {
  const float q = x * y;
  return fmaf(fmaf(-q, b, x), y, q);
}
__device__ __forceinline__ bool div_safe(float least, float most, float b) {
  return least > 1e-30f && most < 1e30f && b > 1e-7f && b < 1e7f;
}
__device__ __forceinline__ float min3abs(float a, float b, float c) { return fminf(fminf(fabsf(a), fabsf(b)), fabsf(c)); }
__device__ __forceinline__ float max3abs(float a, float b, float c) { return fmaxf(fmaxf(fabsf(a), fabsf(b)), fabsf(c)); }

// primitives v = m/rho, p of one cell
template <bool FAST>
__device__ __forceinline__ void fl_prim(float r, float y, float m1, float m2, float m3, float en, float g, float u[5]) {
  auto div = [&](float x) { return FAST ? div_by(x, r, y) : x / r; };
  u[0] = r;
  u[1] = div(m1);
  u[2] = div(m2);
  u[3] = div(m3);
  const float p = (en - div(0.5f * ((m1 * m1 + m2 * m2) + m3 * m3))) * (g - 1.0f);
  u[4] = p > 0.0f ? p : 0.0f;
}
// conserved variables, flux and sound speed of an interface state
template <bool FAST>
__device__ __forceinline__ void fl_side(const float b[5], float y, float g, float yg, float h[5], float f[5], float& v, float& s) {
  auto div = [&](float x) { return FAST ? div_by(x, b[0], y) : x / b[0]; };
  h[0] = b[0]; h[1] = h[0] * b[1]; h[2] = h[0] * b[2]; h[3] = h[0] * b[3];
  const float k = div(0.5f * ((h[1] * h[1] + h[2] * h[2]) + h[3] * h[3]));
  h[4] = (FAST ? div_by(b[4], g - 1.0f, yg) : b[4] / (g - 1.0f)) + k;
  const float p0 = (h[4] - k) * (g - 1.0f), p = p0 > 0.0f ? p0 : 0.0f;
  v = div(h[1]);
  f[0] = h[1];
  f[1] = h[1] * v + p;
  f[2] = h[1] * div(h[2]);
  f[3] = h[1] * div(h[3]);
  f[4] = h[4] * v;
  s = sqrtf(FAST && p > 1e-30f && p < 1e30f ? div_by(p, b[0], y) : p / b[0]);
}

// One sweep along axis AX over W adjacent lines of nc = 2^lnc cells, W nc <=
// FL_SNT FL_SPER.  The normal momentum is the sweep's first momentum component
// and the two others follow in the reference's swapped order (x: x,y,z; y:
// y,x,z; z: z,y,x).  LDS holds the primitives (rho, v1, v2, v3, p) of the
// lines, then their interface fluxes; rows are `pitch` apart, 64/W banks from
// a whole number of rows for the strided sweeps, whose lanes run over the
// lines first.
//   Bound by VALU issue (1.09, 0.97 and 0.78 instructions per SIMD and four
// cycles along x, y and z at 256^3 cells; at 512^3, with strips of 4 lines, 1.15,
// 0.72 and 0.59, where 16-byte pieces of rows wait for memory): 30 divisions of
// some 14 issue slots each per cell were over half of it.  256^3 cells take
// 0.24, 0.27 and 0.33 ms; with a division each and strips of 4 lines 0.32, 0.36
// and 0.48.
template <int AX, int W>
__global__ __launch_bounds__(FL_SNT) void k_fl_sweep(float* F, int nc, int lnc, int pitch, float g, float yg, float dt, float ydx) {
  extern __shared__ float sm[];
  const int64_t n3 = (int64_t)nc * nc * nc;
  const int nla = nc / W;
  // XCD-contiguous order: the line groups adjacent in x that share cache
  // lines (strided sweeps) run on the same XCD's L2
  const uint32_t lb = xcd_remap(blockIdx.x, gridDim.x);
  const int a0 = (int)(lb % nla) * W, b = (int)(lb / nla);
  const int c1 = AX == 0 ? 1 : (AX == 1 ? 2 : 3), c2 = AX == 1 ? 1 : 2, c3 = AX == 2 ? 1 : 3;
  const int L = W * nc;
  auto elem = [&](int e, int& t, int& w) {
    if (AX == 0) { t = e & (nc - 1); w = e >> lnc; }
    else { w = e % W; t = e / W; }
  };
  auto cell = [&](int t, int w) -> int64_t {
    const int a = a0 + w;
    if (AX == 0) return ((int64_t)b * nc + a) * nc + t;
    if (AX == 1) return ((int64_t)b * nc + t) * nc + a;
    return ((int64_t)t * nc + b) * nc + a;
  };
  auto S = [&](int q, int w, int t) -> float& { return sm[(q * W + w) * pitch + t]; };
  // pass 1: primitives into LDS
#pragma unroll
  for (int k = 0; k < FL_SPER; k++) {
    const int e = threadIdx.x + k * FL_SNT;
    if (e >= L) continue;
    int t, w;
    elem(e, t, w);
    const int64_t c = cell(t, w);
    const float r = F[c], m1 = F[(int64_t)c1 * n3 + c], m2 = F[(int64_t)c2 * n3 + c], m3 = F[(int64_t)c3 * n3 + c],
                en = F[4 * n3 + c];
    float u[5];
    // the momenta and half the sum of their squares are divided
    const float least = min3abs(m1, m2, m3), most = max3abs(m1, m2, m3);
    if (div_safe(least * least, 2.0f * (most * most), r)) fl_prim<true>(r, 1.0f / r, m1, m2, m3, en, g, u);
    else fl_prim<false>(r, 0.0f, m1, m2, m3, en, g, u);
#pragma unroll
    for (int q = 0; q < 5; q++) S(q, w, t) = u[q];
  }
  __syncthreads();
  // pass 2: HLL flux at the interface t+1/2 of each element, held in registers
  float fx[FL_SPER][5];
#pragma unroll
  for (int k = 0; k < FL_SPER; k++) {
    const int e = threadIdx.x + k * FL_SNT;
    if (e >= L) continue;
    int t, w;
    elem(e, t, w);
    const int tm = (t - 1) & (nc - 1), tp = (t + 1) & (nc - 1), tq = (t + 2) & (nc - 1);
    float bl[5], br[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const float u0 = S(q, w, tm), u1 = S(q, w, t), u2 = S(q, w, tp), u3 = S(q, w, tq);
      const float l = H_LIM * (u2 - u1);
      bl[q] = u1 + 0.5f * minmod(H_LIM * (u1 - u0), 0.5f * (u2 - u0), l);
      br[q] = u2 - 0.5f * minmod(l, 0.5f * (u3 - u1), H_LIM * (u3 - u2));
    }
    float hl[5], hr[5], fl[5], fr[5], vl, vr, sl, sr;
    // momenta, half the sum of their squares, and pressures (by gamma - 1)
    const float mh = fminf(min3abs(bl[1], bl[2], bl[3]) * bl[0], min3abs(br[1], br[2], br[3]) * br[0]);
    const float xh = fmaxf(max3abs(bl[1], bl[2], bl[3]) * bl[0], max3abs(br[1], br[2], br[3]) * br[0]);
    const bool fast = div_safe(fminf(fminf(bl[4], br[4]), mh * mh), fmaxf(fmaxf(bl[4], br[4]), 2.0f * (xh * xh)), bl[0]) &&
                      div_safe(1.0f, 1.0f, br[0]) && g < 1e7f;
    if (fast) {
      fl_side<true>(bl, 1.0f / bl[0], g, yg, hl, fl, vl, sl);
      fl_side<true>(br, 1.0f / br[0], g, yg, hr, fr, vr, sr);
    } else {
      fl_side<false>(bl, 0.0f, g, yg, hl, fl, vl, sl);
      fl_side<false>(br, 0.0f, g, yg, hr, fr, vr, sr);
    }
    const float ap = fmaxf(fmaxf(0.0f, vl + sl), vr + sr);
    const float am = fmaxf(fmaxf(0.0f, -vl + sl), -vr + sr);
    const float as = ap + am;
    float nu[5], least = 1.0f, most = 1.0f;
#pragma unroll
    for (int q = 0; q < 5; q++) {
      nu[q] = ap * fl[q] + am * fr[q] - ap * am * (hr[q] - hl[q]);
      least = fminf(least, fabsf(nu[q]));
      most = fmaxf(most, fabsf(nu[q]));
    }
    if (div_safe(least, most, as)) {
      const float ya = 1.0f / as;
#pragma unroll
      for (int q = 0; q < 5; q++) fx[k][q] = div_by(nu[q], as, ya);
    } else {
#pragma unroll
      for (int q = 0; q < 5; q++) fx[k][q] = nu[q] / as;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < FL_SPER; k++) {
    const int e = threadIdx.x + k * FL_SNT;
    if (e >= L) continue;
    int t, w;
    elem(e, t, w);
#pragma unroll
    for (int q = 0; q < 5; q++) S(q, w, t) = fx[k][q];
  }
  __syncthreads();
  // pass 3: h += dt*(F(t-1/2) - F(t+1/2))/dx in the sweep's variable order;
  // dx is a power of two, so the product with ydx = 1/dx is the quotient
#pragma unroll
  for (int k = 0; k < FL_SPER; k++) {
    const int e = threadIdx.x + k * FL_SNT;
    if (e >= L) continue;
    int t, w;
    elem(e, t, w);
    const int tm = (t - 1) & (nc - 1);
    const int64_t c = cell(t, w);
    const int64_t off[5] = {0, (int64_t)c1 * n3, (int64_t)c2 * n3, (int64_t)c3 * n3, 4 * n3};
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const float rq = -fx[k][q] + S(q, w, tm);
      F[off[q] + c] = F[off[q] + c] + dt * rq * ydx;
    }
  }
}

// ---------------------------------------------------------------- timestep
// h3_timestep: per x-line, cfl*dx/(max|v| + max c_s); the minimum over lines
// (positive floats order as their bit patterns).
// A wavefront per line and pass; the quotient falls as v + c_s grows, so the
// least of it over a wavefront's lines is that of their largest sum, and a
// workgroup takes the minimum once (one atomic per line of 256^3 cells met on
// one address: 0.75 ms, now 0.07).
__global__ __launch_bounds__(FL_NT) void k_fl_dt(const float* __restrict__ F, int nc, float g, float dx, uint32_t* dtbits) {
  __shared__ float rm[FL_NT / 64];
  const int64_t n3 = (int64_t)nc * nc * nc;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float most = 0.0f;
  for (int line = blockIdx.x * (FL_NT / 64) + wv; line < nc * nc; line += gridDim.x * (FL_NT / 64)) {
    float v = 0.0f, s = 0.0f;
    for (int i = lane; i < nc; i += 64) {
      const int64_t c = (int64_t)line * nc + i;
      const float r = F[c], m1 = F[n3 + c], m2 = F[2 * n3 + c], m3 = F[3 * n3 + c], en = F[4 * n3 + c];
      v = fmaxf(v, fmaxf(fmaxf(fabsf(m1 / r), fabsf(m2 / r)), fabsf(m3 / r)));
      s = fmaxf(s, sqrtf(press(r, m1, m2, m3, en, g) / r));
    }
    const float vm = __uint_as_float(wave_max_bits(__float_as_uint(v))), sm = __uint_as_float(wave_max_bits(__float_as_uint(s)));
    most = fmaxf(most, vm + sm);
  }
  if (lane == 0) rm[wv] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < FL_NT / 64; i++) most = fmaxf(most, rm[i]);
    atomicMin(dtbits, __float_as_uint(H_CFL * dx / most));
  }
}

// ---------------------------------------------------------------- density
struct FlSet {  // the three fluids of the dispersive sum
  const float* rho[3];
  int nc[3];
  float w[3];
};
// hg_density (CIC) of the fluid of DX fine cells per cell at the centres of
// fine cells 4a..4a+3 of row (y, z): the cells' x taps start 0, (j 's share)
// nodes apart and y and z are uniform
template <int DX>
__device__ __forceinline__ void fl_density_quad(const float* __restrict__ rho, int nc, int a, int y, int z, float d[4]) {
  constexpr int NN = DX == 2 ? 4 : (DX == 4 ? 3 : 2);  // nodes the four cells touch along x
  const float xx0 = ((float)(4 * a) + 0.5f) * (1.0f / DX) - 0.5f;
  const int f0 = (int)floorf(xx0);
  float w[2][2];
  int yz[2][2];
  const int p[2] = {y, z};
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const float xx = ((float)p[e] + 0.5f) * (1.0f / DX) - 0.5f;  // exact: DX is a power of two
    const int f = (int)floorf(xx);
    w[e][0] = (float)(f + 1) - xx;
    w[e][1] = 1.0f - w[e][0];
    yz[e][0] = f & (nc - 1);
    yz[e][1] = (f + 1) & (nc - 1);
  }
  float v[2][2][NN];  // [z][y][x]
#pragma unroll
  for (int cz = 0; cz < 2; cz++)
#pragma unroll
    for (int cy = 0; cy < 2; cy++) {
      const float* row = rho + (size_t)(yz[1][cz] * nc + yz[0][cy]) * nc;
#pragma unroll
      for (int n = 0; n < NN; n++) v[cz][cy][n] = row[(f0 + n) & (nc - 1)];
    }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int o = DX == 2 ? (j + 1) / 2 : (DX == 4 ? j / 2 : 0);  // first node of cell j, from f0
    const float xx = ((float)(4 * a + j) + 0.5f) * (1.0f / DX) - 0.5f;
    const float d1 = (float)(f0 + o + 1) - xx, d2 = 1.0f - d1;
    d[j] = v[0][0][o] * d1 * w[0][0] * w[1][0] + v[0][0][o + 1] * d2 * w[0][0] * w[1][0] +
           v[0][1][o] * d1 * w[0][1] * w[1][0] + v[0][1][o + 1] * d2 * w[0][1] * w[1][0] +
           v[1][0][o] * d1 * w[0][0] * w[1][1] + v[1][0][o + 1] * d2 * w[0][0] * w[1][1] +
           v[1][1][o] * d1 * w[0][1] * w[1][1] + v[1][1][o + 1] * d2 * w[0][1] * w[1][1];
  }
}
// dfld_density at every fine-cell centre n+0.5 into D (rows of pitch nf+2):
// the three fluids have 2, 4 and 8 fine cells per cell.  A wavefront per row,
// four cells a lane, so that a lane loads 36 nodes for four cells instead of
// 24 for each (512^3 centres: 0.43 instead of 1.5 ms).
__global__ __launch_bounds__(256) void k_fl_density_centres(FlSet s, int nf, float* D) {
  const int row = (int)xcd_remap(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int y = row & (nf - 1), z = row / nf;
  float* out = D + (size_t)row * (nf + 2);
  for (int a = threadIdx.x & 63; a < nf / 4; a += 64) {
    float d0[4], d1[4], d2[4];
    fl_density_quad<2>(s.rho[0], s.nc[0], a, y, z, d0);
    fl_density_quad<4>(s.rho[1], s.nc[1], a, y, z, d1);
    fl_density_quad<8>(s.rho[2], s.nc[2], a, y, z, d2);
#pragma unroll
    for (int j = 0; j < 4; j++) d0[j] = ((0.0f + s.w[0] * d0[j]) + s.w[1] * d1[j]) + s.w[2] * d2[j];
    *(float2*)(out + 4 * a) = make_float2(d0[0], d0[1]);
    *(float2*)(out + 4 * a + 2) = make_float2(d0[2], d0[3]);
  }
}
// fine mesh (pm.f90:57-72): node n gets f_nu * density(n + 0.5), or the
// homogeneous f_nu before the fluid starts.  Per-block sums of what was
// added go to part[blockIdx.x]: the reference's testrhof sums rho_f after
// the fluid is in (pm.f90:107).
template <typename T>
__global__ __launch_bounds__(256) void k_fl_add_fine(T* R, const float* D, int64_t nf, int lnf, float fnu, int homog, double* part) {
  __shared__ double red[4];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double added = 0;
  if (i < nf * nf * nf) {
    const int64_t row = i >> lnf, q = row * (nf + 2) + (i & (nf - 1));  // nf = 2^lnf
    const T v = (T)(homog ? fnu : D[q] * fnu);
    R[q] = R[q] + v;
    added = (double)v;
  }
  for (int o = 32; o > 0; o >>= 1) added += __shfl_xor(added, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = added;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}
// coarse mesh (pm.f90:198-242): every fine-cell centre's f_nu*density CIC
// onto coarse nodes at cell centres, gathered per node (2*ncell taps per
// dimension, the reference's dx1/dx2 weights).  Per-block sums of what was
// added go to part[blockIdx.x] (testrhoc sums r3 with the fluid in,
// pm.f90:280).
template <typename T>
__device__ __forceinline__ double fl_coarse_node(T* Rc, const float* D, int64_t nf, int ncc, float fnu, int homog, int64_t i);
template <typename T>
__global__ __launch_bounds__(256) void k_fl_add_coarse(T* Rc, const float* D, int64_t nf, int ncc, float fnu, int homog,
                                                       double* part) {
  __shared__ double red[4];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double added = i < (int64_t)ncc * ncc * ncc ? fl_coarse_node(Rc, D, nf, ncc, fnu, homog, i) : 0.0;
  for (int o = 32; o > 0; o >>= 1) added += __shfl_xor(added, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = added;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}
template <typename T>
__device__ __forceinline__ double fl_coarse_node(T* Rc, const float* D, int64_t nf, int ncc, float fnu, int homog, int64_t i) {
  const int cx = (int)(i % ncc), cy = (int)((i / ncc) % ncc), cz = (int)(i / ((int64_t)ncc * ncc));
  const int64_t q = ((int64_t)cz * ncc + cy) * (ncc + 2) + cx;
  if (homog) {
    const T v = (T)(fnu * (float)(CUBE_NCELL * CUBE_NCELL * CUBE_NCELL));
    Rc[q] = Rc[q] + v;
    return (double)v;
  }
  // node c takes the fine-cell centres 4c-2..4c+5 per dimension, whose
  // weights ((m+0.5)/4 - 0.5 against c, exact in float) are these eighths
  const float wt[2 * CUBE_NCELL] = {0.125f, 0.375f, 0.625f, 0.875f, 0.875f, 0.625f, 0.375f, 0.125f};
  double acc = 0;
  const int mask = (int)nf - 1, x0 = CUBE_NCELL * cx - CUBE_NCELL / 2;
  for (int jz = 0; jz < 2 * CUBE_NCELL; jz++) {
    const int mz = (CUBE_NCELL * cz - CUBE_NCELL / 2 + jz) & mask;
#pragma unroll
    for (int jy = 0; jy < 2 * CUBE_NCELL; jy++) {
      const int my = (CUBE_NCELL * cy - CUBE_NCELL / 2 + jy) & mask;
      const float* row = D + ((size_t)mz * nf + my) * (nf + 2);
      float2 v[CUBE_NCELL];  // x0 is even, so pairs do not straddle the wrap
#pragma unroll
      for (int h = 0; h < CUBE_NCELL; h++) v[h] = *(const float2*)(row + ((x0 + 2 * h) & mask));
#pragma unroll
      for (int jx = 0; jx < 2 * CUBE_NCELL; jx++) {
        const float rnu = (jx & 1 ? v[jx >> 1].y : v[jx >> 1].x) * fnu;
        acc += (double)(rnu * wt[jx] * wt[jy] * wt[jz]);
      }
    }
  }
  Rc[q] = Rc[q] + (T)acc;
  return (double)(T)acc;
}

// ---------------------------------------------------------------- gravity
// Fill A_d (row pitch p_d) with component d of the coarse force
// CIC-interpolated at every fine-cell centre, times a_mid*dt/6/pi
// (pm.f90:387-404).  Fc holds the three components [3][ncc^3].
// A wavefront per row and four cells a lane: cells 4a..4a+3 lie between the
// nodes a-1, a and a+1, so 36 loads serve what took 96, and y and z are
// uniform (512^3 centres: 0.47 instead of 1.12 ms).
template <typename T>
__global__ __launch_bounds__(256) void k_fl_coarse_at_centres(const T* __restrict__ Fc, int ncc, int nf, float a_mid, float dt, float* A0,
                                                              float* A1, float* A2, int64_t p0, int64_t p1, int64_t p2) {
  const int row = (int)xcd_remap(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int yz[2] = {row & (nf - 1), row / nf};
  float c[2][2];
  int k[2][2];
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const float xc = ((float)yz[e] + 0.5f) / (float)CUBE_NCELL - 0.5f;
    const int f = (int)floorf(xc);
    c[e][0] = (float)(f + 1) - xc;
    c[e][1] = 1.0f - c[e][0];
    k[e][0] = f & (ncc - 1);
    k[e][1] = (f + 1) & (ncc - 1);
  }
  const float kf = a_mid * dt / 6.0f / PI_F;
  const size_t n3c = (size_t)ncc * ncc * ncc;
  float* const out[3] = {A0 + row * p0, A1 + row * p1, A2 + row * p2};
  for (int a = threadIdx.x & 63; a < nf / 4; a += 64) {
    const float cx[4] = {0.375f, 0.125f, 0.875f, 0.625f};  // weight of a cell's lower node, 1 minus it of its upper
    const int x[3] = {(a - 1) & (ncc - 1), a, (a + 1) & (ncc - 1)};
#pragma unroll
    for (int d = 0; d < 3; d++) {
      float v[2][2][3];
#pragma unroll
      for (int oz = 0; oz < 2; oz++)
#pragma unroll
        for (int oy = 0; oy < 2; oy++) {
          const T* r = Fc + d * n3c + (size_t)(k[1][oz] * ncc + k[0][oy]) * ncc;
#pragma unroll
          for (int n = 0; n < 3; n++) v[oz][oy][n] = (float)r[x[n]] * kf;
        }
      float res[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int o = j >> 1;
        double acc = 0;
#pragma unroll
        for (int t = 0; t < 8; t++) {
          const int ox = t & 1, oy = (t >> 1) & 1, oz = t >> 2;
          acc += (double)(v[oz][oy][o + ox] * (ox ? 1.0f - cx[j] : cx[j]) * c[0][oy] * c[1][oz]);
        }
        res[j] = (float)acc;
      }
      *(float2*)(out[d] + 4 * a) = make_float2(res[0], res[1]);
      *(float2*)(out[d] + 4 * a + 2) = make_float2(res[2], res[3]);
    }
  }
}

// cell i: m += rho J, E += m0.J + rho/2 (|J|^2 + Q)
__device__ __forceinline__ void fl_impulse(float* F, int64_t n3, int64_t i, const double J[3], double Q) {
  const double r = F[i];
  double mj = 0, jj = 0;
  float m[3];
  for (int d = 0; d < 3; d++) {
    m[d] = F[(int64_t)(1 + d) * n3 + i];
    mj += (double)m[d] * J[d];
    jj += J[d] * J[d];
  }
  F[4 * n3 + i] = (float)((double)F[4 * n3 + i] + mj + 0.5 * r * (jj + Q));
  for (int d = 0; d < 3; d++) F[(int64_t)(1 + d) * n3 + i] = (float)((double)m[d] + r * J[d]);
}

// The gather of all three components at once, as separable sums.  With
// dV = w(jx) w(jy) w(jz) and a_d the acceleration on fine cell (jx,jy,jz)
// of the window,
//   J_d = sum_z w sum_y w sum_x w a_d,
//   Q   = sum dV |a|^2 - sum dV^2 |a|^2   (both separable, weights w and w^2),
// so each fine value enters three 1-D passes instead of (2 DX)^3 products.
// A workgroup owns a TXY x TXY column of fluid cells and CZ cells of it in
// z, and marches through the (CZ+1) DX fine planes those cells reach:
// per plane, the x pass (one item per window row and cell, reading the
// three components from HBM) writes five partial sums per row to LDS, and
// one thread per cell folds them along y and adds the plane, weighted, to
// the two cells whose z windows hold it.  Sums are in double in a fixed
// order, whatever CZ is; they differ from the per-tap products only by
// rounding.
// Cells whose sums one thread holds (256 a column) are updated at once
// (fl_impulse); the 8-cell windows, 64 cells a column, spread a cell's sums
// over four wavefronts and leave them in acc.
//   512^3 fine cells, fine-force gather: 0.84, 0.98 and 1.30 ms for windows of 4,
// 8 and 16 (1.02, 0.96 and 1.57 with 64-bit indices, single loads and a
// quarter of the lanes in the 16-fold; the update took another 0.33 ms).  The
// loads' address work bounds the widest windows: four values a load give 1.30
// instead of 1.57 ms there, but cost the narrow windows (0.84 -> 1.34), whose
// loads are misaligned more often than not.  No gain came from 576 threads with
// two buffers, from padded LDS rows, or from more, shorter columns than one
// workgroup a CU (each column reads (CZ+1)/CZ of its planes).
#define FG_NT 256
template <typename T, bool FINE, int DX, int TXY>
__global__ __launch_bounds__(FG_NT) void k_fl_grav_sep(const T* __restrict__ A0, const T* __restrict__ A1, const T* __restrict__ A2,
                                                       int64_t p0, int64_t p1, int64_t p2, int nf, int nc, int CZ, float a_mid,
                                                       float dt, double* acc, float* F) {
  constexpr int SPAN = 2 * DX, EY = (TXY + 1) * DX, NX = EY * TXY;
  constexpr int KW = 256 / (TXY * TXY);  // wavefront groups that share a cell's five sums: 1 or 4
  static_assert(KW == 1 || KW == 4, "256 or 64 cells a column");
  constexpr int VL = DX == 8 ? 4 : 1;
  __shared__ double X[5][NX];
  const int ncol = nc / TXY, mask = nf - 1;  // nf is a power of two
  // XCD-contiguous order: columns adjacent in x share the cache lines of
  // their window edges on one L2
  const uint32_t lb = xcd_remap(blockIdx.x, gridDim.x);
  const int bx = lb % ncol, by = (lb / ncol) % ncol, bz = lb / (ncol * ncol);
  const int c0x = bx * TXY, c0y = by * TXY, c0z = bz * CZ;
  constexpr int s = FINE ? 1 : 0;  // fine force: node on the cell's right edge
  const int m0x = c0x * DX - DX / 2 + s, m0y = c0y * DX - DX / 2 + s, m0z = c0z * DX - DX / 2 + s;
  const bool wraps = m0x < 0 || m0x + EY > nf;  // some row window of the column crosses the box edge
  const float kf = a_mid * dt / 6.0f / PI_F;
  const double inv3 = 1.0 / ((double)DX * (double)DX * (double)DX);
  double w[SPAN];
#pragma unroll
  for (int j = 0; j < SPAN; j++) w[j] = j < DX ? ((double)j + 0.5) / DX : 2.0 - ((double)j + 0.5) / DX;
  const int cell = threadIdx.x % (TXY * TXY), kw = threadIdx.x / (TXY * TXY);
  const int tx = cell % TXY, ty = cell / TXY;
  double cur[5] = {0, 0, 0, 0, 0}, prev[5] = {0, 0, 0, 0, 0};
  const int64_t n3 = (int64_t)nc * nc * nc;
  for (int pz = 0; pz < (CZ + 1) * DX; pz++) {
    const int mz = (m0z + pz) & mask;
    const T* const P0 = A0 + (int64_t)mz * nf * p0;
    const T* const P1 = A1 + (int64_t)mz * nf * p1;
    const T* const P2 = A2 + (int64_t)mz * nf * p2;
    for (int e = threadIdx.x; e < NX; e += FG_NT) {
      const int ry = e / TXY, cx = e % TXY;
      const int my = (m0y + ry) & mask;
      const uint32_t r0 = (uint32_t)(my * (int)p0), r1 = (uint32_t)(my * (int)p1), r2 = (uint32_t)(my * (int)p2);
      double x0 = 0, x1 = 0, x2 = 0, s1 = 0, s2 = 0;
      const int mx0 = m0x + cx * DX;
      // VL consecutive values per component and load
#pragma unroll
      for (int h = 0; h < SPAN; h += VL) {
        T v[3][VL];
        if (VL == 1 || wraps) {
#pragma unroll
          for (int jx = 0; jx < VL; jx++) {
            const uint32_t mx = (uint32_t)((mx0 + h + jx) & mask);
            v[0][jx] = P0[r0 + mx];
            v[1][jx] = P1[r1 + mx];
            v[2][jx] = P2[r2 + mx];
          }
        } else {
          __builtin_memcpy(v[0], P0 + (r0 + mx0 + h), sizeof(v[0]));
          __builtin_memcpy(v[1], P1 + (r1 + mx0 + h), sizeof(v[0]));
          __builtin_memcpy(v[2], P2 + (r2 + mx0 + h), sizeof(v[0]));
        }
#pragma unroll
        for (int jx = h; jx < h + VL; jx++) {
          float f0 = (float)v[0][jx - h], f1 = (float)v[1][jx - h], f2 = (float)v[2][jx - h];
          if (FINE) {
            f0 = f0 * kf;
            f1 = f1 * kf;
            f2 = f2 * kf;
          }
          const double a0 = (double)f0 * inv3, a1 = (double)f1 * inv3, a2 = (double)f2 * inv3;
          const double q = a0 * a0 + a1 * a1 + a2 * a2;
          x0 += w[jx] * a0;
          x1 += w[jx] * a1;
          x2 += w[jx] * a2;
          s1 += w[jx] * q;
          s2 += w[jx] * w[jx] * q;
        }
      }
      X[0][e] = x0;
      X[1][e] = x1;
      X[2][e] = x2;
      X[3][e] = s1;
      X[4][e] = s2;
    }
    __syncthreads();
    // plane pz is position j of cell l = pz / DX's window and j + DX of
    // cell l - 1's
    const int j = pz % DX, l = pz / DX;
    const double wa = ((double)j + 0.5) * (1.0 / DX), wb = 2.0 - ((double)(j + DX) + 0.5) * (1.0 / DX);  // w[j], w[j + DX]
    // sum k of this thread's cell: all five, or k = kw (and 4 beside 3)
    auto fold = [&](int k) {
      double y = 0;
#pragma unroll
      for (int jy = 0; jy < SPAN; jy++) y += (k == 4 ? w[jy] * w[jy] : w[jy]) * X[k][(ty * DX + jy) * TXY + tx];
      return y;
    };
    if (KW == 1) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const double y = fold(k);
        cur[k] += wa * y;
        prev[k] += wb * y;
      }
    } else {
      const double y = fold(kw);
      cur[0] += wa * y;
      prev[0] += wb * y;
    }
    if (KW == 1 || kw == 3) {
      const double y = fold(4);
      cur[4] += wa * wa * y;
      prev[4] += wb * wb * y;
    }
    if (j == DX - 1) {
      if (l >= 1) {
        const int64_t i = ((int64_t)(c0z + l - 1) * nc + (c0y + ty)) * nc + (c0x + tx);
        if (KW == 1) {
          const double J[3] = {prev[0], prev[1], prev[2]};
          fl_impulse(F, n3, i, J, prev[3] - prev[4]);
        } else {
          acc[kw * n3 + i] += kw == 3 ? prev[0] - prev[4] : prev[0];
        }
      }
#pragma unroll
      for (int k = 0; k < 5; k++) {
        prev[k] = cur[k];
        cur[k] = 0;
      }
    }
    __syncthreads();
  }
}

// whether the separable gather covers fluid n, and whether it updates the
// fluid itself (else it leaves its sums in acc)
static bool fl_sep_covers(const NuState& s, int n) {
  const int dx = (int)s.dx[n], nc = s.nc[n];
  return nc % 2 == 0 && ((dx == 2 && nc % 16 == 0) || (dx == 4 && nc % 16 == 0) || (dx == 8 && nc % 8 == 0));
}
static bool fl_sep_applies(const NuState& s, int n) { return fl_sep_covers(s, n) && (int)s.dx[n] < 8; }

template <typename T, bool FINE, int DX, int TXY>
static void fl_grav_sep_dx(cube_handle* h, const T* const A[3], const int64_t pa[3], int n, float a_mid, float dt) {
  NuState& s = h->nu;
  const int nc = s.nc[n], cols = (nc / TXY) * (nc / TXY);
  // cells of a column per workgroup: 8, or fewer (down to 2) while there is
  // less than a workgroup per CU
  int cz = 8;
  while (cz > 2 && (nc % cz || cols * (nc / cz) < 256)) cz /= 2;
  k_fl_grav_sep<T, FINE, DX, TXY><<<(unsigned)(cols * (nc / cz)), FG_NT, 0, h->stream>>>(
      A[0], A[1], A[2], pa[0], pa[1], pa[2], (int)h->nf, nc, cz, a_mid, dt, s.acc[n], s.F[n]);
}
template <typename T, bool FINE>
static bool fl_grav_sep(cube_handle* h, const T* const A[3], const int64_t pa[3], int n, float a_mid, float dt) {
  if (!fl_sep_covers(h->nu, n)) return false;
  switch ((int)h->nu.dx[n]) {
    case 2: fl_grav_sep_dx<T, FINE, 2, 16>(h, A, pa, n, a_mid, dt); break;
    case 4: fl_grav_sep_dx<T, FINE, 4, 16>(h, A, pa, n, a_mid, dt); break;
    default: fl_grav_sep_dx<T, FINE, 8, 8>(h, A, pa, n, a_mid, dt);
  }
  return true;
}

// Gather of J_d and Q over one fluid's cells from an acceleration field on
// fine-cell centres (row pitch ap).  FINE: A is the fine force component at
// nodes, the cell n taking the node n+1 on its right edge (pm.f90:163-165),
// scaled by a_mid*dt/6/pi in float; else A already holds the acceleration.
// accr = a/dx^3 (hydrogr.f90:142).  acc: [4][nc^3] doubles (J0, J1, J2, Q).
template <typename T, bool FINE>
__global__ void k_fl_grav_gather(const T* A, int64_t ap, int64_t nf, int nc, float dx, int d, float a_mid, float dt, double* acc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n3 = (int64_t)nc * nc * nc;
  if (i >= n3) return;
  const int c[3] = {(int)(i % nc), (int)((i / nc) % nc), (int)(i / ((int64_t)nc * nc))};
  const int span = 2 * (int)dx;  // fine cells per dimension reaching this fluid cell
  const double inv3 = 1.0 / ((double)dx * (double)dx * (double)dx);
  const float kf = a_mid * dt / 6.0f / PI_F;
  double J = 0, Q = 0;
  int m0[3];
  for (int e = 0; e < 3; e++) m0[e] = (int)(c[e] * dx - dx / 2);
  for (int jz = 0; jz < span; jz++) {
    const int mz = m0[2] + jz;
    float wz;
    {
      const float xx = ((float)mz + 0.5f) / dx - 0.5f;
      const int f = (int)floorf(xx);
      const float d1 = (float)(f + 1) - xx;
      wz = f == c[2] ? d1 : (f + 1 == c[2] ? 1.0f - d1 : 0.0f);
    }
    if (wz == 0.0f) continue;
    for (int jy = 0; jy < span; jy++) {
      const int my = m0[1] + jy;
      float wy;
      {
        const float xx = ((float)my + 0.5f) / dx - 0.5f;
        const int f = (int)floorf(xx);
        const float d1 = (float)(f + 1) - xx;
        wy = f == c[1] ? d1 : (f + 1 == c[1] ? 1.0f - d1 : 0.0f);
      }
      if (wy == 0.0f) continue;
      for (int jx = 0; jx < span; jx++) {
        const int mx = m0[0] + jx;
        float wx;
        {
          const float xx = ((float)mx + 0.5f) / dx - 0.5f;
          const int f = (int)floorf(xx);
          const float d1 = (float)(f + 1) - xx;
          wx = f == c[0] ? d1 : (f + 1 == c[0] ? 1.0f - d1 : 0.0f);
        }
        if (wx == 0.0f) continue;
        const float dV = wx * wy * wz;
        const int s = FINE ? 1 : 0;  // fine force: node on the cell's right edge
        const int64_t ax = ((int64_t)mx + s + nf) % nf, ay = ((int64_t)my + s + nf) % nf, az = ((int64_t)mz + s + nf) % nf;
        const float fv = (float)A[(az * nf + ay) * ap + ax];
        const double a = (double)(FINE ? fv * kf : fv) * inv3;
        J += (double)dV * a;
        Q += (double)dV * (1.0 - (double)dV) * a * a;
      }
    }
  }
  acc[(int64_t)d * n3 + i] += J;
  acc[3 * n3 + i] += Q;
}

// applies and clears the accumulators
__global__ void k_fl_grav_apply(float* F, int nc, double* acc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n3 = (int64_t)nc * nc * nc;
  if (i >= n3) return;
  const double J[3] = {acc[i], acc[n3 + i], acc[2 * n3 + i]};
  fl_impulse(F, n3, i, J, acc[3 * n3 + i]);
  for (int d = 0; d < 4; d++) acc[(int64_t)d * n3 + i] = 0;
}

__global__ void k_fl_set_u32(uint32_t* p, uint32_t v) { p[threadIdx.x] = v; }

// ------------------------------------------------------------------- host
// hydrodf.f90:17-31 constants
static const float kGLv[3] = {0.41577456f, 2.29428036f, 6.28994508f};
static const float kGLw[3] = {0.71109301f, 0.27851773f, 0.01038926f};

static inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

extern "C" int cube_nu_init(cube_handle* h, const cube_nu_params* p) {
  CUBE_EXCLUSIVE;
  if (!h || !p) return CUBE_ERR_ARG;
  if (hipSetDevice(h->p.device) != hipSuccess) return cube_fail(h, CUBE_ERR_HIP, "hipSetDevice failed");
  if (!(p->m_ev > 0) || !(p->f_neu > 0) || !(p->gamma > 1))
    return cube_fail(h, CUBE_ERR_ARG, "neutrino mass, f_neu and gamma must be positive (gamma > 1)");
  if (h->nf / 8 < FL_W) return cube_fail(h, CUBE_ERR_ARG, "fine mesh too small for the fluids");
  NuState& s = h->nu;
  s.on = true;
  s.par = *p;
  // hydrogr.f90:14 velocity unit, hydrodf.f90:9-13 start of evolution
  const float nf = (float)h->nf;
  const float dv = (2 * nf) / (3.0f * 100.0f * sqrtf(p->omega_m) * p->box);
  const float beta = 5966.34f * p->m_ev;
  const float ai_kms = (8.0f * PI_F * PI_F / 3.0f) / (p->box * p->box * (p->h0 * 100.0f) * (p->h0 * 100.0f) * p->omega_m) / (dv * dv) / 2.0f;
  const float ai_max = 1.0f / (1.0f + p->z_i_nu);
  float wsum = 0;
  for (int n = 0; n < 3; n++) {
    const float v = kGLv[n] / beta * 2.998e5f;  // km/s
    s.nc[n] = (int)(h->nf >> (n + 1));
    s.dx[n] = nf / (float)s.nc[n];
    s.cs2[n] = fmaxf(1e-6f, (v * dv) * (v * dv));
    const float x = kGLv[n];
    s.w[n] = kGLw[n] * (x * x / (expf(x) + 1.0f)) * expf(x);
    wsum += s.w[n];
    float ai = fminf(ai_kms * s.cs2[n], ai_max);
    if (p->neutrino_ic && ai < ai_max) ai = ai_max;  // NEUTRINO_IC: dfld_ai_min = dfld_ai_max
    s.ai[n] = ai;
  }
  for (int n = 0; n < 3; n++) s.w[n] /= wsum;
  for (int n = 0; n < 3; n++) {
    const int64_t n3 = (int64_t)s.nc[n] * s.nc[n] * s.nc[n];
    if (!s.F[n]) HIP_TRY(h, hipMalloc(&s.F[n], sizeof(float) * 5 * n3));
    if (!fl_sep_applies(s, n)) {
      if (!s.acc[n]) HIP_TRY(h, hipMalloc(&s.acc[n], sizeof(double) * 4 * n3));
      HIP_TRY(h, hipMemsetAsync(s.acc[n], 0, sizeof(double) * 4 * n3, h->stream));
    }
    // hg_setup: rho = 1, m = 0, E = cs2 rho/(g-1) (q equation of state)
    std::vector<float> init(5 * n3, 0.0f);
    for (int64_t i = 0; i < n3; i++) {
      init[i] = 1.0f;
      init[4 * n3 + i] = s.cs2[n] * 1.0f / (p->gamma - 1.0f);
    }
    HIP_TRY(h, hipMemcpy(s.F[n], init.data(), sizeof(float) * 5 * n3, hipMemcpyHostToDevice));
  }
  return CUBE_OK;
}

extern "C" int cube_nu_info(cube_handle* h, int n, int32_t* nc, float* dx, float* cs2, float* weight) {
  if (!h || !h->nu.on || n < 0 || n > 2) return CUBE_ERR_ARG;
  if (nc) *nc = h->nu.nc[n];
  if (dx) *dx = h->nu.dx[n];
  if (cs2) *cs2 = h->nu.cs2[n];
  if (weight) *weight = h->nu.w[n];
  return CUBE_OK;
}

extern "C" int cube_nu_set_fluid(cube_handle* h, int n, const float* fld) {
  CUBE_EXCLUSIVE;
  if (!h || !h->nu.on || n < 0 || n > 2 || !fld) return CUBE_ERR_ARG;
  const int64_t n3 = (int64_t)h->nu.nc[n] * h->nu.nc[n] * h->nu.nc[n];
  HIP_TRY(h, hipMemcpy(h->nu.F[n], fld, sizeof(float) * 5 * n3, hipMemcpyHostToDevice));
  return CUBE_OK;
}

extern "C" int cube_nu_get_fluid(cube_handle* h, int n, float* fld) {
  CUBE_EXCLUSIVE;
  if (!h || !h->nu.on || n < 0 || n > 2 || !fld) return CUBE_ERR_ARG;
  const int64_t n3 = (int64_t)h->nu.nc[n] * h->nu.nc[n] * h->nu.nc[n];
  HIP_TRY(h, hipStreamSynchronize(h->stream));
  HIP_TRY(h, hipMemcpy(fld, h->nu.F[n], sizeof(float) * 5 * n3, hipMemcpyDeviceToHost));
  return CUBE_OK;
}

template <int W>
static void fl_sweep_w(cube_handle* h, int n, int ax, float dt) {
  NuState& s = h->nu;
  const int nc = s.nc[n];
  int lnc = 0;
  while ((1 << lnc) < nc) lnc++;
  const int pitch = ax == 0 ? nc : (nc + 63) / 64 * 64 + 64 / W;
  const unsigned grid = (unsigned)((int64_t)(nc / W) * nc);
  const size_t lds = sizeof(float) * 5 * W * pitch;
  const float g = s.par.gamma, yg = 1.0f / (g - 1.0f), ydx = 1.0f / s.dx[n];
  if (ax == 0) k_fl_sweep<0, W><<<grid, FL_SNT, lds, h->stream>>>(s.F[n], nc, lnc, pitch, g, yg, dt, ydx);
  if (ax == 1) k_fl_sweep<1, W><<<grid, FL_SNT, lds, h->stream>>>(s.F[n], nc, lnc, pitch, g, yg, dt, ydx);
  if (ax == 2) k_fl_sweep<2, W><<<grid, FL_SNT, lds, h->stream>>>(s.F[n], nc, lnc, pitch, g, yg, dt, ydx);
}
// The widest strip of lines whose cells a workgroup holds, up to 16 (64-byte
// pieces of the strided sweeps' rows); nc is a power of two
static int fl_sweep(cube_handle* h, int n, int ax, float dt) {
  const int nc = h->nu.nc[n];
  if (nc * FL_W > FL_SPER * FL_SNT)
    return cube_fail(h, CUBE_ERR_ARG, "fluid of %d cells per dimension exceeds the sweep kernel", nc);
  const int most = std::min(FL_SPER * FL_SNT / nc, nc);
  if (most >= 16) fl_sweep_w<16>(h, n, ax, dt);
  else if (most >= 8) fl_sweep_w<8>(h, n, ax, dt);
  else fl_sweep_w<4>(h, n, ax, dt);
  HIP_TRY(h, hipGetLastError());
  return 0;
}

// dfld_evolve (hydrodf.f90:90-110): each active fluid swept x,y,z (dir > 0)
// or z,y,x, then its timestep folded into dt_neu
extern "C" int cube_fluid_evolve(cube_handle* h, float dt, int dir, float a, float* dt_neu) {
  if (!h || !h->nu.on) return CUBE_ERR_ARG;
  if (hipSetDevice(h->p.device) != hipSuccess) return cube_fail(h, CUBE_ERR_HIP, "hipSetDevice failed");
  NuState& s = h->nu;
  int pr = prof_begin(h, PS_FLUID);
  for (int n = 0; n < 3; n++) {
    if (!(a >= s.ai[n])) continue;
    for (int k = 0; k < 3; k++) {
      const int ax = dir > 0 ? k : 2 - k;
      int r = fl_sweep(h, n, ax, dt);
      if (r) return r;
    }
    uint32_t* dtb = h->uflags + 48;
    k_fl_set_u32<<<1, 1, 0, h->stream>>>(dtb, 0x4e6e6b28u);  // 1e9f, the reference's start value
    const int lines = s.nc[n] * s.nc[n];
    k_fl_dt<<<(unsigned)std::min((lines + FL_NT / 64 - 1) / (FL_NT / 64), 2048), FL_NT, 0, h->stream>>>(s.F[n], s.nc[n], s.par.gamma, s.dx[n], dtb);
    HIP_TRY(h, hipGetLastError());
    uint32_t hb;
    HIP_TRY(h, hipMemcpyAsync(&hb, dtb, 4, hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    float dtn;
    memcpy(&dtn, &hb, 4);
    if (dtn == 1e9f) dtn = 1.0f;
    if (dt_neu) *dt_neu = fminf(*dt_neu, dtn);
  }
  prof_end(h, pr);
  return CUBE_OK;
}

// ---- coupling to the PM step (called from cube_pm)
static FlSet fl_set(const NuState& s) {
  FlSet f{};
  for (int n = 0; n < 3; n++) {
    f.rho[n] = s.F[n];
    f.nc[n] = s.nc[n];
    f.w[n] = s.w[n];
  }
  return f;
}

// Coarse-mesh density (before the coarse FFT); leaves the fine-cell-centre
// density in fine.W for fl_density_fine.
int fl_density_coarse(cube_handle* h, float a_mid, double* mass_added, double* mass_dev) {
  NuState& s = h->nu;
  const int homog = 1.0f / a_mid - 1.0f > s.par.z_i_nu;
  const int64_t nf = h->nf;
  float* D = (float*)h->fine.W;
  if (!homog) {
    k_fl_density_centres<<<(unsigned)(nf * nf / 4), 256, 0, h->stream>>>(fl_set(s), (int)nf, D);
    HIP_TRY(h, hipGetLastError());
  }
  const int64_t n3c = h->n3c;
  const int64_t nb = (int64_t)nblk(n3c);
  if (nb > h->dred_n - 16) return cube_fail(h, CUBE_ERR_ARG, "reduction buffer too small");
  if (h->prec == 4)
    k_fl_add_coarse<float><<<(unsigned)nb, 256, 0, h->stream>>>((float*)h->coarse.R, D, nf, (int)h->nc, s.par.f_neu, homog,
                                                                h->dred);
  else
    k_fl_add_coarse<double><<<(unsigned)nb, 256, 0, h->stream>>>((double*)h->coarse.R, D, nf, (int)h->nc, s.par.f_neu, homog,
                                                                 h->dred);
  HIP_TRY(h, hipGetLastError());
  if (mass_dev) return reduce_doubles_dev(h, h->dred, nb, 1, mass_dev);
  if (mass_added) return reduce_doubles(h, h->dred, nb, 1, mass_added);
  return 0;
}

int fl_density_fine(cube_handle* h, float a_mid, double* mass_added, double* mass_dev) {
  NuState& s = h->nu;
  const int homog = 1.0f / a_mid - 1.0f > s.par.z_i_nu;
  const int64_t nf = h->nf;
  const int64_t nb = (int64_t)nblk(nf * nf * nf);
  int lnf = 0;
  while (((int64_t)1 << lnf) < nf) lnf++;
  if (nb > h->dred_n - 16) return cube_fail(h, CUBE_ERR_ARG, "reduction buffer too small");
  if (h->prec == 4)
    k_fl_add_fine<float><<<(unsigned)nb, 256, 0, h->stream>>>((float*)h->fine.R, (const float*)h->fine.W, nf, lnf, s.par.f_neu, homog,
                                                              h->dred);
  else
    k_fl_add_fine<double><<<(unsigned)nb, 256, 0, h->stream>>>((double*)h->fine.R, (const float*)h->fine.W, nf, lnf, s.par.f_neu,
                                                               homog, h->dred);
  HIP_TRY(h, hipGetLastError());
  if (mass_dev) return reduce_doubles_dev(h, h->dred, nb, 1, mass_dev);
  if (mass_added) return reduce_doubles(h, h->dred, nb, 1, mass_added);
  return 0;
}

// The three fine-force components (Ff[d], row pitch pf[d]) into every active
// fluid, or into its accumulators where the gather does not update it itself.
int fl_gravity_fine(cube_handle* h, const void* const Ff[3], const int64_t pf[3], float a_mid, float dt) {
  NuState& s = h->nu;
  for (int n = 0; n < 3; n++) {
    if (!(a_mid >= s.ai[n])) continue;
    const int64_t n3 = (int64_t)s.nc[n] * s.nc[n] * s.nc[n];
    if (h->prec == 4) {
      const float* A[3] = {(const float*)Ff[0], (const float*)Ff[1], (const float*)Ff[2]};
      if (fl_grav_sep<float, true>(h, A, pf, n, a_mid, dt)) {
        HIP_TRY(h, hipGetLastError());
        continue;
      }
    } else {
      const double* A[3] = {(const double*)Ff[0], (const double*)Ff[1], (const double*)Ff[2]};
      if (fl_grav_sep<double, true>(h, A, pf, n, a_mid, dt)) {
        HIP_TRY(h, hipGetLastError());
        continue;
      }
    }
    for (int d = 0; d < 3; d++) {
      if (h->prec == 4)
        k_fl_grav_gather<float, true><<<nblk(n3), 256, 0, h->stream>>>((const float*)Ff[d], pf[d], h->nf, s.nc[n], s.dx[n], d,
                                                                      a_mid, dt, s.acc[n]);
      else
        k_fl_grav_gather<double, true><<<nblk(n3), 256, 0, h->stream>>>((const double*)Ff[d], pf[d], h->nf, s.nc[n], s.dx[n],
                                                                       d, a_mid, dt, s.acc[n]);
      HIP_TRY(h, hipGetLastError());
    }
  }
  return 0;
}

static int fl_apply(cube_handle* h, float a_mid) {
  NuState& s = h->nu;
  for (int n = 0; n < 3; n++) {
    if (!(a_mid >= s.ai[n]) || fl_sep_applies(s, n)) continue;
    const int64_t n3 = (int64_t)s.nc[n] * s.nc[n] * s.nc[n];
    k_fl_grav_apply<<<nblk(n3), 256, 0, h->stream>>>(s.F[n], s.nc[n], s.acc[n]);
    HIP_TRY(h, hipGetLastError());
  }
  return 0;
}

// After the fine kicks: apply the fine impulses that accumulators hold, then
// gather and apply the coarse ones (pm.f90:374-422 runs after the fine phase).
// The coarse acceleration at fine-cell centres goes into the fine-force buffers
// Ff[d] (row pitch pf[d]), which the fine phase no longer needs.
int fl_gravity_finish(cube_handle* h, void* const Ff[3], const int64_t pf[3], float a_mid, float dt) {
  NuState& s = h->nu;
  bool any = false;
  for (int n = 0; n < 3; n++) any = any || a_mid >= s.ai[n];
  if (!any) return 0;
  int r;
  if ((r = fl_apply(h, a_mid))) return r;
  const int64_t nf = h->nf;
  float* A[3] = {(float*)Ff[0], (float*)Ff[1], (float*)Ff[2]};
  if (h->prec == 4)
    k_fl_coarse_at_centres<float><<<(unsigned)(nf * nf / 4), 256, 0, h->stream>>>((const float*)h->fc, (int)h->nc, (int)nf, a_mid,
                                                                                  dt, A[0], A[1], A[2], pf[0], pf[1], pf[2]);
  else
    k_fl_coarse_at_centres<double><<<(unsigned)(nf * nf / 4), 256, 0, h->stream>>>((const double*)h->fc, (int)h->nc, (int)nf, a_mid,
                                                                                   dt, A[0], A[1], A[2], pf[0], pf[1], pf[2]);
  HIP_TRY(h, hipGetLastError());
  const float* Ac[3] = {A[0], A[1], A[2]};
  for (int n = 0; n < 3; n++) {
    if (!(a_mid >= s.ai[n])) continue;
    const int64_t n3 = (int64_t)s.nc[n] * s.nc[n] * s.nc[n];
    if (!fl_grav_sep<float, false>(h, Ac, pf, n, a_mid, dt))
      for (int d = 0; d < 3; d++)
        k_fl_grav_gather<float, false><<<nblk(n3), 256, 0, h->stream>>>(A[d], pf[d], nf, s.nc[n], s.dx[n], d, a_mid, dt,
                                                                        s.acc[n]);
    HIP_TRY(h, hipGetLastError());
  }
  return fl_apply(h, a_mid);
}

void fl_free(NuState& s) {
  for (int n = 0; n < 3; n++) {
    if (s.F[n]) (void)hipFree(s.F[n]);
    if (s.acc[n]) (void)hipFree(s.acc[n]);
    s.F[n] = nullptr;
    s.acc[n] = nullptr;
  }
  s.on = false;
}
