// Level-set kernels: pressure extrapolation into the solid (the path the
// reference's advectLevelSet really runs) and WENO5 / SSP-RK3 advection of
// phi (cuAdvectLsJB).  Both work on the 5-cell mirror-padded domain that
// advect_CUDA builds (src/LevelSet/lsTransportEc.cu:39-166), with the
// reference's per-point boundary substitutions on the outermost padded
// layers restated exactly.  Unlike the reference (floor-divided grids,
// lsTransportEc.cu:58-79), every point is computed, for any size.
#include <cmath>

#include "ops.hpp"

namespace emx {

namespace {

constexpr int GC = 5;  // gcells, lsTransportEc.cu:39

struct PDims {
  int x, y, z;
  __host__ __device__ long long N() const { return (long long)x * y * z; }
};

__device__ __forceinline__ int mirror(int i, int n) {
  // padded index -> interior index of the even mirror used by
  // cuGhostCellsMirror3d{X,Y,Z} (lsTools.cu:482-585)
  int s = i < GC ? 2 * GC - 1 - i : (i >= n + GC ? 2 * (n + GC) - 1 - i : i);
  return s - GC;
}

// cuSwapToGhost + the three mirror passes, as one gather.
__global__ void k_pad(const double* in, int nx, int ny, int nz, double* out,
                      PDims g) {
  const long long NG = g.N();
  for (long long p = (long long)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; p < NG;
       p += (long long)gridDim.x * blockDim.x) {
    const unsigned up = (unsigned)p, row = up / (unsigned)g.x;  // NG < 2^32
    const int i = (int)(up - row * (unsigned)g.x), j = (int)(row % (unsigned)g.y),
              k = (int)(row / (unsigned)g.y);
    const int is = mirror(i, nx), js = mirror(j, ny), ks = mirror(k, nz);
    out[p] = in[(long long)is + (long long)nx * ((long long)js + (long long)ny * ks)];
  }
}

// cuSwapFromGhost (lsTools.cu:798-822).
__global__ void k_unpad(const double* in, PDims g, int nx, int ny, int nz,
                        double* out) {
  const long long N = (long long)nx * ny * nz;
  for (long long p = (long long)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; p < N;
       p += (long long)gridDim.x * blockDim.x) {
    const unsigned up = (unsigned)p, row = up / (unsigned)nx;
    const int i = (int)(up - row * (unsigned)nx), j = (int)(row % (unsigned)ny),
              k = (int)(row / (unsigned)ny);
    out[p] = in[(long long)(i + GC) + (long long)g.x * ((long long)(j + GC) + (long long)g.y * (k + GC))];
  }
}

// DevFirstOrder_LS (src/LevelSet/extrapol.cu:105-153) at padded point id:
// the metric-scaled central difference of S along each axis, one-sided with
// factor 1 for all three when the point lies on any face of the padded grid.
__device__ __forceinline__ void ls_grad1_point(const double* S, const double m[3], PDims g,
                                               double iX, double iY, double iZ, long long id,
                                               int x, int y, int z, double dphi[3]) {
  const long long sxy = (long long)g.x * g.y;
  long long ip = id + 1, im = id - 1, jp = id + g.x, jm = id - g.x, kp = id + sxy,
            km = id - sxy;
  double factor = 0.5;
  if (x == 0) { im = id; factor = 1.0; }
  if (y == 0) { jm = id; factor = 1.0; }
  if (z == 0) { km = id; factor = 1.0; }
  if (x == g.x - 1) { ip = id; factor = 1.0; }
  if (y == g.y - 1) { jp = id; factor = 1.0; }
  if (z == g.z - 1) { kp = id; factor = 1.0; }
  dphi[0] = factor * iX * m[0] * (S[ip] - S[im]);
  dphi[1] = factor * iY * m[1] * (S[jp] - S[jm]);
  dphi[2] = factor * iZ * m[2] * (S[kp] - S[km]);
}

// extrapolKernel (extrapol.cu:5-103, extFlag>0) at one solid point (phiS >
// 0) of the padded grid: the upwind metric-scaled one-sided differences of
// ext along the sign of the solid's gradient.  Elsewhere the reference's rs
// is exactly zero (so = 0 and finite operands).  geo: the point's metrics
// 1, 5, 9 and gradient of the solid (k_ls_solid_geom).
__device__ __forceinline__ double ls_extrap_rs(long long id, const double* ext,
                                               const double* geo, PDims g, double iX,
                                               double iY, double iZ) {
  const long long sxy = (long long)g.x * g.y;
  const unsigned uid = (unsigned)id, row = uid / (unsigned)g.x;  // NG < 2^32
  const int x = (int)(uid - row * (unsigned)g.x), y = (int)(row % (unsigned)g.y),
            z = (int)(row / (unsigned)g.y);
  long long ip = id + 1, im = id - 1, jp = id + g.x, jm = id - g.x, kp = id + sxy,
            km = id - sxy;
  long long id2 = id;
  if (x == 0) { id2 = ip; im = id; }
  if (y == 0) { id2 = jp; jm = id; }
  if (z == 0) { id2 = kp; km = id; }
  if (x == g.x - 1) { id2 = im; ip = id; }
  if (y == g.y - 1) { id2 = jm; jp = id; }
  if (z == g.z - 1) { id2 = km; kp = id; }
  const double so = 1.0;
  const double m1 = geo[0], m5 = geo[1], m9 = geo[2];
  const double pdx = so * geo[3], pdy = so * geo[4], pdz = so * geo[5];
  const double e2 = ext[id2];
  const double xd = iX * m1 * (e2 - ext[im]);
  const double yd = iY * m5 * (e2 - ext[jm]);
  const double zd = iZ * m9 * (e2 - ext[km]);
  const double xu = iX * m1 * (ext[ip] - e2);
  const double yu = iY * m5 * (ext[jp] - e2);
  const double zu = iZ * m9 * (ext[kp] - e2);
  double s = (double)(pdx > 0.0) - (double)(pdx < 0.0);
  double r = (0.5 * (s + 1.0) * xd + 0.5 * fabs(s - 1.0) * xu) * pdx;
  s = (double)(pdy > 0.0) - (double)(pdy < 0.0);
  r += (0.5 * (s + 1.0) * yd + 0.5 * fabs(s - 1.0) * yu) * pdy;
  s = (double)(pdz > 0.0) - (double)(pdz < 0.0);
  r += (0.5 * (s + 1.0) * zd + 0.5 * fabs(s - 1.0) * zu) * pdz;
  return r;
}

// Ordered list of the solid points (S > 0) of the padded grid: per-chunk
// counts, one exclusive scan, then each chunk writes its indices in order
// (wavefront ballots, no atomics).
constexpr int LS_CHUNK = 4096;

__global__ void k_ls_solid_count(const double* S, long long NG, int* bcount) {
  __shared__ int wsum[4];
  const long long base = (long long)blockIdx.x * LS_CHUNK;
  int c = 0;
  for (int t = threadIdx.x; t < LS_CHUNK; t += 256) {
    const long long id = base + t;
    c += (id < NG && S[id] > 0.0) ? 1 : 0;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) bcount[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

// Exclusive scan of nb chunk counts in place (one workgroup of 1024); the
// total into *total.
__global__ void __launch_bounds__(1024) k_ls_scan(int* bcount, int nb, int* total) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  const int per = (nb + 1023) / 1024;
  const int b0 = t * per < nb ? t * per : nb;
  const int b1 = b0 + per < nb ? b0 + per : nb;
  int s = 0;
  for (int b = b0; b < b1; b++) s += bcount[b];
  part[t] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = t > 0 ? part[t - 1] : 0;
  for (int b = b0; b < b1; b++) {
    const int c = bcount[b];
    bcount[b] = run;
    run += c;
  }
  if (t == 1023) *total = part[1023];
}

__global__ void k_ls_solid_write(const double* S, long long NG, const int* boff, int* list) {
  __shared__ int wsum[4];
  const long long base = (long long)blockIdx.x * LS_CHUNK;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int run = boff[blockIdx.x];
  for (int r = 0; r < LS_CHUNK / 256; r++) {
    const long long id = base + r * 256 + threadIdx.x;
    const bool f = id < NG && S[id] > 0.0;
    const unsigned long long m = __ballot(f);
    const int pre = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[wv] = __popcll(m);
    __syncthreads();
    int off = run;
    for (int w = 0; w < wv; w++) off += wsum[w];
    if (f) list[off + pre] = (int)id;
    run += wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
  }
}

__global__ void k_copy2(const double* a, double* b, double* c, long long n) {
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (long long)gridDim.x * blockDim.x) {
    const double v = a[p];
    b[p] = v;
    c[p] = v;
  }
}

// One SSP-RK3 stage of the extrapolation (RunGK_{First,Second,Third}S,
// extrapol.cu:155-212) at the listed solid points:
//   stage 0: out = ext - dt*rs
//   stage 1: out = 0.75*P + 0.25*(ext - dt*rs)
//   stage 2: out = (P + 2*(ext - dt*rs))/3      (out may alias P)
// The fluid points keep P in all three buffers: their rs is zero, and the
// stages only re-round them (0.75*P + 0.25*P, (P + 2*P)/3), which the
// reference does and this build does not.
// The metrics 1, 5, 9 (read from the interior grid through the mirror map
// of the padding) and DevFirstOrder_LS's gradient of S at each listed solid
// point, six doubles per entry: the only points where the pseudo-stages use
// them.
__global__ void k_ls_solid_geom(const int* list, const int* count, const double* S,
                                const double* jbn, int nx, int ny, int nz, PDims g, double iX,
                                double iY, double iZ, double* geo) {
  const int n = *count;
  const long long N = (long long)nx * ny * nz;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
    const long long id = list[t];
    const unsigned uid = (unsigned)id, row = uid / (unsigned)g.x;  // NG < 2^32
    const int x = (int)(uid - row * (unsigned)g.x), y = (int)(row % (unsigned)g.y),
              z = (int)(row / (unsigned)g.y);
    const long long q = mirror(x, nx) + (long long)nx * (mirror(y, ny) + (long long)ny * mirror(z, nz));
    const double m[3] = {jbn[q], jbn[4 * N + q], jbn[8 * N + q]};
    double dphi[3];
    ls_grad1_point(S, m, g, iX, iY, iZ, id, x, y, z, dphi);
    double* e = geo + 6 * (long long)t;
    e[0] = m[0];
    e[1] = m[1];
    e[2] = m[2];
    e[3] = dphi[0];
    e[4] = dphi[1];
    e[5] = dphi[2];
  }
}

__global__ void k_ls_extrap_list(int stage, const int* list, const int* count, const double* ext,
                                 const double* P, const double* geo, PDims g, double iX,
                                 double iY, double iZ, double dt, double* out) {
  const int n = *count;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
    const long long id = list[t];
    const double rs = ls_extrap_rs(id, ext, geo + 6 * (long long)t, g, iX, iY, iZ);
    const double ev = ext[id];
    if (stage == 0) out[id] = ev - dt * rs;
    else if (stage == 1) out[id] = 0.75 * P[id] + 0.25 * (ev - dt * rs);
    else out[id] = (P[id] + 2.0 * (ev - dt * rs)) / 3.0;
  }
}

// 1/x for x in the normal range: the hardware reciprocal r (e = 1 - x r of
// about 2^-27) refined by r (1 + e + e^2), within an ulp of the correctly
// rounded quotient.
__device__ __forceinline__ double recip_nr(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// 1/sqrt(x) for x > 0, by the same third-order step: r (1 + e/2 + 3 e^2/8),
// e = 1 - x r^2, given xr = x r.
__device__ __forceinline__ double rsqrt_step(double r, double xr) {
  const double e = __builtin_fma(-xr, r, 1.0);
  return __builtin_fma(r * e, __builtin_fma(e, 0.375, 0.5), r);
}

// At infinity r = 0, and the largest number takes the place of x in x r (0,
// not NaN): the result is 0.
__device__ __forceinline__ double rsqrt_nr(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  return rsqrt_step(r, __builtin_fmin(x, 0x1.fffffffffffffp1023) * r);
}

// sqrt(x) for x >= 0: x/sqrt(x) and one residual step where x is a positive
// finite number; 0, infinity and NaN are their own roots.
__device__ __forceinline__ double sqrt_nr(double x) {
  const double r0 = __builtin_amdgcn_rsq(x), r = rsqrt_step(r0, x * r0);
  const double s = x * r;
  const double t = __builtin_fma(__builtin_fma(-s, s, x), 0.5 * r, s);
  return __builtin_amdgcn_class(x, 0x180) ? t : x;
}

// Phi_x_WENO (src/LevelSet/lsTools.cu:9-50), written in the differences
// e_i = b_{i+1} - b_i of its operands:
//   4 beta_k = (13/3) dd_k^2 + g_k^2,  dd_k = e_{k+1} - e_k,
//     g = 3 e2 - e1,  e2 + e3,  3 e3 - e4
//   6 p_k = 6 b3 + q_k,  q = 5 e2 - 2 e1,  e2 + 2 e3,  4 e3 - e4
// (p_k the three third-order candidates), so that with weights a_k =
// c_k/t_k^2 (t_k = 4 (beta_k + 1e-6)) the derivative is
// b3 + sum(a_k q_k)/(6 sum(a_k)), and with the weights multiplied by
// (t_1 t_2 t_3)^2 it takes one reciprocal.  42 FP64 instructions (70 as the
// reference writes the sums).  t_k lies in [4e-6, ~1e9], so the products
// stay far from the double range's ends.
__device__ __forceinline__ double weno5_e(double b3, double e1, double e2, double e3, double e4) {
  const double d1 = e2 - e1, d2 = e3 - e2, d3 = e4 - e3;
  const double g1 = __builtin_fma(3.0, e2, -e1), g2 = e2 + e3, g3 = __builtin_fma(3.0, e3, -e4);
  const double t1 = __builtin_fma((13.0 / 3.0) * d1, d1, __builtin_fma(g1, g1, 4.0e-6));
  const double t2 = __builtin_fma((13.0 / 3.0) * d2, d2, __builtin_fma(g2, g2, 4.0e-6));
  const double t3 = __builtin_fma((13.0 / 3.0) * d3, d3, __builtin_fma(g3, g3, 4.0e-6));
  const double u1 = t2 * t3, u2 = t1 * t3, u3 = t1 * t2;
  const double w1 = u1 * u1, w2 = 6.0 * (u2 * u2), w3 = 3.0 * (u3 * u3);
  const double q1 = __builtin_fma(2.0, g1, -e2), q2 = g2 + e3, q3 = g3 + e3;
  const double num = __builtin_fma(w1, q1, __builtin_fma(w2, q2, w3 * q3));
  return __builtin_fma(num * (1.0 / 6.0), recip_nr(w1 + w2 + w3), b3);
}

// Whether any of the three candidates 6 b3 + q_k may be positive (a NaN
// counts as one).
__device__ __forceinline__ bool weno5_positive(double b3, double e1, double e2, double e3,
                                               double e4) {
  const double lim = -6.0 * b3;
  const double q1 = __builtin_fma(5.0, e2, -2.0 * e1), q2 = __builtin_fma(2.0, e3, e2),
               q3 = __builtin_fma(4.0, e3, -e4);
  return !(q1 <= lim && q2 <= lim && q3 <= lim);
}

__device__ __forceinline__ double weno5(double b1, double b2, double b3, double b4, double b5) {
  return weno5_e(b3, b2 - b1, b3 - b2, b4 - b3, b5 - b4);
}

// ---------------------------------------------------------------------------
// Level-set reinitialisation (cuReinitLsJB, lsTransportEc.cu:422-676).

// The padded coordinates whose mirror image (cuGhostCellsMirror3d{Z,Y,X},
// lsTools.cu:482-585, applied over the full padded ranges) is the interior
// padded coordinate X of a line of n interior points: X itself, its
// reflection into the low ghost layers and into the high ones.
__device__ __forceinline__ int mirror_images(int X, int n, int c[3]) {
  int k = 0;
  c[k++] = X;
  if (X < 2 * GC) c[k++] = 2 * GC - 1 - X;
  if (X >= n) c[k++] = 2 * (n + GC) - 1 - X;
  return k;
}

// One axis of the Godunov gradient, max(max(L, 0), max(-R, 0)), from the
// axis' six metric-scaled differences bd (offsets -2..+3) multiplied by
// sign(phi0).  (With that sign s, the reference's max(max(L,0)^2, min(R,0)^2)
// for s > 0 and max(max(R,0)^2, min(L,0)^2) for s < 0 are both the square
// of this.)  L takes bd[0..4] (the fifth given as l5), R takes bd[5..1].
// A WENO derivative is a convex combination of its three candidates, so a
// side whose candidates are all <= 0 (left) or all >= 0 (right) gives 0
// and is not formed.  Away from kinks of phi that is one of the two
// sides: the operands of the side that counts are selected and one
// derivative is evaluated; a second one only where a lane of the wavefront
// needs both.  The differences e of R's operands are L's in the opposite
// order and sign, so -R = -bd[3] + (the sum L adds to its b3).
__device__ __forceinline__ double godunov_axis(const double bd[6], double l5) {
  const double e1 = bd[1] - bd[0], e2 = bd[2] - bd[1], e3 = bd[3] - bd[2], e4 = l5 - bd[3],
               r4 = bd[4] - bd[3], r5 = bd[5] - bd[4];
  const bool left = weno5_positive(bd[2], e1, e2, e3, e4);
  const bool right = weno5_positive(-bd[3], r5, r4, e3, e2);
  const double v = weno5_e(left ? bd[2] : -bd[3], left ? e1 : r5, left ? e2 : r4, e3,
                           left ? e4 : e2);
  double c = v > 0.0 ? v : 0.0;
  if (left && right) {
    const double r = weno5_e(-bd[3], r5, r4, e3, e2);
    c = r > c ? r : c;
  }
  return c;
}

// The reference's edge rules for the six metric-scaled backward differences
// bd (offsets -2..+3) of position q of n: the index-0 rule of
// Dev1thO_Downwind (lsTools.cu:53-95, the forward difference) and the
// substitutions of PhiDevPlusParameterJB (:587-673, operands bd[0..4]) and
// PhiDevMinusParameterJB (:676-770, operands bd[5..1]).  Past the low face
// the first difference is repeated, past the high face they are mirrored.
__device__ __forceinline__ void edge_bd(double bd[6], int q, int n) {
  if (q == 0) bd[2] = bd[3];
  if (q <= 1) bd[1] = bd[2];
  if (q <= 2) bd[0] = bd[1];
  if (q == n - 1) bd[3] = bd[2];
  if (q == n - 1) bd[4] = bd[1];
  if (q == n - 2) bd[4] = bd[3];
  if (q == n - 1) bd[5] = bd[0];
  if (q == n - 2) bd[5] = bd[2];
  if (q == n - 3) bd[5] = bd[4];
}

// The plane of a z-marching workgroup of 256 work-items in LDS: a tile of
// 2^ltx x 2^(8-ltx) columns (x, y) and three more on either side along each
// axis (the stencils are along the axes, so no corners), in two buffers taken
// in turn.  A work-item has its own column's value in registers and loads at
// most one halo column, so a plane costs two loads per point; read from
// memory the stencils took 13, and a stage's 19 to 21 loads and stores per
// point kept the address units 90% busy.
struct StencilTile {
  static constexpr int CELLS = 38 * 14;  // 32 x 8; 16 x 16 takes 22 x 22
  int w, own, halo;  // row stride; cells of the column and of its halo column
  int hx, hy;        // that column's place in the tile (halo < 0: none)
  __device__ __forceinline__ StencilTile(int ltx) {
    const int tx = 1 << ltx, ty = 256 >> ltx;
    int t = threadIdx.x;
    w = tx + 6;
    own = ((t >> ltx) + 3) * w + (t & (tx - 1)) + 3;
    if (t < 6 * tx) {
      const int r = t >> ltx;
      hx = t & (tx - 1);
      hy = r < 3 ? r - 3 : ty + r - 3;
    } else {
      t -= 6 * tx;
      const int r = t % 6;
      hx = r < 3 ? r - 3 : tx + r - 3;
      hy = t / 6;
    }
    halo = (int)threadIdx.x < 6 * tx || hy < ty ? (hy + 3) * w + hx + 3 : -1;
  }
  __device__ __forceinline__ void put(double* c, double v, double h) const {
    c[own] = v;
    if (halo >= 0) c[halo] = h;
  }
  // The seven stencil values along x and y around the own column.
  __device__ __forceinline__ void get(const double* c, double v, double vx[7],
                                      double vy[7]) const {
#pragma unroll
    for (int o = 0; o < 7; o++) {
      vx[o] = o == 3 ? v : c[own + o - 3];
      vy[o] = o == 3 ? v : c[own + (o - 3) * w];
    }
  }
};

// One SSP-RK3 stage of the reinitialisation: the two JB WENO derivatives per
// axis, the Godunov |grad phi| by the sign of phi0 and rs = S(phi0)
// (|grad phi| - 1), S = phi0/sqrt(phi0^2 + dmin^2) (reini_RS_WENOJB,
// lsTools.cu:824-900), then RunGK_{First,Second,Third}S
// (extrapol.cu:155-212).  src is the stage input, P the iteration's phi,
// which is also its phi0 (the reference copies phi to phi0 at the start of
// every iteration).  Stage 0 computes every padded point, stage 1 all but
// the two outermost ghost layers (the last stage's stencils do not reach
// them), stage 2 the interior points, each written into out, a different
// array, together with its mirror images in the ghost layers: out is then
// the next iteration's phi with the ghost mirroring that iteration would
// start with already applied (given phi, the last iteration, only the
// interior, into phi).  dmin and jbn (1, 5, 9 used) are interior fields, read
// at a ghost point's mirror image.
//
// A workgroup owns a 32 x 8 tile of (x, y) and marches z through a slab of
// kz planes with the stencil's z values and differences in registers and the
// plane in LDS (StencilTile).  At 218 x 186 x 170 padded points a stage takes
// 94-99 us: 182 us with one point per work-item and both WENO derivatives of
// every axis, 100-121 us with the x and y stencils read from memory and
// padded copies of dmin and the metrics (five passes of 28 us a call, now
// one).  About 400 VALU instructions per point-wave bound it, with the memory
// floor (24 B per padded and 32 B per interior point) close behind.  Wider
// tiles waste lanes at the row ends (64 x 4: 10% slower), 16 x 16 tiles 3%.
constexpr int RI_TX = 32, RI_TY = 8;

template <int STAGE>
__global__ void __launch_bounds__(256)
k_ls_reinit_stage(const double* src, const double* P, const double* dmin, const double* jbn,
                  PDims g, int kz, double iX, double iY, double iZ, double dt, double* out,
                  double* phi) {
  constexpr int LO = STAGE == 0 ? 0 : (STAGE == 1 ? GC - 3 : GC);
  const int nbx = (g.x - 2 * LO + RI_TX - 1) / RI_TX, nby = (g.y - 2 * LO + RI_TY - 1) / RI_TY;
  const int b = (int)xcd_block(blockIdx.x, gridDim.x);
  const int x0 = LO + (b % nbx) * RI_TX, y0 = LO + (b / nbx % nby) * RI_TY;
  const int x = x0 + (int)threadIdx.x % RI_TX, y = y0 + (int)threadIdx.x / RI_TX;
  const int z0 = LO + b / (nbx * nby) * kz, z1 = min(z0 + kz, g.z - LO);
  const bool own = x < g.x - LO && y < g.y - LO;
  // positions past the padded grid's faces are clamped: work-items there
  // store nothing, and a difference over one is never used
  const int xc = min(x, g.x - 1), yc = min(y, g.y - 1);
  const unsigned sy = (unsigned)g.x, sz = (unsigned)g.x * (unsigned)g.y;  // NG < 2^32
  const unsigned col = (unsigned)xc + sy * (unsigned)yc;
  const int nx = g.x - 2 * GC, ny = g.y - 2 * GC, nz = g.z - 2 * GC;
  const unsigned vsz = (unsigned)nx * (unsigned)ny;
  const size_t vN = (size_t)vsz * (unsigned)nz;
  const unsigned vcol = (unsigned)mirror(xc, nx) + (unsigned)nx * (unsigned)mirror(yc, ny);
  __shared__ double cells[2][StencilTile::CELLS];
  const StencilTile tile(5);
  const unsigned hcol = (unsigned)min(max(x0 + tile.hx, 0), g.x - 1) +
                        sy * (unsigned)min(max(y0 + tile.hy, 0), g.y - 1);
  const bool edge_x = STAGE < 2 && __any(xc < 3 || xc > g.x - 4);
  const bool edge_y = STAGE < 2 && __any(yc < 3 || yc > g.y - 4);
  auto clampz = [&](int z) { return STAGE < 2 ? min(max(z, 0), g.z - 1) : z; };
  // a field's value at byte offset off (the padded grid has fewer than 2^29
  // points): uniform base, 32-bit offset
  auto at = [](const double* f, unsigned off) {
    return reinterpret_cast<const double*>(reinterpret_cast<const char*>(f) + off);
  };
  auto ld = [&](const double* f, unsigned off) { return *at(f, off); };
  auto plane = [&](int z) { return ld(src, (col + (unsigned)clampz(z) * sz) * 8u); };
  double vz[4], dz[6];  // values of planes z .. z+3; the stencil's differences along z
#pragma unroll
  for (int o = 0; o < 3; o++) vz[o + 1] = plane(z0 + o);
  {
    const double a = plane(z0 - 3), b2 = plane(z0 - 2), c = plane(z0 - 1);
    dz[1] = b2 - a;
    dz[2] = c - b2;
    dz[3] = vz[1] - c;
    dz[4] = vz[2] - vz[1];
    dz[5] = vz[3] - vz[2];
  }
  double hv = ld(src, (hcol + (unsigned)z0 * sz) * 8u);
  for (int z = z0; z < z1; z++) {
#pragma unroll
    for (int o = 0; o < 3; o++) vz[o] = vz[o + 1];
#pragma unroll
    for (int o = 0; o < 5; o++) dz[o] = dz[o + 1];
    vz[3] = plane(z + 3);
    dz[5] = vz[3] - vz[2];
    const unsigned id = col + (unsigned)z * sz, off = id * 8u;
    const unsigned vid = vcol + (unsigned)mirror(z, nz) * vsz, voff = vid * 8u;
    const double sv = vz[0];
    double vx[7], vy[7];
    double* c = cells[(z - z0) & 1];
    tile.put(c, sv, hv);
    lds_barrier();
    if (z + 1 < z1) hv = ld(src, (hcol + (unsigned)(z + 1) * sz) * 8u);
    tile.get(c, sv, vx, vy);
    const double p0 = STAGE == 0 ? sv : ld(P, off);
    // metric / spacing with the sign of phi0 (at phi0 = 0, S and with it rs
    // vanish)
    auto signed_by_p0 = [&](double s) {
      return __longlong_as_double(__double_as_longlong(s) ^
                                  (__double_as_longlong(p0) & (long long)(1ull << 63)));
    };
    const double sx = signed_by_p0(iX * ld(jbn, voff)),
                 sY = signed_by_p0(iY * ld(jbn + 4 * vN, voff)),
                 sZ = signed_by_p0(iZ * ld(jbn + 8 * vN, voff)), d = ld(dmin, voff);
    double bx[6], by[6], bz[6];
#pragma unroll
    for (int o = 0; o < 6; o++) {
      bx[o] = sx * (vx[o + 1] - vx[o]);
      by[o] = sY * (vy[o + 1] - vy[o]);
      bz[o] = sZ * dz[o];
    }
    if (edge_x) edge_bd(bx, xc, g.x);
    if (edge_y) edge_bd(by, yc, g.y);
    double z5 = bz[4];
    if (STAGE < 2 && (z < 3 || z > g.z - 4)) {
      edge_bd(bz, z, g.z);
      z5 = bz[4];
      if (z == g.z - 1) {
        // on the last plane L's fifth operand is the z difference one row
        // down (id_kp2 = id_jm1, lsTools.cu:636)
        const unsigned row = (unsigned)xc + sy * (unsigned)(yc == 0 ? 0 : yc - 1);
        z5 = sZ * (ld(src, (row + (unsigned)z * sz) * 8u) - ld(src, (row + (unsigned)(z - 1) * sz) * 8u));
      }
    }
    const double rx = godunov_axis(bx, bx[4]), ry = godunov_axis(by, by[4]),
                 rz = godunov_axis(bz, z5);
    const double grad = sqrt_nr(__builtin_fma(rx, rx, __builtin_fma(ry, ry, rz * rz)));
    const double so = p0 * rsqrt_nr(__builtin_fma(p0, p0, d * d));
    const double step = __builtin_fma(-dt * so, grad - 1.0, sv);  // sv - dt*rs
    if (!own) continue;
    if constexpr (STAGE == 0) {
      out[id] = step;
    } else if constexpr (STAGE == 1) {
      out[id] = 0.75 * p0 + 0.25 * step;
    } else {
      // (P + 2 step)/3, the quotient corrected by its residual
      const double t = p0 + 2.0 * step, o3 = t * (1.0 / 3.0);
      const double o = __builtin_fma(__builtin_fma(-3.0, o3, t), 1.0 / 3.0, o3);
      if (phi) {
        phi[vid] = o;
        continue;
      }
      int cx[3], cy[3], cz[3];
      const int kx = mirror_images(x, g.x - 2 * GC, cx), ky = mirror_images(y, g.y - 2 * GC, cy),
                kk = mirror_images(z, g.z - 2 * GC, cz);
      for (int c = 0; c < kk; c++)
        for (int e = 0; e < ky; e++)
          for (int a = 0; a < kx; a++)
            out[(unsigned)cx[a] + sy * (unsigned)cy[e] + sz * (unsigned)cz[c]] = o;
    }
  }
}

template <int STAGE>
void launch_reinit_stage(hipStream_t st, const double* src, const double* P, const double* dmin,
                         const double* jbn, PDims g, double iX, double iY, double iZ, double dt,
                         double* out, double* phi = nullptr) {
  constexpr int LO = STAGE == 0 ? 0 : (STAGE == 1 ? GC - 3 : GC);
  const long long cols = (long long)((g.x - 2 * LO + RI_TX - 1) / RI_TX) *
                         ((g.y - 2 * LO + RI_TY - 1) / RI_TY);
  const int nz = g.z - 2 * LO;
  // 8 planes a slab (16: 4% slower, a longer last round of workgroups), fewer
  // while the chip's 256 compute units would get less than four workgroups
  int kz = 8;
  while (kz > 2 && cols * ((nz + kz - 1) / kz) < 1024) kz /= 2;
  hipLaunchKernelGGL(k_ls_reinit_stage<STAGE>, dim3((unsigned)(cols * ((nz + kz - 1) / kz))),
                     dim3(256), 0, st, src, P, dmin, jbn, g, kz, iX, iY, iZ, dt, out, phi);
}

// ---------------------------------------------------------------------------
// Level-set advection (cuAdvectLsJB, lsTransportEc.cu:243-399).

// First point of the range that stage 0, 1, 2 computes in every direction of
// the padded grid (it ends as far from the other face).  The last stage
// computes the interior; its stencils reach three points further, so the
// second stage skips the two outermost ghost layers (whose values the
// reference computes and never uses for the interior), and that stage's
// points reach the outermost layer of the first one.
constexpr int adv_first(int stage) { return stage == 0 ? 0 : (stage == 1 ? GC - 3 : GC); }

// Workgroup tiles of the advection: 2^ltx x 2^(8-ltx) columns (x, y), 32 x 8
// unless 16 x 16 leaves fewer work-items past the ends of the rows and
// columns.
int adv_ltx(const PDims& g) {
  auto covered = [&](int l) {
    return (long long)(((g.x + (1 << l) - 1) >> l) << l) *
           (((g.y + (256 >> l) - 1) >> (8 - l)) << (8 - l));
  };
  return covered(4) < covered(5) ? 4 : 5;
}

// Slabs of 8 planes (16: 3% slower on 48 boxes of 25.7 M points), fewer while
// the chip's 256 compute units would get less than four workgroups.
int adv_blocks(const PDims& g, int stage, int ltx, int kz) {
  const int lo = adv_first(stage);
  return ((g.x - 2 * lo + (1 << ltx) - 1) >> ltx) *
         ((g.y - 2 * lo + (256 >> ltx) - 1) >> (8 - ltx)) * ((g.z - 2 * lo + kz - 1) / kz);
}

// One fused SSP-RK3 stage for the columns of workgroup b of a grid: backward
// differences, the upwind JB WENO derivative, the right-hand side
// advect_RS_WENO (lsTools.cu:361-417) and the stage update.  phi, vel (3
// components) and jbn (11; 1, 5, 9 used) are interior fields, read at a
// ghost point's mirror image, so the padded copies of the reference are not
// made: stage 0 takes its stencils straight from phi.  Stages 0 and 1 write
// the padded arrays T1 and T2 (out), the next stage's src; stage 2 writes
// phi in place, whose other points it does not read.
//
// cuAdvectLsJB takes an already padded velocity from a caller the reference
// does not have, so its ghost values are this library's choice: the even
// mirror image of the interior for every component (as phi is padded).  Near
// the faces the advected phi follows that choice (an odd reflection of the
// wall-normal component would be as plausible for a wall); the reference
// does not pin it.
//
// The march along z and the derivative are those of k_ls_reinit_stage.  The
// form with one point per work-item formed every operand from 21 loads and
// found its place by divisions; with the padded copy of phi it took 162 +
// 3 x 694 us on 48 boxes of 25.7 M points (36.4 M padded).  Now
// 497 + 511 + 454 us (3.9 TB/s); 643 + 637 + 498 us with the x and y stencils
// read from memory instead of StencilTile, and 727 + 728 + 566 us with
// nontemporal loads of vel and jbn, whose lines neighbouring tiles share.
template <int STAGE>
__device__ __forceinline__ void ls_advect_tile(const double* src, const double* phi,
                                               const double* vel, const double* jbn, PDims g,
                                               int b, int ltx, int kz, double iX, double iY,
                                               double iZ, double dt, double* out) {
#pragma clang fp contract(fast)
  constexpr int LO = adv_first(STAGE);
  const int nbx = (g.x - 2 * LO + (1 << ltx) - 1) >> ltx,
            nby = (g.y - 2 * LO + (256 >> ltx) - 1) >> (8 - ltx);
  const int x0 = LO + ((b % nbx) << ltx), y0 = LO + ((b / nbx % nby) << (8 - ltx));
  const int x = x0 + ((int)threadIdx.x & ((1 << ltx) - 1)), y = y0 + ((int)threadIdx.x >> ltx);
  const int z0 = LO + b / (nbx * nby) * kz, z1 = min(z0 + kz, g.z - LO);
  const bool own = x < g.x - LO && y < g.y - LO;
  // positions past the padded grid's faces are clamped: work-items there
  // store nothing, and a difference over one is never used
  const int xc = min(x, g.x - 1), yc = min(y, g.y - 1);
  const int nx = g.x - 2 * GC, ny = g.y - 2 * GC, nz = g.z - 2 * GC;
  const unsigned vsz = (unsigned)nx * (unsigned)ny;
  const size_t vN = (size_t)vsz * (unsigned)nz;
  const unsigned vcol = (unsigned)mirror(xc, nx) + (unsigned)nx * (unsigned)mirror(yc, ny);
  // src: the padded grid, or phi through the mirror images
  const unsigned sy = STAGE == 0 ? (unsigned)nx : (unsigned)g.x;
  const unsigned sz = STAGE == 0 ? vsz : (unsigned)g.x * (unsigned)g.y;
  auto place = [&](int t, int gn, int n) {
    t = min(max(t, 0), gn - 1);
    return (unsigned)(STAGE == 0 ? mirror(t, n) : t);
  };
  const unsigned col = place(xc, g.x, nx) + sy * place(yc, g.y, ny);
  __shared__ double cells[2][StencilTile::CELLS];
  const StencilTile tile(ltx);
  const unsigned hcol = place(x0 + tile.hx, g.x, nx) + sy * place(y0 + tile.hy, g.y, ny);
  const bool edge_x = STAGE < 2 && __any(xc < 3 || xc > g.x - 4);
  const bool edge_y = STAGE < 2 && __any(yc < 3 || yc > g.y - 4);
  // a field's value at byte offset off (the padded grid has fewer than 2^29
  // points): uniform base, 32-bit offset
  auto at = [](const double* f, unsigned off) -> decltype(auto) {
    return gref(reinterpret_cast<const double*>(reinterpret_cast<const char*>(f) + off));
  };
  auto ld = [&](const double* f, unsigned off) -> double { return at(f, off); };
  auto plane_of = [&](unsigned c, int z) { return ld(src, (c + place(z, g.z, nz) * sz) * 8u); };
  auto plane = [&](int z) { return plane_of(col, z); };
  double vz[4], dz[6];  // values of planes z .. z+3; the stencil's differences along z
#pragma unroll
  for (int o = 0; o < 3; o++) vz[o + 1] = plane(z0 + o);
  {
    const double a = plane(z0 - 3), b2 = plane(z0 - 2), c = plane(z0 - 1);
    dz[1] = b2 - a;
    dz[2] = c - b2;
    dz[3] = vz[1] - c;
    dz[4] = vz[2] - vz[1];
    dz[5] = vz[3] - vz[2];
  }
  double hv = plane_of(hcol, z0);
  for (int z = z0; z < z1; z++) {
#pragma unroll
    for (int o = 0; o < 3; o++) vz[o] = vz[o + 1];
#pragma unroll
    for (int o = 0; o < 5; o++) dz[o] = dz[o + 1];
    vz[3] = plane(z + 3);
    dz[5] = vz[3] - vz[2];
    const unsigned voff = (vcol + (unsigned)mirror(z, nz) * vsz) * 8u;
    const double sv = vz[0];
    double vx[7], vy[7];
    double* c = cells[(z - z0) & 1];
    tile.put(c, sv, hv);
    lds_barrier();
    if (z + 1 < z1) hv = plane_of(hcol, z + 1);
    tile.get(c, sv, vx, vy);
    const double p0 = STAGE == 0 ? sv : ld(phi, voff);
    // upwinding: the left-biased derivative where the velocity is positive
    // and the right-biased one where it is negative, so only that one is
    // formed: 0.5(s+1) v L + 0.5|s-1| v R  =  v L (v > 0),  v R (v < 0),  0
    auto axis = [&](double v, const double bd[6], double l5) {
      const bool left = v > 0.0;
      const double b1 = left ? bd[0] : bd[5], b2 = left ? bd[1] : bd[4],
                   b3 = left ? bd[2] : bd[3], b4 = left ? bd[3] : bd[2], b5 = left ? l5 : bd[1];
      return v == 0.0 ? 0.0 : v * weno5(b1, b2, b3, b4, b5);
    };
    double bd[6];
    const double mx = iX * ld(jbn, voff), mY = iY * ld(jbn + 4 * vN, voff),
                 mZ = iZ * ld(jbn + 8 * vN, voff);
    const double ux = ld(vel, voff), uy = ld(vel + vN, voff), uz = ld(vel + 2 * vN, voff);
#pragma unroll
    for (int o = 0; o < 6; o++) bd[o] = mx * (vx[o + 1] - vx[o]);
    if (edge_x) edge_bd(bd, xc, g.x);
    double rs = axis(ux, bd, bd[4]);
#pragma unroll
    for (int o = 0; o < 6; o++) bd[o] = mY * (vy[o + 1] - vy[o]);
    if (edge_y) edge_bd(bd, yc, g.y);
    rs += axis(uy, bd, bd[4]);
#pragma unroll
    for (int o = 0; o < 6; o++) bd[o] = mZ * dz[o];
    double z5 = bd[4];
    if (STAGE < 2 && (z < 3 || z > g.z - 4)) {
      edge_bd(bd, z, g.z);
      z5 = bd[4];
      if (z == g.z - 1) {
        // on the last plane L's fifth operand is the z difference one row
        // down (id_kp2 = id_jm1, lsTools.cu:636)
        const unsigned row = place(xc, g.x, nx) + sy * place(yc == 0 ? 0 : yc - 1, g.y, ny);
        z5 = mZ * (plane_of(row, z) - plane_of(row, z - 1));
      }
    }
    rs += axis(uz, bd, z5);
    if (!own) continue;
    double o;
    if (STAGE == 0) o = sv - dt * rs;
    else if (STAGE == 1) o = 0.75 * p0 + 0.25 * (sv - dt * rs);
    else o = (p0 + 2.0 * (sv - dt * rs)) * (1.0 / 3.0);
    gref(out + (STAGE == 2 ? vcol + (unsigned)(z - GC) * vsz
                           : (unsigned)xc + (unsigned)g.x *
                                 ((unsigned)yc + (unsigned)g.y * (unsigned)z))) = o;
  }
}

template <int STAGE>
__global__ void __launch_bounds__(256)
k_ls_advect(const double* src, const double* phi, const double* vel, const double* jbn, PDims g,
            int ltx, int kz, double iX, double iY, double iZ, double dt, double* out) {
  ls_advect_tile<STAGE>(src, phi, vel, jbn, g, (int)xcd_block(blockIdx.x, gridDim.x), ltx, kz, iX,
                        iY, iZ, dt, out);
}

// The same for many grids in one launch (the batched stage): workgroup b
// serves grid gi with blk_start[gi] <= b < blk_start[gi+1].
template <int STAGE>
__global__ void __launch_bounds__(256)
k_batch_advect(const LsBatchGrid* grids, const int* blk_start, int ngrid) {
  const int b = (int)xcd_block(blockIdx.x, gridDim.x);
  int gi = 0, hi = ngrid;
  while (hi - gi > 1) {
    const int mid = (gi + hi) >> 1;
    if (blk_start[mid] <= b) gi = mid;
    else hi = mid;
  }
  const LsBatchGrid& G = grids[gi];
  const PDims g{G.nx + 2 * GC, G.ny + 2 * GC, G.nz + 2 * GC};
  ls_advect_tile<STAGE>(STAGE == 0 ? G.phi : (STAGE == 1 ? G.T1 : G.T2), G.phi, G.vel, G.jbn, g,
                        b - blk_start[gi], G.ltx, G.kz, G.iX, G.iY, G.iZ, G.dt,
                        STAGE == 0 ? G.T1 : (STAGE == 1 ? G.T2 : G.phi));
}

unsigned blocks_for(long long n) {
  long long b = (n + 255) / 256;
  if (b > 131072) b = 131072;
  return (unsigned)(b < 1 ? 1 : b);
}

PDims padded(const Dims& d) { return PDims{d.nx + 2 * GC, d.ny + 2 * GC, d.nz + 2 * GC}; }

}  // namespace

// ten padded fields, then the solid-point list of the extrapolation: chunk
// counts, the count and up to one index per padded point (ints)
size_t ls_scratch_doubles(const Dims& d) {
  const size_t NG = (size_t)padded(d).N();
  const size_t ints = (NG + LS_CHUNK - 1) / LS_CHUNK + 1 + NG;
  return 10 * NG + (ints + 1) / 2 + 1;
}

long long ls_padded_points(int nx, int ny, int nz) {
  return (long long)(nx + 2 * GC) * (ny + 2 * GC) * (nz + 2 * GC);
}

void plan_batch_ls(std::vector<LsBatchGrid>& grids, std::vector<int> blk_start[3]) {
  auto padded_of = [](const LsBatchGrid& G) { return padded(Dims{G.nx, G.ny, G.nz}); };
  int kz = 16;
  long long n;
  do {
    kz /= 2;
    n = 0;
    for (const LsBatchGrid& G : grids) {
      const PDims g = padded_of(G);
      n += adv_blocks(g, 2, adv_ltx(g), kz);
    }
  } while (kz > 2 && n < 1024);
  for (int s = 0; s < 3; s++) {
    blk_start[s].assign(1, 0);
    for (LsBatchGrid& G : grids) {
      const PDims g = padded_of(G);
      G.ltx = adv_ltx(g);
      G.kz = kz;
      blk_start[s].push_back(blk_start[s].back() + adv_blocks(g, s, G.ltx, kz));
    }
  }
}

int op_batch_ls_step(hipStream_t st, const LsBatchGrid* grids, int* const blk_start[3],
                     const int nblk[3], int ngrid) {
  hipLaunchKernelGGL(k_batch_advect<0>, dim3(nblk[0]), dim3(256), 0, st, grids, blk_start[0], ngrid);
  hipLaunchKernelGGL(k_batch_advect<1>, dim3(nblk[1]), dim3(256), 0, st, grids, blk_start[1], ngrid);
  hipLaunchKernelGGL(k_batch_advect<2>, dim3(nblk[2]), dim3(256), 0, st, grids, blk_start[2], ngrid);
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int op_ls_extrapolate(emx_ctx* ctx, double* pres, const double* jbn,
                      const double* sobject, double dx, double dy, double dz,
                      double deltamin) {
  const Dims d = ctx->d;
  const PDims g = padded(d);
  const long long N = d.N(), NG = g.N();
  double* P = ctx->ls_buf;
  double* S = P + NG;
  double* geo = S + NG;  // 6 per solid point, at most 6*NG
  double* D1 = geo + 6 * NG;
  double* D2 = D1 + NG;
  hipStream_t st = ctx->stream;
  const unsigned bg = blocks_for(NG);
  EMX_TIMED(ctx, "ls_pad", 16.0 * NG,
          hipLaunchKernelGGL(k_pad, dim3(bg), dim3(256), 0, st, pres, d.nx, d.ny, d.nz, P, g));
  EMX_TIMED(ctx, "ls_pad", 16.0 * NG,
          hipLaunchKernelGGL(k_pad, dim3(bg), dim3(256), 0, st, sobject, d.nx, d.ny, d.nz, S, g));
  // cuExtrapolation(d_press, d_sobject, d_jbn, deltaX.., NxG.., deltamin*0.5, 1)
  // hands 1.0/deltaX to every kernel (interface.cu:373-421)
  const double iX = 1.0 / dx, iY = 1.0 / dy, iZ = 1.0 / dz, dt = deltamin * 0.5;
  // the solid points, in order; D1 = D2 = P at every point (the fluid
  // points are never written again)
  const int nb = (int)((NG + LS_CHUNK - 1) / LS_CHUNK);
  int* bcount = reinterpret_cast<int*>(D2 + NG);
  int* count = bcount + nb;
  int* list = count + 1;
  EMX_TIMED(ctx, "ls_solid_list", 8.0 * NG,
            hipLaunchKernelGGL(k_ls_solid_count, dim3(nb), dim3(256), 0, st, S, NG, bcount));
  EMX_TIMED(ctx, "ls_solid_list", 0.0,
            hipLaunchKernelGGL(k_ls_scan, dim3(1), dim3(1024), 0, st, bcount, nb, count));
  EMX_TIMED(ctx, "ls_solid_list", 8.0 * NG,
            hipLaunchKernelGGL(k_ls_solid_write, dim3(nb), dim3(256), 0, st, S, NG, bcount, list));
  // algorithmic bytes per solid point (the count is only known on the
  // device; read back while the context records timings): geometry = list
  // entry, S, three metrics in, six values out; a stage = list entry, ext,
  // the six values, P (stages 1, 2), out
  double nsolid = 0.0;
  if (ctx->timing && (ctx->timing_label.empty() || ctx->timing_label == "ls_extrap_stage" ||
                      ctx->timing_label == "ls_solid_geom")) {
    int h = 0;
    EMX_TRY_HIP(hipMemcpyAsync(&h, count, sizeof(int), hipMemcpyDeviceToHost, st));
    EMX_TRY_HIP(hipStreamSynchronize(st));
    nsolid = h;
  }
  const unsigned bl = bg < 4096u ? bg : 4096u;
  EMX_TIMED(ctx, "ls_solid_geom", (4.0 + 8.0 * 10) * nsolid,
            hipLaunchKernelGGL(k_ls_solid_geom, dim3(bl), dim3(256), 0, st, list, count, S, jbn,
                               d.nx, d.ny, d.nz, g, iX, iY, iZ, geo));
  EMX_TIMED(ctx, "ls_copy", 24.0 * NG,
            hipLaunchKernelGGL(k_copy2, dim3(bg), dim3(256), 0, st, P, D1, D2, NG));
  EMX_TRY_HIP(hipGetLastError());
  for (int it = 1; it <= 10; it++) {
    EMX_TIMED(ctx, "ls_extrap_stage", (4.0 + 8.0 * 8) * nsolid,
              hipLaunchKernelGGL(k_ls_extrap_list, dim3(bl), dim3(256), 0, st, 0, list, count, P,
                                 P, geo, g, iX, iY, iZ, dt, D1));
    EMX_TIMED(ctx, "ls_extrap_stage", (4.0 + 8.0 * 9) * nsolid,
              hipLaunchKernelGGL(k_ls_extrap_list, dim3(bl), dim3(256), 0, st, 1, list, count, D1,
                                 P, geo, g, iX, iY, iZ, dt, D2));
    EMX_TIMED(ctx, "ls_extrap_stage", (4.0 + 8.0 * 9) * nsolid,
              hipLaunchKernelGGL(k_ls_extrap_list, dim3(bl), dim3(256), 0, st, 2, list, count, D2,
                                 P, geo, g, iX, iY, iZ, dt, P));
  }
  EMX_TIMED(ctx, "ls_unpad", 16.0 * N,
          hipLaunchKernelGGL(k_unpad, dim3(blocks_for(N)), dim3(256), 0, st, P, g,
                     d.nx, d.ny, d.nz, pres));
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int op_ls_reinit(emx_ctx* ctx, double* phi, const double* jbn, const double* dmin,
                 double dx, double dy, double dz, double deltamin) {
  const Dims d = ctx->d;
  const PDims g = padded(d);
  const long long N = d.N(), NG = g.N();
  double* P = ctx->ls_buf;  // the iteration's phi, ping-pong with Q
  double* Q = P + NG;
  double* T1 = Q + NG;
  double* T2 = T1 + NG;
  hipStream_t st = ctx->stream;
  EMX_TIMED(ctx, "ls_pad", 8.0 * (N + NG),
            hipLaunchKernelGGL(k_pad, dim3(blocks_for(NG)), dim3(256), 0, st, phi, d.nx, d.ny,
                               d.nz, P, g));
  const double iX = 1.0 / dx, iY = 1.0 / dy, iZ = 1.0 / dz, dt = 0.5 * deltamin;
  // the padding already mirrors the ghost layers of the first iteration
  for (int it = 1; it <= 10; it++) {
    // per point: src, phi (= phi0), out; three metrics and dmin, interior
    // fields.  The last iteration writes phi itself.
    EMX_TIMED(ctx, "ls_reinit_stage", 16.0 * NG + 32.0 * N,
              launch_reinit_stage<0>(st, P, P, dmin, jbn, g, iX, iY, iZ, dt, T1));
    EMX_TIMED(ctx, "ls_reinit_stage", 24.0 * NG + 32.0 * N,
              launch_reinit_stage<1>(st, T1, P, dmin, jbn, g, iX, iY, iZ, dt, T2));
    EMX_TIMED(ctx, "ls_reinit_stage", 24.0 * NG + 32.0 * N,
              launch_reinit_stage<2>(st, T2, P, dmin, jbn, g, iX, iY, iZ, dt, Q,
                                     it == 10 ? phi : nullptr));
    std::swap(P, Q);
  }
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int op_ls_advect_weno5(emx_ctx* ctx, double* phi, const double* vel,
                       const double* jbn, double dx, double dy, double dz,
                       double dt) {
  const Dims d = ctx->d;
  const PDims g = padded(d);
  const long long N = d.N(), NG = g.N();
  double* T1 = ctx->ls_buf;
  double* T2 = T1 + NG;
  const double iX = 1.0 / dx, iY = 1.0 / dy, iZ = 1.0 / dz;
  const int ltx = adv_ltx(g);
  int kz = 8;
  while (kz > 2 && adv_blocks(g, 2, ltx, kz) < 1024) kz /= 2;
  auto go = [&](auto kern, int stage, const double* src, double* out) {
    hipLaunchKernelGGL(kern, dim3(adv_blocks(g, stage, ltx, kz)), dim3(256), 0, ctx->stream, src,
                       phi, vel, jbn, g, ltx, kz, iX, iY, iZ, dt, out);
  };
  // per stage: the stage's phi in and out, the step's phi, the velocity and
  // the metrics
  EMX_TIMED(ctx, "ls_weno_stage", 8.0 * NG + 56.0 * N, go(k_ls_advect<0>, 0, phi, T1));
  EMX_TIMED(ctx, "ls_weno_stage", 16.0 * NG + 56.0 * N, go(k_ls_advect<1>, 1, T1, T2));
  EMX_TIMED(ctx, "ls_weno_stage", 8.0 * NG + 64.0 * N, go(k_ls_advect<2>, 2, T2, phi));
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

namespace {

// heviside (solver/advectLS.f90:29-59): the smoothed Heaviside of phi over
// the band |phi| <= eps, in the reference's order of operations.  A point
// that none of the three cases takes (NaN phi) keeps its hevi, as there.
__global__ void k_heviside(const double* phi, long long N, double eps, double* hevi) {
  const double pi = 3.14159265358979323846;  // 2 acos(0) in double
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (long long)gridDim.x * blockDim.x) {
    const double f = phi[p];
    if (f < -eps) hevi[p] = 0.0;
    if (f >= -eps && f <= eps) hevi[p] = 0.5 + f / (2.0 * eps) + sin(pi * f / eps) / (2.0 * pi);
    if (f > eps) hevi[p] = 1.0;
  }
}

}  // namespace

int op_ls_heviside(emx_ctx* ctx, const double* phi, double deltamax, double* hevi) {
  const long long N = ctx->d.N();
  EMX_TIMED(ctx, "ls_heviside", 16.0 * N,
            hipLaunchKernelGGL(k_heviside, dim3(blocks_for(N)), dim3(256), 0, ctx->stream, phi, N,
                               1.5 * deltamax, hevi));
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

}  // namespace emx
