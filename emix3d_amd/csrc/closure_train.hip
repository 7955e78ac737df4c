// Training passes of the learned closure: the network's FP32 forward, the
// gradient of its parameters and the Adam step (layout of the parameters and
// the normalisation: closure.hip).  The reference has no counterpart.
#include <algorithm>

#include "mlp_infer.hpp"

namespace emx {

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float dsilu_f(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}
__device__ __forceinline__ float softplus_f(float z) {
  return z > 20.0f ? z : log1pf(__expf(z));
}

// The training passes run on the FP32 matrix cores,
// v_mfma_f32_16x16x4_f32 (FP32 operands and accumulation), in two layouts
// of a tile of 16 points x 64 neurons; lane l, g = l/16:
//   "point" layout:  a[t][i] is neuron 16t + 4g + i of point l%16;
//   "neuron" layout: a[t][i] is neuron 16t + l%16 of point 4g + i.
// The matrix core takes the operand of row (or column) l%16 at K = l/16 and
// returns rows 4g + i of column l%16.  With K step (t, i) standing for
// neurons 16t + 4g + i, a result in the point layout is the next product's
// operand as it is, and with K step i standing for points 4g + i a result in
// the neuron layout is an operand of a sum over points: no data moves
// between lanes.
//
// These passes replace one-point-per-lane loops whose 64 activations per
// layer, indexed at run time, lived in scratch memory: at 65536 rows 342 us
// forward and 819 us backward, against 32 and 65 us now (the rows'
// pre-activations are 50 MB, 11 us at the copy rate; the products 24 us at
// the FP32 matrix rate of 153 TFLOP/s).  The backward pass is bound by the
// latency of one wavefront per SIMD (75 us before the next tile's reads were
// in flight during a tile).
constexpr int MLP_ACT = 3 * MLP_H + 1;
constexpr int MLP_LDW = MLP_H + 4;  // row stride in LDS: 4 banks between rows
typedef float f32x4u __attribute__((__vector_size__(16), __aligned__(4)));

// Keeps the weight operands of a loop's next part in LDS: without it the
// compiler holds all of them in registers across the loop, and spills.
__device__ __forceinline__ void reread_lds() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Stages the 64 x 64 weight matrix src into LDS with row stride MLP_LDW.
__device__ __forceinline__ void stage_square(float* lw, const float* src) {
  for (int t = threadIdx.x; t < MLP_H * MLP_H; t += blockDim.x)
    lw[(t / MLP_H) * MLP_LDW + t % MLP_H] = src[t];
}

// act[q] = z1[64] z2[64] z3[64] z4 (pre-activations), nu[q].  A wavefront
// takes tiles of 32 points (two 16-point column tiles, so each weight
// operand read from LDS serves two products), the layers chained in the
// point layout.
constexpr int MF_T = 2;
constexpr int MLP_FWD_LDS = 2 * MLP_H * MLP_LDW + 12 * MLP_H + 4 * MLP_H;  // floats

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_mlp_forward(const float* P, const float* norm, const float* feat, int n, float* act,
              float* nu) {
  __shared__ __attribute__((aligned(16))) float lds[MLP_FWD_LDS];
  float* w2 = lds;
  float* w3 = w2 + MLP_H * MLP_LDW;
  float* w1 = w3 + MLP_H * MLP_LDW;  // [12][64]: input k of neuron o, zero rows 10, 11
  float* vb = w1 + 12 * MLP_H;       // b1 b2 b3 W4
  stage_square(w2, P + MW2);
  stage_square(w3, P + MW3);
  for (int t = threadIdx.x; t < 12 * MLP_H; t += blockDim.x) {
    const int k = t / MLP_H, o = t % MLP_H;
    w1[t] = k < MLP_IN ? P[MW1 + o * MLP_IN + k] : 0.0f;
  }
  for (int t = threadIdx.x; t < MLP_H; t += blockDim.x) {
    vb[t] = P[MB1 + t];
    vb[MLP_H + t] = P[MB2 + t];
    vb[2 * MLP_H + t] = P[MB3 + t];
    vb[3 * MLP_H + t] = P[MW4 + t];
  }
  __syncthreads();
  const int l = threadIdx.x & 63, m = l & 15, g = l >> 4;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int nwave = gridDim.x * (blockDim.x >> 6);
  const float b4 = P[MB4], oscale = norm[2 * MLP_IN];
  float shift[3], scale[3];
#pragma unroll
  for (int s = 0; s < 3; s++) {
    const int k = 4 * s + g;
    shift[s] = k < MLP_IN ? norm[k] : 0.0f;
    scale[s] = k < MLP_IN ? norm[MLP_IN + k] : 0.0f;
  }
  const int ntile = (n + 16 * MF_T - 1) / (16 * MF_T);
  for (int tile = wave; tile < ntile; tile += nwave) {
    reread_lds();
    int q[MF_T];  // this lane's points (point layout); clamped rows are not stored
    float h[MF_T][4][4];
    f32x4 c[MF_T][4];
    float x[MF_T][3];
#pragma unroll
    for (int t = 0; t < MF_T; t++) {
      q[t] = tile * 16 * MF_T + 16 * t + m;
      const long long row = (long long)(q[t] < n ? q[t] : n - 1) * MLP_IN;
#pragma unroll
      for (int s = 0; s < 3; s++) {
        const int k = 4 * s + g;
        float f = 0.0f;  // of the zero rows: no feature, which may not be finite
        if (k < MLP_IN) f = feat[row + k];
        x[t][s] = (f - shift[s]) * scale[s];
      }
    }
    // keeps the pre-activations of a layer and forms the next layer's input
    auto finish = [&](int layer) {
#pragma unroll
      for (int t = 0; t < MF_T; t++)
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
          const f32x4 z = c[t][mt];
          if (q[t] < n)
            *reinterpret_cast<f32x4u*>(act + (long long)q[t] * MLP_ACT + layer * MLP_H +
                                       16 * mt + 4 * g) = z;
#pragma unroll
          for (int i = 0; i < 4; i++) h[t][mt][i] = silu_f(z[i]);
        }
    };
    auto bias = [&](int layer) {
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(vb + layer * MLP_H + 16 * mt + 4 * g);
#pragma unroll
        for (int t = 0; t < MF_T; t++) c[t][mt] = b;
      }
    };
    bias(0);
#pragma unroll
    for (int s = 0; s < 3; s++)
#pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        const float a = w1[(4 * s + g) * MLP_H + 16 * mt + m];
#pragma unroll
        for (int t = 0; t < MF_T; t++) c[t][mt] = mfma_f32(a, x[t][s], c[t][mt]);
      }
    finish(0);
#pragma unroll
    for (int layer = 1; layer < 3; layer++) {
      const float* w = layer == 1 ? w2 : w3;
      reread_lds();
      bias(layer);
#pragma unroll
      for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
          const f32x4 a =
              *reinterpret_cast<const f32x4*>(w + (16 * mt + m) * MLP_LDW + 16 * kt + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int t = 0; t < MF_T; t++) c[t][mt] = mfma_f32(a[i], h[t][kt][i], c[t][mt]);
        }
      finish(layer);
    }
    // output neuron: the lane's 16 terms, then the four lane groups
#pragma unroll
    for (int t = 0; t < MF_T; t++) {
      float s = 0.0f;
#pragma unroll
      for (int kt = 0; kt < 4; kt++) {
        const f32x4 w4 = *reinterpret_cast<const f32x4*>(vb + 3 * MLP_H + 16 * kt + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) s += w4[i] * h[t][kt][i];
      }
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      s += b4;
      if (g == 0 && q[t] < n) {
        act[(long long)q[t] * MLP_ACT + 3 * MLP_H] = s;
        nu[q[t]] = oscale * softplus_f(s);
      }
    }
  }
}

// Back-propagation and the weight gradients in one pass over the rows: the
// point derivatives d3, d2, d1 of a 16-point tile stay in registers.  d2 is
// formed in both layouts (the same weight operand, operands exchanged): the
// point layout is the operand of d1, the neuron layout of the sums over
// points, dW_l += d_l h_{l-1}^T, whose 16 x 16 tiles stay in the matrix
// cores' accumulators over all the wavefront's points.  The accumulators
// (144 registers) and a tile's activations leave one wavefront per SIMD;
// the sums of a workgroup's four are added in LDS in a fixed order and leave
// one partial of MNP values per workgroup.
constexpr int MG_WAVES = 4;
constexpr int MLP_GRAD_PAD = 9092;  // MNP rounded up to a multiple of four
static_assert(MLP_GRAD_PAD >= MNP, "partial sums");

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + __expf(-z)); }

__global__ void __launch_bounds__(64 * MG_WAVES)
k_mlp_grad(const float* P, const float* norm, const float* feat, const float* act,
           const float* dnu, int n, float* part) {
  extern __shared__ __attribute__((aligned(16))) float glds[];
  float* w2 = glds;
  float* w3 = w2 + MLP_H * MLP_LDW;
  stage_square(w2, P + MW2);
  stage_square(w3, P + MW3);
  __syncthreads();
  const int l = threadIdx.x & 63, m = l & 15, g = l >> 4, wv = threadIdx.x >> 6;
  const int nwave = gridDim.x * MG_WAVES;
  const int ntile = (n + 15) / 16;
  const float oscale = norm[2 * MLP_IN];
  const int xk = m < MLP_IN ? m : 0;
  const float xshift = norm[xk], xscale = m < MLP_IN ? norm[MLP_IN + xk] : 0.0f;
  // dW tiles [o][k]; layer 1: one tile of 10 inputs and a column of ones
  // (its bias)
  f32x4 g3[4][4], g2[4][4], g1[4];
  float s3[4], s2[4], s4[4], sb4 = 0.0f;  // bias sums of neuron 16t+m; dW4
  float w4p[4][4], w4n[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    s3[t] = s2[t] = s4[t] = 0.0f;
    g1[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    w4n[t] = P[MW4 + 16 * t + m];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      w4p[t][i] = P[MW4 + 16 * t + 4 * g + i];
      g3[t][i] = g2[t][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  // What a lane reads of a tile; rows past the end are clamped to the last
  // one, and their zero output derivatives clear everything they reach.
  struct Tile {
    f32x4 z3p[4], z2p[4];                  // pre-activations, point layout
    float z3n[4][4], z2n[4][4], z1n[4][4]; // neuron layout
    float z4p, dp, z4n[4], dn[4], f[4];    // output neuron, dnu, input xk
  };
  auto load = [&](int tile) {
    Tile T;
    auto row = [&](int p) { return p < n ? p : n - 1; };
    const int rp = row(16 * tile + m);
    const float* ap = act + (long long)rp * MLP_ACT;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      T.z3p[t] = *reinterpret_cast<const f32x4u*>(ap + 2 * MLP_H + 16 * t + 4 * g);
      T.z2p[t] = *reinterpret_cast<const f32x4u*>(ap + MLP_H + 16 * t + 4 * g);
    }
    T.z4p = ap[3 * MLP_H];
    T.dp = dnu[rp];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = row(16 * tile + 4 * g + i);
      const float* an = act + (long long)r * MLP_ACT + m;
#pragma unroll
      for (int t = 0; t < 4; t++) {
        T.z3n[t][i] = an[2 * MLP_H + 16 * t];
        T.z2n[t][i] = an[MLP_H + 16 * t];
        T.z1n[t][i] = an[16 * t];
      }
      T.z4n[i] = an[3 * MLP_H - m];
      T.dn[i] = dnu[r];
      T.f[i] = feat[(long long)r * MLP_IN + xk];
    }
    return T;
  };
  // tiles dealt round robin over all wavefronts, the next one's reads in
  // flight while a tile is worked on
  int tile = wv * gridDim.x + blockIdx.x;
  Tile next;
  if (tile < ntile) next = load(tile);
  for (; tile < ntile; tile += nwave) {
    const Tile T = next;
    if (tile + nwave < ntile) next = load(tile + nwave);
    reread_lds();
    const int p0 = 16 * tile;
    float z3p[4][4], z3n[4][4], z2p[4][4], z2n[4][4], z1n[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        z3p[t][i] = T.z3p[t][i];
        z2p[t][i] = T.z2p[t][i];
        z3n[t][i] = T.z3n[t][i];
        z2n[t][i] = T.z2n[t][i];
        z1n[t][i] = T.z1n[t][i];
      }
    float d4n[4], xn[4];
    // point layout: point m; neuron layout: points 4g + i
    const float d4p = p0 + m < n ? T.dp * oscale * sigmoid_f(T.z4p) : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      d4n[i] = p0 + 4 * g + i < n ? T.dn[i] * oscale * sigmoid_f(T.z4n[i]) : 0.0f;
      xn[i] = m == MLP_IN ? 1.0f : (T.f[i] - xshift) * xscale;
    }
    // layer 3: d3 in both layouts, the output neuron's sums
    float d3p[4][4], d3n[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        d3p[t][i] = d4p * w4p[t][i] * dsilu_f(z3p[t][i]);
        const float z = z3n[t][i], s = sigmoid_f(z);
        const float d = d4n[i] * w4n[t] * (s * (1.0f + z * (1.0f - s)));
        d3n[t][i] = d;
        s3[t] += d;
        s4[t] += d4n[i] * (z * s);
      }
#pragma unroll
    for (int i = 0; i < 4; i++) sb4 += d4n[i];
    // h2, and dsilu(z2) kept in its place
    float hn[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float z = z2n[t][i], s = sigmoid_f(z);
        hn[t][i] = z * s;
        z2n[t][i] = s * (1.0f + z * (1.0f - s));
      }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int o = 0; o < 4; o++)
#pragma unroll
        for (int k = 0; k < 4; k++) g3[o][k] = mfma_f32(d3n[o][i], hn[k][i], g3[o][k]);
    // d2 in both layouts
    reread_lds();
    float d2p[4][4], d2n[4][4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      f32x4 cp{0.0f, 0.0f, 0.0f, 0.0f}, cn{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float w = w3[(16 * t + 4 * g + i) * MLP_LDW + 16 * k + m];
          cp = mfma_f32(w, d3p[t][i], cp);
          cn = mfma_f32(d3p[t][i], w, cn);
        }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        d2p[k][i] = cp[i] * dsilu_f(z2p[k][i]);
        d2n[k][i] = cn[i] * z2n[k][i];
        s2[k] += d2n[k][i];
      }
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float z = z1n[t][i], s = sigmoid_f(z);
        hn[t][i] = z * s;
        z1n[t][i] = s * (1.0f + z * (1.0f - s));
      }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int o = 0; o < 4; o++)
#pragma unroll
        for (int k = 0; k < 4; k++) g2[o][k] = mfma_f32(d2n[o][i], hn[k][i], g2[o][k]);
    // d1 in the neuron layout
    reread_lds();
#pragma unroll
    for (int k = 0; k < 4; k++) {
      f32x4 cn{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          cn = mfma_f32(d2p[t][i], w2[(16 * t + 4 * g + i) * MLP_LDW + 16 * k + m], cn);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        g1[k] = mfma_f32(cn[i] * z1n[k][i], xn[i], g1[k]);
      }
    }
  }
  // the workgroup's sum: one slice of LDS per wavefront (over the weights,
  // no longer needed), then the four slices are added
  auto groups = [](float v) {  // over the four lane groups (points 4g + i)
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
  };
#pragma unroll
  for (int t = 0; t < 4; t++) {
    s3[t] = groups(s3[t]);
    s2[t] = groups(s2[t]);
    s4[t] = groups(s4[t]);
  }
  sb4 = groups(sb4);
  __syncthreads();
  float* red = glds + wv * MLP_GRAD_PAD;
#pragma unroll
  for (int o = 0; o < 4; o++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = 16 * o + 4 * g + i;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        red[MW3 + row * MLP_H + 16 * k + m] = g3[o][k][i];
        red[MW2 + row * MLP_H + 16 * k + m] = g2[o][k][i];
      }
      if (m < MLP_IN) red[MW1 + row * MLP_IN + m] = g1[o][i];
      if (m == MLP_IN) red[MB1 + row] = g1[o][i];
    }
  if (g == 0) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      red[MB2 + 16 * t + m] = s2[t];
      red[MB3 + 16 * t + m] = s3[t];
      red[MW4 + 16 * t + m] = s4[t];
    }
    if (m == 0) red[MB4] = sb4;
  }
  __syncthreads();
  float* out = part + (long long)blockIdx.x * MNP;
  for (int w = threadIdx.x; w < MNP; w += blockDim.x)
    out[w] = (glds[w] + glds[MLP_GRAD_PAD + w]) +
             (glds[2 * MLP_GRAD_PAD + w] + glds[3 * MLP_GRAD_PAD + w]);
}

// Workgroups of k_mlp_grad for n rows: one to a compute unit, each wavefront
// at least one 16-row tile.  Their partial sums are the work area.
static int mlp_grad_blocks(int n) {
  const int tiles = (int)(((long long)n + 15) / 16);
  return std::min(256, (tiles + MG_WAVES - 1) / MG_WAVES);
}

// grad[w] = the sum of the nblk partials: 64 values per workgroup, the
// partials over its sixteen wavefronts (the 64 values are adjacent in memory,
// so each read takes whole cache lines).
__global__ void __launch_bounds__(1024)
k_mlp_reduce(const float* part, int nblk, float* grad) {
  __shared__ float red[16][64];
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int w = blockIdx.x * 64 + l;
  float s = 0.0f;
  if (w < MNP) {
#pragma unroll 4
    for (int b = wv; b < nblk; b += 16) s += part[(long long)b * MNP + w];
  }
  red[wv][l] = s;
  __syncthreads();
  if (wv == 0 && w < MNP) {
    s = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; k++) s += red[k][l];
    grad[w] = s;
  }
}

// Adam (Kingma & Ba 2015) with bias correction.
__global__ void k_adam(float* p, const float* g, float* m, float* v, int n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

}  // namespace emx

extern "C" {

int emx_mlp_forward_f32(const float* params, const float* norm, const float* feat, int n,
                        float* act, float* nu, void* stream) {
  if (!params || !norm || !feat || !act || !nu || n <= 0) {
    emx::set_error("emx_mlp_forward_f32: bad arguments");
    return EMX_ERR_ARG;
  }
  // one wavefront per 32 rows, up to two workgroups per compute unit
  const int tiles = (n + 16 * emx::MF_T - 1) / (16 * emx::MF_T);
  hipLaunchKernelGGL(emx::k_mlp_forward, dim3(std::min(512, (tiles + 3) / 4)), dim3(256), 0,
                     (hipStream_t)stream, params, norm, feat, n, act, nu);
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

// The partial sums of every workgroup.
size_t emx_mlp_backward_work(int n) { return (size_t)emx::mlp_grad_blocks(n) * emx::MNP; }

int emx_mlp_backward_f32(const float* params, const float* norm, const float* feat,
                         const float* act, const float* dnu, int n, float* grad, float* work,
                         size_t work_floats, void* stream) {
  if (!params || !norm || !feat || !act || !dnu || !grad || !work || n <= 0) {
    emx::set_error("emx_mlp_backward_f32: bad arguments");
    return EMX_ERR_ARG;
  }
  if (work_floats < emx_mlp_backward_work(n)) {
    emx::set_error("emx_mlp_backward_f32: work holds %zu floats, %zu needed", work_floats,
                   emx_mlp_backward_work(n));
    return EMX_ERR_SIZE;
  }
  const int nblk = emx::mlp_grad_blocks(n);
  const size_t lds = (size_t)4 * emx::MLP_GRAD_PAD * sizeof(float);
  hipStream_t st = (hipStream_t)stream;
  EMX_TRY_HIP(hipFuncSetAttribute((const void*)emx::k_mlp_grad,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(emx::k_mlp_grad, dim3(nblk), dim3(64 * emx::MG_WAVES), lds, st, params, norm,
                     feat, act, dnu, n, work);
  hipLaunchKernelGGL(emx::k_mlp_reduce, dim3((emx::MNP + 63) / 64), dim3(1024), 0, st, work, nblk,
                     grad);
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int emx_adam_f32(float* params, const float* grad, float* m, float* v, int n, float lr,
                 float beta1, float beta2, float eps, int step, void* stream) {
  if (!params || !grad || !m || !v || n <= 0 || step < 1) {
    emx::set_error("emx_adam_f32: bad arguments");
    return EMX_ERR_ARG;
  }
  const float c1 = 1.0f - powf(beta1, (float)step);
  const float c2 = 1.0f - powf(beta2, (float)step);
  hipLaunchKernelGGL(emx::k_adam, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     params, grad, m, v, n, lr, beta1, beta2, eps, c1, c2);
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

}  // extern "C"
