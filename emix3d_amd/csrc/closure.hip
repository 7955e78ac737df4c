// Learned eddy-viscosity closure: a 10 -> 64 -> 64 -> 64 -> 1 network
// (SiLU hidden activations, softplus output) of the physical velocity
// gradient and the filter width.  The reference has no counterpart.
//
// Parameters (FP32, EMX_MLP_NPARAM values):
//   W1[64][10] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[64] b4
// Normalisation (FP32, EMX_MLP_NNORM): in_shift[10] in_scale[10] out_scale,
//   x_k = (f_k - in_shift_k) * in_scale_k,  nu = out_scale * softplus(z4).
// Features f of a grid point: du_a/dx_b = jbn(1+4b) * dvel(3b+a) at index
// 3a+b, then delta.
//
// Inference (k_mlp_infer) runs the three hidden layers on the matrix cores:
// v_mfma_f32_16x16x32_bf16, BF16 operands, FP32 accumulation.  Each layer
// is computed transposed, H^T[64 x 16 points] = W[64 x K] X^T[K x 16], so
// the 16x16 result tile a lane holds (4 neurons of one point) is already
// the B operand of the next layer once the K order of that layer's weights
// is permuted to match (perm_in below): no data moves between lanes.
// The training passes are in closure_train.hip.
#include <algorithm>

#include "mlp_infer.hpp"
#include "ops_common.hpp"

namespace emx {

// Physical gradient and filter width of point p (the 10 features).
__device__ __forceinline__ void point_features(const double* dvel, const double* jbn,
                                               const double* delta, long long N,
                                               long long p, double f[MLP_IN]) {
  const double m[3] = {jbn[p], jbn[4 * N + p], jbn[8 * N + p]};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) f[3 * a + b] = m[b] * dvel[(3 * b + a) * N + p];
  f[9] = delta[p];
}

// Packs the parameters into per-lane BF16 A operands, one work-item per
// packed value (MLP_PACK_ELEMS of them, in units of 64 lanes x 8):
//   A1[mt][lane][8]      layer 1 (features padded to K = 32)
//   A2[mt][s][lane][8], A3[mt][s][lane][8]   layers 2, 3
//   A4[s][lane][8]       the output neuron's weights (divided by the scale
//                        of the hidden layers) in every row
// lane l holds row m = l%16 (output neuron 16mt+m), K = 8(l/16) + j.
__global__ void k_mlp_pack(const float* P, __bf16* A) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_PACK_ELEMS) return;
  const int j = e & 7, l = (e >> 3) & 63, unit = e >> 9;
  const int m = l % 16, g = l / 16;
  float v;
  if (e < MLP_PACK_A2) {
    // layer 1 in the scaled form of mlp_group64: y = MLP_YS * z
    const int k = 8 * g + j;
    v = k < MLP_IN ? MLP_YS * P[MW1 + (16 * unit + m) * MLP_IN + k] : 0.0f;
  } else if (e < MLP_PACK_A4) {
    const int layer = e < MLP_PACK_A3 ? 0 : 1;
    const int r = unit - 4 - 8 * layer, mt = r >> 1, sk = r & 1;
    v = P[(layer == 0 ? MW2 : MW3) + (16 * mt + m) * MLP_H + perm_in(sk, g, j)];
  } else {
    v = P[MW4 + perm_in(unit - 20, g, j)] / MLP_YS;
  }
  A[e] = (__bf16)v;
}

// nu_t of every grid point: persistent wavefronts, each taking groups of
// 64 consecutive points (one per lane, loads coalesced).  Three wavefronts
// per SIMD (at most 168 registers, no spills) hide one group's loads behind
// the others' networks; keeping the next group's inputs in registers
// instead allows only two and was measured slower (0.97 against 0.88 ms at
// 256^3).  Grids hold at most 2^28 points (emx_create), so every access is
// a uniform field base plus a 32-bit byte offset: no 64-bit address
// arithmetic per load.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
k_mlp_infer(const double* dvel, const double* jbn, const double* delta, long long N,
            const float* P, const float* norm, const __bf16* A, double* nut, double c4,
            double* vis) {
  __shared__ __attribute__((aligned(16))) float vec[MLP_VEC + 2];
  __shared__ double nrm[2 * MLP_IN];  // in_shift, in_scale
  __shared__ float xs[4][MLP_IN * 64];
  __shared__ bf16x8 lw[MLP_LW];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  mlp_stage_weights(lw, A);
  mlp_stage_vectors(vec, P, norm);
  for (int t = threadIdx.x; t < 2 * MLP_IN; t += blockDim.x) nrm[t] = (double)norm[t];
  __syncthreads();
  const long long ngroup = (N + 63) / 64;
  const long long nwave = (long long)gridDim.x * (blockDim.x >> 6);
  for (long long grp = (long long)blockIdx.x * (blockDim.x >> 6) + w; grp < ngroup;
       grp += nwave) {
    const long long p = grp * 64 + l;
    const unsigned off = (unsigned)(p < N ? p : N - 1) * 8u;
    auto at = [off](const double* base) -> const double& {
      return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
    };
    // raw inputs of the point: dvel 1..9, jbn 1, 5, 9, delta
    double r[13];
#pragma unroll
    for (int c = 0; c < 9; c++) r[c] = at(dvel + c * N);
    r[9] = at(jbn);
    r[10] = at(jbn + 4 * N);
    r[11] = at(jbn + 8 * N);
    r[12] = at(delta);
    float x[MLP_IN];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++)
        x[3 * a + b] =
            (float)((r[9 + b] * r[3 * b + a] - nrm[3 * a + b]) * nrm[MLP_IN + 3 * a + b]);
    x[9] = (float)((r[12] - nrm[9]) * nrm[MLP_IN + 9]);
    const float nu = mlp_group64(lw, x, xs[w], vec, l);
    if (p < N) {
      double* const np = reinterpret_cast<double*>(reinterpret_cast<char*>(nut) + off);
      *np = (double)nu;
      if (vis) {
        double* const vp = reinterpret_cast<double*>(reinterpret_cast<char*>(vis) + off);
        *vp = c4 * 1.0 + (double)nu;  // viscosidad (solver/viscosidad_incomp.f90:15-17)
      }
    }
  }
}

// Features of the listed points (training), [n][10] (indices clamped to [0, N)).
__global__ void k_mlp_gather(const double* dvel, const double* jbn, const double* delta,
                             long long N, const long long* idx, int n, float* feat) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
    double f[MLP_IN];
    const long long p = idx[q] < 0 ? 0 : (idx[q] >= N ? N - 1 : idx[q]);
    point_features(dvel, jbn, delta, N, p, f);
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) feat[(long long)q * MLP_IN + k] = (float)f[k];
  }
}

// ---------------------------------------------------------------------------

size_t mlp_pack_elems() { return (size_t)MLP_PACK_ELEMS; }

int op_mlp_pack(emx_ctx* ctx, const float* params, const float* norm) {
  __bf16* A = reinterpret_cast<__bf16*>(ctx->mlp_pack);
  EMX_TIMED(ctx, "mlp_pack", 0.0,
            hipLaunchKernelGGL(k_mlp_pack, dim3((MLP_PACK_ELEMS + 255) / 256), dim3(256), 0,
                               ctx->stream, params, A));
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int op_mlp_nut(emx_ctx* ctx, const float* params, const float* norm, const double* dvel,
               const double* jbn, const double* delta, double* nut, double c4, double* vis) {
  const long long N = ctx->d.N();
  if (N > (1LL << 29)) {  // k_mlp_infer's 32-bit byte offsets
    set_error("emx_mlp_nut: %lld points, at most 2^29", N);
    return EMX_ERR_SIZE;
  }
  __bf16* A = reinterpret_cast<__bf16*>(ctx->mlp_pack);
  EMX_TRY(op_mlp_pack(ctx, params, norm));
  static const int resident = resident_blocks(k_mlp_infer, 0);
  const long long groups = (N + 63) / 64;
  long long blocks = (groups + 3) / 4;
  if (blocks > resident) blocks = resident;
  // reads dvel (9), jbn (3), delta; writes nut (and vis)
  EMX_TIMED(ctx, "mlp_infer", (vis ? 15.0 : 14.0) * 8.0 * N,
            hipLaunchKernelGGL(k_mlp_infer, dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                               dvel, jbn, delta, N, params, norm, A, nut, c4, vis));
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

int op_mlp_gather(emx_ctx* ctx, const double* dvel, const double* jbn, const double* delta,
                  const long long* idx, int n, float* feat) {
  hipLaunchKernelGGL(k_mlp_gather, dim3(std::min(4096, (n + 255) / 256)), dim3(256), 0,
                     ctx->stream, dvel, jbn, delta, ctx->d.N(), idx, n, feat);
  EMX_TRY_HIP(hipGetLastError());
  return EMX_OK;
}

}  // namespace emx
