// Compact filter (FILTRADO, src/MSVSingle/herramientas_incomp2.f90:227-410)
// on the device: each conservative field times J is filtered along the
// three directions in the order itf selects, each pass one tridiagonal
// solve per line (FILTRONPER, src/MSVSingle/filtro_incomp.f90:307-362) with
// an 11-point explicit right-hand side, then times 1/J; u, temp and pres are
// recomputed from the result.  The solves run on the line-solver kernels of
// the derivatives (chunked Thomas with precomputed carries), with the
// filter's matrix in the line table and a 5-point halo.
#include "ops_common.hpp"

namespace emx {

// One field filtered in place along a line: J*f formed at load, the
// filtered value times 1/J stored (a nontemporal store: the pass does not
// read it back, and the hint measured 5% faster over FILTRADO).
struct ProbFilter {
  static constexpr int NV = 1;
  static const char* label() { return "filter"; }
  double* f;
  const double* jac;
  const double* ijac;
  __device__ __forceinline__ void load(long long p, double* v) const { v[0] = f[p] * jac[p]; }
  __device__ __forceinline__ void store(long long p, const double* v) const {
    __builtin_nontemporal_store(v[0] * ijac[p], &f[p]);
  }
  // Q points p + i*sl at once, the 1/J reads first (each would otherwise
  // wait for the store before it)
  static constexpr bool BATCH_STORE = true;
  template <int Q>
  __device__ __forceinline__ void store_batch(long long p, long long sl,
                                              const double (*v)[NV]) const {
    double q[Q];
#pragma unroll
    for (int i = 0; i < Q; i++) q[i] = ijac[p + i * sl];
#pragma unroll
    for (int i = 0; i < Q; i++) __builtin_nontemporal_store(v[i][0] * q[i], &f[p + i * sl]);
  }
};

// The five conservative fields (stride N) in one launch.  The strided kinds
// take them as parts, a line group's five next to each other on one XCD: J
// and 1/J come from memory once and from its L2 four times (96 B per point
// and direction instead of 160).
struct ProbFilterParts {
  using Part = ProbFilter;
  static constexpr int NV = 1;
  static constexpr bool BATCH_STORE = true, INTERLEAVE = true;
  double* f;
  const double* jac;
  const double* ijac;
  long long N;
  static int parts() { return 5; }
  __host__ __device__ __forceinline__ Part part(int m) const { return Part{f + m * N, jac, ijac}; }
};

// The wavefront kind solves a line's five fields one after another, J and
// 1/J read once for all.  Same arithmetic as ProbFilter.
struct ProbFilterLine {
  static constexpr int NV = 5;
  static constexpr bool PREFETCH = true, LINE_STORE = true;
  double* f;
  const double* jac;
  const double* ijac;
  long long N;
  __device__ __forceinline__ void load(long long p, double* v) const {
    const double j = jac[p];
#pragma unroll
    for (int m = 0; m < 5; m++) v[m] = f[m * N + p] * j;
  }
  template <int C>
  __device__ __forceinline__ void store_line(long long base, long long sl, int lane, int n,
                                             const double (*v)[NV]) const {
    double q[C];
#pragma unroll
    for (int i = 0; i < C; i++) q[i] = ijac[base + min(i * 64 + lane, n - 1) * sl];
#pragma unroll
    for (int i = 0; i < C; i++) {
      if (i * 64 + lane >= n) continue;
#pragma unroll
      for (int m = 0; m < 5; m++)
        __builtin_nontemporal_store(v[i][m] * q[i], &f[m * N + base + (i * 64 + lane) * sl]);
    }
  }
};

namespace {

// xi: one wavefront per line, the shortest chunk that covers the line;
// eta, zeta: 32 lines per wavefront, chunks of 16 points.
int filter_shape(int dir, int n, int* kind, int* C) {
  if (dir == 0) {
    int c = 1;
    while (c * 64 < n) c *= 2;
    *kind = KIND_WAVE;
    *C = c == 4 && n <= 192 ? 3 : c;
  } else {
    *kind = KIND_STRIDED32;
    *C = 16;
  }
  return EMX_OK;
}

template <int S>
hipError_t launch_filter(double* um1, const double* jbn, long long N, const LineTab& T,
                         const DirGeom& g, double cfilt, hipStream_t st) {
  const double *jac = jbn + 9 * N, *ijac = jbn + 10 * N;
  if (T.kind == KIND_WAVE) {
    const ProbFilterLine p{um1, jac, ijac, N};
    switch (T.C) {
      case 1: return launch_wave_c<S, 1>(p, T, g, cfilt, st);
      case 2: return launch_wave_c<S, 2>(p, T, g, cfilt, st);
      case 3: return launch_wave_c<S, 3>(p, T, g, cfilt, st);
      case 4: return launch_wave_c<S, 4>(p, T, g, cfilt, st);
    }
    // lines past 256 points: five fields of such a chunk do not fit the
    // registers
    hipError_t e = hipSuccess;
    for (int m = 0; e == hipSuccess && m < 5; m++) {
      const ProbFilter q{um1 + m * N, jac, ijac};
      e = T.C == 8 ? launch_wave_c<S, 8>(q, T, g, cfilt, st)
                   : launch_wave_c<S, 16>(q, T, g, cfilt, st);
    }
    return e;
  }
  return launch_strided_c<S, 16, 32>(ProbFilterParts{um1, jac, ijac, N}, T, g, cfilt, st);
}

}  // namespace

int op_filtrado(emx_ctx* ctx, int itf, double* um1, const double* jbn, double cfilt,
                double mach, double* u, double* pres, double* temp) {
  // direction order of each itf (herramientas_incomp2.f90:245-392)
  static const int order[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2},
                                  {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  const long long N = ctx->d.N();
  LineTab tab[3];
  for (int dir = 0; dir < 3; dir++) {
    const int n = dir == 0 ? ctx->d.nx : (dir == 1 ? ctx->d.ny : ctx->d.nz);
    int kind, C;
    EMX_TRY(filter_shape(dir, n, &kind, &C));
    EMX_TRY(get_line_tab(dir == 2 ? FILTER_P : FILTER_NP, n, C, kind, &tab[dir], cfilt));
  }
  for (int k = 0; k < 3; k++) {
    const int dir = order[itf - 1][k];
    const DirGeom g = dir_geom(ctx->d, dir);
    // five fields in and out, J and 1/J
    LaunchTimer timer(ctx, ProbFilter::label(), dir, 96.0 * (double)N);
    const hipError_t e =
        dir == 2 ? launch_filter<FILTER_P>(um1, jbn, N, tab[dir], g, cfilt, ctx->stream)
                 : launch_filter<FILTER_NP>(um1, jbn, N, tab[dir], g, cfilt, ctx->stream);
    if (e != hipSuccess) {
      set_error("filter launch (dir %d) failed: %s", dir, hipGetErrorString(e));
      return EMX_ERR_HIP;
    }
  }
  // u, temp, pres from the filtered variables (herramientas_incomp2.f90:395-405)
  return op_varc_to_varnc(ctx, um1, mach, u, pres, temp, nullptr);
}

}  // namespace emx
