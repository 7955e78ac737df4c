// Adjoints (transposes) of the spatial operator: the compact derivative,
// the velocity gradient, the divergence and the linearised flux
// divergence of all five equations.  The reference has no adjoint; each
// function here is the exact transpose of the forward operator it names
// (same scheme, same metric projection), up to rounding.
#include "ops_common.hpp"

namespace emx {

// C adjacent values at f, which need not be aligned beyond a double.
typedef double f64x2u __attribute__((__vector_size__(16), __aligned__(8)));
template <int C>
__device__ __forceinline__ void read_w(const double* f, double* v) {
#pragma unroll
  for (int i = 0; i < C; i += 2) {
    const f64x2u t = *reinterpret_cast<const f64x2u*>(f + i);
    v[i] = t[0];
    v[i + 1] = t[1];
  }
}
template <int C>
__device__ __forceinline__ void write_w(double* f, const double* v) {
#pragma unroll
  for (int i = 0; i < C; i += 2) *reinterpret_cast<f64x2u*>(f + i) = f64x2u{v[i], v[i + 1]};
}

// Stores the first m of a chunk's C points (stride st) of one field; with
// add the old values, all read before the first write, are added to.
template <int C, bool XI>
__device__ __forceinline__ void put_chunk(double* f, long long st, int m, double* v, bool add) {
  if (XI && m == C) {
    if (add) {
      double o[C];
      read_w<C>(f, o);
#pragma unroll
      for (int i = 0; i < C; i++) v[i] = o[i] + v[i];
    }
    write_w<C>(f, v);
    return;
  }
  if (add) {
    double o[C];
#pragma unroll
    for (int i = 0; i < C; i++) o[i] = i < m ? f[i * st] : 0.0;
#pragma unroll
    for (int i = 0; i < C; i++) v[i] = o[i] + v[i];
  }
#pragma unroll
  for (int i = 0; i < C; i++)
    if (i < m) f[i * st] = v[i];
}

// Calls f(q, point) for the first m of a chunk's C points.
template <int C, class F>
__device__ __forceinline__ void each_point(long long p, long long st, int m, F f) {
#pragma unroll
  for (int q = 0; q < C; q++)
    if (q < m) f(q, p + q * st);
}

// NV fields, each through D^T along the pass direction; with accumulate
// the result is added to out (the passes of a gradient adjoint).
template <int N_>
struct ProbDerivAdj {
  static constexpr int NV = N_;
  static const char* label() { return "deriv_adj"; }
  double bytes_pt() const { return 8.0 * N_ * (accumulate ? 3 : 2); }
  const double* in[N_];
  double* out[N_];
  bool accumulate;
  __device__ __forceinline__ void load(long long p, double* v) const {
#pragma unroll
    for (int a = 0; a < N_; a++) v[a] = in[a][p];
  }
  template <int C>
  __device__ __forceinline__ void load_w(long long p, double (*v)[NV]) const {
#pragma unroll
    for (int a = 0; a < N_; a++) {
      double t[C];
      read_w<C>(in[a] + p, t);
#pragma unroll
      for (int i = 0; i < C; i++) v[i][a] = t[i];
    }
  }
  template <int C, bool XI>
  __device__ __forceinline__ void store(long long p, long long st, int m,
                                        const double (*v)[NV]) const {
#pragma unroll
    for (int a = 0; a < N_; a++) {
      double t[C];
#pragma unroll
      for (int i = 0; i < C; i++) t[i] = v[i][a];
      put_chunk<C, XI>(out[a] + p, st, m, t, accumulate);
    }
  }
};

// Four fields as two pairs, for chunks of eight: the gradient's adjoint with
// temperature at 300 x 280 x 60 takes 689 us with four fields to a
// work-item, 471 us in pairs.
struct ProbDerivAdjPairs {
  using Part = ProbDerivAdj<2>;
  static const char* label() { return Part::label(); }
  double bytes_pt() const { return 2.0 * lo.bytes_pt(); }
  Part lo, hi;
  static int parts() { return 2; }
  __host__ __device__ __forceinline__ Part part(int z) const { return z == 0 ? lo : hi; }
};

// Transpose of the divergence (solver/divergencia.f90:225-354 forward):
// rs = (1/J) sum_d D_d(J m_d e_d) gives e_d_bar = J m_d D_d^T(rs_bar / J),
// and the same for the viscous pair.  flux_bar holds e,f,g,ev,fv,gv.
struct ProbDivAdj {
  static constexpr int NV = 2;
  static const char* label() { return "divergence_adj"; }
  double bytes_pt() const { return 8.0 * 7; }
  const double* rs_bar;
  const double* rsv_bar;
  const double* jbn;
  double* flux_bar;
  long long N;
  int dir;
  __device__ __forceinline__ void load(long long p, double* v) const {
    const double ij = jbn[10 * N + p];
    v[0] = ij * rs_bar[p];
    v[1] = ij * rsv_bar[p];
  }
  template <int C>
  __device__ __forceinline__ void load_w(long long p, double (*v)[NV]) const {
#pragma unroll
    for (int i = 0; i < C; i++) load(p + i, v[i]);
  }
  template <int C, bool XI>
  __device__ __forceinline__ void store(long long p0, long long st, int m,
                                        const double (*v)[NV]) const {
    each_point<C>(p0, st, m, [&](int q, long long p) {
      const double jm = jbn[9 * N + p] * jbn[(4 * dir) * N + p];
      flux_bar[dir * N + p] = jm * v[q][0];
      flux_bar[(3 + dir) * N + p] = jm * v[q][1];
    });
  }
};

// Transpose of the linearisation of the five-equation flux divergence
// (flujos_compact.f90:20-217 fluxes, divergencia.f90 projection) about
// (um, u, vis, dvel); pres enters linearly, jbn is fixed.  With
// x_d[k] = D_d^T(r_k / J) for the eight adjoints r (convective equations
// 1..5, viscous 2..4), the flux adjoints of direction d are e_d = J m_d x_d,
// and they scatter to the input adjoints:
//   conv 1   e = -um(2+d)                 -> um(2+d)
//   conv 2-4 e = -um(2+d) u(a+1) [-pres]  -> um(2+d), u(a+1), pres (a = d)
//   conv 5   e = -u(1+d) um5              -> u(1+d), um5
//   visc a=d  mu*2*(J m_a D_a)            -> vis, dvel(1+4a)
//   visc a!=d mu*(J_x D_y + J_z D_w)      -> vis, two dvel
// The xi and eta passes only solve: x_0 and x_1 go into the output arrays
// (slot() below), which the two zeta passes (convective, viscous) read at
// the points they overwrite with the results of all three directions.  One
// pass per direction that scattered at once read the primal fields three
// times and added to its outputs in memory: 1008 B per point and 3 x 236 us
// at 128^3, against 832 B and 102 + 97 + 148 + 141 us now (4.1 TB/s in the
// scatter passes, whose registers leave two workgroups on a CU).
struct AdjScratch {
  double* um_bar;    // 5 fields (1 is zero)
  double* u_bar;     // 3 fields
  double* pres_bar;
  double* vis_bar;
  double* dvel_bar;  // 9 fields
  long long N;
  // Where x_d[k] is kept, d = 0, 1.  The convective pass overwrites um_bar,
  // u_bar and pres_bar, the viscous one, which runs after it, the rest.
  __host__ __device__ __forceinline__ double* slot(int d, int k) const {
    if (k >= 5) return dvel_bar + (3 * d + k - 5) * N;
    if (d == 0) return um_bar + k * N;
    return k < 3 ? u_bar + k * N : (k == 3 ? pres_bar : dvel_bar + 6 * N);
  }
};

// The eight solves of the xi or eta pass, four fields to a work-item (all
// eight: 116-128 us a pass, with half the wavefronts).
struct ProbDivAllSolve {
  struct Part {
    static constexpr int NV = 4;
    const double* in[4];
    double* out[4];
    const double* ij;
    __device__ __forceinline__ void load(long long p, double* v) const {
      const double j = ij[p];
#pragma unroll
      for (int a = 0; a < 4; a++) v[a] = j * in[a][p];
    }
    template <int C>
    __device__ __forceinline__ void load_w(long long p, double (*v)[NV]) const {
      double j[C];
      read_w<C>(ij + p, j);
#pragma unroll
      for (int a = 0; a < 4; a++) {
        double t[C];
        read_w<C>(in[a] + p, t);
#pragma unroll
        for (int i = 0; i < C; i++) v[i][a] = j[i] * t[i];
      }
    }
    template <int C, bool XI>
    __device__ __forceinline__ void store(long long p, long long st, int m,
                                          const double (*v)[NV]) const {
#pragma unroll
      for (int a = 0; a < 4; a++) {
        double t[C];
#pragma unroll
        for (int i = 0; i < C; i++) t[i] = v[i][a];
        put_chunk<C, XI>(out[a] + p, st, m, t, false);
      }
    }
  };
  static const char* label() { return "flux_div_all_adj[solve]"; }
  double bytes_pt() const { return 8.0 * 17; }
  static constexpr bool INTERLEAVE = true;  // 1/J
  Part lo, hi;
  static int parts() { return 2; }
  __host__ __device__ __forceinline__ Part part(int z) const { return z == 0 ? lo : hi; }
};

// The convective half of the zeta pass.
struct ProbDivAllConv {
  static constexpr int NV = 5;
  static constexpr int ADJ_WAVES = 4;
  static const char* label() { return "flux_div_all_adj[conv]"; }
  // rs_bar and 1/J; x_0, x_1, um 2..5, u, J and three metrics; um_bar,
  // u_bar, pres_bar
  double bytes_pt() const { return 8.0 * (6 + 10 + 4 + 3 + 4 + 9); }
  FluxIn in;
  const double* rs_bar;
  AdjScratch o;
  __device__ __forceinline__ void load(long long p, double* v) const {
    const double ij = in.J(11, p);
#pragma unroll
    for (int a = 0; a < 5; a++) v[a] = ij * rs_bar[a * in.N + p];
  }
  template <int C, bool XI>
  __device__ __forceinline__ void store(long long p0, long long st, int m,
                                        const double (*v)[NV]) const {
    each_point<C>(p0, st, m, [&](int q, long long p) {
      const long long N = in.N;
      double x[3][5], umd[3], u[3];
#pragma unroll
      for (int k = 0; k < 5; k++) {
        x[0][k] = o.slot(0, k)[p];
        x[1][k] = o.slot(1, k)[p];
        x[2][k] = v[q][k];
      }
      const double J = in.J(10, p);
#pragma unroll
      for (int d = 0; d < 3; d++) {
        umd[d] = in.UM(2 + d, p);
        u[d] = in.U(1 + d, p);
        const double jm = J * in.J(1 + 4 * d, p);
#pragma unroll
        for (int k = 0; k < 5; k++) x[d][k] = jm * x[d][k];
      }
      const double um5 = in.UM(5, p);
      o.um_bar[p] = 0.0;  // um(1) does not enter any flux
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double t = -x[d][0];
#pragma unroll
        for (int a = 0; a < 3; a++) t -= x[d][1 + a] * u[a];
        o.um_bar[(1 + d) * N + p] = t;
      }
      double b5 = 0.0, bp = 0.0, bu[3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
          double g = -x[d][1 + a] * umd[d];
          if (a == d) g -= x[d][4] * um5;
          bu[a] = d == 0 ? g : bu[a] + g;
        }
        b5 = d == 0 ? -x[d][4] * u[d] : b5 + -x[d][4] * u[d];
        bp = d == 0 ? -x[d][1 + d] : bp + -x[d][1 + d];
      }
      o.um_bar[4 * N + p] = b5;
#pragma unroll
      for (int a = 0; a < 3; a++) o.u_bar[a * N + p] = bu[a];
      o.pres_bar[p] = bp;
    });
  }
};

// The viscous half.
struct ProbDivAllVisc {
  static constexpr int NV = 3;
  static constexpr int ADJ_WAVES = 4;
  static const char* label() { return "flux_div_all_adj[visc]"; }
  // rsv_bar 2..4 and 1/J; x_0, x_1, vis, J and three metrics, dvel;
  // vis_bar, dvel_bar
  double bytes_pt() const { return 8.0 * (4 + 6 + 1 + 4 + 9 + 10); }
  FluxIn in;
  const double* rsv_bar;
  AdjScratch o;
  __device__ __forceinline__ void load(long long p, double* v) const {
    const double ij = in.J(11, p);
#pragma unroll
    for (int a = 0; a < 3; a++) v[a] = ij * rsv_bar[(1 + a) * in.N + p];
  }
  template <int C, bool XI>
  __device__ __forceinline__ void store(long long p0, long long st, int m,
                                        const double (*v)[NV]) const {
    each_point<C>(p0, st, m, [&](int q, long long p) {
      const long long N = in.N;
      double e[3][3], Jm[3], D[9], b[9];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        e[0][k] = o.slot(0, 5 + k)[p];
        e[1][k] = o.slot(1, 5 + k)[p];
        e[2][k] = v[q][k];
      }
      const double J = in.J(10, p), mu = in.vis[p];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        Jm[d] = in.J(1 + 4 * d, p);
        const double jm = J * Jm[d];
#pragma unroll
        for (int k = 0; k < 3; k++) e[d][k] = jm * e[d][k];
      }
#pragma unroll
      for (int k = 0; k < 9; k++) D[k] = in.D(1 + k, p);
      const double J1 = Jm[0], J5 = Jm[1], J9 = Jm[2];
      double vis = 0.0;
      bool set[9] = {};  // resolved at compile time
      auto dput = [&](int k, double w) {
        b[k - 1] = set[k - 1] ? b[k - 1] + w : w;
        set[k - 1] = true;
      };
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double vb = 0.0;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const double w = e[d][a];
          if (a == d) {
            vb += w * (2.0 * (Jm[a] * D[4 * a]));
            dput(1 + 4 * a, w * mu * 2.0 * Jm[a]);
          } else if (a + d == 1) {  // J1*D2 + J5*D4
            vb += w * (J1 * D[1] + J5 * D[3]);
            dput(2, w * mu * J1);
            dput(4, w * mu * J5);
          } else if (a + d == 2) {  // J1*D3 + J9*D7
            vb += w * (J1 * D[2] + J9 * D[6]);
            dput(3, w * mu * J1);
            dput(7, w * mu * J9);
          } else {                  // J9*D8 + J5*D6
            vb += w * (J9 * D[7] + J5 * D[5]);
            dput(8, w * mu * J9);
            dput(6, w * mu * J5);
          }
        }
        vis = d == 0 ? vb : vis + vb;
      }
      o.vis_bar[p] = vis;
#pragma unroll
      for (int k = 0; k < 9; k++) o.dvel_bar[k * N + p] = b[k];
    });
  }
};

int adj_ready(emx_ctx* ctx) {
  for (int d = 0; d < 3; d++)
    if (!ctx->adj[d].blob) {
      set_error("adjoint operators need lines of at most %d points (grid %d x %d x %d)",
                ADJ_MAX_N, ctx->d.nx, ctx->d.ny, ctx->d.nz);
      return EMX_ERR_SIZE;
    }
  return EMX_OK;
}

int op_deriv_adj(emx_ctx* ctx, int dir, const double* g, double* out, double ih) {
  EMX_TRY(adj_ready(ctx));
  ProbDerivAdj<1> p{{g}, {out}, false};
  return launch_lines_adj(ctx, dir, p, ih);
}

int op_grad_adj(emx_ctx* ctx, const double* dvel_bar, const double* dtemp_bar,
                double* u_bar, double* temp_bar, const double ih[3]) {
  EMX_TRY(adj_ready(ctx));
  const long long N = ctx->d.N();
  for (int d = 0; d < 3; d++) {
    if (dtemp_bar && ctx->adj[d].C == 8) {
      const double* b = dvel_bar + 3 * d * N;
      ProbDerivAdjPairs p{{{b, b + N}, {u_bar, u_bar + N}, d > 0},
                          {{b + 2 * N, dtemp_bar + d * N}, {u_bar + 2 * N, temp_bar}, d > 0}};
      EMX_TRY(launch_lines_adj(ctx, d, p, ih[d]));
    } else if (dtemp_bar) {
      ProbDerivAdj<4> p{{dvel_bar + (3 * d) * N, dvel_bar + (3 * d + 1) * N,
                         dvel_bar + (3 * d + 2) * N, dtemp_bar + d * N},
                        {u_bar, u_bar + N, u_bar + 2 * N, temp_bar}, d > 0};
      EMX_TRY(launch_lines_adj(ctx, d, p, ih[d]));
    } else {
      ProbDerivAdj<3> p{{dvel_bar + (3 * d) * N, dvel_bar + (3 * d + 1) * N,
                         dvel_bar + (3 * d + 2) * N},
                        {u_bar, u_bar + N, u_bar + 2 * N}, d > 0};
      EMX_TRY(launch_lines_adj(ctx, d, p, ih[d]));
    }
  }
  return EMX_OK;
}

int op_divergence_adj(emx_ctx* ctx, const double* rs_bar, const double* rsv_bar,
                      const double* jbn, const double ih[3], double* flux_bar) {
  EMX_TRY(adj_ready(ctx));
  for (int d = 0; d < 3; d++) {
    ProbDivAdj p{rs_bar, rsv_bar, jbn, flux_bar, ctx->d.N(), d};
    EMX_TRY(launch_lines_adj(ctx, d, p, ih[d]));
  }
  return EMX_OK;
}

int op_flux_div_all_adj(emx_ctx* ctx, const double* rs_bar, const double* rsv_bar,
                        const FluxPtrs& fp, const double ih[3], double* um_bar,
                        double* u_bar, double* pres_bar, double* vis_bar,
                        double* dvel_bar) {
  EMX_TRY(adj_ready(ctx));
  const long long N = ctx->d.N();
  const FluxIn in{fp.um, fp.u, nullptr, fp.vis, fp.jbn, fp.dvel, N};
  const AdjScratch o{um_bar, u_bar, pres_bar, vis_bar, dvel_bar, N};
  for (int d = 0; d < 2; d++) {
    ProbDivAllSolve p;
    p.lo.ij = p.hi.ij = fp.jbn + 10 * N;
    for (int k = 0; k < 8; k++) {
      ProbDivAllSolve::Part& h = k < 4 ? p.lo : p.hi;
      h.in[k % 4] = k < 5 ? rs_bar + k * N : rsv_bar + (k - 4) * N;
      h.out[k % 4] = o.slot(d, k);
    }
    EMX_TRY(launch_lines_adj(ctx, d, p, ih[d]));
  }
  EMX_TRY(launch_lines_adj_as<false>(ctx, 2, ProbDivAllConv{in, rs_bar, o}, ih[2]));
  return launch_lines_adj_as<false>(ctx, 2, ProbDivAllVisc{in, rsv_bar, o}, ih[2]);
}

}  // namespace emx
