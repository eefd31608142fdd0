// march_rows.h -- rows of the implicit-Euler matrix of one instance and of its
// inverse, for the kernels that march with them (march.hip, dense.hip).
#pragma once
#include "device_common.h"
#include "scft_internal.h"

namespace scft {

// The persistent workgroups' next item: its own number first (the caller's
// loop), then from the launch's counter, which is not read when the grid covers
// all items.  Thread 0 takes the index and broadcasts it through LDS; the value
// is workgroup-uniform, so every wave leaves the loop together.  The two
// barriers also separate an instance's use of LDS from the next one's.
__device__ __forceinline__ int next_item(const MarchArgs& a, int tid, int* s_next) {
  const int grid = static_cast<int>(gridDim.x);
  if (a.n_items <= grid) return a.n_items;
  if (tid == 0) *s_next = grid + atomicAdd(a.queue, 1);
  wg_barrier();
  const int it = __builtin_amdgcn_readfirstlane(*s_next);
  wg_barrier();  // everyone has read it before thread 0 overwrites it
  return it;
}

template <int W>
struct MarchShared {
  // forward, then backward wave totals (per step, two sets in turn), and a
  // place for every other lane's write
  double tot[2][W > 1 ? 2 * W + 64 * W : 1];
  double Aw[W];     // forward wave transfer products (per instance)
  double Gw[W];     // backward wave transfer products (per instance)
  double cx[W], ax[W];  // last super-, first sub-diagonal of each wave (setup)
  double hx[W], fx[W];  // last h, first f of each wave (setup)
  double Mx[W][4][2];  // wave products of the determinant matrices, double-double (setup)
  double red[W];    // norm reduction
  double cw[6];     // pairing weights by class (per instance)
  unsigned bad[W];
};


// One row of D = A + dt (B + C) and of the right-hand-side operator A for
// unknown u (node u+1), from its two adjacent elements.  Evaluated without
// FMA contraction and in the same operation order as the CPU restatement:
// the rows of D are nearly identical, so a contracted rounding would shift
// every row the same way and move the diagonal-dominance margin
// b - |a| - |c| ~ h by eps * dt/h^2 relative per step, which adds up over the
// march (~1e-10 after a few hundred steps when dt/h^2 ~ 1e3).
struct Row {
  double a, b, c;  // D = A + dt (B + C): sub-, main and super-diagonal
  double ra, rc;   // A q = ra (q_{i-1} + 2 q_i) + rc (2 q_i + q_{i+1})
};

// Returned by value with every field assigned once (selects, no stores
// through references): conditional stores to two different outputs get
// merged into one store through a pointer phi, which keeps the row arrays
// out of registers.
__device__ __forceinline__ Row assemble_row(const double* __restrict__ x,
                                            const double* __restrict__ w, int n, int M, int u,
                                            double dt, int cmat, double wall0, double wallL) {
#pragma clang fp contract(off)
  const bool live = u < n;
  const int i = live ? u + 1 : 1;  // padding rows read node 1 and are discarded
  const double xl = x[i - 1], xc = x[i];
  const bool has_r = (i + 1 < M);
  const double xr = has_r ? x[i + 1] : xc;
  const double hl = xc - xl, hr = xr - xc;
  const double wi = live ? w[live ? u : 0] : 0.0;  // index clamped: no load past the field
  const double Al = hl / 6.0, Ar = hr / 6.0, Ad = hl / 3.0 + hr / 3.0;
  const double Bl = -1.0 / hl;
  const double Br = has_r ? -1.0 / hr : 0.0;
  const double Bd = 1.0 / hl + (has_r ? 1.0 / hr : 0.0);
  double Cl, Cd, Cr;
  if (cmat == 0) {
    Cl = wi * Al;
    Cd = wi * Ad;
    Cr = wi * Ar;
  } else {
    const double wl = (u > 0 && live) ? w[u - 1] : wall0;
    const double wr = (u + 1 < n) ? w[u + 1] : wallL;
    Cl = hl * (wl + wi) / 12.0;
    Cd = hl * (wl + 3.0 * wi) / 12.0 + hr * (3.0 * wi + wr) / 12.0;
    Cr = hr * (wi + wr) / 12.0;
  }
  const double av = Al + dt * (Bl + Cl);
  const double bv = Ad + dt * (Bd + Cd);
  const double cv = Ar + dt * (Br + Cr);
  // left neighbour of unknown 0 is the Dirichlet wall; right neighbour of
  // unknown n-1 is a wall (DD) or none (DN); padding rows are decoupled
  // identity rows with a zero right-hand side (q stays 0 there)
  Row r;
  r.a = (live && u > 0) ? av : 0.0;
  r.c = (live && u < n - 1) ? cv : 0.0;
  r.b = live ? bv : 1.0;
  r.ra = live ? Al : 0.0;
  r.rc = live ? Ar : 0.0;
  return r;
}

// Rows of the mass matrix A and of D' = B + C for unknown u (node u+1), from
// its two adjacent elements; the same expressions and boundary handling as
// assemble_row's (no FMA contraction).  Padding rows (u >= n) are
// zero in both, and the couplings to Dirichlet nodes or past the last
// unknown are dropped.
struct SplitRow {
  double al, ad, ar;  // A
  double dl, dd, dr;  // D'
};
__device__ __forceinline__ SplitRow assemble_split(const double* __restrict__ x,
                                                   const double* __restrict__ w, int n, int M,
                                                   int u, int cmat, double wall0, double wallL) {
#pragma clang fp contract(off)
  const bool live = u < n;
  const int i = live ? u + 1 : 1;
  const double xl = x[i - 1], xc = x[i];
  const bool has_r = (i + 1 < M);
  const double xr = has_r ? x[i + 1] : xc;
  const double hl = xc - xl, hr = xr - xc;
  const double wi = live ? w[live ? u : 0] : 0.0;
  const double Al = hl / 6.0, Ar = hr / 6.0, Ad = hl / 3.0 + hr / 3.0;
  const double Bl = -1.0 / hl;
  const double Br = has_r ? -1.0 / hr : 0.0;
  const double Bd = 1.0 / hl + (has_r ? 1.0 / hr : 0.0);
  double Cl, Cd, Cr;
  if (cmat == 0) {
    Cl = wi * Al;
    Cd = wi * Ad;
    Cr = wi * Ar;
  } else {
    const double wl = (u > 0 && live) ? w[u - 1] : wall0;
    const double wr = (u + 1 < n) ? w[u + 1] : wallL;
    Cl = hl * (wl + wi) / 12.0;
    Cd = hl * (wl + 3.0 * wi) / 12.0 + hr * (3.0 * wi + wr) / 12.0;
    Cr = hr * (wi + wr) / 12.0;
  }
  const bool has_l = live && u > 0, has_rr = live && u < n - 1;
  SplitRow s;
  s.al = has_l ? Al : 0.0;
  s.ad = live ? Ad : 0.0;
  s.ar = has_rr ? Ar : 0.0;
  s.dl = has_l ? Bl + Cl : 0.0;
  s.dd = live ? Bd + Cd : 0.0;
  s.dr = has_rr ? Br + Cr : 0.0;
  return s;
}

// D is tridiagonal, so its inverse G falls off by fixed factors away from the
// diagonal: G_ii = 1 / (u_i + v_i - b_i), G_ij = f_i G_{i-1,j} below it and
// h_i G_{i+1,j} above it, with f_i = -a_i / v_i, h_i = -c_i / u_i and u, v the
// elimination pivots from above and from below.  Lane tid of the workgroup
// (W waves) holds rows tid K .. tid K + K - 1; gi = 1 / G_ii.
template <int K, int W>
__device__ __forceinline__ void inverse_rows(const double (&av)[K], const double (&bv)[K],
                                             const double (&cv)[K], MarchShared<W>& sh,
                                             const int tid, double (&f)[K], double (&h)[K],
                                             dd (&gi)[K], unsigned& bad) {
  constexpr int P = 64 * W;
  const int lane = tid & 63;
  [[maybe_unused]] const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // c of the row left of this lane's chunk, a of the row right of it
  double cprev = __shfl_up(cv[K - 1], 1), anext = __shfl_down(av[0], 1);
  if constexpr (W > 1) {
    sh.cx[wave] = readlane_d(cv[K - 1], 63);
    sh.ax[wave] = readlane_d(av[0], 0);
    wg_barrier();
    const double cx_prev = (wave > 0) ? sh.cx[wave - 1] : 0.0;
    const double ax_next = (wave < W - 1) ? sh.ax[wave + 1 < W ? wave + 1 : wave] : 0.0;
    cprev = (lane == 0) ? cx_prev : cprev;
    anext = (lane == 63) ? ax_next : anext;
  } else {
    cprev = (lane == 0) ? 0.0 : cprev;
    anext = (lane == 63) ? 0.0 : anext;
  }
  const dd p_left = two_prod(av[0], cprev);        // couples the chunk to the row before it
  const dd p_right = two_prod(anext, cv[K - 1]);   // ... and to the row after it
  // Determinants of the chunk's rows: A of all of them, Cd without the last,
  // Bd without the first, Dd without both (three-term recurrences in the rows)
  dd A = dd_from(bv[0]), Cd = dd_from(1.0), Bd = dd_from(1.0), Dd = dd_from(0.0);
#pragma unroll
  for (int t = 1; t < K; t++) {
    const dd np = dd_neg(two_prod(av[t], cv[t - 1]));
    const dd An = dd_add(dd_mul_d(A, bv[t]), dd_mul(np, Cd));
    const dd Bn = dd_add(dd_mul_d(Bd, bv[t]), dd_mul(np, Dd));
    Cd = A;
    A = An;
    Dd = Bd;
    Bd = Bn;
    // every second row (the last is one): the product of four rows overflows at
    // 1e77, of two where a row's own products do
    if (t % 2 == 1) norm4(A, Cd, Bd, Dd);
  }
  if constexpr (K == 1) norm4(A, Cd, Bd, Dd);
  // Adjacent chunks combine as a 2x2 product, whichever side's matrix carries
  // the coupling: the prefix form T = [[A, C], [-p_left B, -p_left D]] gives
  // the pivot of the last row before a chunk, T00 / T01; the suffix form
  // R = [[A, -p_right C], [B, -p_right D]] the pivot (from below) of the first
  // row after it, R00 / R10.
  // (One after the other, with the scheduler held between them: together
  // they would double the registers of the setup, which set the occupancy of
  // the small variants.)
  dd up = dd_from(1.0), vn = dd_from(1.0);  // no coupling at the two ends: p = 0
  {
    dd T[4] = {A, Cd, dd_neg(dd_mul(p_left, Bd)), dd_neg(dd_mul(p_left, Dd))};
#pragma unroll
    for (int lev = 0; lev < 6; lev++) {
      const int s = 1 << lev;
      dd Tp[4];
#pragma unroll
      for (int e = 0; e < 4; e++) Tp[e] = shfl_up_dd(T[e], s);
      if (lane >= s) mat_mul_norm(Tp, T, T);
    }
    dd pr0 = dd_from(1.0), pr1 = dd_from(0.0);  // row 0 of the product before this wave
    if constexpr (W > 1) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        sh.Mx[wave][e][0] = readlane_d(T[e].h, 63);
        sh.Mx[wave][e][1] = readlane_d(T[e].l, 63);
      }
      wg_barrier();
      for (int v = 0; v < wave; v++) {
        const dd Mv[4] = {{sh.Mx[v][0][0], sh.Mx[v][0][1]}, {sh.Mx[v][1][0], sh.Mx[v][1][1]},
                          {sh.Mx[v][2][0], sh.Mx[v][2][1]}, {sh.Mx[v][3][0], sh.Mx[v][3][1]}};
        row_times_mat(pr0, pr1, Mv);
      }
      wg_barrier();  // Mx is written again below
    }
#pragma unroll
    for (int e = 0; e < 4; e++) T[e] = shfl_up_dd(T[e], 1);
    if (lane > 0) row_times_mat(pr0, pr1, T);
    if (tid > 0) up = dd_div(pr0, pr1);
  }
  __builtin_amdgcn_sched_barrier(0);
  {
    dd R[4] = {A, dd_neg(dd_mul(p_right, Cd)), Bd, dd_neg(dd_mul(p_right, Dd))};
#pragma unroll
    for (int lev = 0; lev < 6; lev++) {
      const int s = 1 << lev;
      dd Rn[4];
#pragma unroll
      for (int e = 0; e < 4; e++) Rn[e] = shfl_down_dd(R[e], s);
      if (lane + s < 64) mat_mul_norm(R, Rn, R);
    }
    dd sc0 = dd_from(1.0), sc1 = dd_from(0.0);  // column 0 of the product after this wave
    if constexpr (W > 1) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        sh.Mx[wave][e][0] = readlane_d(R[e].h, 0);
        sh.Mx[wave][e][1] = readlane_d(R[e].l, 0);
      }
      wg_barrier();
      for (int v = W - 1; v > wave; v--) {
        const dd Mv[4] = {{sh.Mx[v][0][0], sh.Mx[v][0][1]}, {sh.Mx[v][1][0], sh.Mx[v][1][1]},
                          {sh.Mx[v][2][0], sh.Mx[v][2][1]}, {sh.Mx[v][3][0], sh.Mx[v][3][1]}};
        mat_times_col(Mv, sc0, sc1);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) R[e] = shfl_down_dd(R[e], 1);
    if (lane < 63) mat_times_col(R, sc0, sc1);
    if (tid < P - 1) vn = dd_div(sc0, sc1);
  }
  __builtin_amdgcn_sched_barrier(0);

  // Rows of the inverse (f, h and G_ii above).  The pivots stay in
  // double-double through the chunk: u_i + v_i - b_i cancels when the columns
  // fall off slowly, and an error of f shared by like rows is multiplied by
  // the fall-off length and by N.
  {
    dd sl[K];  // u_t - b_t
#pragma unroll
    for (int t = 0; t < K; t++) {
      const dd p = (t == 0) ? p_left : two_prod(av[t], cv[t > 0 ? t - 1 : 0]);
      sl[t] = dd_neg(dd_div(p, up));
      up = dd_add(dd_from(bv[t]), sl[t]);
      if (!(up.h > 0.0) || !isfinite(up.h)) bad |= ST_PIVOT;
      h[t] = -dd_quot(cv[t], up);
    }
#pragma unroll
    for (int t = K - 1; t >= 0; t--) {
      const dd p = (t == K - 1) ? p_right : two_prod(av[t + 1 < K ? t + 1 : 0], cv[t]);
      vn = dd_add(dd_from(bv[t]), dd_neg(dd_div(p, vn)));
      f[t] = -dd_quot(av[t], vn);
      gi[t] = dd_add(sl[t], vn);
    }
  }
}

}  // namespace scft
