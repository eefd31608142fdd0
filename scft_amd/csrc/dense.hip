// dense.hip -- the march of the smallest meshes (up to 64 unknowns) on the FP64
// matrix cores, for both steppers.
//
// With so few unknowns a step q <- T q is a dense 32 x 32 or 64 x 64 product,
// and the scans of march.hip spend their time on the chain of a step (0.145 us
// whatever the size).  Here the contour is cut into blocks of 64 steps:
//
//   1. T, one column per lane: elimination of D (implicit Euler: T = D^-1 A) or
//      of the complex stage matrix S (IRK4: T = I - dt Re(omega S^-1 D')), then
//      one refinement with the residual in double-double, so that T is held as
//      a leading part and a remainder, good to ~2^-100.
//   2. The powers T^2, T^4 .. T^64 by squaring.  A power keeps its remainder:
//      with P = Ph + Pm, Ph the leading 22 bits, Ph Ph is exact in the
//      accumulators (v_mfma_f64_16x16x4f64) and Ph Pm + Pm P is 2^-22 of it, so
//      the square comes out to ~2^-75.  (Squares rounded to 53 bits, and rows of
//      A and D rounded to doubles, would repeat their roundings N times over:
//      phi as far off as the scan march's, or twice.)
//   3. The first 64 columns q_0 .. q_63, doubled with the powers as they come:
//      wave w of four holds columns 16 w .. 16 w + 15, and applies T^16 and T^32
//      as its number says, so no wave waits for another.
//   4. Blocks: q_{j+64} = T^64 q_j.  The accumulator of the product (element e
//      of lane l of row tile t: row 16 t + l / 16 + 4 e, column l % 16) is the
//      operand of the next one (k = 4 s + l / 16, s = 4 t + e): the march never
//      leaves the registers.  The first half is stored, the second pairs with it
//      as in march.hip; the pairing weight of a lane is that of its column.
//
// One workgroup of four waves per instance, instances from a queue.  Bound by
// the matrix pipe of its CU: 16 (64) products of 64 cycles per wave and block.
// One instance against the scan march, us: n = 31, N = 2048: 312 -> 51; n = 59,
// N = 2048: 312 -> 175; IRK4 n = 31, N = 512: 178 -> 49.  phi is within a few
// 1e-16 of an extended-precision march (the scan marches: 1e-14 .. 2e-13).
#include "scft_internal.h"
#include "device_common.h"
#include "march_rows.h"

namespace scft {

typedef double d4 __attribute__((ext_vector_type(4)));

template <int NP, bool IRK>
struct DenseShared {
  double H[NP][NP + 2], L[NP][NP + 2];  // the power: leading part and remainder
  double X[NP][NP + 2];                 // setup: residuals (IRK4: real and imaginary parts)
  double Y[IRK ? NP : 1][NP + 2];
  double row[6][NP];                    // right-hand side: A (IE) or dt D' (IRK4), leading
                                        // parts and remainders of the three diagonals
  double sys[12][NP];                   // D, or the real and imaginary parts of S, likewise
  double lu[6][NP];                     // its elimination
  double part[4][NP];                   // density by wave
  double mx[4];                         // largest entry of the power by wave
  unsigned bad;
};

// a b + (the sum so far) in double-double, b a double
__device__ __forceinline__ void dd_acc(dd& s, dd a, double b) {
  s = dd_add(s, dd_mul_d(a, b));
}

// Rows of the mass matrix A and of dt D' = dt (B + C) for unknown u, as
// assemble_split has them but in double-double: the powers repeat a rounding of
// an entry N times over.
struct RowDD {
  dd v[6];  // A: sub-, main, super-diagonal; dt D' likewise
};
__device__ __forceinline__ RowDD assemble_dd(const double* __restrict__ x,
                                             const double* __restrict__ w, const InstDesc& d,
                                             int u, double dt) {
  const bool live = u < d.n;
  const int i = live ? u + 1 : 1;
  const bool has_r = i + 1 < d.M;
  const dd zero = dd_from(0.0);
  const dd hl = two_sum(x[i], -x[i - 1]), hr = has_r ? two_sum(x[i + 1], -x[i]) : zero;
  const double wi = live ? w[live ? u : 0] : 0.0;
  const dd Al = dd_div(hl, dd_from(6.0)), Ar = dd_div(hr, dd_from(6.0));
  const dd Ad = dd_scale(dd_add(Al, Ar), 2.0);
  const dd Bl = dd_neg(dd_div(dd_from(1.0), hl));
  const dd Br = has_r ? dd_neg(dd_div(dd_from(1.0), hr)) : zero;
  dd Cl, Cd, Cr;
  if (d.cmat == 0) {
    Cl = dd_mul_d(Al, wi);
    Cd = dd_mul_d(Ad, wi);
    Cr = dd_mul_d(Ar, wi);
  } else {
    const double wl = (u > 0 && live) ? w[u - 1] : d.wall0;
    const double wr = (u + 1 < d.n) ? w[u + 1] : d.wallL;
    const dd sl = two_sum(wl, wi), sr = two_sum(wr, wi), w2 = dd_from(2.0 * wi);
    Cl = dd_scale(dd_mul(Al, sl), 0.5);
    Cr = dd_scale(dd_mul(Ar, sr), 0.5);
    Cd = dd_scale(dd_add(dd_mul(Al, dd_add(sl, w2)), dd_mul(Ar, dd_add(sr, w2))), 0.5);
  }
  const bool in_l = live && u > 0, in_r = live && u < d.n - 1;
  RowDD r;
  r.v[0] = in_l ? Al : zero;
  r.v[1] = live ? Ad : zero;
  r.v[2] = in_r ? Ar : zero;
  r.v[3] = in_l ? dd_scale(dd_add(Bl, Cl), dt) : zero;
  r.v[4] = live ? dd_scale(dd_add(dd_neg(dd_add(Bl, Br)), Cd), dt) : zero;
  r.v[5] = in_r ? dd_scale(dd_add(Br, Cr), dt) : zero;
  return r;
}
// The right-hand side's diagonals and the system's: D = A + dt D' for implicit
// Euler; S = A + dt lambda D', lambda = 1/4 + i sqrt3/12, for IRK4 (irk4.hip).
// Padding rows are the identity with a zero right-hand side.
template <int NP, bool IRK>
__device__ __forceinline__ void stage_rows(DenseShared<NP, IRK>& sh, const double* x,
                                           const double* w, const InstDesc& d, const double dt,
                                           const int tid) {
  const dd lam_im = {0.14433756729740643, 8.362570184839086e-18};  // sqrt(3)/12
  if (tid < NP) {
    const RowDD r = assemble_dd(x, w, d, tid, dt);
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const dd rhs = IRK ? dd_neg(r.v[3 + e]) : r.v[e];
      dd re = dd_add(r.v[e], IRK ? dd_scale(r.v[3 + e], 0.25) : r.v[3 + e]);
      if (e == 1 && tid >= d.n) re = dd_from(1.0);
      sh.row[e][tid] = rhs.h;
      sh.row[3 + e][tid] = rhs.l;
      sh.sys[e][tid] = re.h;
      sh.sys[3 + e][tid] = re.l;
      if constexpr (IRK) {
        const dd im = dd_mul(lam_im, r.v[3 + e]);
        sh.sys[6 + e][tid] = im.h;
        sh.sys[9 + e][tid] = im.l;
      }
    }
  }
  if (tid == 0) sh.bad = 0;
  wg_barrier();
}

// 1 / u to ~2 ulp: the elimination only has to be good enough for the
// refinement
__device__ __forceinline__ double recip(double u) {
  double r = __builtin_amdgcn_rcp(u);
  r = fma(fma(-u, r, 1.0), r, r);
  return fma(fma(-u, r, 1.0), r, r);
}

// T in (H, L) for implicit Euler, D T = A; all 256 threads.
template <int NP, bool IRK>
__device__ void step_matrix_ie(DenseShared<NP, IRK>& sh, const double* x, const double* w,
                               const InstDesc& d, const double dt, const int tid) {
#pragma clang fp contract(off)
  stage_rows<NP, IRK>(sh, x, w, d, dt, tid);
  if (tid < 64) {  // every lane follows the pivots, lane 0 keeps them
    double inv = 0.0, cp = 0.0;
    unsigned bad = 0;
#pragma unroll 8
    for (int i = 0; i < NP; i++) {
      const double al = sh.sys[0][i] * inv;
      const double u = fma(-al, cp, sh.sys[1][i]);
      if (!(u > 0.0) || !isfinite(u)) bad = ST_PIVOT;
      inv = recip(u);
      cp = sh.sys[2][i];
      if (tid == 0) {
        sh.lu[0][i] = inv;
        sh.lu[1][i] = sh.sys[0][i] * inv;
        sh.lu[2][i] = cp * inv;
      }
    }
    if (tid == 0) sh.bad = bad;
  }
  wg_barrier();
  const int k = tid;
  if (k < NP) {
    double z = 0.0;
#pragma unroll 8
    for (int i = 0; i < NP; i++) {
      double r = 0.0;
      if (i == k - 1) r = sh.row[2][i];
      if (i == k) r = sh.row[1][i];
      if (i == k + 1) r = sh.row[0][i];
      z = fma(-sh.lu[1][i], z, r * sh.lu[0][i]);
      sh.X[i][k] = z;
    }
    z = 0.0;
#pragma unroll 8
    for (int i = NP - 1; i >= 0; i--) {
      z = fma(-sh.lu[2][i], z, sh.X[i][k]);
      sh.H[i][k] = z;
    }
  }
  wg_barrier();
  for (int e = tid; e < NP * NP; e += 256) {  // residual A - D T, entry by entry
    const int i = e / NP, c = e % NP;
    dd r = dd_from(0.0);
#pragma unroll
    for (int part = 0; part < 3; part++) {
      const int j = i + part - 1;
      const bool in = j >= 0 && j < NP;
      if (c == j) r = dd_add(r, {sh.row[part][i], sh.row[3 + part][i]});
      dd_acc(r, {sh.sys[part][i], sh.sys[3 + part][i]}, in ? -sh.H[in ? j : 0][c] : 0.0);
    }
    sh.X[i][c] = r.h * sh.lu[0][i];
  }
  wg_barrier();
  if (k < NP) {
    double z = 0.0;
#pragma unroll 8
    for (int i = 0; i < NP; i++) {
      z = fma(-sh.lu[1][i], z, sh.X[i][k]);
      sh.X[i][k] = z;
    }
    z = 0.0;
#pragma unroll 8
    for (int i = NP - 1; i >= 0; i--) {
      z = fma(-sh.lu[2][i], z, sh.X[i][k]);
      const dd t = two_sum(sh.H[i][k], z);
      sh.H[i][k] = t.h;
      sh.L[i][k] = t.l;
    }
  }
  wg_barrier();
}

// T in (H, L) for IRK4: S z = -dt D' e_k and T e_k = e_k + Re((1 - i sqrt3) z).
template <int NP, bool IRK>
__device__ void step_matrix_irk4(DenseShared<NP, IRK>& sh, const double* x, const double* w,
                                 const InstDesc& d, const double dt, const int tid) {
#pragma clang fp contract(off)
  const dd root3 = {1.7320508075688772, 1.0035084221806903e-16};
  stage_rows<NP, IRK>(sh, x, w, d, dt, tid);
  if (tid < 64) {
    cd inv = {0.0, 0.0}, cp = {0.0, 0.0};
    unsigned bad = 0;
#pragma unroll 4
    for (int i = 0; i < NP; i++) {
      const cd sa = {sh.sys[0][i], sh.sys[6][i]};
      const cd u = c_fnma(c_mul(sa, inv), cp, {sh.sys[1][i], sh.sys[7][i]});
      const double m2 = u.re * u.re + u.im * u.im;
      if (!(m2 > 0.0) || !isfinite(m2)) bad = ST_PIVOT;
      const double im2 = recip(m2);
      inv = {u.re * im2, -u.im * im2};
      cp = {sh.sys[2][i], sh.sys[8][i]};
      const cd al = c_mul(sa, inv), ga = c_mul(cp, inv);
      if (tid == 0) {
        sh.lu[0][i] = inv.re;
        sh.lu[1][i] = inv.im;
        sh.lu[2][i] = al.re;
        sh.lu[3][i] = al.im;
        sh.lu[4][i] = ga.re;
        sh.lu[5][i] = ga.im;
      }
    }
    if (tid == 0) sh.bad = bad;
  }
  wg_barrier();
  const int k = tid;
  if (k < NP) {
    cd z = {0.0, 0.0};
#pragma unroll 4
    for (int i = 0; i < NP; i++) {
      double r = 0.0;
      if (i == k - 1) r = sh.row[2][i];
      if (i == k) r = sh.row[1][i];
      if (i == k + 1) r = sh.row[0][i];
      z = c_fnma({sh.lu[2][i], sh.lu[3][i]}, z, {r * sh.lu[0][i], r * sh.lu[1][i]});
      sh.X[i][k] = z.re;
      sh.Y[i][k] = z.im;
    }
    z = {0.0, 0.0};
#pragma unroll 4
    for (int i = NP - 1; i >= 0; i--) {
      z = c_fnma({sh.lu[4][i], sh.lu[5][i]}, z, {sh.X[i][k], sh.Y[i][k]});
      sh.H[i][k] = z.re;
      sh.L[i][k] = z.im;
    }
  }
  wg_barrier();
  for (int e = tid; e < NP * NP; e += 256) {  // residual -dt D' - S z, entry by entry
    const int i = e / NP, c = e % NP;
    dd re = dd_from(0.0), im = dd_from(0.0);
#pragma unroll
    for (int part = 0; part < 3; part++) {
      const int j = i + part - 1;
      const bool in = j >= 0 && j < NP;
      if (c == j) re = dd_add(re, {sh.row[part][i], sh.row[3 + part][i]});
      const double zr = in ? sh.H[in ? j : 0][c] : 0.0, zi = in ? sh.L[in ? j : 0][c] : 0.0;
      const dd sr = {sh.sys[part][i], sh.sys[3 + part][i]};
      const dd si = {sh.sys[6 + part][i], sh.sys[9 + part][i]};
      dd_acc(re, sr, -zr);
      dd_acc(re, si, zi);
      dd_acc(im, sr, -zi);
      dd_acc(im, si, -zr);
    }
    const cd r = c_mul({re.h, im.h}, {sh.lu[0][i], sh.lu[1][i]});
    sh.X[i][c] = r.re;
    sh.Y[i][c] = r.im;
  }
  wg_barrier();
  if (k < NP) {
    cd z = {0.0, 0.0};
#pragma unroll 4
    for (int i = 0; i < NP; i++) {
      z = c_fnma({sh.lu[2][i], sh.lu[3][i]}, z, {sh.X[i][k], sh.Y[i][k]});
      sh.X[i][k] = z.re;
      sh.Y[i][k] = z.im;
    }
    z = {0.0, 0.0};
#pragma unroll 4
    for (int i = NP - 1; i >= 0; i--) {
      z = c_fnma({sh.lu[4][i], sh.lu[5][i]}, z, {sh.X[i][k], sh.Y[i][k]});
      dd t = dd_add(dd_from(sh.H[i][k]), dd_mul_d(root3, sh.L[i][k]));
      t = dd_add(t, dd_from(z.re + root3.h * z.im));
      t = dd_add(dd_from(i == k ? 1.0 : 0.0), t);
      sh.H[i][k] = t.h;
      sh.L[i][k] = t.l;
    }
  }
  wg_barrier();
}

// The leading bits of v (sg = 1.5 * 2^52 times their unit)
__device__ __forceinline__ double lead_bits(double v, double sg) {
#pragma clang fp contract(off)
  return (v + sg) - sg;
}

template <int NP, bool IRK>
__device__ void dense_one(const MarchArgs& a, const int inst, const unsigned st0,
                          double* __restrict__ slab, DenseShared<NP, IRK>& sh, const int tid) {
  constexpr int KS = NP / 4, RT = NP / 16;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const InstDesc d = a.desc[inst];
  const int n = __builtin_amdgcn_readfirstlane(d.n);
  const int N = __builtin_amdgcn_readfirstlane(d.N);
  const double dt = 1.0 / N;
  const double* __restrict__ pw = a.pw + d.po;
  if constexpr (IRK)
    step_matrix_irk4<NP, IRK>(sh, a.x + d.xo, a.w + d.uo, d, dt, tid);
  else
    step_matrix_ie<NP, IRK>(sh, a.x + d.xo, a.w + d.uo, d, dt, tid);

  // largest entry: the unit of the leading bits
  double mx = 0.0;
  for (int e = tid; e < NP * NP; e += 256) mx = fmax(mx, fabs(sh.H[e / NP][e % NP]));
  auto share_max = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off));
    sh.mx[wave] = readlane_d(mx, 0);
  };
  share_max();
  wg_barrier();

  double Q[KS];  // rows 4 s + kq of column 16 wave + col (all waves start from column col)
#pragma unroll
  for (int s = 0; s < KS; s++) Q[s] = (col == 0 && 4 * s + kq < n) ? 1.0 : 0.0;
  double A[RT][KS];
  auto load_power = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int s = 0; s < KS; s++) A[t][s] = sh.H[16 * t + col][4 * s + kq];
  };
  auto apply = [&](const double (&q)[KS], double (&out)[KS]) __attribute__((always_inline)) {
    d4 acc[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
      for (int t = 0; t < RT; t++)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[t][s], q[s], acc[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) out[4 * t + e] = acc[t][e];
  };

  for (int c = 1; c < DENSE_COLS; c *= 2) {
    // columns: c .. 2c - 1 of the tile from 0 .. c - 1, then whole tiles
    load_power();
    double Z[KS];
    apply(Q, Z);
#pragma unroll
    for (int s = 0; s < KS; s++) {
      if (c < 16) {
        const double z = (c == 1) ? row_shr<1>(Z[s]) : (c == 2) ? row_shr<2>(Z[s])
                       : (c == 4) ? row_shr<4>(Z[s]) : row_shr<8>(Z[s]);
        Q[s] = (col >= c && col < 2 * c) ? z : Q[s];
      } else {
        Q[s] = (wave & (c / 16)) ? Z[s] : Q[s];
      }
    }
    // the square
    const double m4 = fmax(fmax(sh.mx[0], sh.mx[1]), fmax(sh.mx[2], sh.mx[3]));
    const double sg = (m4 > 0.0 && isfinite(m4)) ? ldexp(1.5, ilogb(m4) + 31) : 0.0;
    constexpr int NT = NP == 64 ? 4 : 1;  // tiles of this wave: one row tile
    const int rt = NP == 64 ? wave : wave >> 1, ct0 = NP == 64 ? 0 : wave & 1;
    d4 hi[NT], lo[NT];
#pragma unroll
    for (int u = 0; u < NT; u++) hi[u] = lo[u] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KS; s++) {
      double ah0 = A[0][s];  // row tile rt of the power just applied
#pragma unroll
      for (int t = 1; t < RT; t++) ah0 = (rt == t) ? A[t][s] : ah0;
      const double al0 = sh.L[16 * rt + col][4 * s + kq];
      const double ah = lead_bits(ah0, sg), am = (ah0 - ah) + al0;
#pragma unroll
      for (int u = 0; u < NT; u++) {
        const double bh0 = sh.H[4 * s + kq][16 * (ct0 + u) + col];
        const double bl0 = sh.L[4 * s + kq][16 * (ct0 + u) + col];
        const double bh = lead_bits(bh0, sg), bm = (bh0 - bh) + bl0;
        hi[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ah, bh, hi[u], 0, 0, 0);
        lo[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ah, bm, lo[u], 0, 0, 0);
        lo[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(am, bh0, lo[u], 0, 0, 0);
      }
    }
    wg_barrier();  // every wave has read the power it squares
    mx = 0.0;
#pragma unroll
    for (int u = 0; u < NT; u++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const dd t = two_sum(hi[u][e], lo[u][e]);
        const int i = 16 * rt + kq + 4 * e, j = 16 * (ct0 + u) + col;
        sh.H[i][j] = t.h;
        sh.L[i][j] = t.l;
        mx = fmax(mx, fabs(t.h));
      }
    share_max();
    wg_barrier();
  }

  // ------------------------------------------------------------------ march
  load_power();
  const int blocks = N / DENSE_COLS;
  const __amdgpu_buffer_rsrc_t srsrc =
      slab_rsrc(slab, static_cast<unsigned>(a.slab_stride * sizeof(double)));
  constexpr unsigned BLOCK_BYTES = DENSE_COLS * NP * 8u;
  const unsigned mine = static_cast<unsigned>(wave * KS * 512 + lane * 8);
  for (int b = 0; b < blocks / 2; b++) {
#pragma unroll
    for (int s = 0; s < KS; s++)
      slab_store(Q[s], srsrc, mine + s * 512u, static_cast<unsigned>(b) * BLOCK_BYTES);
    double Z[KS];
    apply(Q, Z);
#pragma unroll
    for (int s = 0; s < KS; s++) Q[s] = Z[s];
  }
  vmem_drain();  // the second half reads what other waves stored
  wg_barrier();
  // step j = 64 b + 16 wave + col pairs with step N - j, held by another lane
  double acc[KS], cur[KS];
  const int j0 = N / 2 + 16 * wave + col;
  const bool self = j0 == N / 2;  // step N/2 pairs with itself
  const int jp = self ? N / 2 - DENSE_COLS : N - j0;  // (its loads: in range, not used)
  unsigned off = static_cast<unsigned>(jp / DENSE_COLS) * BLOCK_BYTES +
                 static_cast<unsigned>((jp / 16 % 4) * KS * 512 + (kq * 16 + jp % 16) * 8);
  const unsigned next_off = self ? 0u : BLOCK_BYTES;  // self: already the next block's
  const double wgt = pw[(col & 1) ? 1 : (col & 2) ? 2 : (col & 4) ? 4 : col ? 8 : 16];
#pragma unroll
  for (int s = 0; s < KS; s++) {
    cur[s] = slab_load(srsrc, off + s * 512u, 0u);
    acc[s] = 0.0;
  }
  const double w0 = pw[0];
  for (int b = blocks / 2; b < blocks; b++) {
    double nxt[KS];
    off -= (b == blocks / 2) ? next_off : BLOCK_BYTES;
    if (b + 1 < blocks) {
#pragma unroll
      for (int s = 0; s < KS; s++) nxt[s] = slab_load(srsrc, off + s * 512u, 0u);
    }
    const bool me = self && b == blocks / 2;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const double c = me ? w0 : wgt, p = me ? Q[s] : cur[s];
      acc[s] = fma(c * Q[s], p, acc[s]);
    }
    double Z[KS];
    apply(Q, Z);
#pragma unroll
    for (int s = 0; s < KS; s++) {
      Q[s] = Z[s];
      cur[s] = nxt[s];
    }
  }
  if (wave == 0 && col == 0) {  // step N with step 0
    const double ce = pw[N / 2];
#pragma unroll
    for (int s = 0; s < KS; s++) acc[s] = fma(ce, Q[s], acc[s]);
  }
#pragma unroll
  for (int s = 0; s < KS; s++) {
#pragma unroll
    for (int off2 = 8; off2 >= 1; off2 >>= 1) acc[s] += __shfl_xor(acc[s], off2);
    if (col == 0) sh.part[wave][4 * s + kq] = acc[s];
  }
  wg_barrier();

  // --------------------------------------------------------------- residual
  if (wave == 0) {
    unsigned bad = sh.bad;
    double m = 0.0;
    if (lane < n) {
      const double phi = (sh.part[0][lane] + sh.part[1][lane]) +
                         (sh.part[2][lane] + sh.part[3][lane]);
      const double res = phi - a.phit[d.uo + lane];
      a.r[d.uo + lane] = res;
      if (a.phi) a.phi[d.uo + lane] = phi;
      if (!isfinite(res)) bad |= ST_NAN;
      m = fabs(res);
    }
#pragma unroll
    for (int off2 = 32; off2 >= 1; off2 >>= 1) {
      m = fmax(m, __shfl_xor(m, off2));
      bad |= __shfl_xor(bad, off2);
    }
    a.rnorm[inst] = (bad & ST_NAN) ? __builtin_nan("") : m;
    a.status[inst] = st0 | bad;
  }
}

// The work queue of march_kernel.
template <int NP, bool IRK>
__global__ void __launch_bounds__(256, NP == 32 ? 3 : 1) dense_kernel(MarchArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  DenseShared<NP, IRK>& sh = *reinterpret_cast<DenseShared<NP, IRK>*>(lds);
  __shared__ int s_next;
  const int tid = threadIdx.x;
  double* slab = a.slabs + (long long)blockIdx.x * a.slab_stride;
  for (int it = blockIdx.x; it < a.n_items; it = next_item(a, tid, &s_next)) {
    const int inst = __builtin_amdgcn_readfirstlane(a.items[it]);
    const unsigned st = __builtin_amdgcn_readfirstlane(a.status[inst]);
    if (st & ST_DONE_MASK) continue;
    dense_one<NP, IRK>(a, inst, st, slab, sh, tid);
  }
}

// ------------------------------------------------------------------ dispatch
static const void* dense_fn(int np, bool irk4) {
  if (np == 32)
    return irk4 ? reinterpret_cast<const void*>(&dense_kernel<32, true>)
                : reinterpret_cast<const void*>(&dense_kernel<32, false>);
  return irk4 ? reinterpret_cast<const void*>(&dense_kernel<64, true>)
              : reinterpret_cast<const void*>(&dense_kernel<64, false>);
}
static size_t dense_lds(int np, bool irk4) {
  if (np == 32) return irk4 ? sizeof(DenseShared<32, true>) : sizeof(DenseShared<32, false>);
  return irk4 ? sizeof(DenseShared<64, true>) : sizeof(DenseShared<64, false>);
}

hipError_t launch_dense(int np, bool irk4, const MarchArgs& a, int grid, hipStream_t s) {
  MarchArgs arg = a;
  void* params[] = {&arg};
  return hipLaunchKernel(dense_fn(np, irk4), dim3(grid), dim3(256), params, dense_lds(np, irk4),
                         s);
}

int dense_max_grid(int np, bool irk4) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, dense_fn(np, irk4), 256,
                                                   dense_lds(np, irk4)) != hipSuccess)
    return 0;
  return per * cus;
}

}  // namespace scft
