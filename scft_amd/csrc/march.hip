// march.hip -- the hot path of the SCFT field evaluation on gfx950, FP64.
//
// One workgroup of W wavefronts (P = 64 W lanes) evaluates one instance at a
// time; lane p owns K consecutive unknowns, so n <= P K.  Per instance:
//
//   1. assembly  (1D_FEM.c:84-186, simple_FEM_1D_transient.m:28-79,
//                 scft.cc:641-651): every lane builds its own rows of
//                 D = A + dt (B + C) and of the right-hand-side operator A from
//                 the node coordinates and the field (no atomics: a row reads
//                 its two adjacent elements itself).
//   2. factor:   D is tridiagonal, so its inverse G falls off by fixed factors
//                away from the diagonal: G_ii = 1 / (u_i + v_i - b_i),
//                G_ij = f_i G_{i-1,j} below it and h_i G_{i+1,j} above it, with
//                f_i = -a_i / v_i, h_i = -c_i / u_i and u, v the elimination
//                pivots from above and from below.  The pivots are ratios of
//                determinants of leading and trailing blocks; a lane takes the
//                four determinants its chunk needs, and a prefix and a suffix
//                product of 2x2 matrices over the lanes (and a fold over waves)
//                give the pivots at its two ends.  All of it in double-double,
//                once per evaluation (20-40 us).
//   3. march:    N implicit-Euler steps D q^{j+1} = A q^j (1D_FEM.c:208-228,
//                step count of DEALII_SCFT/drivescft.cc:130) as q = G (A q): a
//                recurrence downwards and one upwards that do not wait for each
//                other.  Each is split into a lane-local pass, a scan of the
//                lanes' affine maps over the wave (four DPP row levels, then
//                two cross-row levels: broadcast DPP moves forward, LDS-
//                crossbar permutes backward; every multiplier is fixed per
//                instance, so a level costs one FMA per step), a fold over
//                waves through LDS, and the rows from the two inflows.
//   4. density:  phi_i = sum_j c_j q_j(i) q_{N-j}(i) (drivescft.cc:184-193 with
//                romint.c's weights, symmetric in j).  Slabs q_0..q_{N/2-1}
//                stream to HBM (coalesced, raw-buffer stores and loads with
//                non-temporal hints); from step N/2 on each new slab is paired
//                with slab N-j.  Either every slab is kept (SEG = 1: loaded a
//                few steps ahead through a register ring), or every fourth, and
//                the second half recomputes the others, four at a time into LDS
//                (SEG = 4).
//   5. residual: r = phi - phi_t (1D_FEM.c:274-277), ||r||_inf per instance.
//
// What bounds it, and what that gave against a two-sweep solve (elimination
// down, substitution up, every slab kept) on the same variants:
//   * one instance, or few: the chain of a step.  The two-sweep solve scans
//     twice and meets twice at a barrier; here once (one exchange through LDS
//     costs 0.1-0.2 us).  A step of 255 / 1023 / 2047 / 4095 unknowns takes
//     0.20 / 0.37 / 0.49 / 0.69 us (0.24 / 0.49 / 0.60 / 0.81 before).
//   * a full chip: HBM.  Stores and loads of all slabs reach ~5.1 TB/s
//     whatever the variant (640 G node-steps/s), and at that traffic the clock
//     falls to 1.6 GHz.  With every fourth slab and 1.375 N steps the vector
//     units bound it (72% busy at 1.9 GHz): 970-1120 G node-steps/s.
//   * accuracy: the rows of G are computed in double-double and rounded once.
//     Where neighbours couple negatively (dt > h^2 / 6) every weight is positive
//     and nothing cancels; where they do not, f and h are negative, but below
//     0.27 in size on a uniform mesh, so a row reaches a few neighbours only.
//     phi against an extended-precision march, uniform, m = 4095: 1.1e-14 for
//     N = 128, 5e-14 for N = 4096 (2.9e-13 and 2.1e-12 with pivots rounded to
//     double).
// No MFMA: nothing here is a dense contraction.
#include "scft_internal.h"
#include "device_common.h"
#include "march_rows.h"

namespace scft {

template <int K, int W, int SEG>
__device__ void march_one(const MarchArgs& a, const int inst, const unsigned st0,
                          double* __restrict__ slab, MarchShared<W>& sh,
                          double* __restrict__ seg_lds, const int tid) {
  constexpr int P = 64 * W;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const InstDesc d = a.desc[inst];
  const int n = __builtin_amdgcn_readfirstlane(d.n);
  const int N = __builtin_amdgcn_readfirstlane(d.N);
  const int M = __builtin_amdgcn_readfirstlane(d.M);
  const double dt = 1.0 / N;
  const double* __restrict__ x = a.x + d.xo;
  const double* __restrict__ w = a.w + d.uo;
  const double* __restrict__ pw = a.pw + d.po;
  const int cmat = __builtin_amdgcn_readfirstlane(d.cmat);
  const int u0 = tid * K;

  // The pairing weight of step j depends on how often 2 divides j, up to four
  // times (the five trapezoid levels), except for the last step: six values
  // in LDS instead of the table of N/2 + 1, which at N = 8192 kept all but
  // four workgroups off a CU.  (Small N never read the higher classes.)
  const int half = N >> 1;
  if (tid < 6) {
    const int t = (tid == 5) ? half : 1 << tid;
    sh.cw[tid] = pw[t < half ? t : half];
  }
  wg_barrier();
  auto weight = [&](const int i) __attribute__((always_inline)) {  // of step N/2 + i
    return sh.cw[(i == half) ? 5 : min(__builtin_ctz(half + i), 4)];
  };

  // ---------------------------------------------------------------- assembly
  double av[K], bv[K], cv[K], ra[K], rc[K];
#pragma unroll
  for (int t = 0; t < K; t++) {
    const Row rw = assemble_row(x, w, n, M, u0 + t, dt, cmat, d.wall0, d.wallL);
    av[t] = rw.a;
    bv[t] = rw.b;
    cv[t] = rw.c;
    ra[t] = rw.ra;
    rc[t] = rw.rc;
  }

  // ------------------------------------------------------------ factor scan
  unsigned bad = 0;
  double f[K], h[K], rd[K];
  {
    dd gi[K];
    inverse_rows<K, W>(av, bv, cv, sh, tid, f, h, gi, bad);
#pragma unroll
    for (int t = 0; t < K; t++) {
      ra[t] = dd_quot(ra[t], gi[t]);
      rc[t] = dd_quot(rc[t], gi[t]);
      rd[t] = 2.0 * (ra[t] + rc[t]);
    }
  }

  // -------------------------------------------- scan constants of the march
  // A lane's chunk is an affine map in each direction: F leaves it as
  // Af F_in + B, Y leaves it (upwards) as Gb Y_in + C, with Af = prod f and
  // Gb = prod h fixed for the instance.  The two scans of a step run side by
  // side: a Hillis-Steele scan inside each 16-lane row (DPP row_shr / row_shl
  // by 1, 2, 4, 8), then two row-to-row levels (forward: DPP row_bcast:15 and
  // row_bcast:31; backward: ds_bpermute from the first lane of the next
  // rows), then (several waves) one fold over the wave totals of both in
  // LDS.  All multipliers are precomputed here; a step costs one FMA per level.
  const int rl = lane & 15;   // lane within its row
  const int row = lane >> 4;  // row within the wave
  // Pf_t = f_0 .. f_t and Ph_t = h_t .. h_{K-1}: what the inflows add to row t
  double Pf[K], Ph[K];
  Pf[0] = f[0];
  Ph[K - 1] = h[K - 1];
#pragma unroll
  for (int t = 1; t < K; t++) {
    Pf[t] = Pf[t - 1] * f[t];
    Ph[K - 1 - t] = Ph[K - t] * h[K - 1 - t];
  }
  double Af = Pf[K - 1], Gb = Ph[0];
  double mf[4], mb[4];
  {
    double Ap, Gp;
    Ap = row_shr<1>(Af); Gp = row_shl<1>(Gb);
    mf[0] = (rl >= 1) ? Af : 0.0; mb[0] = (rl + 1 < 16) ? Gb : 0.0;
    Af = (rl >= 1) ? Af * Ap : Af; Gb = (rl + 1 < 16) ? Gb * Gp : Gb;
    Ap = row_shr<2>(Af); Gp = row_shl<2>(Gb);
    mf[1] = (rl >= 2) ? Af : 0.0; mb[1] = (rl + 2 < 16) ? Gb : 0.0;
    Af = (rl >= 2) ? Af * Ap : Af; Gb = (rl + 2 < 16) ? Gb * Gp : Gb;
    Ap = row_shr<4>(Af); Gp = row_shl<4>(Gb);
    mf[2] = (rl >= 4) ? Af : 0.0; mb[2] = (rl + 4 < 16) ? Gb : 0.0;
    Af = (rl >= 4) ? Af * Ap : Af; Gb = (rl + 4 < 16) ? Gb * Gp : Gb;
    Ap = row_shr<8>(Af); Gp = row_shl<8>(Gb);
    mf[3] = (rl >= 8) ? Af : 0.0; mb[3] = (rl + 8 < 16) ? Gb : 0.0;
    Af = (rl >= 8) ? Af * Ap : Af; Gb = (rl + 8 < 16) ? Gb * Gp : Gb;
  }
  // Af = product over the row from its first lane to this lane, Gb = product
  // from this lane to the row's last lane; row totals as uniform scalars
  const double Arow0 = readlane_d(Af, 15), Arow1 = readlane_d(Af, 31);
  const double Arow2 = readlane_d(Af, 47), Arow3 = readlane_d(Af, 63);
  const double Grow0 = readlane_d(Gb, 0), Grow1 = readlane_d(Gb, 16);
  const double Grow2 = readlane_d(Gb, 32), Grow3 = readlane_d(Gb, 48);
  // DPP reads are made with every lane active: a DPP move in a conditional
  // arm runs under a partial EXEC mask and reads 0 from disabled lanes.
  const double Af_sh = row_shr<1>(Af), Gb_sh = row_shl<1>(Gb);
  const double Ashift = (rl > 0) ? Af_sh : 0.0;   // row product to lane-1
  const double Gshift = (rl < 15) ? Gb_sh : 0.0;  // row product from lane+1
  // products over whole rows before / after this lane's row
  const double Abefore = (row == 0) ? 1.0 : (row == 1) ? Arow0
                         : (row == 2) ? Arow0 * Arow1 : Arow0 * Arow1 * Arow2;
  const double Gafter = (row == 3) ? 1.0 : (row == 2) ? Grow3
                        : (row == 1) ? Grow2 * Grow3 : Grow1 * Grow2 * Grow3;
  // wave prefix over lanes 0..lane-1 and suffix over lane+1..63 (wave folds)
  const double Apre_m1 = ((rl > 0) ? Ashift : 1.0) * Abefore;
  // multipliers of the forward scan's two broadcast levels: rows 1 and 3 take
  // the prefix ending at lane 15 / 47 times their own row product up to the
  // lane; then rows 2 and 3 take the prefix ending at lane 31 times the
  // product from lane 32 up to the lane
  const double mf5 = Af;
  const double mf6 = (row == 3) ? Arow2 * Af : Af;
  // the backward scan's two cross-row levels, mirror images of those (DPP has
  // no downward broadcast: the values come through ds_bpermute): rows 0 and 2
  // take the suffix starting at lane 16 / 48 times their own row product
  // from the lane on; then rows 0 and 1 take the suffix starting at lane 32
  // times the product from the lane to lane 31.  0 for rows that do not take.
  const double mbA = (row == 0 || row == 2) ? Gb : 0.0;
  const double mbB = (row == 0) ? Gb * Grow1 : (row == 1) ? Gb : 0.0;
  const int srcA = ((row + 1) & 3) * 64;  // byte address of lane 16 (row + 1)
  const int srcB = 32 * 4;
  const double Gsuf_p1 = ((rl < 15) ? Gshift : 1.0) * Gafter;
  // h of the row left of the chunk, f of the row right of it
  double hl = __shfl_up(h[K - 1], 1), fr = __shfl_down(f[0], 1);
  // Fold multipliers.  The forward carry into this wave from the waves before
  // it is Z = sum_{v < wave} fz[v] Bw[v] with fz[v] = prod_{v < u < wave} Aw[u];
  // the backward carry from the waves after it is X = sum_{v > wave} fx[v] Cw[v]
  // with fx[v] = prod_{wave < u < v} Gw[u].  Fixed per instance (0 where the
  // wave does not read) and held as wave-uniform values, so a step reads all
  // wave totals at once: one LDS round trip instead of one per earlier wave.
  [[maybe_unused]] double fz[W], fx[W];
  if constexpr (W > 1) {
    sh.Aw[wave] = Arow0 * Arow1 * Arow2 * Arow3;
    sh.hx[wave] = readlane_d(h[K - 1], 63);
    sh.fx[wave] = readlane_d(f[0], 0);
    sh.Gw[wave] = Grow0 * Grow1 * Grow2 * Grow3;
    wg_barrier();
    const double hx_prev = (wave > 0) ? sh.hx[wave - 1] : 0.0;
    const double fx_next = (wave < W - 1) ? sh.fx[wave + 1 < W ? wave + 1 : wave] : 0.0;
    hl = (lane == 0) ? hx_prev : hl;
    fr = (lane == 63) ? fx_next : fr;
    double p = 1.0;
#pragma unroll
    for (int v = W - 1; v >= 0; v--) {
      fz[v] = readlane_d((v < wave) ? p : 0.0, 0);
      p = (v < wave) ? p * sh.Aw[v] : p;
    }
    p = 1.0;
#pragma unroll
    for (int v = 0; v < W; v++) {
      fx[v] = readlane_d((v > wave) ? p : 0.0, 0);
      p = (v > wave) ? p * sh.Gw[v] : p;
    }
  } else {
    hl = (lane == 0) ? 0.0 : hl;
    fr = (lane == 63) ? 0.0 : fr;
  }

  // ------------------------------------------------------------------ march
  double q[K], acc[K];
#pragma unroll
  for (int t = 0; t < K; t++) {
    q[t] = (u0 + t < n) ? 1.0 : 0.0;
    acc[t] = 0.0;
  }
  double ql = (u0 - 1 >= 0 && u0 - 1 < n) ? 1.0 : 0.0;
  double qr = (u0 + K < n) ? 1.0 : 0.0;

  // One implicit-Euler step q <- G (A q) for the whole instance: with r the
  // right-hand side scaled by G_ii (ra, rd, rc),
  //   F_i = r_i + f_i F_{i-1},  Y_i = r_i + h_i Y_{i+1},  q_i = F_i + h_i Y_{i+1},
  // two recurrences that do not wait for each other, so the lane-local
  // passes, the scans and the fold over waves (one barrier) overlap; ql / qr
  // become the new values of the unknowns left of q[0] and right of q[K-1].
  // How the inflows reach the rows: with the products Pf, Ph (KEEP_P) two
  // independent FMAs per row after them, which is the shorter chain; without,
  // the passes run again (the same FMAs, one after the other), which saves 4 K
  // registers.
  constexpr bool KEEP_P = SEG == 1 && W < 8;
  int par = 0;
  [[maybe_unused]] const int tot_at = (lane == 0) ? W + wave : (lane == 63) ? wave : 2 * W + tid;
  auto advance = [&](double (&q)[K], double& ql, double& qr) __attribute__((always_inline)) {
    double r[K];
#pragma unroll
    for (int t = 0; t < K; t++) {
      const double qm = (t == 0) ? ql : q[t - 1];
      const double qp = (t == K - 1) ? qr : q[t + 1];
      r[t] = fma(ra[t], qm, fma(rc[t], qp, rd[t] * q[t]));
    }
    // local passes from zero inflow: what the chunk adds to its outflows
    double B = r[0], Cc = r[K - 1];
    double F0[K], Y0[K];  // (KEEP_P only)
    F0[0] = B;
    Y0[K - 1] = Cc;
#pragma unroll
    for (int t = 1; t < K; t++) {
      B = fma(f[t], B, r[t]);
      Cc = fma(h[K - 1 - t], Cc, r[K - 1 - t]);
      F0[t] = B;
      Y0[K - 1 - t] = Cc;
    }
    if constexpr (KEEP_P) {  // the chunk's own part of its rows, ready before the inflows are
#pragma unroll
      for (int t = 0; t + 1 < K; t++) F0[t] = fma(h[t], Y0[t + 1], F0[t]);
    }
    const double Bk = B, Ck = Cc;
    B = fma(mf[0], row_shr<1>(B), B);
    Cc = fma(mb[0], row_shl<1>(Cc), Cc);
    B = fma(mf[1], row_shr<2>(B), B);
    Cc = fma(mb[1], row_shl<2>(Cc), Cc);
    B = fma(mf[2], row_shr<4>(B), B);
    Cc = fma(mb[2], row_shl<4>(Cc), Cc);
    B = fma(mf[3], row_shr<8>(B), B);
    Cc = fma(mb[3], row_shl<8>(Cc), Cc);
    // carries into rows 0..2 of the backward scan: the suffix from the first
    // lane of the row after; rows to the whole wave forward: broadcast levels
    Cc = fma(mbA, bpermute_d(srcA, Cc), Cc);
    B = fma(mf5, row_bcast15(B), B);
    Cc = fma(mbB, bpermute_d(srcB, Cc), Cc);
    B = fma(mf6, row_bcast31(B), B);
    // wave-inclusive now: this lane's inflows are lane - 1's and lane + 1's
    double Fin = wave_shr1(B), Yin = wave_shl1(Cc);
    if constexpr (W > 1) {
      // two sets of slots in turn: a wave writes the next step's set while a
      // slower one still reads this step's, and the barrier in between keeps
      // any wave from being two steps ahead
      // (lane 63 writes the forward total, lane 0 the backward one, the other
      // lanes a place of their own: a branch around the write costs 50 ns)
      sh.tot[par][tot_at] = (lane == 0) ? Cc : B;
      wg_barrier();
      double Z0 = 0.0, Z1 = 0.0, X0 = 0.0, X1 = 0.0;
#pragma unroll
      for (int v = 0; v + 1 < W; v += 2) {
        Z0 = fma(fz[v], sh.tot[par][v], Z0);
        if (v + 2 < W) Z1 = fma(fz[v + 1], sh.tot[par][v + 1], Z1);
        X0 = fma(fx[v + 1], sh.tot[par][W + v + 1], X0);
        if (v + 2 < W) X1 = fma(fx[v + 2], sh.tot[par][W + v + 2], X1);
      }
      Fin = fma(Apre_m1, Z0 + Z1, Fin);
      Yin = fma(Gsuf_p1, X0 + X1, Yin);
      par ^= 1;
    }
    if constexpr (KEEP_P) {
      ql = fma(hl, fma(Ph[0], Yin, Ck), Fin);
      qr = fma(fr, fma(Pf[K - 1], Fin, Bk), Yin);
#pragma unroll
      for (int t = 0; t < K; t++) q[t] = fma(Pf[t], Fin, fma(Ph[t], Yin, F0[t]));
    } else {
      // the passes again from the true inflows
      double Y = Yin, F = Fin;
#pragma unroll
      for (int t = K - 1; t >= 0; t--) {
        q[t] = Y;
        Y = fma(h[t], Y, r[t]);
      }
#pragma unroll
      for (int t = 0; t < K; t++) {
        F = fma(f[t], F, r[t]);
        q[t] = fma(h[t], q[t], F);
      }
      ql = fma(hl, Y, Fin);
      qr = fma(fr, F, Yin);
    }
  };

  // Slabs.  Slab s is q after step s (slab 0: the initial condition).  With
  // SEG = 1 the slabs 0 .. N/2 - 1 are all kept; with SEG > 1 every SEG-th, and
  // the second half of the march recomputes the ones between from the kept
  // one below them.  Kept slab number g starts at g * slab_len; within it row
  // t of lane tid sits at (t / 2) * 2P + 2 tid + t % 2 (K >= 2: 16 bytes per
  // lane and access) or at tid (K = 1).  Lanes whose rows are all padding
  // (u0 >= n) store nothing (one exec mask for the whole loop) and load from
  // lane 0's address, so a wave's dead lanes share one cache line; their
  // values are replaced by 0.  The region is accessed as a raw buffer
  // (slab_rsrc): the step and element select a scalar offset, the lane a fixed
  // 32-bit offset.  First half: nothing here waits on memory.
  const bool lane_live = u0 < n;
  const __amdgpu_buffer_rsrc_t srsrc =
      slab_rsrc(slab, static_cast<unsigned>(a.slab_stride * sizeof(double)));
  const unsigned off_dst = static_cast<unsigned>(tid) * slab_lane_bytes<K>();
  const unsigned off_src = lane_live ? off_dst : 0u;
  constexpr unsigned SLAB_BYTES = march_slab_len(K, W, SEG) * 8u;
  if constexpr (SEG == 1) {
    auto store_slab = [&](const int j) __attribute__((always_inline)) {
      if (lane_live) slab_put<K>(q, srsrc, off_dst, static_cast<unsigned>(j) * SLAB_BYTES, P);
    };
    for (int j = 0; j < half; j++) {
      store_slab(j);
      advance(q, ql, qr);
    }
    // step N/2 pairs with itself
    {
      const double c0 = pw[0];
#pragma unroll
      for (int t = 0; t < K; t++) acc[t] = c0 * q[t] * q[t];
    }

    // Second half: step N/2 + i pairs with slab N/2 - i (i = 1 .. N/2).  Slabs
    // come through a ring of PD register sets, each loaded PD steps before its
    // use (indices below 0 reload slab 0 and are never used).  PD divides N/2
    // (N is a power of two >= 16).  What dead lanes load only ever multiplies
    // their q = 0.
    constexpr int PD = (K <= 2) ? 8 : (K == 4) ? 4 : 2;
    double ring[PD][K];
    auto fetch = [&](const int s, double (&dstv)[K]) __attribute__((always_inline)) {
      slab_get<K>(dstv, srsrc, off_src, static_cast<unsigned>(max(s, 0)) * SLAB_BYTES, P);
    };
    // The loop below waits on each ring set by the count of loads issued after
    // it.  That count is exact only if nothing else is in flight (the first
    // half's slab stores are drained here) and the sets are issued in ring
    // order (the scheduler may not reorder them across the barrier).
    vmem_drain();
#pragma unroll
    for (int e = 0; e < PD; e++) {
      fetch(half - 1 - e, ring[e]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // (a step's pairing stands before the next step, whose scans leave time
    // for it; the step after N is computed and not used)
    advance(q, ql, qr);
    for (int i0 = 1; i0 <= half; i0 += PD) {
#pragma unroll
      for (int e = 0; e < PD; e++) {
        const int i = i0 + e;
        const double cj = weight(i);
#pragma unroll
        for (int t = 0; t < K; t++) acc[t] = fma(cj * q[t], ring[e][t], acc[t]);
        fetch(half - i - PD, ring[e]);
        advance(q, ql, qr);
      }
    }
  } else {
    // A kept slab carries the values beyond each wave's two ends behind its
    // rows (2 per wave): a step started from it needs them.
    const unsigned off_edge =
        static_cast<unsigned>(P * K + 2 * wave + (lane == 63 ? 1 : 0)) * 8u;
    for (int g = 0; g < half / SEG; g++) {
      const unsigned o = static_cast<unsigned>(g) * SLAB_BYTES;
      if (lane_live) slab_put<K>(q, srsrc, off_dst, o, P);
      if constexpr (W > 1) {
        if (lane == 0 || lane == 63) slab_store(lane == 0 ? ql : qr, srsrc, off_edge, o);
      }
#pragma unroll 1
      for (int e = 0; e < SEG; e++) advance(q, ql, qr);
    }
    {
      const double c0 = pw[0];
#pragma unroll
      for (int t = 0; t < K; t++) acc[t] = c0 * q[t] * q[t];
    }
    // Second half, segment by segment: the slabs g SEG .. g SEG + SEG - 1 into
    // this lane's own places in LDS (the kept one, loaded a segment ahead,
    // then SEG - 1 steps from it: those of the first half to rounding, since a
    // lane's two outer neighbours are read from the lanes beside it here and
    // come out of its own inflows there), then SEG steps of the march that pair
    // with them from the top down.
    auto lds_slot = [&](const int e) __attribute__((always_inline)) {
      return seg_lds + e * (P * K) + (K >= 2 ? 2 * tid : tid);
    };
    auto put_lds = [&](const double (&v)[K], const int e) __attribute__((always_inline)) {
      double* d = lds_slot(e);
      if constexpr (K >= 2) {
#pragma unroll
        for (int t = 0; t < K; t += 2)
          *reinterpret_cast<f64x2*>(d + t * P) = f64x2{v[t], v[t + 1]};
      } else {
        d[0] = v[0];
      }
    };
    double kept[K], edge = 0.0;
    auto fetch = [&](const int g) __attribute__((always_inline)) {
      const unsigned o = static_cast<unsigned>(max(g, 0)) * SLAB_BYTES;
      slab_get<K>(kept, srsrc, off_src, o, P);
      if constexpr (W > 1) edge = slab_load(srsrc, off_edge, o);
    };
    int g = half / SEG - 1;
    fetch(g);
    for (; g >= 0; g--) {
      {
        double s[K];
#pragma unroll
        for (int t = 0; t < K; t++) s[t] = lane_live ? kept[t] : 0.0;
        double sl = wave_shr1(s[K - 1]), sr = wave_shl1(s[0]);
        if constexpr (W > 1) {
          sl = (lane == 0) ? edge : sl;
          sr = (lane == 63) ? edge : sr;
        }
        put_lds(s, 0);
        fetch(g - 1);
#pragma unroll 1
        for (int e = 1; e < SEG; e++) {
          advance(s, sl, sr);
          put_lds(s, e);
        }
      }
#pragma unroll 1
      for (int e = SEG - 1; e >= 0; e--) {
        advance(q, ql, qr);
        const double cj = weight(half - (g * SEG + e));
        const double* p = lds_slot(e);
        if constexpr (K >= 2) {
#pragma unroll
          for (int t = 0; t < K; t += 2) {
            const f64x2 v = *reinterpret_cast<const f64x2*>(p + t * P);
            acc[t] = fma(cj * q[t], v.x, acc[t]);
            acc[t + 1] = fma(cj * q[t + 1], v.y, acc[t + 1]);
          }
        } else {
          acc[0] = fma(cj * q[0], p[0], acc[0]);
        }
      }
    }
  }

  // --------------------------------------------------------------- residual
  const double* __restrict__ pt = a.phit + d.uo;
  double* __restrict__ r = a.r + d.uo;
  double* __restrict__ phi = a.phi ? a.phi + d.uo : nullptr;
  double mx = 0.0;
#pragma unroll
  for (int t = 0; t < K; t++) {
    const int u = u0 + t;
    if (u < n) {
      const double res = acc[t] - pt[u];
      r[u] = res;
      if (phi) phi[u] = acc[t];
      if (!isfinite(res)) bad |= ST_NAN;
      mx = fmax(mx, fabs(res));
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off));
    bad |= __shfl_xor(bad, off);
  }
  mx = readlane_d(mx, 0);
  bad = __builtin_amdgcn_readfirstlane(bad);
  if constexpr (W > 1) {
    sh.red[wave] = mx;
    sh.bad[wave] = bad;
    wg_barrier();
    for (int v = 0; v < W; v++) {
      mx = fmax(mx, sh.red[v]);
      bad |= sh.bad[v];
    }
    wg_barrier();  // sh.red / sh.bad are reused by the next instance
  }
  // every lane of wave 0 stores the same (uniform) values: no lane branch
  if (wave == 0) {
    a.rnorm[inst] = (bad & ST_NAN) ? __builtin_nan("") : mx;
    a.status[inst] = st0 | bad;
  }
}

// Persistent workgroups take items (sorted by cost, largest first) from a
// per-bucket counter: greedy list scheduling, which also rebalances as
// instances converge.  Thread 0 takes the next index and broadcasts it
// through LDS; the exit test is on that workgroup-uniform value, so every
// wave leaves the loop together once the counter passes n_items.
template <int K, int W, int SEG>
__global__ void __launch_bounds__(64 * W, K == 8 ? 2 : 1) march_kernel(MarchArgs a) {
  __shared__ MarchShared<W> sh;
  __shared__ int s_next;
  extern __shared__ __align__(16) double seg_lds[];  // SEG > 1: one segment's slabs
  const int tid = threadIdx.x;
  double* slab = a.slabs + (long long)blockIdx.x * a.slab_stride;
  for (int it = blockIdx.x; it < a.n_items; it = next_item(a, tid, &s_next)) {
    const int inst = __builtin_amdgcn_readfirstlane(a.items[it]);
    const unsigned st = __builtin_amdgcn_readfirstlane(a.status[inst]);
    if (st & ST_DONE_MASK) continue;
    march_one<K, W, SEG>(a, inst, st, slab, sh, seg_lds, tid);
  }
}

// The same queue for instances of up to 512 unknowns of any size, one wave
// each: a sweep over many sizes then needs four launches for the four
// hardware queues instead of seven, and no small bucket waits for another to
// finish.  Costs the smallest sizes their occupancy (two waves per SIMD, the
// registers of K = 8), so a batch that has queues left launches its buckets
// one by one.
template <int SEG>
__global__ void __launch_bounds__(64, 2) march_small_kernel(MarchArgs a) {
  __shared__ MarchShared<1> sh;
  __shared__ int s_next;
  extern __shared__ __align__(16) double seg_lds[];
  const int tid = threadIdx.x;
  double* slab = a.slabs + (long long)blockIdx.x * a.slab_stride;
  for (int it = blockIdx.x; it < a.n_items; it = next_item(a, tid, &s_next)) {
    const int inst = __builtin_amdgcn_readfirstlane(a.items[it]);
    const unsigned st = __builtin_amdgcn_readfirstlane(a.status[inst]);
    if (st & ST_DONE_MASK) continue;
    const int n = __builtin_amdgcn_readfirstlane(a.desc[inst].n);
    if (n <= 64)
      march_one<1, 1, SEG>(a, inst, st, slab, sh, seg_lds, tid);
    else if (n <= 128)
      march_one<2, 1, SEG>(a, inst, st, slab, sh, seg_lds, tid);
    else if (n <= 256)
      march_one<4, 1, SEG>(a, inst, st, slab, sh, seg_lds, tid);
    else
      march_one<8, 1, SEG>(a, inst, st, slab, sh, seg_lds, tid);
  }
}

// ------------------------------------------------------------------ dispatch
// (K, W) variants: one wave per instance up to 512 unknowns, then 4 or 8 rows
// per lane.  Fewer rows per lane lose more to the scans than the shorter
// lane-local passes give (a step of 512 unknowns: <8, 1> 0.29 us, <4, 2>
// 0.35, <2, 4> 0.36), 16 spill.
#define SCFT_MARCH_VARIANTS(X) \
  X(1, 1) X(2, 1) X(4, 1) X(8, 1) X(4, 2) X(8, 2) X(4, 4) X(8, 4) X(4, 8) X(8, 8)

static const void* march_fn(int K, int W, int seg) {
#define X(k, w)                                                                  \
  if (K == k && W == w)                                                          \
    return seg == 1 ? reinterpret_cast<const void*>(&march_kernel<k, w, 1>)      \
                    : reinterpret_cast<const void*>(&march_kernel<k, w, MARCH_SEG>);
  SCFT_MARCH_VARIANTS(X)
#undef X
  return nullptr;
}

static size_t march_lds_bytes(int K, int W, int seg) {
  return seg > 1 ? static_cast<size_t>(seg) * 64 * W * K * sizeof(double) : 0;
}

bool march_variant_exists(int K, int W) { return march_fn(K, W, 1) != nullptr; }

hipError_t launch_march(int K, int W, const MarchArgs& a, int grid, hipStream_t s) {
  const size_t lds = march_lds_bytes(K, W, a.seg);
#define X(k, w)                                                                          \
  if (K == k && W == w) {                                                                \
    if (a.seg == 1)                                                                      \
      hipLaunchKernelGGL((march_kernel<k, w, 1>), dim3(grid), dim3(64 * w), lds, s, a);  \
    else                                                                                 \
      hipLaunchKernelGGL((march_kernel<k, w, MARCH_SEG>), dim3(grid), dim3(64 * w), lds, \
                         s, a);                                                          \
    return hipGetLastError();                                                            \
  }
  SCFT_MARCH_VARIANTS(X)
#undef X
  return hipErrorInvalidValue;
}

static int resident_grid(const void* f, int threads, size_t lds) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, threads, lds) != hipSuccess) return 0;
  if (per < 1) per = 1;
  return per * cus;
}

int march_max_grid(int K, int W, int seg) {
  const void* f = march_fn(K, W, seg);
  return f ? resident_grid(f, 64 * W, march_lds_bytes(K, W, seg)) : 0;
}

hipError_t launch_march_small(const MarchArgs& a, int grid, hipStream_t s) {
  const size_t lds = march_lds_bytes(8, 1, a.seg);
  if (a.seg == 1)
    hipLaunchKernelGGL(march_small_kernel<1>, dim3(grid), dim3(64), lds, s, a);
  else
    hipLaunchKernelGGL(march_small_kernel<MARCH_SEG>, dim3(grid), dim3(64), lds, s, a);
  return hipGetLastError();
}

int march_small_max_grid(int seg) {
  const void* f = seg == 1 ? reinterpret_cast<const void*>(&march_small_kernel<1>)
                           : reinterpret_cast<const void*>(&march_small_kernel<MARCH_SEG>);
  return resident_grid(f, 64, march_lds_bytes(8, 1, seg));
}

}  // namespace scft
