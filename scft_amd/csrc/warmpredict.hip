// warmpredict.hip -- the learned warm start's last step on the device: the
// network's outputs mapped onto every instance's unknowns and written into
// the batch's resident field, so no field crosses PCIe between the
// prediction and the solve.  No counterpart in the reference.
//
// Per instance (one 256-thread workgroup): the outputs y' ys + ym (FP32, as
// the network produces them) become FP64 values; the grid part is
// interpolated by the not-a-knot cubic spline of DEALII_SCFT/src/spline_chen.c
// (the tridiagonal form and evaluation of host_math.cpp's spline_not_a_knot /
// spline_eval), the leading wall unknowns by the samples asinh(w / s)
// interpolated linearly in the node number.  All instances are in flight at
// once, so the time is the longest chain in one: 12 us for 1160 instances of
// 128 grid points, 125 us with one thread eliminating (a division and three LDS
// trips per row); 25 us for 888 of which some have thousands of unknowns, 97 us
// before.
#include "scft_internal.h"

namespace scft {

namespace {

constexpr int WM_THREADS = 256;
static_assert(WARM_MAX_GRID <= WM_THREADS, "a thread per row of the spline's system");

struct alignas(16) Row {  // of the spline's system: below, on, above the diagonal, rhs
  double l, d, u, r;
};

__device__ double spline_value(int n, const double* gx, const double* gy, const double* M,
                               double xp) {
  int klo = 0, khi = n - 1;
  while (khi - klo > 1) {
    const int k = (khi + klo) >> 1;
    if (gx[k] > xp)
      khi = k;
    else
      klo = k;
  }
  const double h = gx[khi] - gx[klo];
  const double a = (gx[khi] - xp) / h, b = (xp - gx[klo]) / h;
  return a * gy[klo] + b * gy[khi] +
         ((a * a * a - a) * M[klo] + (b * b * b - b) * M[khi]) * (h * h) / 6.0;
}

__global__ void __launch_bounds__(WM_THREADS) warm_map_kernel(WarmMapArgs a) {
  const int row = blockIdx.x;  // row of the plan; the batch instance it writes:
  const int inst = a.sel ? a.sel[row] : row;
  const int tid = threadIdx.x;
  __shared__ double gx[WARM_MAX_GRID], gy[WARM_MAX_GRID], M[WARM_MAX_GRID];
  __shared__ Row rows[WARM_MAX_GRID];
  __shared__ double sv[WARM_MAX_NODES];
  const int ng = a.n_grid;
  const float* yr = a.y + static_cast<long long>(row) * a.n_out;
  for (int i = tid; i < ng; i += WM_THREADS) {
    gx[i] = a.grid[static_cast<long long>(row) * ng + i];
    const float v = a.ys ? yr[i] * a.ys[i] + a.ym[i] : yr[i];
    gy[i] = static_cast<double>(v);
  }
  for (int j = tid; j < a.n_node; j += WM_THREADS) {
    const int o = ng + j;
    const float v = a.ys ? yr[o] * a.ys[o] + a.ym[o] : yr[o];
    sv[j] = static_cast<double>(v);
  }
  __syncthreads();
  // Second derivatives, not-a-knot ends folded into the end rows: row i of the
  // ng - 2 stands at thread i, and cyclic reduction of all rows at once
  // (diagonally dominant: no pivoting) solves them in log2(ng) steps.
  const int k = ng - 2;
  const double h0 = gx[1] - gx[0], h1 = gx[2] - gx[1];
  const double ha = gx[ng - 2] - gx[ng - 3], hb = gx[ng - 1] - gx[ng - 2];
  double l = 0.0, dg = 1.0, up = 0.0, r = 0.0;
  if (tid < k) {
    const double hl = gx[tid + 1] - gx[tid], hr = gx[tid + 2] - gx[tid + 1];
    l = hl / 6.0;
    dg = (hl + hr) / 3.0;
    up = hr / 6.0;
    r = (gy[tid + 2] - gy[tid + 1]) / hr - (gy[tid + 1] - gy[tid]) / hl;
    const double lf = l, uf = up;
    if (tid == 0) {
      dg += lf * (1.0 + h0 / h1);
      up -= lf * (h0 / h1);
      l = 0.0;
    }
    if (tid == k - 1) {
      dg += uf * (1.0 + hb / ha);
      l -= uf * (hb / ha);
      up = 0.0;
    }
  }
  for (int s = 1; s < k; s <<= 1) {
    if (tid < k) rows[tid] = {l, dg, up, r};
    __syncthreads();
    if (tid < k) {
      const bool has_l = tid >= s, has_r = tid + s < k;
      const Row pl = rows[has_l ? tid - s : tid], pr = rows[has_r ? tid + s : tid];
      const double fl = has_l ? l / pl.d : 0.0, fr = has_r ? up / pr.d : 0.0;
      dg -= fl * pl.u + fr * pr.l;
      r -= fl * pl.r + fr * pr.r;
      l = -fl * pl.l;
      up = -fr * pr.u;
    }
    __syncthreads();
  }
  if (tid < k) M[tid + 1] = r / dg;
  __syncthreads();
  if (tid == 0) {
    M[0] = (1.0 + h0 / h1) * M[1] - (h0 / h1) * M[2];
    M[ng - 1] = (1.0 + hb / ha) * M[ng - 2] - (hb / ha) * M[ng - 3];
  }
  __syncthreads();
  const InstDesc d = a.desc[inst];
  const double* xn = a.x + d.xo;
  double* w = a.w + d.uo;
  const int nwall = a.wall_count[row];
  for (int u = tid; u < d.n; u += WM_THREADS) {
    const int node = u + 1;
    double v;
    if (u < nwall) {
      // bracket of the node number among the samples (clamped to the ends)
      int j = 0;
      while (j + 2 < a.n_node && a.node_idx[j + 1] <= node) j++;
      const double t = static_cast<double>(node - a.node_idx[j]) /
                       static_cast<double>(a.node_idx[j + 1] - a.node_idx[j]);
      const double tc = t < 0.0 ? 0.0 : (t > 1.0 ? 1.0 : t);
      v = a.node_scale * sinh((1.0 - tc) * sv[j] + tc * sv[j + 1]);
    } else {
      v = spline_value(ng, gx, gy, M, xn[node]);
    }
    w[u] = v;
  }
}

}  // namespace

hipError_t launch_warm_map(const WarmMapArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(warm_map_kernel, dim3(a.n_inst), dim3(WM_THREADS), 0, s, a);
  return hipGetLastError();
}

}  // namespace scft
