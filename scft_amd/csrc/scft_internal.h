// scft_internal.h -- device data layout shared by the kernels and the host
// side of libscft_hip.so (not part of the public C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace scft {

// One SCFT instance as the kernels see it.  Unknown u <-> mesh node u+1.
struct InstDesc {
  int n;          // unknowns (M-2 for DD, M-1 for DN)
  int N;          // implicit-Euler contour steps, 2^k >= 16
  int M;          // mesh nodes
  int bc;         // SCFT_BC_DD / SCFT_BC_DN
  int cmat;       // SCFT_C_ROWSCALED / SCFT_C_CONSISTENT
  int pad;
  long long xo;   // offset of the M node coordinates in `x`
  long long uo;   // offset of the n unknowns in w / phi_t / phi / r
  long long po;   // offset of the N/2+1 pairing weights in `pw`
  long long ho;   // offset of the history ring (S*n doubles) of the mixer
  double wall0;   // field at node 0 (only the consistent C reads it)
  double wallL;   // field at node M-1 for DD (consistent C only)
};

// Arguments of one persistent march launch (one size bucket).
struct MarchArgs {
  const InstDesc* desc;
  const double* x;        // node coordinates
  const double* w;        // field on unknowns
  const double* phit;     // target on unknowns
  const double* pw;       // Romberg pairing weights
  double* phi;            // out: density on unknowns (nullable)
  double* r;              // out: residual phi - phi_t on unknowns
  double* rnorm;          // out: ||r||_inf per instance
  unsigned* status;       // per-instance status word
  double* slabs;          // q-slab scratch, one region per workgroup
  long long slab_stride;  // doubles per workgroup region (N_max/2 slabs)
  const int* items;       // instance ids of this bucket, largest first
  int* queue;             // items taken past the grid's first (zeroed before a launch of more)
  int n_items;
  int half_max;           // largest N/2 of the bucket (IRK4: LDS weight table size - 1)
  int seg;                // 1: every slab is kept, MARCH_SEG: every MARCH_SEG-th (march.hip)
};

constexpr unsigned ST_CONVERGED = 1u;
constexpr unsigned ST_NAN = 2u;
constexpr unsigned ST_PIVOT = 4u;
constexpr unsigned ST_MAXITER = 8u;
constexpr unsigned ST_FALLBACK = 16u;
constexpr unsigned ST_FAILED = 32u;
constexpr unsigned ST_PLAIN_FORM = 64u;  // left the ground-state form
constexpr unsigned ST_RATIONAL = 128u;   // reached the rational form's threshold
// instances the march skips: converged, out of iterations, or given up by the
// mixer (FAILED without a NaN: growth with no halvings left)
constexpr unsigned ST_DONE_MASK = ST_CONVERGED | ST_NAN | ST_PIVOT | ST_MAXITER | ST_FAILED;

struct MixState {
  int k;         // evaluations so far
  int head;      // next ring slot
  int stored;    // valid ring entries
  int restarts;
  double best;   // best ||r||_inf so far
  double eacc;   // ||r||_inf of the last accepted iterate (inf: none yet)
  int halvings;  // consecutive backtracking halvings
  int pad;
};

struct AndersonArgs {
  const int* order;  // instance of workgroup g: largest n first (nullable: g)
  const InstDesc* desc;
  double* w;            // field on unknowns (updated in place)
  const double* r;      // plain residual phi - phi_t from the march
  const double* rnorm;  // ||r||_inf from the march
  const double* phit;   // target on unknowns
  const double* x;      // node coordinates (preconditioner stencil)
  const double* wcold;  // cold-start fields (nullable)
  double* hw;           // history of fields   (S * n per instance at ho)
  double* hr;           // history of residuals
  MixState* st;
  unsigned* status;
  int* iters;           // evaluations used (written at convergence / stop)
  int* active;          // count of instances still running after this sweep
  int n_inst;
  int history;          // m (ring of m+1 slots)
  int transform;        // 0 plain, 1 relative, 2 log
  int max_iter;
  double beta, tol, step_cap, restart_factor, reg, floor;
  double fallback_thresh;  // absolute threshold (<= 0: off), first sweep only
  double precond;          // Laplacian preconditioner coefficient (0: off)
  double backtrack;        // growth factor that triggers a halving (0: off)
  int max_halvings;
  double field_floor;      // w >= -field_floor * N after each update (0: off)
  double gs_precond;       // ground-state form coefficient (0: off)
  double gs_field_weight;  // its field weight c
  int gs_switch;           // evaluations allowed in that form (0: no limit)
  double gs_switch_growth; // leave it when ||r|| > growth * best (0: never)
  double gs_shift;         // g > 0: the rational ground-state form (0: linear)
  double gs_shift_below;   // > 0: rational only once ||r|| < this (linear before)
  double* tri;             // 4 x tri_stride doubles at desc.uo: the factors of
  long long tri_stride;    // g I + G0 (1/pivot, lower/pivot, upper/pivot), work
};

// Size bucket of an instance with n unknowns: the power of two >= n (at
// least 64) = 64 * W * K lanes-times-rows of the workgroup that marches it.
inline int bucket_capacity(int n) {
  int c = 64;
  while (c < n) c *= 2;
  return c;
}
// Rows per lane of a bucket of `items` instances before any tuning.  Implicit
// Euler: one wave up to 512 unknowns, then waves of 8 rows per lane; the 1024
// bucket takes 4 waves of 4 rows while every instance finds a CU of its own
// (a step 0.37 us against 0.47 us at <8, 2>), and <8, 2> beyond (1030 against
// 860 G node-steps/s with the chip full).  IRK4 keeps ~11 doubles per row and
// is bound by a wave's own instructions, so there the 512 bucket does likewise
// (600-1000 unknowns, <= 256 instances, 512 steps: <4, 4> 0.50-0.58 ms against
// <8, 2> 0.65-0.69; 300 unknowns <4, 2> 0.40-0.43 against <8, 1> 0.41-0.47; with
// 1024 instances 0.93 against 0.61).
inline int bucket_default_K(int cap, bool irk4, int items, int cus) {
  if ((cap == 1024 || (irk4 && cap == 512)) && items <= cus) return 4;
  const int k = cap / 64;
  return k < 8 ? k : 8;
}

// Slabs of a workgroup that keeps every seg-th, and the doubles of one kept
// slab (seg > 1: two more per wave).
constexpr int MARCH_SEG = 4;
constexpr int march_slab_len(int K, int W, int seg) { return 64 * W * K + (seg > 1 ? 2 * W : 0); }

// Launch one bucket.  Returns hipSuccess or the launch error.
hipError_t launch_march(int K, int W, const MarchArgs& a, int grid,
                        hipStream_t s);
// Largest grid of co-resident workgroups for a variant (persistent launch).
int march_max_grid(int K, int W, int seg);
bool march_variant_exists(int K, int W);
// Instances of up to 512 unknowns of any size in one launch of single waves
// (rows per lane by n, as bucket_default_K).
hipError_t launch_march_small(const MarchArgs& a, int grid, hipStream_t s);
int march_small_max_grid(int seg);
// Instances of up to 64 unknowns as dense products on the matrix cores, 32 or
// 64 unknowns wide (dense.hip); kept slabs: N/2 x width doubles.
hipError_t launch_dense(int np, bool irk4, const MarchArgs& a, int grid, hipStream_t s);
int dense_max_grid(int np, bool irk4);
constexpr int DENSE_COLS = 64;  // steps per block
// Width for `items` instances of at most n unknowns and at least N steps, or 0:
// the scan march.  The powers cost 30-40 us (width 32) or 100-120 us, then 64
// steps take 0.5 or 1.8 us, one workgroup of each CU at a time; a scan step
// takes 0.15 us (IRK4 0.31) however many there are, up to 1024 waves.  Sweeps
// of 1 / 512 / 1024 / 4096 instances in us, dense against scan:
//   n = 31, N = 256   37 /  59 / 102 / 357       52 /  65 /  81 / 182
//           N = 512   39 /  65 / 112 / 399       89 / 115 / 129 / 301
//           N = 1024  43 /  76 / 128 / 461      163 / 212 / 223 / 534
//   n = 59, N = 1024 145 / 307 /   - /   -      163 / 180 / 201 / 639
//   n = 59, N = 512, IRK4, 158 / 332 against 180 / 202.
inline int dense_width(int n, int N, int items, int cus, bool irk4) {
  if (n <= 32) {
    const int most = N >= 1024 || (irk4 && N >= 512) ? items : N >= 512 ? 4 * cus : 2 * cus;
    return N >= 256 && items <= most ? 32 : 0;
  }
  return n <= 64 && N >= (irk4 ? 512 : 1024) && items <= cus ? 64 : 0;
}
// The same for the two-stage Gauss (IRK4) march (irk4.hip).
hipError_t launch_irk4(int K, int W, const MarchArgs& a, int grid, hipStream_t s);
int irk4_max_grid(int K, int W, int half_max);  // 0: the workgroup does not fit
bool irk4_variant_exists(int K, int W);
// The Thomas factors of the rational preconditioner's g I + G0 (once per
// batch and shift).
hipError_t launch_gs_pivots(const AndersonArgs& a, hipStream_t s);
hipError_t launch_anderson(const AndersonArgs& a, hipStream_t s);
hipError_t launch_reset(int* counters, int n, hipStream_t s);
constexpr int MIX_MAX_HISTORY = 16;

// Mapping of the warm-start network's outputs onto a batch's unknowns
// (warmpredict.hip): instance k's row of raw outputs y (before the output
// normalisation y' ys + ym) holds n_grid values at its grid points, then
// n_node wall samples asinh(w / node_scale) at the 1-based node numbers
// node_idx; its first wall_count[k] unknowns come from the samples
// (linear in the node number), the others from the not-a-knot cubic spline
// through the grid values.  One workgroup per instance.
constexpr int WARM_MAX_GRID = 256;
constexpr int WARM_MAX_NODES = 32;
struct WarmMapArgs {
  const InstDesc* desc;
  const double* x;         // the batch's node coordinates
  double* w;               // out: the batch's field on unknowns
  const float* y;          // network outputs, one row per instance of the plan
  const float* ym;         // output shift and scale (nullable: none)
  const float* ys;
  const double* grid;      // n_grid grid points per row, increasing
  const int* node_idx;     // n_node sample node numbers, increasing
  const int* wall_count;   // per row
  const int* sel;          // batch instance of each row (nullable: row k is instance k)
  double node_scale;
  int n_inst, n_out, n_grid, n_node;  // n_inst: rows
};
hipError_t launch_warm_map(const WarmMapArgs& a, hipStream_t s);

}  // namespace scft

// The network's forward pass on rows already normalised and resident in
// device memory (mlp.hip): *d_out receives its raw output activations
// (batch x dims.back(), before the output normalisation), *ym / *ys its
// output shift and scale as host arrays (nullptr: none).  Waits for the
// network's stream.
struct scft_mlp;
int scft_mlp_forward_resident(scft_mlp* m, int batch, const float* d_xn, const float** d_out,
                              const float** ym, const float** ys, int* n_out, int* n_in);
int scft_mlp_normalise_inputs(const scft_mlp* m, const float* X, int rows, float* out);

namespace scft {

}  // namespace scft
