// mlp.hip -- the warm-start MLP: dense FP32 layers (tanh on hidden layers,
// linear output), mean-squared-error loss and Adam, trained and evaluated on
// the device by the kernels below.  No reference counterpart: the reference
// has no learned warm start.  Parameters are packed as the FP64 restatement in
// oracle/oracle_mlp.c packs them: per layer W (dout x din, row-major), then
// b (dout).
//
// Networks whose activations of 16 rows fit in LDS run whole: one launch takes
// the rows through all layers (in training also through the loss and the
// deltas), one makes all gradients and the Adam step (net_kernel,
// grad_kernel).  Wider or deeper ones go product by product: `gemm_kernel` is
// C[m][n] = sum_k A(m,k) B(k,n) with arbitrary element strides for A and B,
// FP32 operands and FP32 accumulation on the matrix cores
// (v_mfma_f32_16x16x4f32), and a fused epilogue (bias + tanh for hidden
// layers, bias for the output layer, the tanh derivative for back-propagated
// deltas, or nothing).  Workgroups of 4 waves own a 32 x 32 tile of C, each
// wave one 16 x 16 block; K advances in chunks of 64 staged in LDS, each
// operand loaded along whichever of its strides is 1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/scft.h"

namespace scft {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 32;
constexpr int KC = 64;  // k chunk staged per iteration
enum Epilogue { EP_NONE = 0, EP_BIAS = 1, EP_BIAS_TANH = 2, EP_DTANH = 3 };

struct GemmArgs {
  const float* A;
  long long a_m, a_k;  // A(m, k) = A[m * a_m + k * a_k]
  const float* B;
  long long b_k, b_n;  // B(k, n) = B[k * b_k + n * b_n]
  float* C;            // C[m * ldc + n]
  long long ldc;
  int M, N, K;
  int epilogue;
  const float* bias;   // EP_BIAS*: bias[n]
  const float* act;    // EP_DTANH: C *= 1 - act[m * ldc + n]^2
};

__global__ void __launch_bounds__(256) gemm_kernel(GemmArgs g) {
  __shared__ float As[TILE][KC + 1];
  __shared__ float Bs[KC][TILE + 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
  const int wm = (wave >> 1) * 16, wn = (wave & 1) * 16;  // the wave's block
  // consecutive threads walk the operand's contiguous index
  const bool a_kfast = g.a_k == 1, b_nfast = g.b_n == 1;
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = 0; k0 < g.K; k0 += KC) {
    // stage A[m0:m0+32, k0:k0+64] and B[k0:k0+64, n0:n0+32], zero outside
#pragma unroll
    for (int e = tid; e < TILE * KC; e += 256) {
      const int mm = a_kfast ? e / KC : e % TILE;
      const int kk = a_kfast ? e % KC : e / TILE;
      const int m = m0 + mm, k = k0 + kk;
      As[mm][kk] = (m < g.M && k < g.K) ? g.A[m * g.a_m + k * g.a_k] : 0.f;
    }
#pragma unroll
    for (int e = tid; e < TILE * KC; e += 256) {
      const int kk = b_nfast ? e / TILE : e % KC;
      const int nn = b_nfast ? e % TILE : e / KC;
      const int k = k0 + kk, n = n0 + nn;
      Bs[kk][nn] = (n < g.N && k < g.K) ? g.B[k * g.b_k + n * g.b_n] : 0.f;
    }
    __syncthreads();
    // 16 x 16 x 4 MFMA operands: lane l supplies A(row l % 16, k l / 16) and
    // B(k l / 16, col l % 16); the result's lane l holds rows
    // 4 (l / 16) + 0..3 of column l % 16.
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int ks = 0; ks < KC; ks += 4)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(As[wm + r][ks + q], Bs[ks + q][wn + r], acc,
                                                 0, 0, 0);
    __syncthreads();
  }

  const int col = lane & 15, rq = (lane >> 4) * 4;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int m = m0 + wm + rq + e;
    const int n = n0 + wn + col;
    if (m >= g.M || n >= g.N) continue;
    float v = acc[e];
    if (g.epilogue == EP_BIAS || g.epilogue == EP_BIAS_TANH) v += g.bias[n];
    if (g.epilogue == EP_BIAS_TANH) v = tanhf(v);
    if (g.epilogue == EP_DTANH) {
      const float a = g.act[m * g.ldc + n];
      v *= 1.f - a * a;
    }
    g.C[m * g.ldc + n] = v;
  }
}

// gb[o] = sum_b delta[b][o]: a workgroup takes 64 columns, its 4 waves
// every 4th row each (lanes on consecutive columns, loads coalesced), then
// the 4 partial sums meet in LDS
__global__ void __launch_bounds__(256) colsum_kernel(const float* __restrict__ delta, int batch,
                                                     int dout, float* __restrict__ gb) {
  __shared__ float part[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int o = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (o < dout)
    for (int b = wave; b < batch; b += 4) s += delta[(long long)b * dout + o];
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && o < dout) gb[o] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

// delta = 2 (y - t) / (batch * dout); loss partial sums into *loss (FP64)
__global__ void mse_kernel(const float* __restrict__ y, const float* __restrict__ t, long long n,
                           float scale, float* __restrict__ delta, double* __restrict__ loss) {
  __shared__ double red[4];
  double s = 0.0;
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n;
       k += (long long)gridDim.x * blockDim.x) {
    const float e = y[k] - t[k];
    delta[k] = scale * e;
    s += (double)e * e;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int v = 0; v < (int)(blockDim.x >> 6); v++) tot += red[v];
    atomicAdd(loss, tot);
  }
}

// Adam (Kingma & Ba 2015, Algorithm 1) with bias corrections c1, c2
struct AdamArgs {
  float *p, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};

__device__ __forceinline__ float adam_update(const AdamArgs& a, long long k, float gk, float pk,
                                             float mo, float vo) {
  const float mk = a.b1 * mo + (1.f - a.b1) * gk;
  const float vk = a.b2 * vo + (1.f - a.b2) * gk * gk;
  a.m[k] = mk;
  a.v[k] = vk;
  const float pn = pk - a.lr * (mk / a.c1) / (sqrtf(vk / a.c2) + a.eps);
  a.p[k] = pn;
  return pn;
}

__global__ void adam_kernel(long long n, const float* __restrict__ g, AdamArgs a) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n;
       k += (long long)gridDim.x * blockDim.x)
    adam_update(a, k, g[k], a.p[k], a.m[k], a.v[k]);
}

// rows idx[0..batch) of src (row length len) into dst
__global__ void gather_kernel(const float* __restrict__ src, const int* __restrict__ idx,
                              int batch, int len, float* __restrict__ dst) {
  const long long n = (long long)batch * len;
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n;
       k += (long long)gridDim.x * blockDim.x) {
    const long long b = k / len, c = k % len;
    dst[k] = src[(long long)idx[b] * len + c];
  }
}

// ------------------------------------------------------- whole networks
// The rows of a batch are independent up to the weight gradients, so one
// launch takes 16 rows per workgroup through all layers, and in training on
// through the loss and the deltas of every layer, with the activations in LDS:
// a launch per product spent 13-21 us each on 64 workgroups and four memory
// round trips, for 0.5 us of matrix work.
//
// The weights are read in the order of the matrix instruction's operand: tile
// (output block n, input block j) holds, for lane l and element e,
// W(16 n + l % 16, 16 j + 4 e + l / 16): one 16-byte load per lane feeds four
// instructions, and the products are summed in ascending k as gemm_kernel
// does (same bits).  A second copy holds the transpose for the deltas.  Both
// are written with the parameters.  A row of tiles is padded to kRing blocks,
// the loads that a wave keeps in flight: 16 waves x 8 KB cover the latency of
// L2, and the next tile's loads start before the barrier between layers.
//
// Bound by the matrix instructions of the 16 compute units that a batch of 256
// occupies (27 us at 2.4 GHz of the 50 us that 133 - 4 x 256 - 136 takes there,
// forward and deltas; the rest is the barrier and the result of each of the
// nine products).  16 rows are the instruction's least, so a batch of 256
// cannot use more units; rows split over units would meet at every layer.
// With grad_kernel's 12 us a step takes 62 us, 322 us in 23 launches before;
// a forward pass of 592 rows 100 -> 28 us.
constexpr int ROWS = 16;       // rows of a workgroup
constexpr int NET_WAVES = 16;  // waves of a workgroup, one 16-column tile each at a time
static_assert(NET_WAVES == ROWS && NET_WAVES >= 8, "a wave stages a row, and a layer's bias");
constexpr int kRing = 8;
constexpr int kMaxLayers = 8;
constexpr int kMaxLds = 150 * 1024;

inline int blocks16(int n) { return (n + 15) / 16; }
inline long long packed_size(int dout, int din) {  // floats
  return (long long)blocks16(dout) * ((blocks16(din) + kRing - 1) / kRing * kRing) * 256;
}

struct NetPhase {      // one product: forward layer l, then the deltas of layer l
  const float* w;      // packed tiles
  const float* bias;   // forward
  float* out;          // global copy of the result (nullptr: none)
  int J, NB;           // blocks of 16 along the sum and along the outputs
  int cols;            // outputs
  int in, dst, act;    // LDS offsets (floats): input, result; bias or activation (deltas)
};

struct NetArgs {
  int L, phases, batch, din, lds0;
  const float* x;      // input rows
  const int* idx;      // nullptr: row b is x + b * din, else x + idx[b] * din
  float* x_out;        // training: the gathered rows
  const float* t;      // training: targets, indexed as x
  float scale;         // delta = scale (y - t)
  double* loss;
  NetPhase ph[2 * kMaxLayers - 1];
};

__device__ __forceinline__ floatx4 mfma4(float4 a, float4 b, floatx4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
}

template <bool TRAIN>
__global__ void __launch_bounds__(64 * NET_WAVES) net_kernel(NetArgs g) {
  extern __shared__ __align__(16) float lds[];
  __shared__ double red[NET_WAVES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int row0 = blockIdx.x * ROWS;

  auto tile_row = [&](int ph, int nb) {
    const int jp = (g.ph[ph].J + kRing - 1) / kRing * kRing;
    return reinterpret_cast<const float4*>(g.ph[ph].w) + (size_t)nb * jp * 64 + lane;
  };
  // the wave's first tile of a phase at or after `ph`
  int ph_w = 0;
  while (ph_w < g.phases && wave >= g.ph[ph_w].NB) ph_w++;
  const float4* w = tile_row(ph_w < g.phases ? ph_w : 0, ph_w < g.phases ? wave : 0);
  float4 ring[kRing];
#pragma unroll
  for (int e = 0; e < kRing; e++) ring[e] = w[e * 64];

  // Input rows, targets (where their deltas will be) and biases to LDS: wave v
  // loads row v and the bias of layer v, all loads of 256 columns before the
  // first use.  Rows with k = 16 j + 4 e + q at 16 j + 4 q + e, zeros outside.
  {
    const NetPhase& last = g.ph[g.L - 1];
    const NetPhase& mine = g.ph[min(wave, g.L - 1)];
    const int cx = g.ph[0].J * 16, ct = TRAIN ? last.NB * 16 : 0;
    const int cb = wave < g.L ? mine.NB * 16 : 0;
    const int row = row0 + wave;
    const bool live = row < g.batch;
    const long long src = !live ? 0 : g.idx ? g.idx[row] : row;
    const float* px = g.x + src * g.din;
    const float* pt = TRAIN ? g.t + src * last.cols : nullptr;
    for (int k0 = 0; k0 < max(max(cx, ct), cb); k0 += 256) {
      float x[4], t[4], b[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int k = k0 + 64 * c + lane;
        x[c] = t[c] = b[c] = 0.f;
        if (k < cb && k < mine.cols) b[c] = mine.bias[k];
        if (live && k < g.din) x[c] = px[k];
        if (TRAIN && live && k < last.cols) t[c] = pt[k];
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int k = k0 + 64 * c + lane, pos = (k & ~15) + 4 * (k & 3) + ((k >> 2) & 3);
        if (k < cb) lds[mine.act + k] = b[c];
        if (k < cx) lds[g.lds0 + wave * (cx + 4) + pos] = x[c];
        if (k < ct) lds[last.dst + wave * (ct + 4) + pos] = t[c];
        if (TRAIN && live && k < g.din) g.x_out[(long long)row * g.din + k] = x[c];
      }
    }
  }
  __syncthreads();

  double sq = 0.0;
  for (int ph = 0; ph < g.phases; ph++) {
    const NetPhase& f = g.ph[ph];
    const int J = f.J, SA = J * 16 + 4, SO = f.NB * 16 + 4;
    const float4* a = reinterpret_cast<const float4*>(lds + f.in + r * SA + 4 * q);
    for (int nb = wave; nb < f.NB; nb += NET_WAVES) {
      const float4* next = w;  // (no tile left: any)
      if (nb + NET_WAVES < f.NB) {
        next = tile_row(ph, nb + NET_WAVES);
      } else {
        int p2 = ph + 1;
        while (p2 < g.phases && wave >= g.ph[p2].NB) p2++;
        if (p2 < g.phases) next = tile_row(p2, wave);
      }
      floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
      int j0 = 0;
      float4 av[2] = {a[0], a[min(1, J - 1) * 4]};
      for (; j0 + kRing <= J; j0 += kRing) {
        const float4* nx = j0 + kRing < J ? w + (j0 + kRing) * 64 : next;
#pragma unroll
        for (int e = 0; e < kRing; e++) {
          acc = mfma4(av[e & 1], ring[e], acc);
          // after their use: the same registers; and not moved to the group's
          // end, where the scheduler would put them
          ring[e] = nx[e * 64];
          av[e & 1] = a[min(j0 + e + 2, J - 1) * 4];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (j0 < J) {  // the last, partly filled group
#pragma unroll
        for (int e = 0; e < kRing; e++) {
          if (j0 + e < J) {
            acc = mfma4(av[e & 1], ring[e], acc);
            av[e & 1] = a[min(j0 + e + 2, J - 1) * 4];
          }
          ring[e] = next[e * 64];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      w = next;
      // lane holds rows 4 q + e of column n; what the result needs is in LDS: a
      // wait for a load from memory would be one for the ring's, too
      const int n = nb * 16 + r;
      const bool in = n < f.cols;
      const float bias = ph < g.L ? lds[f.act + n] : 0.f;
      const int pos = nb * 16 + 4 * (r & 3) + (r >> 2);
      float* o = lds + f.dst + 4 * q * SO + pos;  // rows 4 q + e: every SO
      const int live = in ? g.batch - row0 - 4 * q : 0;  // rows of the four in the batch
      float v[4];
      if (ph < g.L) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = acc[e] + bias;
        if (ph < g.L - 1) {
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = tanhf(v[e]);
        } else if (TRAIN) {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float err = e < live ? v[e] - o[e * SO] : 0.f;  // o: the target
            v[e] = g.scale * err;
            sq += (double)err * err;
          }
        }
      } else {
        const float* act = lds + f.act + 4 * q * SO + pos;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float y = act[e * SO];
          v[e] = acc[e] * (1.f - y * y);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) o[e * SO] = in ? v[e] : 0.f;
      if (f.out) {
        float* out = f.out + (long long)(row0 + 4 * q) * f.cols + n;
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (e < live) out[(long long)e * f.cols] = v[e];
      }
    }
    __syncthreads();
  }
  if (TRAIN) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sq += __shfl_xor(sq, off);
    if (lane == 0) red[wave] = sq;
    __syncthreads();
    if (tid == 0) {
      double tot = 0.0;
      for (int v = 0; v < NET_WAVES; v++) tot += red[v];
      atomicAdd(g.loss, tot);
    }
  }
}

// The two packed copies of one weight (o, i); `jf`, `jb`: padded blocks of a
// row of tiles.
__device__ __forceinline__ void store_packed(float* wf, float* wb, int jf, int jb, int o, int i,
                                             float v) {
  wf[((long long)(o >> 4) * jf + (i >> 4)) * 256 + ((i & 3) * 16 + (o & 15)) * 4 +
     ((i >> 2) & 3)] = v;
  wb[((long long)(i >> 4) * jb + (o >> 4)) * 256 + ((o & 3) * 16 + (i & 15)) * 4 +
     ((o >> 2) & 3)] = v;
}

struct GradLayer {
  const float *delta, *act;  // batch x dout, batch x din
  float *wf, *wb;            // packed copies
  long long off;             // of the layer's parameters
  int dout, din, jf, jb, tile0, tiles_n;
};

struct GradArgs {
  int L, batch;
  float* g;
  AdamArgs adam;
  GradLayer l[kMaxLayers];
};

// All layers' weight and bias gradients of a batch, and with ADAM the step
// itself: a workgroup takes a 32 x 32 tile of one layer's weights, a wave a
// 16 x 16 block; both operands are contiguous along the block's rows or
// columns, so they go from L2 to the matrix cores without LDS, 16 steps of
// the sum in flight.  The bias gradient is the running sum of the operand
// that the lane loads anyway, in the order of colsum_kernel (rows b = q mod
// 4, then the four parts), the sum over the batch that of gemm_kernel.
template <bool ADAM>
__global__ void __launch_bounds__(256) grad_kernel(GradArgs g) {
  constexpr int G = 16;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int li = 0;
  while (li + 1 < g.L && (int)blockIdx.x >= g.l[li + 1].tile0) li++;
  const GradLayer& l = g.l[li];
  const int tile = blockIdx.x - l.tile0;
  const int o0 = (tile / l.tiles_n) * 32 + (wave >> 1) * 16;
  const int i0 = (tile % l.tiles_n) * 32 + (wave & 1) * 16;
  if (o0 >= l.dout || i0 >= l.din) return;
  const int r = lane & 15, q = lane >> 4;
  // columns outside the layer repeat its last one; their results are dropped
  const float* pa = l.delta + min(o0 + r, l.dout - 1);
  const float* pb = l.act + min(i0 + r, l.din - 1);
  const int i = i0 + r, ob = o0 + 4 * q;  // the lane's column and first row of the result
  float po[4], mo[4], vo[4];
  if (ADAM) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const long long k = l.off + (long long)min(ob + e, l.dout - 1) * l.din + min(i, l.din - 1);
      po[e] = g.adam.p[k];
      mo[e] = g.adam.m[k];
      vo[e] = g.adam.v[k];
    }
  }
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  float sum = 0.f;
  auto load = [&](int b0, float (&a)[G], float (&b)[G]) {
#pragma unroll
    for (int s = 0; s < G; s++) {  // rows past the batch: zeros
      const int row = b0 + 4 * s + q, rc = min(row, g.batch - 1);
      a[s] = pa[(long long)rc * l.dout];
      b[s] = pb[(long long)rc * l.din];
      if (row >= g.batch) a[s] = b[s] = 0.f;
    }
  };
  float a[G], b[G], a2[G], b2[G];
  load(0, a, b);
  for (int b0 = 0; b0 < g.batch; b0 += 4 * G) {
    if (b0 + 4 * G < g.batch) load(b0 + 4 * G, a2, b2);
#pragma unroll
    for (int s = 0; s < G; s++) {
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], acc, 0, 0, 0);
      sum += a[s];
    }
#pragma unroll
    for (int s = 0; s < G; s++) {
      a[s] = a2[s];
      b[s] = b2[s];
    }
  }
  if (i < l.din) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (ob + e >= l.dout) continue;
      const long long k = l.off + (long long)(ob + e) * l.din + i;
      g.g[k] = acc[e];
      if (ADAM) {
        const float pn = adam_update(g.adam, k, acc[e], po[e], mo[e], vo[e]);
        store_packed(l.wf, l.wb, l.jf, l.jb, ob + e, i, pn);
      }
    }
  }
  if (i0 == 0) {
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    const int o = o0 + r;
    if (q == 0 && o < l.dout) {
      const long long k = l.off + (long long)l.dout * l.din + o;
      g.g[k] = sum;
      if (ADAM) adam_update(g.adam, k, sum, g.adam.p[k], g.adam.m[k], g.adam.v[k]);
    }
  }
}

struct PackArgs {
  int L;
  long long n;
  const float *p, *g;  // (g: with ADAM)
  AdamArgs adam;
  struct {
    long long off;
    float *wf, *wb;
    int dout, din, jf, jb;
  } l[kMaxLayers];
};

// The packed copies of all layers' weights, after the parameters were set or,
// with ADAM, together with the step on the gradient held: one launch (an Adam
// step of 133 - 4 x 256 - 136 takes 15 us; with a launch per layer for the
// copies it took 28).
template <bool ADAM>
__global__ void pack_kernel(PackArgs a) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < a.n;
       k += (long long)gridDim.x * blockDim.x) {
    const float v = ADAM ? adam_update(a.adam, k, a.g[k], a.p[k], a.adam.m[k], a.adam.v[k]) : a.p[k];
    int li = 0;
    while (li + 1 < a.L && k >= a.l[li + 1].off) li++;
    const auto& l = a.l[li];
    const int i = static_cast<int>(k - l.off);
    if (i < l.dout * l.din)  // (the layer's bias follows)
      store_packed(l.wf, l.wb, l.jf, l.jb, i / l.din, i % l.din, v);
  }
}

}  // namespace
}  // namespace scft

// ------------------------------------------------------------------ host
using namespace scft;

struct scft_mlp {
  std::vector<int> dims;           // dims[0] inputs ... dims[L] outputs
  std::vector<long long> off;      // parameter offset of each layer
  long long n_params = 0;
  int cap_batch = 0, cap_train = 0;  // rows that the buffers of each pass hold
  float *d_p = nullptr, *d_g = nullptr, *d_m = nullptr, *d_v = nullptr;
  std::vector<float*> d_act;       // L + 1 activation buffers [cap_batch x dims[l]]
  float *d_delta0 = nullptr, *d_delta1 = nullptr, *d_t = nullptr;
  // networks that net_kernel takes: packed weights, deltas of every layer
  bool whole = false;
  int lds_fwd = 0, lds_train = 0;  // bytes
  float* d_pack = nullptr;
  std::vector<long long> pack_f, pack_b;  // offsets in d_pack
  std::vector<float*> d_delta;
  double* d_loss = nullptr;
  int adam_t = 0;
  hipStream_t stream = nullptr;
  // input / output normalisation: x' = (x - xm) / xs, y = y' * ys + ym
  std::vector<float> xm, xs, ym, ys;
};

namespace {
#define MLPCHK(expr)                                                         \
  do {                                                                       \
    hipError_t e_ = (expr);                                                  \
    if (e_ != hipSuccess) {                                                  \
      fprintf(stderr, "scft mlp: %s failed: %s\n", #expr, hipGetErrorString(e_)); \
      return SCFT_E_HIP;                                                     \
    }                                                                        \
  } while (0)

int mlp_dalloc(float** p, long long n) {
  return hipMalloc(reinterpret_cast<void**>(p), sizeof(float) * (n > 0 ? n : 1)) == hipSuccess
             ? SCFT_OK
             : SCFT_E_NOMEM;
}

// Row buffers of a forward pass (the hidden activations of a whole network stay
// in LDS), and what training needs beside them.  A forward pass of many rows
// then does not pay for deltas: 200 000 rows of 133 - 4 x 256 - 136 take 0.2 GB,
// 2.1 GB with everything.
void free_forward(scft_mlp* m) {
  for (size_t l = 0; l < m->d_act.size(); l++) {
    if (m->whole && l > 0 && l + 1 < m->d_act.size()) continue;
    (void)hipFree(m->d_act[l]);
    m->d_act[l] = nullptr;
  }
  m->cap_batch = 0;
}

void free_train(scft_mlp* m) {
  for (size_t l = 1; m->whole && l + 1 < m->d_act.size(); l++) {
    (void)hipFree(m->d_act[l]);
    m->d_act[l] = nullptr;
  }
  for (auto p : m->d_delta) (void)hipFree(p);
  (void)hipFree(m->d_delta0);
  (void)hipFree(m->d_delta1);
  (void)hipFree(m->d_t);
  m->d_delta.assign(m->dims.size() - 1, nullptr);
  m->d_delta0 = m->d_delta1 = m->d_t = nullptr;
  m->cap_train = 0;
}

int ensure_batch(scft_mlp* m, int batch, bool train) {
  const size_t L = m->dims.size() - 1;
  m->d_act.resize(L + 1, nullptr);
  if (batch > m->cap_batch) {
    free_forward(m);
    for (size_t l = 0; l <= L; l++)
      if ((!m->whole || l == 0 || l == L) &&
          mlp_dalloc(&m->d_act[l], (long long)batch * m->dims[l]))
        return SCFT_E_NOMEM;
    m->cap_batch = batch;
  }
  if (train && batch > m->cap_train) {
    free_train(m);
    int widest = 0;
    for (size_t l = 0; l <= L; l++) {
      widest = std::max(widest, m->dims[l]);
      if (m->whole && l > 0 && l < L && mlp_dalloc(&m->d_act[l], (long long)batch * m->dims[l]))
        return SCFT_E_NOMEM;
      if (m->whole && l > 0 && mlp_dalloc(&m->d_delta[l - 1], (long long)batch * m->dims[l]))
        return SCFT_E_NOMEM;
    }
    if (!m->whole && (mlp_dalloc(&m->d_delta0, (long long)batch * widest) ||
                      mlp_dalloc(&m->d_delta1, (long long)batch * widest)))
      return SCFT_E_NOMEM;
    if (mlp_dalloc(&m->d_t, (long long)batch * m->dims.back())) return SCFT_E_NOMEM;
    m->cap_train = batch;
  }
  return SCFT_OK;
}

int ring16(int n) { return (blocks16(n) + kRing - 1) / kRing * kRing; }

// net_kernel takes networks of at most kMaxLayers layers whose activations of
// 16 rows fit in LDS beside two buffers for the running input and delta; the
// default shape (133, 4 x 256, 136) needs 102 KB.  Others go layer by layer.
void plan_whole(scft_mlp* m) {
  const int L = static_cast<int>(m->dims.size()) - 1;
  long long hidden = 0, bias = 0;
  int widest = 0;
  for (int l = 0; l <= L; l++) {
    const int row = blocks16(m->dims[l]) * 16 + 4;
    widest = std::max(widest, row);
    if (l > 0 && l < L) hidden += row;
    if (l > 0) bias += row - 4;
  }
  const long long fwd = (long long)sizeof(float) * (ROWS * 2 * widest + bias);
  const long long train = fwd + (long long)sizeof(float) * ROWS * hidden;
  m->whole = L <= kMaxLayers && train <= kMaxLds;
  m->lds_fwd = m->whole ? static_cast<int>(fwd) : 0;
  m->lds_train = m->whole ? static_cast<int>(train) : 0;
}

// the packed copies of a whole network, with `adam` after a step
int pack(scft_mlp* m, const AdamArgs* adam) {
  if (!m->whole) return SCFT_OK;
  PackArgs a{};
  a.L = static_cast<int>(m->dims.size()) - 1;
  a.n = m->n_params;
  a.p = m->d_p;
  a.g = m->d_g;
  if (adam) a.adam = *adam;
  for (int l = 0; l < a.L; l++) {
    auto& t = a.l[l];
    t.off = m->off[l];
    t.wf = m->d_pack + m->pack_f[l];
    t.wb = m->d_pack + m->pack_b[l];
    t.din = m->dims[l];
    t.dout = m->dims[l + 1];
    t.jf = ring16(t.din);
    t.jb = ring16(t.dout);
  }
  const int grid = static_cast<int>(std::min<long long>(1024, (a.n + 255) / 256));
  if (adam)
    hipLaunchKernelGGL(pack_kernel<true>, dim3(grid), dim3(256), 0, m->stream, a);
  else
    hipLaunchKernelGGL(pack_kernel<false>, dim3(grid), dim3(256), 0, m->stream, a);
  MLPCHK(hipGetLastError());
  return SCFT_OK;
}

// `batch` rows of x (idx: gathered) through the network; t == nullptr: the
// outputs into d_act.back(), else the loss onto *d_loss and every layer's
// input and delta into d_act and d_delta.
int run_net(scft_mlp* m, int batch, const float* x, const float* t, const int* idx) {
  const int L = static_cast<int>(m->dims.size()) - 1;
  NetArgs g{};
  g.L = L;
  g.phases = t ? 2 * L - 1 : L;
  g.batch = batch;
  g.din = m->dims[0];
  g.x = x;
  g.idx = idx;
  g.x_out = t ? m->d_act[0] : nullptr;
  g.t = t;
  g.scale = 2.f / static_cast<float>((long long)batch * m->dims[L]);
  g.loss = m->d_loss;
  int widest = 0;
  for (int d : m->dims) widest = std::max(widest, blocks16(d) * 16 + 4);
  const int buf[2] = {0, ROWS * widest};  // the inputs go to buf[0]
  int act[kMaxLayers];                    // LDS offset of d_act[l]
  act[0] = buf[0];
  int lds = 2 * ROWS * widest;
  for (int l = 0; l < L; l++) {
    g.ph[l].act = lds;
    lds += blocks16(m->dims[l + 1]) * 16;
  }
  for (int l = 1; l < L; l++) {
    act[l] = t ? lds : buf[l & 1];
    lds += ROWS * (blocks16(m->dims[l]) * 16 + 4);
  }
  g.lds0 = act[0];
  for (int l = 0; l < L; l++) {
    NetPhase& f = g.ph[l];
    f.w = m->d_pack + m->pack_f[l];
    f.bias = m->d_p + m->off[l] + (long long)m->dims[l + 1] * m->dims[l];
    f.cols = m->dims[l + 1];
    f.J = blocks16(m->dims[l]);
    f.NB = blocks16(f.cols);
    f.in = act[l];
    f.dst = l + 1 < L ? act[l + 1] : t ? buf[1] : buf[L & 1];
    f.out = t ? (l + 1 < L ? m->d_act[l + 1] : m->d_delta[l]) : l + 1 < L ? nullptr : m->d_act[L];
  }
  for (int l = L - 1, ph = L, k = 1; t && l > 0; l--, ph++, k ^= 1) {  // deltas of layer l - 1
    NetPhase& f = g.ph[ph];
    f.w = m->d_pack + m->pack_b[l];
    f.cols = m->dims[l];
    f.J = blocks16(m->dims[l + 1]);
    f.NB = blocks16(f.cols);
    f.in = buf[k];
    f.dst = buf[k ^ 1];
    f.act = act[l];
    f.out = m->d_delta[l - 1];
  }
  const dim3 grid((batch + ROWS - 1) / ROWS), block(64 * NET_WAVES);
  if (t)
    hipLaunchKernelGGL(net_kernel<true>, grid, block, m->lds_train, m->stream, g);
  else
    hipLaunchKernelGGL(net_kernel<false>, grid, block, m->lds_fwd, m->stream, g);
  MLPCHK(hipGetLastError());
  return SCFT_OK;
}

AdamArgs adam_args(const scft_mlp* m, float lr) {
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)m->adam_t);
  const float c2 = 1.f - std::pow(b2, (float)m->adam_t);
  return AdamArgs{m->d_p, m->d_m, m->d_v, lr, b1, b2, 1e-8f, c1, c2};
}

// the gradients of the batch that run_net left, and with `adam` the step
int run_grad(scft_mlp* m, int batch, const AdamArgs* adam) {
  GradArgs g{};
  g.L = static_cast<int>(m->dims.size()) - 1;
  g.batch = batch;
  g.g = m->d_g;
  if (adam) g.adam = *adam;
  int tiles = 0;
  for (int l = 0; l < g.L; l++) {
    GradLayer& a = g.l[l];
    a.delta = m->d_delta[l];
    a.act = m->d_act[l];
    a.wf = m->d_pack + m->pack_f[l];
    a.wb = m->d_pack + m->pack_b[l];
    a.off = m->off[l];
    a.din = m->dims[l];
    a.dout = m->dims[l + 1];
    a.jf = ring16(a.din);
    a.jb = ring16(a.dout);
    a.tile0 = tiles;
    a.tiles_n = (a.din + 31) / 32;
    tiles += a.tiles_n * ((a.dout + 31) / 32);
  }
  if (adam)
    hipLaunchKernelGGL(grad_kernel<true>, dim3(tiles), dim3(256), 0, m->stream, g);
  else
    hipLaunchKernelGGL(grad_kernel<false>, dim3(tiles), dim3(256), 0, m->stream, g);
  MLPCHK(hipGetLastError());
  return SCFT_OK;
}

hipError_t gemm(hipStream_t s, const float* A, long long a_m, long long a_k, const float* B,
                long long b_k, long long b_n, float* C, long long ldc, int M, int N, int K,
                int ep, const float* bias, const float* act) {
  GemmArgs g{A, a_m, a_k, B, b_k, b_n, C, ldc, M, N, K, ep, bias, act};
  dim3 grid((N + TILE - 1) / TILE, (M + TILE - 1) / TILE);
  hipLaunchKernelGGL(gemm_kernel, grid, dim3(256), 0, s, g);
  return hipGetLastError();
}

// forward of `batch` rows already in d_act[0], layer by layer; activations kept
// for backward
int forward(scft_mlp* m, int batch) {
  const int L = static_cast<int>(m->dims.size()) - 1;
  for (int l = 0; l < L; l++) {
    const int din = m->dims[l], dout = m->dims[l + 1];
    const float* W = m->d_p + m->off[l];
    const float* b = W + (long long)dout * din;
    MLPCHK(gemm(m->stream, m->d_act[l], din, 1, W, 1, din, m->d_act[l + 1], dout, batch, dout,
                din, l < L - 1 ? EP_BIAS_TANH : EP_BIAS, b, nullptr));
  }
  return SCFT_OK;
}

// loss and gradient for the rows in d_act[0] against targets in d_t; the
// squared error is added to *d_loss, which is cleared first unless the
// caller accumulates over several batches
int backward(scft_mlp* m, int batch, bool clear_loss = true) {
  const int L = static_cast<int>(m->dims.size()) - 1;
  const int dl = m->dims[L];
  const long long n = (long long)batch * dl;
  if (clear_loss) MLPCHK(hipMemsetAsync(m->d_loss, 0, sizeof(double), m->stream));
  hipLaunchKernelGGL(mse_kernel, dim3(64), dim3(256), 0, m->stream, m->d_act[L], m->d_t, n,
                     2.f / static_cast<float>(n), m->d_delta0, m->d_loss);
  MLPCHK(hipGetLastError());
  float* delta = m->d_delta0;
  float* other = m->d_delta1;
  for (int l = L - 1; l >= 0; l--) {
    const int din = m->dims[l], dout = m->dims[l + 1];
    const float* W = m->d_p + m->off[l];
    float* gW = m->d_g + m->off[l];
    float* gb = gW + (long long)dout * din;
    // gW[o][i] = sum_b delta[b][o] act_l[b][i]
    MLPCHK(gemm(m->stream, delta, 1, dout, m->d_act[l], din, 1, gW, din, dout, din, batch,
                EP_NONE, nullptr, nullptr));
    hipLaunchKernelGGL(colsum_kernel, dim3((dout + 63) / 64), dim3(256), 0, m->stream, delta,
                       batch, dout, gb);
    MLPCHK(hipGetLastError());
    if (l > 0) {  // delta_prev[b][i] = sum_o delta[b][o] W[o][i] * (1 - act_l[b][i]^2)
      MLPCHK(gemm(m->stream, delta, dout, 1, W, din, 1, other, din, batch, din, dout, EP_DTANH,
                  nullptr, m->d_act[l]));
      std::swap(delta, other);
    }
  }
  return SCFT_OK;
}

void normalise_rows(const scft_mlp* m, const float* X, int rows, std::vector<float>& out) {
  const int din = m->dims[0];
  out.resize((size_t)rows * din);
  for (int r = 0; r < rows; r++)
    for (int i = 0; i < din; i++) {
      const float v = X[(size_t)r * din + i];
      out[(size_t)r * din + i] = m->xm.empty() ? v : (v - m->xm[i]) / m->xs[i];
    }
}

uint64_t splitmix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
}  // namespace

extern "C" int scft_mlp_create(scft_mlp** out, int n_layers, const int* dims,
                               unsigned long long seed) {
  if (!out || n_layers < 1 || !dims) return SCFT_E_ARG;
  for (int l = 0; l <= n_layers; l++)
    if (dims[l] < 1 || dims[l] > 4096) return SCFT_E_ARG;
  scft_mlp* m = new scft_mlp;
  m->dims.assign(dims, dims + n_layers + 1);
  m->off.resize(n_layers + 1);
  long long o = 0;
  for (int l = 0; l < n_layers; l++) {
    m->off[l] = o;
    o += (long long)dims[l + 1] * dims[l] + dims[l + 1];
  }
  m->off[n_layers] = o;
  m->n_params = o;
  plan_whole(m);
  long long np = 0;
  for (int l = 0; l < n_layers && m->whole; l++) {
    m->pack_f.push_back(np);
    np += packed_size(dims[l + 1], dims[l]);
    m->pack_b.push_back(np);
    np += packed_size(dims[l], dims[l + 1]);
  }
  // Glorot-uniform weights, zero biases, from splitmix64(seed)
  std::vector<float> p(o, 0.f);
  uint64_t s = seed;
  for (int l = 0; l < n_layers; l++) {
    const double lim = std::sqrt(6.0 / (dims[l] + dims[l + 1]));
    for (long long k = 0; k < (long long)dims[l + 1] * dims[l]; k++) {
      const double u = (splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
      p[m->off[l] + k] = static_cast<float>((2.0 * u - 1.0) * lim);
    }
  }
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
      mlp_dalloc(&m->d_p, o) || mlp_dalloc(&m->d_g, o) || mlp_dalloc(&m->d_m, o) ||
      mlp_dalloc(&m->d_v, o) || mlp_dalloc(&m->d_pack, np) ||
      hipMalloc(reinterpret_cast<void**>(&m->d_loss), sizeof(double)) != hipSuccess) {
    delete m;
    return SCFT_E_NOMEM;
  }
  if (hipMemcpy(m->d_p, p.data(), sizeof(float) * o, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(m->d_m, 0, sizeof(float) * o) != hipSuccess ||
      hipMemset(m->d_v, 0, sizeof(float) * o) != hipSuccess ||
      (np > 0 && hipMemset(m->d_pack, 0, sizeof(float) * np) != hipSuccess) ||
      hipStreamSynchronize(nullptr) != hipSuccess || pack(m, nullptr)) {
    delete m;
    return SCFT_E_HIP;
  }
  if (m->whole) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(net_kernel<true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(net_kernel<false>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
  }
  *out = m;
  return SCFT_OK;
}

extern "C" int scft_mlp_destroy(scft_mlp* m) {
  if (!m) return SCFT_OK;
  (void)hipStreamSynchronize(m->stream);
  free_forward(m);
  free_train(m);
  (void)hipFree(m->d_pack);
  (void)hipFree(m->d_p);
  (void)hipFree(m->d_g);
  (void)hipFree(m->d_m);
  (void)hipFree(m->d_v);
  (void)hipFree(m->d_loss);
  (void)hipStreamDestroy(m->stream);
  delete m;
  return SCFT_OK;
}

extern "C" int scft_mlp_param_count(const scft_mlp* m, long long* count) {
  if (!m || !count) return SCFT_E_ARG;
  *count = m->n_params;
  return SCFT_OK;
}

extern "C" int scft_mlp_get_params(const scft_mlp* m, float* out) {
  if (!m || !out) return SCFT_E_ARG;
  MLPCHK(hipStreamSynchronize(m->stream));
  MLPCHK(hipMemcpy(out, m->d_p, sizeof(float) * m->n_params, hipMemcpyDeviceToHost));
  return SCFT_OK;
}

extern "C" int scft_mlp_set_params(scft_mlp* m, const float* in) {
  if (!m || !in) return SCFT_E_ARG;
  const size_t bytes = sizeof(float) * m->n_params;
  MLPCHK(hipMemcpyAsync(m->d_p, in, bytes, hipMemcpyHostToDevice, m->stream));
  MLPCHK(hipMemsetAsync(m->d_m, 0, bytes, m->stream));
  MLPCHK(hipMemsetAsync(m->d_v, 0, bytes, m->stream));
  m->adam_t = 0;
  if (int rc = pack(m, nullptr)) return rc;
  MLPCHK(hipStreamSynchronize(m->stream));
  return SCFT_OK;
}

extern "C" int scft_mlp_set_normalisation(scft_mlp* m, const float* x_mean, const float* x_std,
                                          const float* y_mean, const float* y_std) {
  if (!m) return SCFT_E_ARG;
  const int din = m->dims.front(), dout = m->dims.back();
  if (!x_mean || !x_std || !y_mean || !y_std) {
    m->xm.clear();
    m->xs.clear();
    m->ym.clear();
    m->ys.clear();
    return SCFT_OK;
  }
  for (int i = 0; i < din; i++)
    if (!(x_std[i] > 0.f)) return SCFT_E_ARG;
  for (int i = 0; i < dout; i++)
    if (!(y_std[i] > 0.f)) return SCFT_E_ARG;
  m->xm.assign(x_mean, x_mean + din);
  m->xs.assign(x_std, x_std + din);
  m->ym.assign(y_mean, y_mean + dout);
  m->ys.assign(y_std, y_std + dout);
  return SCFT_OK;
}

extern "C" int scft_mlp_forward(scft_mlp* m, int batch, const float* X, float* Y) {
  if (!m || batch < 1 || !X || !Y) return SCFT_E_ARG;
  if (int rc = ensure_batch(m, batch, false)) return rc;
  std::vector<float> xn;
  normalise_rows(m, X, batch, xn);
  MLPCHK(hipMemcpyAsync(m->d_act[0], xn.data(), sizeof(float) * xn.size(),
                        hipMemcpyHostToDevice, m->stream));
  if (int rc = m->whole ? run_net(m, batch, m->d_act[0], nullptr, nullptr) : forward(m, batch))
    return rc;
  const int dout = m->dims.back();
  MLPCHK(hipMemcpyAsync(Y, m->d_act.back(), sizeof(float) * (size_t)batch * dout,
                        hipMemcpyDeviceToHost, m->stream));
  MLPCHK(hipStreamSynchronize(m->stream));
  if (!m->ym.empty())
    for (int r = 0; r < batch; r++)
      for (int o = 0; o < dout; o++) Y[(size_t)r * dout + o] = Y[(size_t)r * dout + o] *
                                                                    m->ys[o] + m->ym[o];
  return SCFT_OK;
}

// Forward pass for the device-side warm-start prediction (scft_internal.h).
int scft_mlp_forward_resident(scft_mlp* m, int batch, const float* d_xn, const float** d_out,
                              const float** ym, const float** ys, int* n_out, int* n_in) {
  if (!m || batch < 1 || !d_xn || !d_out) return SCFT_E_ARG;
  if (int rc = ensure_batch(m, batch, false)) return rc;
  const int din = m->dims.front();
  if (m->whole) {
    if (int rc = run_net(m, batch, d_xn, nullptr, nullptr)) return rc;
  } else {
    MLPCHK(hipMemcpyAsync(m->d_act[0], d_xn, sizeof(float) * (size_t)batch * din,
                          hipMemcpyDeviceToDevice, m->stream));
    if (int rc = forward(m, batch)) return rc;
  }
  MLPCHK(hipStreamSynchronize(m->stream));
  *d_out = m->d_act.back();
  if (ym) *ym = m->ym.empty() ? nullptr : m->ym.data();
  if (ys) *ys = m->ys.empty() ? nullptr : m->ys.data();
  if (n_out) *n_out = m->dims.back();
  if (n_in) *n_in = din;
  return SCFT_OK;
}

// x' = (x - xm) / xs of `rows` host rows, as scft_mlp_forward applies it.
int scft_mlp_normalise_inputs(const scft_mlp* m, const float* X, int rows, float* out) {
  if (!m || !X || !out || rows < 0) return SCFT_E_ARG;
  std::vector<float> xn;
  normalise_rows(m, X, rows, xn);
  std::copy(xn.begin(), xn.end(), out);
  return SCFT_OK;
}

// Loss and gradient on raw (already normalised) rows, for gradient checks:
// no normalisation is applied here.
extern "C" int scft_mlp_loss_grad(scft_mlp* m, int batch, const float* X, const float* T,
                                  double* loss, float* grad) {
  if (!m || batch < 1 || !X || !T) return SCFT_E_ARG;
  if (int rc = ensure_batch(m, batch, true)) return rc;
  const int din = m->dims.front(), dout = m->dims.back();
  MLPCHK(hipMemcpyAsync(m->d_act[0], X, sizeof(float) * (size_t)batch * din,
                        hipMemcpyHostToDevice, m->stream));
  MLPCHK(hipMemcpyAsync(m->d_t, T, sizeof(float) * (size_t)batch * dout, hipMemcpyHostToDevice,
                        m->stream));
  if (m->whole) {
    MLPCHK(hipMemsetAsync(m->d_loss, 0, sizeof(double), m->stream));
    if (int rc = run_net(m, batch, m->d_act[0], m->d_t, nullptr)) return rc;
    if (int rc = run_grad(m, batch, nullptr)) return rc;
  } else {
    if (int rc = forward(m, batch)) return rc;
    if (int rc = backward(m, batch)) return rc;
  }
  double l = 0.0;
  MLPCHK(hipMemcpyAsync(&l, m->d_loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  if (grad)
    MLPCHK(hipMemcpyAsync(grad, m->d_g, sizeof(float) * m->n_params, hipMemcpyDeviceToHost,
                          m->stream));
  MLPCHK(hipStreamSynchronize(m->stream));
  if (loss) *loss = l / ((double)batch * dout);
  return SCFT_OK;
}

// One Adam step on the gradient currently held (after scft_mlp_loss_grad).
extern "C" int scft_mlp_adam_step(scft_mlp* m, float lr) {
  if (!m) return SCFT_E_ARG;
  m->adam_t++;
  const AdamArgs adam = adam_args(m, lr);
  if (m->whole) {
    if (int rc = pack(m, &adam)) return rc;
  } else {
    hipLaunchKernelGGL(adam_kernel, dim3(256), dim3(256), 0, m->stream, m->n_params, m->d_g, adam);
    MLPCHK(hipGetLastError());
  }
  MLPCHK(hipStreamSynchronize(m->stream));
  return SCFT_OK;
}

// Mini-batch Adam over n_samples rows (normalised with the object's
// statistics when set), reshuffled every epoch from splitmix64(seed); the
// last partial batch of an epoch is used as is.  epoch_loss[e] (nullable)
// receives the mean loss of epoch e in normalised units.
extern "C" int scft_mlp_train(scft_mlp* m, int n_samples, const float* X, const float* Y,
                              int epochs, int batch, float lr, unsigned long long seed,
                              double* epoch_loss) {
  if (!m || n_samples < 1 || !X || !Y || epochs < 1 || batch < 1 || !(lr > 0.f))
    return SCFT_E_ARG;
  const int din = m->dims.front(), dout = m->dims.back();
  if (int rc = ensure_batch(m, batch, true)) return rc;
  std::vector<float> xn, yn((size_t)n_samples * dout);
  normalise_rows(m, X, n_samples, xn);
  for (int r = 0; r < n_samples; r++)
    for (int o = 0; o < dout; o++) {
      const float v = Y[(size_t)r * dout + o];
      yn[(size_t)r * dout + o] = m->ym.empty() ? v : (v - m->ym[o]) / m->ys[o];
    }
  float *dX = nullptr, *dY = nullptr;
  int* dIdx = nullptr;
  if (mlp_dalloc(&dX, (long long)n_samples * din) || mlp_dalloc(&dY, (long long)n_samples * dout) ||
      hipMalloc(reinterpret_cast<void**>(&dIdx), sizeof(int) * n_samples) != hipSuccess) {
    (void)hipFree(dX);
    (void)hipFree(dY);
    return SCFT_E_NOMEM;
  }
  int rc = SCFT_OK;
  std::vector<int> idx(n_samples);
  for (int i = 0; i < n_samples; i++) idx[i] = i;
  uint64_t s = seed;
  if (hipMemcpy(dX, xn.data(), sizeof(float) * xn.size(), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dY, yn.data(), sizeof(float) * yn.size(), hipMemcpyHostToDevice) != hipSuccess)
    rc = SCFT_E_HIP;
  for (int e = 0; e < epochs && rc == SCFT_OK; e++) {
    for (int i = n_samples - 1; i > 0; i--) {  // Fisher-Yates
      const int j = static_cast<int>(splitmix(s) % static_cast<uint64_t>(i + 1));
      std::swap(idx[i], idx[j]);
    }
    if (hipMemcpyAsync(dIdx, idx.data(), sizeof(int) * n_samples, hipMemcpyHostToDevice,
                       m->stream) != hipSuccess) {
      rc = SCFT_E_HIP;
      break;
    }
    // the epoch's squared error accumulates on the device and is read once
    // at its end: the steps queue without a host round trip between them
    if (hipMemsetAsync(m->d_loss, 0, sizeof(double), m->stream) != hipSuccess) {
      rc = SCFT_E_HIP;
      break;
    }
    for (int b0 = 0; b0 < n_samples && rc == SCFT_OK; b0 += batch) {
      const int nb = std::min(batch, n_samples - b0);
      if (m->whole) {  // two launches: rows, then weights
        m->adam_t++;
        const AdamArgs adam = adam_args(m, lr);
        if (run_net(m, nb, dX, dY, dIdx + b0) || run_grad(m, nb, &adam)) rc = SCFT_E_HIP;
        continue;
      }
      hipLaunchKernelGGL(gather_kernel, dim3(128), dim3(256), 0, m->stream, dX, dIdx + b0, nb,
                         din, m->d_act[0]);
      hipLaunchKernelGGL(gather_kernel, dim3(128), dim3(256), 0, m->stream, dY, dIdx + b0, nb,
                         dout, m->d_t);
      if (hipGetLastError() != hipSuccess || forward(m, nb) || backward(m, nb, false)) {
        rc = SCFT_E_HIP;
        break;
      }
      m->adam_t++;
      hipLaunchKernelGGL(adam_kernel, dim3(256), dim3(256), 0, m->stream, m->n_params, m->d_g,
                         adam_args(m, lr));
      if (hipGetLastError() != hipSuccess) rc = SCFT_E_HIP;
    }
    // also orders the next epoch's host shuffle after this epoch's index copy
    double esum = 0.0;
    if (rc == SCFT_OK &&
        (hipMemcpyAsync(&esum, m->d_loss, sizeof(double), hipMemcpyDeviceToHost, m->stream) !=
             hipSuccess ||
         hipStreamSynchronize(m->stream) != hipSuccess))
      rc = SCFT_E_HIP;
    if (epoch_loss && rc == SCFT_OK)
      epoch_loss[e] = esum / (static_cast<double>(n_samples) * dout);
  }
  (void)hipStreamSynchronize(m->stream);
  (void)hipFree(dX);
  (void)hipFree(dY);
  (void)hipFree(dIdx);
  return rc;
}
