// diff.hip -- differentiable full render (training mode) and its adjoint.
//
// Forward, for a list of pixels (y * W + x) of one camera, with FP32
// parameter blocks in the nerfacc layout (hash table [entries][2], density
// MLP W1|W2|W3, colour MLP H1|H2, row-major [out][in]) owned by the caller:
//   k_diff_count   ray setup (initRayPayloads_split_kernel, renderer.cu:86-
//                  134) and the occupancy march of sample_performance_kernel
//                  (performance_renderer.cu:15-69) to the far bound, counting
//                  the occupied samples per ray;
//   exclusive scan of the counts (hipCUB);
//   k_diff_emit    the same march again, writing each sample's contracted
//                  midpoint, step size and ray;
//   k_diff_net_fwd hash-grid encoding + both MLPs in FP32 on the 16x16x4 f32
//                  MFMA: (colour logits, log density) per sample;
//   k_diff_composite  accumulate_performance_kernel (performance_renderer.cu:
//                  71-125) per ray, stopping at T < 1e-4; output C + T (the
//                  white background of applyWhiteBackground).
// Backward, for dL/d(C + T):
//   k_diff_composite_bwd  per ray, dL/d(logits, log density) per sample:
//                  dC/dc_i = w_i and dC/dsigma_i = dt_i (T_{i+1} c_i - S_i),
//                  S_i = (C + T) - sum_{j<=i} w_j c_j; sigmoid' and exp';
//   k_diff_net_bwd per 16 samples: the forward recomputed (no activation is
//                  stored), the chain back through the colour MLP, the
//                  density MLP (ReLU' = [pre-activation > 0]) and the
//                  encoding, on MFMA with transposed-weight fragments; weight
//                  gradients dW = sum_s dY_s X_s^T as MFMA over the samples
//                  (operands transposed through LDS), summed in registers,
//                  then added to the caller's gradient;
//   k_diff_scatter the encoding's gradients through the trilinear weights
//                  into the hash table's gradient with FP32 atomics.
// Samples skipped by alpha_thre and samples after termination carry no
// gradient (the branch decisions are constants of the forward pass).
//
// MFMA operand layout (v_mfma_f32_16x16x4_f32, transposed formulation
// D[neuron][sample] = W[neuron][k] X[k][sample]): lane l = (col = l % 16,
// g = l / 16); A: W[row(i = col)][k(slot, g)], B: X[k(slot, g)][sample col],
// D: rows 4g..4g+3 of a 16-row block for sample col.  A layer's D blocks are
// the next layer's B slots (slot 4 nb + e = block nb element e), so each
// weight matrix is packed once per call into fragments whose k order
// follows the slots (k_diff_pack, from index tables built on the host).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "fvc_internal.h"
#include "march.h"
#include "mlp_mfma.h"
#include "render_common.h"
#include "wave.h"

namespace fvc {

// ------------------------------------------------------------ fragments
enum {
  F_W1 = 0,     // 4 blocks x 8 slots (encoding)
  F_W2 = 32,    // 4 x 16
  F_W3 = 96,    // 1 x 16
  F_H1 = 112,   // 4 x 8 (head input)
  F_H2 = 144,   // 1 x 16
  B_H2T = 160,  // 4 blocks (d hidden) x 4 slots (16 outputs)
  B_H1T = 176,  // 1 block (latent / padding inputs) x 16 slots
  B_W3T = 192,  // 4 x 4
  B_W2T = 208,  // 4 x 16
  B_W1T = 272,  // 2 blocks (encoding, quad-level order) x 16
  N_DIFF_FRAGS = 304,
  N_FWD_FRAGS = 160,             // the forward's fragments come first
  N_HEAD_FRAGS = B_W3T - F_H1    // the colour MLP's, forward and backward
};

// k index of slot m in lane group g
static int k_chain(int m, int g) { return 16 * (m / 4) + 4 * g + (m % 4); }
static int k_enc(int m, int g) { return 2 * (g + 4 * (m / 2)) + (m % 2); }  // level g + 4 (m/2), feature m % 2
static int k_head(int m, int g) {                                        // head input column
  if (m >= 4) return 8 + 4 * g + (m - 4);                                // SH coefficient
  const int r = 4 * g + m;                                               // base output row
  if (r >= 1 && r <= 8) return r - 1;                                    // latent r - 1
  return r == 0 ? 24 : r + 16;                                           // 1.0 padding columns
}
// encoding feature of row i of d_enc block nb (the encoder's slot order)
static int row_enc(int nb, int i) { return k_enc(4 * nb + (i % 4), i / 4); }
// head input feature of row i of the d_head_input block
static int row_head(int i) { return k_head(i % 4, i / 4); }

// Index of every fragment value in the concatenated parameters
// [mlp_base | mlp_head] (-1: zero).  Fragments f .. f + 3 (f a multiple of 4,
// slots m .. m + 3 of one block) lie together per lane, so a lane reads four
// slots' operands with one 16-byte load.
std::vector<int> diff_frag_index() {
  const int n_base = 32 * 64 + 64 * 64 + 64 * 16;
  const int W1 = 0, W2 = 32 * 64, W3 = 32 * 64 + 64 * 64, H1 = n_base, H2 = n_base + 32 * 64;
  std::vector<int> t((size_t)N_DIFF_FRAGS * 64, -1);
  auto put = [&](int f0, int n_blocks, int n_slots, auto val) {
    for (int nb = 0; nb < n_blocks; nb++)
      for (int m = 0; m < n_slots; m++)
        for (int lane = 0; lane < 64; lane++) {
          const size_t f = (size_t)(f0 + nb * n_slots + m);
          t[((f >> 2) * 64 + lane) * 4 + (f & 3)] = val(nb, m, lane % 16, lane / 16);
        }
  };
  // forward: A = W[16 nb + i][k(m, g)]
  put(F_W1, 4, 8, [&](int nb, int m, int i, int g) { return W1 + (16 * nb + i) * 32 + k_enc(m, g); });
  put(F_W2, 4, 16, [&](int nb, int m, int i, int g) { return W2 + (16 * nb + i) * 64 + k_chain(m, g); });
  put(F_W3, 1, 16, [&](int, int m, int i, int g) { return W3 + i * 64 + k_chain(m, g); });
  put(F_H1, 4, 8, [&](int nb, int m, int i, int g) { return H1 + (16 * nb + i) * 32 + k_head(m, g); });
  put(F_H2, 1, 16, [&](int, int m, int i, int g) { return H2 + i * 64 + k_chain(m, g); });
  // backward: A = W^T[row][k(m, g)] = W[k(m, g)][row]
  put(B_H2T, 4, 4, [&](int nb, int m, int i, int g) { return H2 + k_chain(m, g) * 64 + 16 * nb + i; });
  put(B_H1T, 1, 16, [&](int, int m, int i, int g) { return H1 + k_chain(m, g) * 32 + row_head(i); });
  put(B_W3T, 4, 4, [&](int nb, int m, int i, int g) { return W3 + k_chain(m, g) * 64 + 16 * nb + i; });
  put(B_W2T, 4, 16, [&](int nb, int m, int i, int g) { return W2 + k_chain(m, g) * 64 + 16 * nb + i; });
  put(B_W1T, 2, 16, [&](int nb, int m, int i, int g) { return W1 + k_chain(m, g) * 32 + row_enc(nb, i); });
  return t;
}

__global__ void k_diff_pack(const int* __restrict__ idx, const float* __restrict__ base,
                            const float* __restrict__ head, int n_base, float* __restrict__ frags) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= N_DIFF_FRAGS * 64) return;
  const int k = idx[s];
  frags[s] = k < 0 ? 0.0f : (k < n_base ? base[k] : head[k - n_base]);
}

// ------------------------------------------------------------ device math
__device__ __forceinline__ f4 mma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// NB output blocks from M input slots with the fragments of a layer at fr (in
// LDS; slots 4q..4q+3 of block nb at fr[(nb * M / 4 + q) * 64 + lane]).  The
// lane index is made opaque per call so that the reads of a layer are not
// hoisted into registers across the sample loop.
template <int NB, int M>
__device__ __forceinline__ void dense4(const float4* fr, int lane_, const float* x, f4* y) {
  const int lane = opaque(lane_);
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    f4 acc = f4zero();
#pragma unroll
    for (int q = 0; q < M / 4; q++) {
      const float4 a = fr[(nb * (M / 4) + q) * 64 + lane];
      acc = mma4(a.x, x[4 * q], acc);
      acc = mma4(a.y, x[4 * q + 1], acc);
      acc = mma4(a.z, x[4 * q + 2], acc);
      acc = mma4(a.w, x[4 * q + 3], acc);
    }
    y[nb] = acc;
  }
}
// the fragments [f0, f0 + n) of the packed table into LDS (every thread of the block)
__device__ __forceinline__ void stage_diff_frags(const float* __restrict__ frags, int f0, int n, float4* lds) {
  const float4* src = reinterpret_cast<const float4*>(frags) + f0 * 16;
  for (int i = threadIdx.x; i < n * 16; i += blockDim.x) lds[i] = src[i];
}
template <int NB> __device__ __forceinline__ void relu_slots(const f4* y, float* x) {
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int e = 0; e < 4; e++) x[4 * nb + e] = relu_bits(y[nb][e]);
}
template <int NB> __device__ __forceinline__ void relu_grad(const f4* pre, f4* d) {
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int e = 0; e < 4; e++) d[nb][e] = pre[nb][e] > 0.0f ? d[nb][e] : 0.0f;
}

// SH degree 4 coefficients 4g..4g+3 of dir01 * 2 - 1 in FP32
// (my_fully_fused_mlp.cu:206-234)
__device__ __forceinline__ void sh4_quarter_f32(V3 d01, int g, float* o) {
  const float x = d01.x * 2.0f - 1.0f, y = d01.y * 2.0f - 1.0f, z = d01.z * 2.0f - 1.0f;
  const float xy = x * y, xz = x * z, yz = y * z, x2 = x * x, y2 = y * y, z2 = z * z;
  if (g == 0) {
    o[0] = 0.28209479177387814f;
    o[1] = -0.48860251190291987f * y;
    o[2] = 0.48860251190291987f * z;
    o[3] = -0.48860251190291987f * x;
  } else if (g == 1) {
    o[0] = 1.0925484305920792f * xy;
    o[1] = -1.0925484305920792f * yz;
    o[2] = 0.94617469575755997f * z2 - 0.31539156525251999f;
    o[3] = -1.0925484305920792f * xz;
  } else if (g == 2) {
    o[0] = 0.54627421529603959f * x2 - 0.54627421529603959f * y2;
    o[1] = 0.59004358992664352f * y * (-3.0f * x2 + y2);
    o[2] = 2.8906114426405538f * xy * z;
    o[3] = 0.45704579946446572f * y * (1.0f - 5.0f * z2);
  } else {
    o[0] = 0.3731763325901154f * z * (5.0f * z2 - 3.0f);
    o[1] = 0.45704579946446572f * x * (1.0f - 5.0f * z2);
    o[2] = 1.4453057213202769f * z * (x2 - y2);
    o[3] = 0.59004358992664352f * x * (-x2 + 3.0f * y2);
  }
}

// Corners of levels g, g+4, g+8, g+12 at p (clamped to [0,1]^3): entry
// index (table entries) and trilinear weight, corner bits x=1, y=2, z=4
// (tcnn GridEncoding, the hash of the iNGP paper).
__device__ __forceinline__ void quad_corners(const GridLevel* __restrict__ lv, const GridParams& gp, V3 p, int g,
                                             uint32_t (&idx)[4][8], float (&w)[4][8]) {
  const float px = fminf_(fmaxf_(p.x, 0.0f), 1.0f);
  const float py = fminf_(fmaxf_(p.y, 0.0f), 1.0f);
  const float pz = fminf_(fmaxf_(p.z, 0.0f), 1.0f);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int l = 4 * j + g;
    const GridLevel L = lv[l];
    const float ax = px * L.scale + 0.5f, ay = py * L.scale + 0.5f, az = pz * L.scale + 0.5f;
    const float fx = floorf(ax), fy = floorf(ay), fz = floorf(az);
    const uint32_t gx = (uint32_t)(int)fx, gy = (uint32_t)(int)fy, gz = (uint32_t)(int)fz;
    const float wx = ax - fx, wy = ay - fy, wz = az - fz;
    const float ux = 1.0f - wx, uy = 1.0f - wy, uz = 1.0f - wz;
    const float wxy[4] = {ux * uy, wx * uy, ux * wy, wx * wy};
    const bool dense = (gp.dense_mask >> l) & 1u;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const uint32_t x = gx + (c & 1), y = gy + ((c >> 1) & 1), z = gz + (c >> 2);
      uint32_t t;
      if (dense) {
        t = x + y * L.res + z * L.res2;
        t = t % L.size;
      } else {
        t = (x ^ (y * 2654435761u) ^ (z * 805459861u)) & (L.size - 1u);
      }
      idx[j][c] = L.offset + t;
      w[j][c] = wxy[c & 3] * ((c & 4) ? wz : uz);
    }
  }
}

// network forward of one 16-sample tile; activations kept for the backward
struct FwdActs {
  float enc[8];
  f4 a1[4], a2[4], out, z1[4], o;
  float xh[8];
};

// colour MLP on the base-output rows 4g..4g+3 in `rows` (rows 1..8 are the
// latents; row 0 and rows 9..15 give way to the 1.0 padding inputs)
// fr: the staged fragments from fragment F0 on
template <int F0>
__device__ __forceinline__ void head_forward(const float4* fr, int lane, int g, f4 rows, V3 d01, FwdActs& a) {
  float sh[4], h[16];
  sh4_quarter_f32(d01, g, sh);
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const int r = 4 * g + m;
    a.xh[m] = (r >= 1 && r <= 8) ? rows[m] : 1.0f;
    a.xh[4 + m] = sh[m];
  }
  dense4<4, 8>(fr + (F_H1 - F0) * 16, lane, a.xh, a.z1);
  relu_slots<4>(a.z1, h);
  dense4<1, 16>(fr + (F_H2 - F0) * 16, lane, h, &a.o);
}

__device__ __forceinline__ void net_forward(const float4* fr, const float* __restrict__ table,
                                            const GridLevel* __restrict__ lv, const GridParams& gp, V3 p, V3 d01,
                                            int lane, int g, FwdActs& a) {
  uint32_t idx[4][8];
  float w[4][8];
  quad_corners(lv, gp, p, g, idx, w);
  const float2* t2 = reinterpret_cast<const float2*>(table);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float e0 = 0.0f, e1 = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const float2 v = t2[idx[j][c]];
      e0 = e0 + w[j][c] * v.x;
      e1 = e1 + w[j][c] * v.y;
    }
    a.enc[2 * j] = e0;
    a.enc[2 * j + 1] = e1;
  }
  float h[16];
  dense4<4, 8>(fr + F_W1 * 16, lane, a.enc, a.a1);
  relu_slots<4>(a.a1, h);
  dense4<4, 16>(fr + F_W2 * 16, lane, h, a.a2);
  relu_slots<4>(a.a2, h);
  dense4<1, 16>(fr + F_W3 * 16, lane, h, &a.out);
  head_forward<0>(fr, lane, g, a.out, d01, a);
}

__device__ __forceinline__ V3 ray_dir01(const RayState& r) { return unit_to_01(V3{r.dx, r.dy, r.dz}); }

// ------------------------------------------------------------ march
// Every ray is marched to its far bound, by G lanes each (group_lanes; a
// batch of a few thousand rays would otherwise wait for its longest ray).
// each(is, t0): is: the lane holds a sample, of start t0; called by all lanes
// of a group together, in march order.
template <int G, class Each>
__device__ __forceinline__ void march_all(const MarchGrid& mg, const uint32_t* coarse, MarchRay& mr, Each&& each) {
  int bins = 0, cnt = 0;
  const int sub = lane_id() & (G - 1);
  if (G > 1 && group_usable(mg, mr)) {
    march_group_steps<(G > 1 ? G : 2)>(mg, coarse, mr, 0x7fffffff, cnt, bins, [&](uint32_t samples, int, float t0) {
      each(((samples >> sub) & 1u) != 0u, t0);
    });
    return;
  }
  while (true) {
    float t0;
    const int res = march_trip(mg, coarse, mr, t0, bins);
    if (res == TRIP_END) break;
    if (res == TRIP_SAMPLE) each(sub == 0, t0);
  }
}
// lanes of the group with is set below this one, and in all
template <int G> __device__ __forceinline__ int group_rank(bool is, int& total) {
  const int lane = lane_id(), sub = lane & (G - 1), sh = lane & ~(G - 1);
  const uint32_t m = (uint32_t)(__ballot(is) >> sh) & ((1u << G) - 1u);
  total = __popc(m);
  return __popc(m & ((1u << sub) - 1u));
}

template <int G>
__global__ __launch_bounds__(256) void k_diff_count(fvc_raymarch_info rm, V3 aabb_from, V3 aabb_to,
                                                    const int* __restrict__ pix, int n, MarchGrid mg,
                                                    const uint32_t* __restrict__ coarse_g,
                                                    RayState* __restrict__ rays, int* __restrict__ counts) {
  __shared__ uint32_t coarse[16 * COARSE_WORDS];
  load_coarse(coarse_g, mg.occ.nlvl, coarse);
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G, sub = threadIdx.x & (G - 1);
  if (i >= n) return;
  const int W = rm.cam_info.res_x;
  RayState r;
  const bool hit = init_ray_state(rm, aabb_from, aabb_to, pix[i] % W, pix[i] / W, r);
  if (sub == 0) rays[i] = r;
  int cnt = 0;
  if (hit) {
    MarchRay mr = march_ray(r, mg.tab);
    march_all<G>(mg, coarse, mr, [&](bool is, float) {
      int total;
      group_rank<G>(is, total);
      cnt += total;
    });
  }
  if (sub == 0) counts[i] = cnt;
}

template <int G>
__global__ __launch_bounds__(256) void k_diff_emit(int n, MarchGrid mg, ContractParams con,
                                                   const uint32_t* __restrict__ coarse_g,
                                                   const RayState* __restrict__ rays, const int* __restrict__ counts,
                                                   const int64_t* __restrict__ offsets, float* __restrict__ s_pos,
                                                   float* __restrict__ s_dt, int* __restrict__ s_ray) {
  __shared__ uint32_t coarse[16 * COARSE_WORDS];
  load_coarse(coarse_g, mg.occ.nlvl, coarse);
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G;
  if (i >= n || counts[i] == 0) return;
  const RayState r = rays[i];
  MarchRay mr = march_ray(r, mg.tab);
  const V3 o = {r.ox, r.oy, r.oz}, d = {r.dx, r.dy, r.dz};
  int q0 = (int)offsets[i];  // the batch holds fewer than 2^31 samples
  march_all<G>(mg, coarse, mr, [&](bool is, float t0) {
    int total;
    const int q = q0 + group_rank<G>(is, total);
    q0 += total;
    if (!is) return;
    const float dt = step_dt(mg.st, t0);
    const float tm = (t0 + (t0 + dt)) * 0.5f;
    const V3 p = contract(o + tm * d, con);
    s_pos[3 * (int64_t)q] = p.x; s_pos[3 * (int64_t)q + 1] = p.y; s_pos[3 * (int64_t)q + 2] = p.z;
    s_dt[q] = dt;
    s_ray[q] = i;
  });
}

// ------------------------------------------------------------ network
__global__ __launch_bounds__(256) void k_diff_net_fwd(int n, const int* __restrict__ list,
                                                      const float* __restrict__ s_pos,
                                                      const int* __restrict__ s_ray,
                                                      const RayState* __restrict__ rays,
                                                      const float* __restrict__ table, GridParams gp,
                                                      const float* __restrict__ frags, float4* __restrict__ out4) {
  __shared__ GridLevel lv[MAX_LEVELS];
  __shared__ float4 fr[N_FWD_FRAGS * 16];
  if (threadIdx.x < MAX_LEVELS) lv[threadIdx.x] = gp.lv[threadIdx.x];
  stage_diff_frags(frags, 0, N_FWD_FRAGS, fr);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int n_groups = (n + 15) / 16;
  for (int grp = blockIdx.x * 4 + wave; grp < n_groups; grp += gridDim.x * 4) {
    const int j = grp * 16 + col;
    const bool valid = j < n;
    const int sl = list ? list[valid ? j : n - 1] : (valid ? j : n - 1);
    const V3 p = {s_pos[3 * sl], s_pos[3 * sl + 1], s_pos[3 * sl + 2]};
    const V3 d01 = ray_dir01(rays[s_ray[sl]]);
    FwdActs a;
    net_forward(fr, table, lv, gp, p, d01, lane, g, a);
    if (g == 0 && valid) out4[sl] = make_float4(a.o[0], a.o[1], a.o[2], a.out[0]);
  }
}

// ------------------------------------------------------------ compositing
__device__ __forceinline__ void sample_terms(float4 o4, float dt, float& sigma, float& alpha, float (&c)[3]) {
  sigma = expf(o4.w);
  alpha = fminf_(fmaxf_(1.0f - expf(-sigma * dt), 0.0f), 1.0f);
  c[0] = 1.0f / (1.0f + expf(-o4.x));
  c[1] = 1.0f / (1.0f + expf(-o4.y));
  c[2] = 1.0f / (1.0f + expf(-o4.z));
}

// Both composites: G = 16 lanes per ray, lane k taking sample k of the next G
// (group_transmittance, group_add); the next samples are loaded while these
// are composited.  Bound by a ray's chain of steps: a training ray brings all
// its samples (57 on average in the small scene), so 16 lanes serve large
// batches too.  Measured, forward + backward, 4 lanes above 32768 rays and
// broadcasts by LDS permutes / 4 lanes / 16 lanes: 262144 rays 1.40 / 1.49 /
// 1.07 ms, 65521 rays 0.54 / 0.55 /
// 0.34, 4096 rays (16 lanes before too) 0.212 / - / 0.093.
static const int COMPOSITE_LANES = 16;
static dim3 composite_grid(int n) { return dim3((unsigned)(((int64_t)n * COMPOSITE_LANES + 255) / 256)); }
__global__ __launch_bounds__(256) void k_diff_composite(int n, float alpha_thre, const int* __restrict__ counts,
                                                        const int64_t* __restrict__ offsets,
                                                        const float4* __restrict__ out4,
                                                        const float* __restrict__ s_dt, float* __restrict__ rgb,
                                                        float4* __restrict__ ray_out, int* __restrict__ n_used) {
  constexpr int G = COMPOSITE_LANES;
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G, sub = threadIdx.x & (G - 1);
  if (i >= n) return;
  const int off = (int)offsets[i], cnt = counts[i];
  float C[3] = {0.0f, 0.0f, 0.0f}, T = 1.0f;
  int k = 0;  // samples walked
  bool ended = false;
  // the next samples are loaded while these are composited
  auto at = [&](int j) { return off + min(j, cnt - 1); };
  float4 v_next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float dt_next = 0.0f;
  if (cnt > 0) { v_next = out4[at(sub)]; dt_next = s_dt[at(sub)]; }
  for (int k0 = 0; k0 < cnt && !ended; k0 += G) {
    float sigma, alpha, c[3];
    const float4 v = v_next;
    const float dt = dt_next;
    v_next = out4[at(k0 + G + sub)];
    dt_next = s_dt[at(k0 + G + sub)];
    sample_terms(v, dt, sigma, alpha, c);
    const int m = cnt - k0;
    const bool counts = sub < m && alpha > alpha_thre;
    const float factor = counts ? 1.0f - alpha : 1.0f;
    const float before = group_transmittance<G>(factor, T);
    const float after = before * factor;
    const int sh = lane_id() & ~(G - 1);
    const uint32_t ends = (uint32_t)(__ballot(sub < m && after < 1e-4f) >> sh) & ((1u << G) - 1u);
    const int last = ends ? __ffs(ends) - 1 : G - 1;
    const bool adds = counts && sub <= last;
    const float w = alpha * before;
    for (int ch = 0; ch < 3; ch++) C[ch] = group_add<G>(C[ch], adds ? w * c[ch] : 0.0f);
    k += min(m, last + 1);
    ended = ends != 0;
    if (ended) T = __shfl(after, last, G);
  }
  if (sub != 0) return;
  const float4 res = make_float4(C[0] + T, C[1] + T, C[2] + T, T);
  ray_out[i] = res;
  n_used[i] = k;  // the backward walks the same ones
  rgb[3 * i] = res.x; rgb[3 * i + 1] = res.y; rgb[3 * i + 2] = res.z;
}

__global__ __launch_bounds__(256) void k_diff_composite_bwd(int n, float alpha_thre, const int* __restrict__ counts,
                                                            const int64_t* __restrict__ offsets,
                                                            const int* __restrict__ n_walk,
                                                            const float4* __restrict__ out4,
                                                            const float* __restrict__ s_dt,
                                                            const float4* __restrict__ ray_out,
                                                            const float* __restrict__ d_rgb,
                                                            float4* __restrict__ d_out4) {
  constexpr int G = COMPOSITE_LANES;
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G, sub = threadIdx.x & (G - 1);
  if (i >= n) return;
  const int off = (int)offsets[i], cnt = counts[i], walk = n_walk[i];
  const float4 ro = ray_out[i];
  const float tot[3] = {ro.x, ro.y, ro.z};
  const float dr[3] = {d_rgb[3 * i], d_rgb[3 * i + 1], d_rgb[3 * i + 2]};
  float T = 1.0f, pre[3] = {0.0f, 0.0f, 0.0f};
  auto at = [&](int j) { return off + min(j, walk - 1); };
  float4 v_next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float dt_next = 0.0f;
  if (walk > 0) { v_next = out4[at(sub)]; dt_next = s_dt[at(sub)]; }
  for (int k0 = 0; k0 < cnt; k0 += G) {
    const int k = k0 + sub;
    float4 d = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (k0 < walk) {
      float sigma, alpha, c[3];
      const float4 v = v_next;
      const float dt = dt_next;
      v_next = out4[at(k + G)];
      dt_next = s_dt[at(k + G)];
      sample_terms(v, dt, sigma, alpha, c);
      // the lane's own sample: weight, transmittance after it, colour up to it
      const bool counts = k < walk && alpha > alpha_thre;
      const float factor = counts ? 1.0f - alpha : 1.0f;
      const float before = group_transmittance<G>(factor, T);
      const float wk = counts ? alpha * before : 0.0f, T1 = before * factor;
      float pk[3];
      for (int ch = 0; ch < 3; ch++) {
        const float x = counts ? wk * c[ch] : 0.0f;
        float own = 0.0f;
        each<G>([&](auto u) {
          pre[ch] = pre[ch] + group_lane<G, u>(x);
          own = sub == u ? pre[ch] : own;
        });
        pk[ch] = own;
      }
      if (k < walk && alpha > alpha_thre) {
        float dsig = 0.0f, dc[3];
        for (int ch = 0; ch < 3; ch++) {
          const float S = tot[ch] - pk[ch];
          dsig = dsig + dr[ch] * (T1 * c[ch] - S);
          dc[ch] = dr[ch] * wk * c[ch] * (1.0f - c[ch]);
        }
        d = make_float4(dc[0], dc[1], dc[2], dsig * dt * sigma);
      }
    }
    if (k < cnt) d_out4[off + k] = d;
  }
}

// ------------------------------------------------------------ backward
// where a layer's gradient starts in its parameter block (row-major [out][in])
enum { G_W1 = 0, G_W2 = 64 * 32, G_W3 = 64 * 32 + 64 * 64, G_H1 = 0, G_H2 = 64 * 32 };

// Weight gradients dW[out][in] = sum over samples of dY[out] X[in], by the
// eight waves of a block over the block's 128 samples: every wave writes its
// tile's dY and X to LDS as rows of samples, then the 16x16 blocks of dW are
// shared out among the waves, each kept in a wave's registers over the whole
// sample loop (40 blocks: 24 registers a lane) and added to the caller's
// gradient once, at the end.  A lane reads its operands of four MFMA steps
// (samples 16 q + 4 g .. + 3) as one float4; the row stride of 132 floats
// spreads the 16 rows of such a read, and the four lane groups of a write,
// over all LDS banks.
// Bound by the f32 MFMA issue (464 steps of 32 cycles per tile with the
// forward's recomputation); measured at 2^18 rays (14 M samples) against one
// LDS atomic per tile and weight: training step 88.0 -> 80.3 ms, 4096 rays
// 5.30 -> 5.05 ms.
static const int BWD_WAVES = 8, BWD_SAMPLES = 16 * BWD_WAVES;
static const int STG = BWD_SAMPLES + 4;  // LDS row stride (floats)

template <int NB> __device__ __forceinline__ void stage_rows(float* rows, const f4* y, int g, int smp) {
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int e = 0; e < 4; e++) rows[(16 * nb + 4 * g + e) * STG + smp] = y[nb][e];
}
template <int MX, class KCol>
__device__ __forceinline__ void stage_cols(float* rows, const float* x, KCol kcol, int g, int smp) {
#pragma unroll
  for (int m = 0; m < MX; m++) rows[kcol(m, g) * STG + smp] = x[m];
}
// acc += block (jb, kb) of dY X^T over samples [16 q0, 16 q1)
__device__ __forceinline__ void wgrad_block(const float* ys, const float* xs, int jb, int kb, int q0, int q1, int col,
                                            int g, f4& acc) {
  const float* yr = ys + (16 * jb + col) * STG + 4 * g;
  const float* xr = xs + (16 * kb + col) * STG + 4 * g;
#pragma unroll 4
  for (int q = q0; q < q1; q++) {
    const float4 a = *reinterpret_cast<const float4*>(yr + 16 * q);
    const float4 b = *reinterpret_cast<const float4*>(xr + 16 * q);
    acc = mma4(a.x, b.x, acc);
    acc = mma4(a.y, b.y, acc);
    acc = mma4(a.z, b.z, acc);
    acc = mma4(a.w, b.w, acc);
  }
}
// block (jb, kb) of dW added to the caller's gradient (rows of n_in)
__device__ __forceinline__ void add_block(float* gw, int jb, int kb, int n_in, int col, int g, f4 acc) {
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (acc[e] != 0.0f) unsafeAtomicAdd(&gw[(16 * jb + 4 * g + e) * n_in + 16 * kb + col], acc[e]);
}

// column maps of the B slots (device copies of k_chain, k_enc, k_head)
struct KChain {
  __device__ int operator()(int m, int g) const { return 16 * (m / 4) + 4 * g + (m % 4); }
};
struct KEnc {
  __device__ int operator()(int m, int g) const { return 2 * (g + 4 * (m / 2)) + (m % 2); }
};
struct KHead {
  __device__ int operator()(int m, int g) const {
    if (m >= 4) return 8 + 4 * g + (m - 4);
    const int r = 4 * g + m;
    if (r >= 1 && r <= 8) return r - 1;
    return r == 0 ? 24 : r + 16;
  }
};

// Hash-table gradient of samples [j0, n): entry (x, y, z) of level l gets
// w d_enc for the sample's two features.  d_enc[l][j - j0] (level rows of
// `cap` samples) is the network backward's gradient of the encoding.
//
// Bound by the L2's atomics: about 21 G requests/s whatever the address
// range, where the lanes of one instruction that touch different words of
// one 64-byte line make one request.  So (1) a lane quad takes one sample,
// its lanes the two x corners times the two features, whose four words lie
// together on dense levels and, hashed, for all but the x that carry past a
// group of 8 entries; and (2) every quad walks SCATTER_SEG consecutive
// samples (neighbours along a ray) and keeps the sums of the cell's four
// (y, z) rows in registers until the cell changes, so a run of samples in
// one cell costs four requests in all.  A wave works on one level (uniform
// index arithmetic); the levels rotate over the blocks so that each XCD gets
// coarse and fine ones.
static const int SCATTER_SEG = 32;
struct LevelList {
  int n;
  int l[MAX_LEVELS];
};
__global__ __launch_bounds__(256) void k_diff_scatter(int j0, int n, const int* __restrict__ list,
                                                      const float* __restrict__ s_pos, GridParams gp, LevelList ll,
                                                      const float* __restrict__ d_enc, int64_t cap,
                                                      float* __restrict__ g_pos) {
  const int grp = blockIdx.x / ll.n;
  const int l = ll.l[(blockIdx.x + grp) % ll.n];
  const GridLevel L = gp.lv[l];
  const bool dense = (gp.dense_mask >> l) & 1u;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int xc = (lane >> 1) & 1, f = lane & 1;
  const int64_t seg = ((int64_t)grp * 4 + wave) * 16 + (lane >> 2);
  const int64_t first = j0 + seg * SCATTER_SEG;
  const int cnt = (int)(first >= n ? 0 : (n - first < SCATTER_SEG ? n - first : SCATTER_SEG));
  const float* de = d_enc + 2 * ((int64_t)l * cap) + f;
  float* gl = g_pos + 2 * (size_t)L.offset + f;
  uint32_t cx = 0u, cy = 0u, cz = 0u;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  auto flush = [&] {
    const uint32_t x = cx + (uint32_t)xc;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t y = cy + (uint32_t)(r & 1), z = cz + (uint32_t)(r >> 1);
      uint32_t t;
      if (dense) {
        t = x + y * L.res + z * L.res2;
        t = min(t, t - L.size);  // t < 2 * size
      } else {
        t = (x ^ (y * 2654435761u) ^ (z * 805459861u)) & (L.size - 1u);
      }
      if (acc[r] != 0.0f) unsafeAtomicAdd(gl + 2 * (size_t)t, acc[r]);
    }
  };
  static const int U = 4;  // samples loaded together
  for (int k0 = 0; k0 < cnt; k0 += U) {
    V3 p[U];
    float d[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t j = first + min(k0 + u, cnt - 1);
      const int sl = list ? list[j] : (int)j;
      p[u] = V3{s_pos[3 * (int64_t)sl], s_pos[3 * (int64_t)sl + 1], s_pos[3 * (int64_t)sl + 2]};
      d[u] = de[2 * (j - j0)];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (k0 + u >= cnt) break;
      const float px = fminf_(fmaxf_(p[u].x, 0.0f), 1.0f);
      const float py = fminf_(fmaxf_(p[u].y, 0.0f), 1.0f);
      const float pz = fminf_(fmaxf_(p[u].z, 0.0f), 1.0f);
      const float ax = px * L.scale + 0.5f, ay = py * L.scale + 0.5f, az = pz * L.scale + 0.5f;
      const float fx = floorf(ax), fy = floorf(ay), fz = floorf(az);
      const uint32_t gx = (uint32_t)(int)fx, gy = (uint32_t)(int)fy, gz = (uint32_t)(int)fz;
      if (gx != cx || gy != cy || gz != cz) {
        flush();
        cx = gx; cy = gy; cz = gz;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = 0.0f;
      }
      const float wx = ax - fx, wy = ay - fy, wz = az - fz;
      const float vx = xc ? wx : 1.0f - wx, uy = 1.0f - wy, uz = 1.0f - wz;
      const float w0 = vx * uy, w1 = vx * wy;
      acc[0] = acc[0] + (w0 * uz) * d[u];
      acc[1] = acc[1] + (w1 * uz) * d[u];
      acc[2] = acc[2] + (w0 * wz) * d[u];
      acc[3] = acc[3] + (w1 * wz) * d[u];
    }
  }
  flush();
}

// Table gradient of the hashed levels without global atomics, in two kernels
// over a chunk of samples.  k_diff_bin walks runs of BIN_SEG consecutive
// samples per thread as k_diff_scatter does and turns each finished cell row
// (y, z) into a record: the entries of corners x and x + 1 and the four sums
// to add there.  Records are collected in LDS and written out sorted by
// table slice of BIN_ENTRIES entries (one counter request per slice and
// flush).  k_diff_bin_add gives each slice to one block, which sums its
// records in LDS and adds the slice to the gradient with plain loads and
// stores.  Entries x and x + 1 differ in the bits below the carry only
// (res < BIN_ENTRIES), so a record has one slice.  LDS sums are FP64: on
// gfx950 ds_add_f64 takes 26 cycles for a wave's random addresses,
// ds_add_f32 185.
//
// Bound by the records' traffic (40 bytes each, written and read) in the
// place of one 21 G/s atomic request per row: measured at 2^18 rays (14 M
// samples, T 2^19), the table gradient 21.1 ms with k_diff_scatter alone, 9.2
// ms with the 11 hashed levels in slices (4.5 + 2.6 ms here, 2.0 ms for the
// dense levels in k_diff_scatter).
// A slice holds `cap` records of a chunk; what does not fit (rays that
// crowd into few cells) is added with atomics.
static const int BIN_ENTRIES = 8192, BIN_SEG = 16, BIN_THREADS = 256;
static const int BIN_BUF = 3072;                 // records buffered per block
static const int BIN_MAX = 256;                  // slices of a level
struct BinLevels {
  int n;
  int l[MAX_LEVELS], n_bins[MAX_LEVELS], first[MAX_LEVELS];  // first: the level's first slice
};
__global__ __launch_bounds__(BIN_THREADS) void k_diff_bin(int64_t j0, int n, int64_t d_off,
                                                          const int* __restrict__ list,
                                                          const float* __restrict__ s_pos, GridParams gp,
                                                          BinLevels bl, const float2* __restrict__ d_enc,
                                                          int64_t d_cap, int cap, int* __restrict__ cursor,
                                                          float4* __restrict__ rec_val,
                                                          uint32_t* __restrict__ rec_key,
                                                          float* __restrict__ g_pos) {
  __shared__ float4 s_val[BIN_BUF];
  __shared__ uint32_t s_key[BIN_BUF];   // entry of corner x, trailing ones of x above bit 24
  __shared__ int s_hist[BIN_MAX], s_base[BIN_MAX];
  __shared__ int s_cnt;
  const int li = blockIdx.x % bl.n, grp = blockIdx.x / bl.n;
  const int l = bl.l[li], n_bins = bl.n_bins[li], bin0 = bl.first[li];
  const GridLevel L = gp.lv[l];
  const int lane = threadIdx.x & 63;
  if (threadIdx.x == 0) s_cnt = 0;
  const int64_t first = ((int64_t)grp * BIN_THREADS + threadIdx.x) * BIN_SEG;  // in the chunk
  const int cnt = (int)(first >= n ? 0 : (n - first < BIN_SEG ? n - first : BIN_SEG));
  const float2* de = d_enc + (int64_t)l * d_cap + d_off;
  uint32_t cx = 0u, cy = 0u, cz = 0u;
  float4 acc[4];  // row r: (x, feature 0), (x, 1), (x + 1, 0), (x + 1, 1)
#pragma unroll
  for (int r = 0; r < 4; r++) acc[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto entry = [&](uint32_t x, uint32_t y, uint32_t z) {
    return (x ^ (y * 2654435761u) ^ (z * 805459861u)) & (L.size - 1u);
  };
  auto other = [&](uint32_t i0, uint32_t ones) { return (i0 ^ ((2u << ones) - 1u)) & (L.size - 1u); };
  // sorts the buffered records by slice and writes them out
  auto flush = [&](int c) {
    for (int b = threadIdx.x; b < n_bins; b += BIN_THREADS) s_hist[b] = 0;
    __syncthreads();
    int rank[BIN_BUF / BIN_THREADS];
#pragma unroll
    for (int u = 0; u < BIN_BUF / BIN_THREADS; u++) {
      const int i = u * BIN_THREADS + threadIdx.x;
      if (i < c) rank[u] = atomicAdd(&s_hist[(s_key[i] & 0xffffffu) / BIN_ENTRIES], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < n_bins; b += BIN_THREADS)
      s_base[b] = s_hist[b] > 0 ? atomicAdd(&cursor[bin0 + b], s_hist[b]) : 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BIN_BUF / BIN_THREADS; u++) {
      const int i = u * BIN_THREADS + threadIdx.x;
      if (i >= c) break;
      const uint32_t k = s_key[i], i0 = k & 0xffffffu, i1 = other(i0, k >> 24);
      const int b = (int)(i0 / BIN_ENTRIES), at = s_base[b] + rank[u];
      const float4 v = s_val[i];
      if (at < cap) {
        const int64_t q = (int64_t)(bin0 + b) * cap + at;
        rec_val[q] = v;
        rec_key[q] = (i0 & (BIN_ENTRIES - 1u)) | ((i1 & (BIN_ENTRIES - 1u)) << 16);
      } else {
        float* g0 = g_pos + 2 * ((size_t)L.offset + i0);
        float* g1 = g_pos + 2 * ((size_t)L.offset + i1);
        unsafeAtomicAdd(g0, v.x);
        unsafeAtomicAdd(g0 + 1, v.y);
        unsafeAtomicAdd(g1, v.z);
        unsafeAtomicAdd(g1 + 1, v.w);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
  };
  __syncthreads();
  for (int k = 0; k <= BIN_SEG; k++) {
    const bool in = k < cnt;
    float2 d = make_float2(0.0f, 0.0f);
    uint32_t gx = 0u, gy = 0u, gz = 0u;
    float wx = 0.0f, wy = 0.0f, wz = 0.0f;
    if (in) {
      const int64_t j = j0 + first + k;
      const int64_t sl = list ? list[j] : j;
      const float px = fminf_(fmaxf_(s_pos[3 * sl], 0.0f), 1.0f);
      const float py = fminf_(fmaxf_(s_pos[3 * sl + 1], 0.0f), 1.0f);
      const float pz = fminf_(fmaxf_(s_pos[3 * sl + 2], 0.0f), 1.0f);
      d = de[first + k];
      const float ax = px * L.scale + 0.5f, ay = py * L.scale + 0.5f, az = pz * L.scale + 0.5f;
      const float fx = floorf(ax), fy = floorf(ay), fz = floorf(az);
      gx = (uint32_t)(int)fx; gy = (uint32_t)(int)fy; gz = (uint32_t)(int)fz;
      wx = ax - fx; wy = ay - fy; wz = az - fz;
    }
    // a finished cell with something to add becomes four records
    bool emit = !in || gx != cx || gy != cy || gz != cz;
    if (emit) {
      bool any = false;
#pragma unroll
      for (int r = 0; r < 4; r++)
        any = any || acc[r].x != 0.0f || acc[r].y != 0.0f || acc[r].z != 0.0f || acc[r].w != 0.0f;
      emit = any;
    }
    const unsigned long long m = __ballot(emit);
    const int ne = __popcll(m);
    int base = 0;
    if (lane == 0 && ne > 0) base = atomicAdd(&s_cnt, 4 * ne);
    base = __shfl(base, 0, 64);
    if (emit) {
      const int at = base + __popcll(m & ((1ull << lane) - 1ull));
      const uint32_t ones = (uint32_t)__builtin_ctz(~cx);  // x < 2^24
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s_val[at + r * ne] = acc[r];
        s_key[at + r * ne] = entry(cx, cy + (r & 1), cz + (r >> 1)) | (ones << 24);
      }
    }
    if (!in || gx != cx || gy != cy || gz != cz) {
      cx = gx; cy = gy; cz = gz;
#pragma unroll
      for (int r = 0; r < 4; r++) acc[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    const float ux = 1.0f - wx, uy = 1.0f - wy, uz = 1.0f - wz;
    const float wxy[4] = {ux * uy, wx * uy, ux * wy, wx * wy};
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float w = (r & 2) ? wz : uz, w0 = wxy[2 * (r & 1)] * w, w1 = wxy[2 * (r & 1) + 1] * w;
      acc[r].x = acc[r].x + w0 * d.x;
      acc[r].y = acc[r].y + w0 * d.y;
      acc[r].z = acc[r].z + w1 * d.x;
      acc[r].w = acc[r].w + w1 * d.y;
    }
    __syncthreads();
    const int c = s_cnt;
    __syncthreads();
    // a step adds at most 4 records a thread
    if (c > BIN_BUF - 4 * BIN_THREADS || (k == BIN_SEG && c > 0)) flush(c);
  }
}

__global__ void k_diff_zero(int* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// one slice of one level: its records summed in LDS, then added to the
// gradient (the block is the only one that touches these entries)
__global__ __launch_bounds__(1024) void k_diff_bin_add(GridParams gp, BinLevels bl, int cap,
                                                       int* __restrict__ cursor,
                                                       const float4* __restrict__ rec_val,
                                                       const uint32_t* __restrict__ rec_key,
                                                       float* __restrict__ g_pos) {
  __shared__ double acc[2 * BIN_ENTRIES];
  // the finest levels, with the most records, first
  int li = bl.n - 1, b = blockIdx.x;
  while (b >= bl.n_bins[li]) b -= bl.n_bins[li--];
  const GridLevel L = gp.lv[bl.l[li]];
  const int bin = bl.first[li] + b;
  const int c = min(cursor[bin], cap);
  if (c <= 0) return;
  const int n_ent = min((int)L.size - b * BIN_ENTRIES, BIN_ENTRIES);
  for (int i = threadIdx.x; i < 2 * n_ent; i += 1024) acc[i] = 0.0;
  __syncthreads();
  if (threadIdx.x == 0) cursor[bin] = 0;  // for the next chunk
  const float4* rv = rec_val + (int64_t)bin * cap;
  const uint32_t* rk = rec_key + (int64_t)bin * cap;
  for (int i = threadIdx.x; i < c; i += 1024) {
    const uint32_t k = rk[i];
    const float4 v = rv[i];
    double* a0 = acc + 2 * (k & 0xffffu);
    double* a1 = acc + 2 * (k >> 16);
    unsafeAtomicAdd(a0, (double)v.x);
    unsafeAtomicAdd(a0 + 1, (double)v.y);
    unsafeAtomicAdd(a1, (double)v.z);
    unsafeAtomicAdd(a1 + 1, (double)v.w);
  }
  __syncthreads();
  float* g = g_pos + 2 * ((size_t)L.offset + (size_t)b * BIN_ENTRIES);
  for (int i = threadIdx.x; i < 2 * n_ent; i += 1024)
    if (acc[i] != 0.0) g[i] = g[i] + (float)acc[i];
}

// colour MLP backward of a tile: d_o (output rows 4g..4g+3), d_z1
// (hidden pre-activations) and d_xh (head inputs in the rows of the
// base output, row r = latent r - 1 for r in 1..8)
template <int F0>
__device__ __forceinline__ void head_backward(const float4* fr, int lane, int g, const FwdActs& a, float4 dq,
                                              f4& d_o, f4* d_z1, f4& d_xh) {
  d_o = g == 0 ? f4{dq.x, dq.y, dq.z, 0.0f} : f4zero();
  float x[16];
#pragma unroll
  for (int e = 0; e < 4; e++) x[e] = d_o[e];
  dense4<4, 4>(fr + (B_H2T - F0) * 16, lane, x, d_z1);
  relu_grad<4>(a.z1, d_z1);
#pragma unroll
  for (int nb = 0; nb < 4; nb++)
#pragma unroll
    for (int e = 0; e < 4; e++) x[4 * nb + e] = d_z1[nb][e];
  dense4<1, 16>(fr + (B_H1T - F0) * 16, lane, x, &d_xh);
}

// colour MLP weight gradients of the block's samples: wave w takes block
// w % 4 of H2 over half w / 4 of the samples, and block (w / 2, w % 2) of H1.
// Every thread of the block calls it; it ends with a barrier.
struct HeadAcc { f4 h2, h1; };
__device__ __forceinline__ void head_wgrad(float* stage, const FwdActs& a, const f4& d_o, const f4* d_z1, int wave,
                                           int col, int g, HeadAcc& acc) {
  const int smp = 16 * wave + col;
  float h[16];
  relu_slots<4>(a.z1, h);
  stage_rows<1>(stage, &d_o, g, smp);
  stage_cols<16>(stage + 16 * STG, h, KChain(), g, smp);
  __syncthreads();
  wgrad_block(stage, stage + 16 * STG, 0, wave & 3, (wave >> 2) * 4, (wave >> 2) * 4 + 4, col, g, acc.h2);
  __syncthreads();
  stage_rows<4>(stage, d_z1, g, smp);
  stage_cols<8>(stage + 64 * STG, a.xh, KHead(), g, smp);
  __syncthreads();
  wgrad_block(stage, stage + 64 * STG, wave >> 1, wave & 1, 0, BWD_WAVES, col, g, acc.h1);
  __syncthreads();
}
__device__ __forceinline__ void flush_head(float* g_head, int wave, int col, int g, const HeadAcc& acc) {
  add_block(g_head + G_H2, 0, wave & 3, 64, col, g, acc.h2);
  add_block(g_head + G_H1, wave >> 1, wave & 1, 32, col, g, acc.h1);
}

// samples [j0, n) of the list; d_feat: [16 levels][cap] gradients of the encoding
__global__ __launch_bounds__(64 * BWD_WAVES) void k_diff_net_bwd(int j0, int n, const int* __restrict__ list,
                                                      const float* __restrict__ s_pos,
                                                      const int* __restrict__ s_ray,
                                                      const RayState* __restrict__ rays,
                                                      const float* __restrict__ table, GridParams gp,
                                                      const float* __restrict__ frags,
                                                      const float4* __restrict__ d_out4,
                                                      float2* __restrict__ d_feat, int64_t cap,
                                                      float* __restrict__ g_base, float* __restrict__ g_head) {
  __shared__ GridLevel lv[MAX_LEVELS];
  __shared__ float4 fr[N_DIFF_FRAGS * 16];
  __shared__ __attribute__((aligned(16))) float stage[128 * STG];
  if (threadIdx.x < MAX_LEVELS) lv[threadIdx.x] = gp.lv[threadIdx.x];
  stage_diff_frags(frags, 0, N_DIFF_FRAGS, fr);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int smp = 16 * wave + col;  // the lane's sample among the block's
  HeadAcc acc_h{f4zero(), f4zero()};
  f4 acc_w3 = f4zero(), acc_w2[2] = {f4zero(), f4zero()}, acc_w1 = f4zero();
  // every wave of the block takes part in every iteration (barriers); lanes
  // past the last sample carry zero gradients
  for (int base = j0 + blockIdx.x * BWD_SAMPLES; base < n; base += gridDim.x * BWD_SAMPLES) {
    const int j = base + smp;
    const bool valid = j < n;
    const int sl = list ? list[valid ? j : n - 1] : (valid ? j : n - 1);
    const float4 dq = valid ? d_out4[sl] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const V3 p = {s_pos[3 * sl], s_pos[3 * sl + 1], s_pos[3 * sl + 2]};
    const V3 d01 = ray_dir01(rays[s_ray[sl]]);
    FwdActs a;
    net_forward(fr, table, lv, gp, p, d01, lane, g, a);
    // colour MLP
    f4 d_o, d_z1[4], d_xh;
    head_backward<0>(fr, lane, g, a, dq, d_o, d_z1, d_xh);
    head_wgrad(stage, a, d_o, d_z1, wave, col, g, acc_h);
    float x[16];
    // density MLP: output rows 4g + e (0: log density, 1..8: latents)
    f4 d_out;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 4 * g + e;
      d_out[e] = r == 0 ? dq.w : ((r >= 1 && r <= 8) ? d_xh[e] : 0.0f);
    }
    f4 d_a2[4], d_a1[4], d_enc[2];
    for (int e = 0; e < 4; e++) x[e] = d_out[e];
    dense4<4, 4>(fr + B_W3T * 16, lane, x, d_a2);
    relu_grad<4>(a.a2, d_a2);
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int e = 0; e < 4; e++) x[4 * nb + e] = d_a2[nb][e];
    dense4<4, 16>(fr + B_W2T * 16, lane, x, d_a1);
    relu_grad<4>(a.a1, d_a1);
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int e = 0; e < 4; e++) x[4 * nb + e] = d_a1[nb][e];
    dense4<2, 16>(fr + B_W1T * 16, lane, x, d_enc);
    // gradient of the encoding: slot 2i + k of level 4i + g is d_enc[i / 2][2 (i % 2) + k]
    if (valid) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        d_feat[(4 * i + g) * cap + (j - j0)] = make_float2(d_enc[i >> 1][2 * (i & 1)], d_enc[i >> 1][2 * (i & 1) + 1]);
    }
    // density MLP weight gradients (activations as the forward's B slots)
    float h[16];
    relu_slots<4>(a.a2, h);
    stage_rows<1>(stage, &d_out, g, smp);
    stage_cols<16>(stage + 16 * STG, h, KChain(), g, smp);
    __syncthreads();
    wgrad_block(stage, stage + 16 * STG, 0, wave & 3, (wave >> 2) * 4, (wave >> 2) * 4 + 4, col, g, acc_w3);
    __syncthreads();
    relu_slots<4>(a.a1, h);
    stage_rows<4>(stage, d_a2, g, smp);
    stage_cols<16>(stage + 64 * STG, h, KChain(), g, smp);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; k++)
      wgrad_block(stage, stage + 64 * STG, wave >> 1, 2 * (wave & 1) + k, 0, BWD_WAVES, col, g, acc_w2[k]);
    __syncthreads();
    stage_rows<4>(stage, d_a1, g, smp);
    stage_cols<8>(stage + 64 * STG, a.enc, KEnc(), g, smp);
    __syncthreads();
    wgrad_block(stage, stage + 64 * STG, wave >> 1, wave & 1, 0, BWD_WAVES, col, g, acc_w1);
    __syncthreads();
  }
  flush_head(g_head, wave, col, g, acc_h);
  add_block(g_base + G_W3, 0, wave & 3, 64, col, g, acc_w3);
#pragma unroll
  for (int k = 0; k < 2; k++) add_block(g_base + G_W2, wave >> 1, 2 * (wave & 1) + k, 64, col, g, acc_w2[k]);
  add_block(g_base + G_W1, wave >> 1, wave & 1, 32, col, g, acc_w1);
}

// ------------------------------------------------------------ cached mode
// Differentiable cached render: classification of every occupied sample as
// in the cache marcher (classify_sample); resample samples take the network
// (k_diff_net_fwd / _bwd over list_r), cache samples the trilinear lookup of
// the brick pool and the colour MLP (k_diffc_head_fwd / _bwd over list_c).
// The adjoint of the lookup (generateNetworkInput_cache_shfl_perf_kernel_cg,
// cache_performance_renderer.cu:678-787): with s = log(max(sum_c w_c
// sigma_c, 1e-6)) and l_i = sum_c w_c l_c,i / sum_c w_c isset_c,
//   dL/dsigma_c = w_c dL/ds / sum (0 when the clamp is active),
//   dL/dl_c,i   = w_c dL/dl_i / sum_c w_c isset_c;
// isset is a mask.  Voxel gradients go to g_pool [slot][512][10] (8 latents,
// density, isset = 0) with FP32 atomics.
template <int G>
__global__ __launch_bounds__(256) void k_diffc_count(fvc_raymarch_info rm, V3 aabb_from, V3 aabb_to,
                                                     const int* __restrict__ pix, int n, MarchGrid mg, CacheView cv,
                                                     const uint32_t* __restrict__ coarse_g,
                                                     RayState* __restrict__ rays, int* __restrict__ counts_r,
                                                     int* __restrict__ counts_c) {
  __shared__ uint32_t coarse[16 * COARSE_WORDS];
  load_coarse(coarse_g, mg.occ.nlvl, coarse);
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G, sub = threadIdx.x & (G - 1);
  if (i >= n) return;
  const int W = rm.cam_info.res_x;
  RayState r;
  const bool hit = init_ray_state(rm, aabb_from, aabb_to, pix[i] % W, pix[i] / W, r);
  if (sub == 0) rays[i] = r;
  int nr = 0, nc = 0;
  if (hit) {
    MarchRay mr = march_ray(r, mg.tab);
    const V3 oc = transform(cv.cam.world2cam, mr.o.x, mr.o.y, mr.o.z, 1.0f);
    const V3 dc = transform(cv.cam.world2cam, mr.d.x, mr.d.y, mr.d.z, 0.0f);
    march_all<G>(mg, coarse, mr, [&](bool is, float t0) {
      const int k = is ? classify_sample(cv, oc, dc, t0, step_dt(mg.st, t0)) : SAMPLE_SKIP;
      int tr, tc;
      group_rank<G>(k == SAMPLE_RESAMPLE, tr);
      group_rank<G>(k == SAMPLE_CACHE, tc);
      nr += tr;
      nc += tc;
    });
  }
  if (sub == 0) {
    counts_r[i] = nr;
    counts_c[i] = nc;
  }
}

template <int G>
__global__ __launch_bounds__(256) void k_diffc_emit(int n, MarchGrid mg, ContractParams con, CacheView cv,
                                                    const uint32_t* __restrict__ coarse_g,
                                                    const RayState* __restrict__ rays,
                                                    const int* __restrict__ counts_r, const int* __restrict__ counts_c,
                                                    const int64_t* __restrict__ off_r,
                                                    const int64_t* __restrict__ off_c, int* __restrict__ counts,
                                                    int64_t* __restrict__ offsets, float* __restrict__ s_pos,
                                                    float* __restrict__ s_dt, int* __restrict__ s_ray,
                                                    int* __restrict__ list_r, int* __restrict__ list_c) {
  __shared__ uint32_t coarse[16 * COARSE_WORDS];
  load_coarse(coarse_g, mg.occ.nlvl, coarse);
  const int i = blockIdx.x * (256 / G) + threadIdx.x / G, sub = threadIdx.x & (G - 1);
  if (i >= n) return;
  const int nr = counts_r[i], nc = counts_c[i];
  int q0 = (int)(off_r[i] + off_c[i]);  // the batch holds fewer than 2^31 samples
  if (sub == 0) {
    counts[i] = nr + nc;
    offsets[i] = q0;
  }
  if (nr + nc == 0) return;
  const RayState r = rays[i];
  MarchRay mr = march_ray(r, mg.tab);
  const V3 o = {r.ox, r.oy, r.oz}, d = {r.dx, r.dy, r.dz};
  const V3 oc = transform(cv.cam.world2cam, o.x, o.y, o.z, 1.0f);
  const V3 dc = transform(cv.cam.world2cam, d.x, d.y, d.z, 0.0f);
  int kr0 = (int)off_r[i], kc0 = (int)off_c[i];
  march_all<G>(mg, coarse, mr, [&](bool is, float t0) {
    const float dt = step_dt(mg.st, t0);
    const int k = is ? classify_sample(cv, oc, dc, t0, dt) : SAMPLE_SKIP;
    int tr, tc;
    const int kr = kr0 + group_rank<G>(k == SAMPLE_RESAMPLE, tr), kc = kc0 + group_rank<G>(k == SAMPLE_CACHE, tc);
    const int q = q0 + (kr - kr0) + (kc - kc0);
    kr0 += tr;
    kc0 += tc;
    q0 += tr + tc;
    if (k == SAMPLE_SKIP) return;
    // network inputs at t0 + dt / 2 (cache_performance_renderer.cu:198-313)
    const float tm2 = t0 + dt * 0.5f;
    V3 p;
    if (k == SAMPLE_RESAMPLE) {
      p = contract(o + tm2 * d, con);
      list_r[kr] = q;
    } else {
      float tf;
      p = cam2froxel(oc + tm2 * dc, cv.cam, cv.st, tf);
      list_c[kc] = q;
    }
    s_pos[3 * (int64_t)q] = p.x; s_pos[3 * (int64_t)q + 1] = p.y; s_pos[3 * (int64_t)q + 2] = p.z;
    s_dt[q] = dt;
    s_ray[q] = i;
  });
}

// trilinear lookup of one sample by its 4 lanes: lane group g fetches the
// corners (x, y) = (g >> 1, g & 1), z = 0 / 1; every lane ends with the sums
struct LookupLane {
  float w[2];
  int64_t v[2];  // voxel index in the reference's order (g_pool), -1: outside or unset brick
  float wsum, dsum, lat[8];
};
__device__ __forceinline__ void lookup_f32(const CacheView& cv, V3 f, int g, LookupLane& L) {
  const float fcx = f.x - 0.5f, fcy = f.y - 0.5f, fcz = f.z - 0.5f;
  const float ix = floorf(fcx), iy = floorf(fcy), iz = floorf(fcz);
  const float lx = fcx - ix, ly = fcy - iy, lz = fcz - iz;
  const float ox = (float)(g >> 1), oy = (float)(g & 1);
  const float px = ix + ox, py = iy + oy;
  const float wx = (1.0f - ox) * (1.0f - 2.0f * lx) + lx;
  const float wy = (1.0f - oy) * (1.0f - 2.0f * ly) + ly;
  const float wxy = wx * wy;
  const bool in_xy = px >= 0.0f && px < (float)cv.fx && py >= 0.0f && py < (float)cv.fy;
  float wd = 0.0f, dd = 0.0f, ld[8];
#pragma unroll
  for (int cc = 0; cc < 2; cc++) {
    const float pz = iz + (float)cc;
    const float wz = cc == 0 ? (1.0f - 2.0f * lz) + lz : lz;
    const float w = wxy * wz;
    L.w[cc] = w;
    L.v[cc] = -1;
    float cw = 0.0f, cd = 0.0f, cl[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (in_xy && pz >= 0.0f && pz < (float)cv.fz) {
      const int vx = (int)px, vy = (int)py, vz = (int)pz;
      const int slot = cv.table[((int64_t)(vz >> 3) * cv.by + (vy >> 3)) * cv.bx + (vx >> 3)];
      if (slot >= 0) {
        L.v[cc] = (int64_t)slot * BRICK_VOXELS + canon_voxel(vx, vy, vz);
        const Voxel vox = cv.pool[(int64_t)slot * BRICK_VOXELS + brick_voxel(vx, vy, vz)];
        cw = w * vox.isset;
        cd = w * vox.density;
#pragma unroll
        for (int k = 0; k < 8; k++) cl[k] = w * h2f(vox.lat[k]);
      }
    }
    if (cc == 0) {
      wd = cw; dd = cd;
#pragma unroll
      for (int k = 0; k < 8; k++) ld[k] = cl[k];
    } else {
      wd = wd + cw; dd = dd + cd;
#pragma unroll
      for (int k = 0; k < 8; k++) ld[k] = ld[k] + cl[k];
    }
  }
  L.wsum = xor32_sum(xor16_sum(wd));
  L.dsum = xor32_sum(xor16_sum(dd));
#pragma unroll
  for (int k = 0; k < 8; k++) L.lat[k] = xor32_sum(xor16_sum(ld[k])) / L.wsum;
}

// base-output rows 4g..4g+3 of a cache sample: latents in rows 1..8
__device__ __forceinline__ f4 lookup_rows(const LookupLane& L, int g) {
  f4 r;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int k = 4 * g + e - 1;
    float v = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) v = k == i ? L.lat[i] : v;
    r[e] = v;
  }
  return r;
}

__global__ __launch_bounds__(256) void k_diffc_head_fwd(int n, const int* __restrict__ list,
                                                        const float* __restrict__ s_pos,
                                                        const int* __restrict__ s_ray,
                                                        const RayState* __restrict__ rays, CacheView cv,
                                                        const float* __restrict__ frags,
                                                        float4* __restrict__ out4) {
  __shared__ float4 fr[(B_H2T - F_H1) * 16];
  stage_diff_frags(frags, F_H1, B_H2T - F_H1, fr);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int n_groups = (n + 15) / 16;
  for (int grp = blockIdx.x * 4 + wave; grp < n_groups; grp += gridDim.x * 4) {
    const int j = grp * 16 + col;
    const bool valid = j < n;
    const int sl = list[valid ? j : n - 1];
    const V3 f = {s_pos[3 * sl], s_pos[3 * sl + 1], s_pos[3 * sl + 2]};
    const V3 d01 = ray_dir01(rays[s_ray[sl]]);
    LookupLane L;
    lookup_f32(cv, f, g, L);
    FwdActs a;
    head_forward<F_H1>(fr, lane, g, lookup_rows(L, g), d01, a);
    if (g == 0 && valid) out4[sl] = make_float4(a.o[0], a.o[1], a.o[2], logf(fmaxf_(L.dsum, 1e-6f)));
  }
}

// Voxel gradients of a tile of 16 samples.  Bound by atomic requests (21 G/s;
// the lanes of an instruction within one 64-byte line are one request): lane
// (2 y + x) * 9 + k takes value k (8 latents, density) of corner column
// (x, y), so a voxel's nine words, and its x neighbour's, go in one
// instruction; and a ray's next sample is usually one froxel further in z,
// so the sum for corner z + 1 waits for the next sample's corner z.
// Measured at 65521 rays (3.8 M cache samples) against one atomic per corner
// and value, a corner's values in one lane: k_diffc_head_bwd 11.3 -> 1.2 ms.
static const uint32_t NO_VOXEL = 0xffffffffu;  // outside the frustum or unset; indices stay below
struct PoolTile {
  uint32_t v[16][2][4];   // voxel in the order of g_pool [sample][z][2 x + y]
  float wl[16][2][4], wd[16][2][4];
  float d[16][9];
};
__device__ __forceinline__ void scatter_pool(const PoolTile& pt, int lane, float* __restrict__ g_pool) {
  if (lane >= 36) return;
  const int k = lane % 9, c = lane / 9, g = 2 * (c & 1) + (c >> 1);
  auto add = [&](uint32_t v, float x) {
    if (v != NO_VOXEL && x != 0.0f) unsafeAtomicAdd(&g_pool[(size_t)v * 10 + k], x);
  };
  uint32_t pv = NO_VOXEL;
  float pend = 0.0f;
  for (int s = 0; s < 16; s++) {
    const uint32_t v0 = pt.v[s][0][g], v1 = pt.v[s][1][g];
    const float d = pt.d[s][k];
    float x0 = (k < 8 ? pt.wl[s][0][g] : pt.wd[s][0][g]) * d;
    const float x1 = (k < 8 ? pt.wl[s][1][g] : pt.wd[s][1][g]) * d;
    if (v0 == pv) x0 = x0 + pend;
    else add(pv, pend);
    add(v0, x0);
    pv = v1;
    pend = x1;
  }
  add(pv, pend);
}

__global__ __launch_bounds__(64 * BWD_WAVES) void k_diffc_head_bwd(int n, const int* __restrict__ list,
                                                        const float* __restrict__ s_pos,
                                                        const int* __restrict__ s_ray,
                                                        const RayState* __restrict__ rays, CacheView cv,
                                                        const float* __restrict__ frags,
                                                        const float4* __restrict__ d_out4,
                                                        float* __restrict__ g_head, float* __restrict__ g_pool) {
  __shared__ float4 fr[N_HEAD_FRAGS * 16];
  __shared__ __attribute__((aligned(16))) float stage[96 * STG];
  stage_diff_frags(frags, F_H1, N_HEAD_FRAGS, fr);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, g = lane >> 4;
  HeadAcc acc_h{f4zero(), f4zero()};
  for (int base = blockIdx.x * BWD_SAMPLES; base < n; base += gridDim.x * BWD_SAMPLES) {
    const int j = base + 16 * wave + col;
    const bool valid = j < n;
    const int sl = list[valid ? j : n - 1];
    const float4 dq = valid ? d_out4[sl] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const V3 f = {s_pos[3 * sl], s_pos[3 * sl + 1], s_pos[3 * sl + 2]};
    const V3 d01 = ray_dir01(rays[s_ray[sl]]);
    LookupLane L;
    lookup_f32(cv, f, g, L);
    FwdActs a;
    head_forward<F_H1>(fr, lane, g, lookup_rows(L, g), d01, a);
    f4 d_o, d_z1[4], d_xh;
    head_backward<F_H1>(fr, lane, g, a, dq, d_o, d_z1, d_xh);
    head_wgrad(stage, a, d_o, d_z1, wave, col, g, acc_h);
    // the tile's corner voxels, their weights and the samples' gradients
    // (dL/dl_i of latent i is row i + 1 of d_xh), then the scatter
    static_assert(BWD_WAVES * sizeof(PoolTile) <= sizeof(stage), "the tiles share the staging rows");
    PoolTile* pt = reinterpret_cast<PoolTile*>(stage) + wave;
#pragma unroll
    for (int cc = 0; cc < 2; cc++) {
      pt->v[col][cc][g] = valid && L.v[cc] >= 0 ? (uint32_t)L.v[cc] : NO_VOXEL;
      pt->wl[col][cc][g] = L.w[cc] / L.wsum;
      pt->wd[col][cc][g] = L.w[cc];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 4 * g + e;
      if (r >= 1 && r <= 8) pt->d[col][r - 1] = d_xh[e];
    }
    if (g == 0) pt->d[col][8] = L.dsum > 1e-6f ? dq.w / L.dsum : 0.0f;
    wave_sync();
    scatter_pool(*pt, lane, g_pool);
    __syncthreads();  // the staging rows are free again
  }
  flush_head(g_head, wave, col, g, acc_h);
}

// ------------------------------------------------------------ host
static int persistent_blocks(int64_t n_groups) {
  const int64_t blocks = (n_groups + 3) / 4;
  return (int)std::max<int64_t>(1, std::min<int64_t>(blocks, 256 * 8));
}

// the kernel of G lanes per ray
#define BY_LANES(G, k) ((G) == 16 ? k<16> : ((G) == 4 ? k<4> : k<1>))

// blocks of the backward kernels: one per CU (their fragments and staging
// rows fill its LDS), 128 samples per block and iteration
static int bwd_blocks(int64_t n) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((n + BWD_SAMPLES - 1) / BWD_SAMPLES, 256));
}

// exclusive scan of counts[0..n) into offs[0..n] (offs[n] = total)
static int64_t scan_counts(DiffState& D, int* counts, int64_t* offs, int n, hipStream_t s) {
  FVC_HIP(hipMemsetAsync(counts + n, 0, sizeof(int), s));
  size_t tmp = 0;
  FVC_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, counts, offs, n + 1, s));
  D.scan_tmp.ensure(std::max<size_t>(tmp, 16));
  FVC_HIP(hipcub::DeviceScan::ExclusiveSum(D.scan_tmp.p, tmp, counts, offs, n + 1, s));
  int64_t total = 0;
  FVC_HIP(hipMemcpyAsync(&total, offs + n, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  FVC_HIP(hipStreamSynchronize(s));
  return total;
}

// the encoding's gradients of samples [j0, j0 + n) into the table's gradient:
// hashed levels through the slice bins, the others (and all of a small
// batch) with atomics.  Bins pay for reading and writing every slice once
// per chunk: measured at T 2^19 (16 to 140 thousand samples) the two are equal at 35 to
// 65 thousand, below that atomics are ahead.
// Levels of more than BIN_MAX slices (T > 2^21) would fill a slice's place in
// a flush with less than a cache line.
static const int64_t BIN_MIN_SAMPLES = 1 << 16, BIN_CHUNK = 1 << 19;
static void scatter_table(DiffState& D, const GridParams& gp, const int* list, int64_t j0, int64_t n, int64_t d_cap,
                          float* g_pos, hipStream_t s) {
  LevelList ll{};
  BinLevels bl{};
  int n_bins = 0, most = 1;
  auto plan = [&](bool bins) {
    ll = LevelList{};
    bl = BinLevels{};
    n_bins = 0;
    for (int l = 0; l < gp.n_levels; l++) {
      const GridLevel& L = gp.lv[l];
      const int nb = (int)((L.size + BIN_ENTRIES - 1) / BIN_ENTRIES);
      if (!bins || ((gp.dense_mask >> l) & 1u) || nb > BIN_MAX || L.res >= (uint32_t)BIN_ENTRIES) {
        ll.l[ll.n++] = l;
        continue;
      }
      bl.l[bl.n] = l;
      bl.n_bins[bl.n] = nb;
      bl.first[bl.n++] = n_bins;
      n_bins += nb;
      most = std::max(most, nb);
    }
  };
  plan(n >= BIN_MIN_SAMPLES);
  // room for a quarter more than an even spread of four records a sample
  const int64_t chunk = std::min<int64_t>(n, BIN_CHUNK);
  const int cap = (int)(5 * chunk / most + 1024);
  if (bl.n > 0 && !(D.bin_cursor.try_ensure((size_t)n_bins * sizeof(int)) &&
                    D.bin_val.try_ensure((size_t)n_bins * cap * sizeof(float4)) &&
                    D.bin_key.try_ensure((size_t)n_bins * cap * sizeof(uint32_t)))) {
    D.bin_val.release();  // no room for the records: by atomics
    D.bin_key.release();
    plan(false);
  }
  if (ll.n > 0) {
    const int64_t per_block = 4 * 16 * SCATTER_SEG;
    hipLaunchKernelGGL(k_diff_scatter, dim3((unsigned)(ll.n * ((n + per_block - 1) / per_block))), dim3(256), 0, s,
                       (int)j0, (int)(j0 + n), list, D.s_pos.as<float>(), gp, ll, D.d_enc.as<float>(), d_cap, g_pos);
    FVC_HIP(hipGetLastError());
  }
  if (bl.n == 0) return;
  hipLaunchKernelGGL(k_diff_zero, dim3((n_bins + 255) / 256), dim3(256), 0, s, D.bin_cursor.as<int>(), n_bins);
  for (int64_t c0 = 0; c0 < n; c0 += chunk) {
    const int64_t nc = std::min<int64_t>(chunk, n - c0);
    const int64_t per_block = (int64_t)BIN_THREADS * BIN_SEG;
    hipLaunchKernelGGL(k_diff_bin, dim3((unsigned)(bl.n * ((nc + per_block - 1) / per_block))), dim3(BIN_THREADS), 0, s,
                       j0 + c0, (int)nc, c0, list, D.s_pos.as<float>(), gp, bl, D.d_enc.as<float2>(), d_cap, cap,
                       D.bin_cursor.as<int>(), D.bin_val.as<float4>(), D.bin_key.as<uint32_t>(), g_pos);
    FVC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_diff_bin_add, dim3(n_bins), dim3(1024), 0, s, gp, bl, cap, D.bin_cursor.as<int>(),
                       D.bin_val.as<float4>(), D.bin_key.as<uint32_t>(), g_pos);
    FVC_HIP(hipGetLastError());
  }
}

void diff_forward(Renderer& r, const fvc_raymarch_info& rm, const int* pix, int n, const float* pos,
                  const float* base, const float* head, float* rgb, fvc_diff_stats* stats, bool cached) {
  const Model& m = *r.model;
  DiffState& D = r.diff;
  hipStream_t s = r.stream();
  if (cached && !r.caches[r.render_idx].initialized) throw Error(FVC_E_NOT_INITIALIZED, "Cache is not initialized!");
  if (cached && r.caches[r.render_idx].lat8)
    throw Error(FVC_E_UNSUPPORTED, "the differentiable cached render needs FP16 cache latents");
  if (D.frag_index.p == nullptr) {
    const std::vector<int> t = diff_frag_index();
    D.frag_index.ensure(t.size() * sizeof(int));
    FVC_HIP(hipMemcpy(D.frag_index.p, t.data(), t.size() * sizeof(int), hipMemcpyHostToDevice));
    D.frags.ensure((size_t)N_DIFF_FRAGS * 64 * sizeof(float));
  }
  D.pos = nullptr;  // set once the forward pass has completed
  D.n = n;
  D.cached = cached;
  D.n_samples = D.n_r = D.n_c = 0;
  if (stats) std::memset(stats, 0, sizeof(*stats));
  if (n == 0) {
    D.pos = pos; D.base = base; D.head = head;
    return;
  }
  D.rays.ensure((size_t)n * sizeof(RayState));
  D.counts.ensure(((size_t)n + 1) * sizeof(int));
  D.offsets.ensure(((size_t)n + 1) * sizeof(int64_t));
  D.ray_out.ensure((size_t)n * sizeof(float4));
  D.n_walk.ensure((size_t)n * sizeof(int));
  hipLaunchKernelGGL(k_diff_pack, dim3((N_DIFF_FRAGS * 64 + 255) / 256), dim3(256), 0, s, D.frag_index.as<int>(), base,
                     head, (int)m.n_base, D.frags.as<float>());
  const MarchGrid mg = march_grid(r, &rm, 1);
  const V3 af = {m.scene.aabb_from.x, m.scene.aabb_from.y, m.scene.aabb_from.z};
  const V3 at = {m.scene.aabb_to.x, m.scene.aabb_to.y, m.scene.aabb_to.z};
  const int G = mg.tab.n_rows > 0 ? group_lanes(n) : 1;
  const dim3 grid((unsigned)(((int64_t)n * G + 255) / 256));
  int64_t total64 = 0;
  if (!cached) {
    hipLaunchKernelGGL(BY_LANES(G, k_diff_count), grid, dim3(256), 0, s, rm, af, at, pix, n, mg, m.coarse.as<uint32_t>(),
                       D.rays.as<RayState>(), D.counts.as<int>());
    FVC_HIP(hipGetLastError());
    total64 = scan_counts(D, D.counts.as<int>(), D.offsets.as<int64_t>(), n, s);
    D.n_r = total64;
  } else {
    D.cv = cache_view(r.caches[r.render_idx]);
    D.counts_c.ensure(((size_t)n + 1) * sizeof(int));
    D.off_r.ensure(((size_t)n + 1) * sizeof(int64_t));
    D.off_c.ensure(((size_t)n + 1) * sizeof(int64_t));
    hipLaunchKernelGGL(BY_LANES(G, k_diffc_count), grid, dim3(256), 0, s, rm, af, at, pix, n, mg, D.cv, m.coarse.as<uint32_t>(),
                       D.rays.as<RayState>(), D.counts.as<int>(), D.counts_c.as<int>());
    FVC_HIP(hipGetLastError());
    D.n_r = scan_counts(D, D.counts.as<int>(), D.off_r.as<int64_t>(), n, s);
    D.n_c = scan_counts(D, D.counts_c.as<int>(), D.off_c.as<int64_t>(), n, s);
    total64 = D.n_r + D.n_c;
  }
  if (total64 >= ((int64_t)1 << 31) / 3)
    throw Error(FVC_E_INVALID, "more than 2^31 / 3 samples in one differentiable batch: pass fewer rays");
  const int total = (int)total64;
  D.n_samples = total;
  const size_t ns = (size_t)std::max(total, 1);
  D.s_pos.ensure(ns * 3 * sizeof(float));
  D.s_dt.ensure(ns * sizeof(float));
  D.s_ray.ensure(ns * sizeof(int));
  D.out4.ensure(ns * sizeof(float4));
  D.d_out4.ensure(ns * sizeof(float4));
  if (!cached) {
    hipLaunchKernelGGL(BY_LANES(G, k_diff_emit), grid, dim3(256), 0, s, n, mg, m.con, m.coarse.as<uint32_t>(),
                       D.rays.as<RayState>(), D.counts.as<int>(), D.offsets.as<int64_t>(), D.s_pos.as<float>(),
                       D.s_dt.as<float>(), D.s_ray.as<int>());
  } else {
    D.list_r.ensure((size_t)std::max<int64_t>(D.n_r, 1) * sizeof(int));
    D.list_c.ensure((size_t)std::max<int64_t>(D.n_c, 1) * sizeof(int));
    D.counts_all.ensure((size_t)n * sizeof(int));
    hipLaunchKernelGGL(BY_LANES(G, k_diffc_emit), grid, dim3(256), 0, s, n, mg, m.con, D.cv, m.coarse.as<uint32_t>(),
                       D.rays.as<RayState>(), D.counts.as<int>(), D.counts_c.as<int>(), D.off_r.as<int64_t>(),
                       D.off_c.as<int64_t>(), D.counts_all.as<int>(), D.offsets.as<int64_t>(), D.s_pos.as<float>(),
                       D.s_dt.as<float>(), D.s_ray.as<int>(), D.list_r.as<int>(), D.list_c.as<int>());
  }
  FVC_HIP(hipGetLastError());
  const int* list_r = cached ? D.list_r.as<int>() : nullptr;
  if (D.n_r > 0) {
    hipLaunchKernelGGL(k_diff_net_fwd, dim3(persistent_blocks((D.n_r + 15) / 16)), dim3(256), 0, s, (int)D.n_r,
                       list_r, D.s_pos.as<float>(), D.s_ray.as<int>(), D.rays.as<RayState>(), pos, m.grid,
                       D.frags.as<float>(), D.out4.as<float4>());
    FVC_HIP(hipGetLastError());
  }
  if (D.n_c > 0) {
    hipLaunchKernelGGL(k_diffc_head_fwd, dim3(persistent_blocks((D.n_c + 15) / 16)), dim3(256), 0, s, (int)D.n_c,
                       D.list_c.as<int>(), D.s_pos.as<float>(), D.s_ray.as<int>(), D.rays.as<RayState>(), D.cv,
                       D.frags.as<float>(), D.out4.as<float4>());
    FVC_HIP(hipGetLastError());
  }
  const int* counts = cached ? D.counts_all.as<int>() : D.counts.as<int>();
  hipLaunchKernelGGL(k_diff_composite, composite_grid(n), dim3(256), 0, s, n, m.scene.alpha_thre, counts, D.offsets.as<int64_t>(),
                     D.out4.as<float4>(), D.s_dt.as<float>(), rgb, D.ray_out.as<float4>(), D.n_walk.as<int>());
  FVC_HIP(hipGetLastError());
  FVC_HIP(hipStreamSynchronize(s));
  D.pos = pos;
  D.base = base;
  D.head = head;
  if (stats) {
    stats->n_rays = n;
    stats->n_samples = total;
    stats->n_cache_samples = D.n_c;
  }
}

void diff_backward(Renderer& r, const float* d_rgb, float* g_pos, float* g_base, float* g_head, float* g_pool) {
  const Model& m = *r.model;
  DiffState& D = r.diff;
  if (D.pos == nullptr) throw Error(FVC_E_NOT_INITIALIZED, "no differentiable forward pass to differentiate");
  if (D.cached && D.n_c > 0 && g_pool == nullptr) throw Error(FVC_E_INVALID, "the cached backward needs g_pool");
  hipStream_t s = r.stream();
  const int n = D.n;
  if (n == 0) return;
  const int* counts = D.cached ? D.counts_all.as<int>() : D.counts.as<int>();
  hipLaunchKernelGGL(k_diff_composite_bwd, composite_grid(n), dim3(256), 0, s, n, m.scene.alpha_thre, counts,
                     D.offsets.as<int64_t>(), D.n_walk.as<int>(), D.out4.as<float4>(), D.s_dt.as<float>(),
                     D.ray_out.as<float4>(), d_rgb, D.d_out4.as<float4>());
  FVC_HIP(hipGetLastError());
  if (D.n_r > 0) {
    // the encoding's gradients pass through memory in chunks (at most 512 MiB,
    // less where the device has no room)
    int64_t cap = std::min<int64_t>(D.n_r, (int64_t)1 << 22);
    while (cap > 4096 && !D.d_enc.try_ensure((size_t)cap * 16 * sizeof(float2))) cap = (cap + 1) / 2;
    D.d_enc.ensure((size_t)cap * 16 * sizeof(float2));
    const int* list = D.cached ? D.list_r.as<int>() : nullptr;
    for (int64_t j0 = 0; j0 < D.n_r; j0 += cap) {
      const int64_t nc = std::min<int64_t>(cap, D.n_r - j0);
      hipLaunchKernelGGL(k_diff_net_bwd, dim3(bwd_blocks(nc)), dim3(64 * BWD_WAVES), 0, s, (int)j0, (int)(j0 + nc),
                         list, D.s_pos.as<float>(), D.s_ray.as<int>(), D.rays.as<RayState>(), D.pos, m.grid,
                         D.frags.as<float>(), D.d_out4.as<float4>(), D.d_enc.as<float2>(), cap, g_base, g_head);
      FVC_HIP(hipGetLastError());
      scatter_table(D, m.grid, list, j0, nc, cap, g_pos, s);
    }
  }
  if (D.n_c > 0) {
    hipLaunchKernelGGL(k_diffc_head_bwd, dim3(2 * bwd_blocks(D.n_c)), dim3(64 * BWD_WAVES), 0, s, (int)D.n_c,
                       D.list_c.as<int>(), D.s_pos.as<float>(), D.s_ray.as<int>(), D.rays.as<RayState>(), D.cv,
                       D.frags.as<float>(), D.d_out4.as<float4>(), g_head, g_pool);
    FVC_HIP(hipGetLastError());
  }
  FVC_HIP(hipStreamSynchronize(s));
}

}  // namespace fvc
