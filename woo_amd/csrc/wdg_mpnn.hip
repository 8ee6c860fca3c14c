// Learned coarse step: a message-passing network on the contact graph, trained and run by
// hand-written BF16 MFMA kernels (v_mfma_f32_16x16x32_bf16, FP32 accumulation).
//
// Network (hidden width H = 64):
//   h0 = relu(X W_enc + b_enc)                       X: node inputs, 32 columns (5 used)
//   for l in 0, 1:
//     m_e   = relu([h_recv(e), h_send(e), F_e] W_m,l + b_m,l)   F_e: edge inputs, 32 columns (9 used)
//     agg_i = sum over edges e received by i of m_e
//     u_i   = relu([h_i, agg_i] W_u,l + b_u,l);  h_i <- h_i + u_i
//   a_i = h_i W_dec + b_dec                          (3 outputs: acceleration / g)
// Storage: activations that feed a GEMM are BF16 (h, m, agg, u); GEMMs accumulate in FP32;
// the residual sum is formed in FP32 and rounded once; parameters are FP32 master copies with
// BF16 images (transposed for the forward GEMM operand, row-major for the input-gradient one).
//
// Graph: edges in CSR by receiver (rowOff, recv, send), both directions of every pair, and
// rev[e] = the opposite edge; every sum over edges follows this order (deterministic).
//
// Kernels: a wavefront owns 16 nodes and all the edges they receive. One kernel per layer forms the
// messages, sums them and updates the nodes (k_layer); nothing per edge is written but, for
// training, one 64-bit word of relu signs. Because the message GEMM is linear in its three inputs,
// its backward needs no per-edge gradient either: with S1_i = sum of dY_e over the edges received
// by i and S2_i over those sent by i (FP32 sums of the same BF16 values), the activation gradients
// are S1 W_recv^T + S2 W_send^T and the weight gradients h^T S1, h^T S2: GEMMs over nodes, of which
// there are seven times fewer. S1 and S2 enter the matrix cores as three BF16 terms that add up to
// the FP32 value exactly.
//
// MFMA operands for 64-wide wavefronts (16x16x32): lane l supplies row (l mod 16) and 8 values of k
// from group l/16. Which 8 k they are is free as long as both operands agree, so the result of one
// product (rows 4*(l/16) + q) is fed to the next from registers, without a transpose through LDS:
// messages to the segmented sum, the sum to the update, the update to the decoder.
#include <algorithm>
#include <cstring>
#include <vector>

#include "wdg_internal.hpp"

namespace wdg {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef uint16_t bf16;

constexpr int H = 64;     // hidden width
constexpr int KX = 32;    // node input columns (NIN used)
constexpr int KE = 32;    // edge input columns (NEI used)
constexpr int NIN = 7, NEI = 15;
constexpr int XP = 8, EP = 16;  // stored columns of the node and edge inputs (the others are zero)
constexpr int ONE = 15;         // free operand row of the input GEMMs: ones, for the bias gradient
constexpr int KM = 2 * H + KE;  // message GEMM inner dimension (160)
constexpr int KU = 2 * H;       // update GEMM inner dimension (128)
constexpr int NOUT = 3;
// input scales: lengths by R0, velocities by V0 (outputs are accelerations in units of MPNN_A0)
// overlaps (fractions of the contact distance, 1e-3 .. 1e-2) are scaled by MPNN_OV so that BF16
// resolves them, and clipped to +-MPNN_OV_CLIP as inputs of their own (gaps of spheres that are
// far apart would otherwise dominate the first layers); the force inputs use them unclipped
constexpr double MPNN_R0 = 2.5e-3, MPNN_V0 = 1.0, MPNN_OV = 100.0, MPNN_OV_CLIP = 2.0;
// unit of the outputs and targets: 100 g, the order of contact accelerations, so that outputs are
// of order one
constexpr double MPNN_A0 = 100.0 * 9.81;

// Inputs of edge e (receiver i, sender j), all scaled, computed in double:
//   0-2   (x_j - x_i) / (r_i + r_j)
//   3     overlap ov = (1 - d / (r_i + r_j)) OV, clipped to +-OV_CLIP
//   4-6   (v_j - v_i) / V0
//   7, 8  r_i / R0, r_j / R0
//   9-11  -n ov+^(3/2) sqrt(a b) (a + b) / a^3            (n = (x_j - x_i) / d, a = r_i / R0,
//                                                          b = r_j / R0, ov+ = max(ov, 0)):
//         the direction and radius scaling of a Hertz force on i, divided by i's mass
//   12-14 n vN ov+^(1/4) (a + b)^(1/4) sqrt(mb sqrt(Rb)) / a^3   (vN = (v_j - v_i).n / V0,
//         mb = a^3 b^3 / (a^3 + b^3), Rb = a b / (a + b)): the same for the viscous term
// Inputs of node i (floor at height zf, h = z_i - zf):
//   0-2   v_i / V0;  3  r_i / R0;  4  clip((1 - h / r_i) OV, +-OV_CLIP)
//   5     ovf+^(3/2) / a;  6  (v_i)_z / V0 ovf+^(1/4) / a   (ovf+ = max((1 - h / r_i) OV, 0))
// The same expressions, in the same order, build host graphs (woo_amd/surrogate.py).
__host__ __device__ inline void edge_inputs(double xi, double yi, double zi, double xj, double yj, double zj,
                                            double vxi, double vyi, double vzi, double vxj, double vyj,
                                            double vzj, double ri, double rj, float* f) {
  const double rs = ri + rj;
  const double dx = (xj - xi) / rs, dy = (yj - yi) / rs, dz = (zj - zi) / rs;
  const double dn = sqrt((dx * dx + dy * dy) + dz * dz);
  const double ov = (1. - dn) * MPNN_OV;
  const double wx = (vxj - vxi) / MPNN_V0, wy = (vyj - vyi) / MPNN_V0, wz = (vzj - vzi) / MPNN_V0;
  const double a = ri / MPNN_R0, b = rj / MPNN_R0;
  const double nx = dn > 0 ? dx / dn : 0., ny = dn > 0 ? dy / dn : 0., nz = dn > 0 ? dz / dn : 0.;
  const double ovp = ov > 0 ? ov : 0.;
  const double a3 = a * a * a, b3 = b * b * b;
  const double hz = ovp * sqrt(ovp) * (sqrt(a * b) * (a + b) / a3);
  const double mb = a3 * b3 / (a3 + b3), Rb = a * b / (a + b);
  const double vn = (wx * nx + wy * ny) + wz * nz;
  const double dp = vn * sqrt(sqrt(ovp)) * (sqrt(sqrt(a + b)) * sqrt(mb * sqrt(Rb)) / a3);
  const double ovc = fmin(fmax(ov, -MPNN_OV_CLIP), MPNN_OV_CLIP);
  const double v[NEI] = {dx, dy, dz, ovc, wx, wy, wz, a, b, -nx * hz, -ny * hz, -nz * hz, nx * dp, ny * dp, nz * dp};
  for (int q = 0; q < NEI; q++) f[q] = (float)v[q];
}
__host__ __device__ inline void node_inputs(double vx, double vy, double vz, double r, double h, float* f) {
  const double a = r / MPNN_R0;
  const double ov = (1. - h / r) * MPNN_OV;
  const double ovp = ov > 0 ? ov : 0.;
  const double v[NIN] = {vx / MPNN_V0, vy / MPNN_V0, vz / MPNN_V0, a, fmin(fmax(ov, -MPNN_OV_CLIP), MPNN_OV_CLIP),
                         ovp * sqrt(ovp) / a, vz / MPNN_V0 * sqrt(sqrt(ovp)) / a};
  for (int q = 0; q < NIN; q++) f[q] = (float)v[q];
}

// round to nearest even (finite inputs)
__host__ __device__ inline bf16 f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16 b) {
  uint32_t u = (uint32_t)b << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// ------------------------------------------------------------------ parameter layout (floats)
struct PLayout {
  size_t encW, encB, mW[2], mB[2], uW[2], uB[2], decW, decB, total;
  PLayout() {
    size_t o = 0;
    encW = o; o += (size_t)KX * H;
    encB = o; o += H;
    for (int l = 0; l < 2; l++) {
      mW[l] = o; o += (size_t)KM * H;
      mB[l] = o; o += H;
      uW[l] = o; o += (size_t)KU * H;
      uB[l] = o; o += H;
    }
    decW = o; o += (size_t)H * NOUT;
    decB = o; o += NOUT;
    total = o;
  }
};

__device__ __forceinline__ bf16x8 as_bf8(uint4 v) {
  bf16x8 r;
  memcpy(&r, &v, 16);
  return r;
}
__device__ __forceinline__ uint32_t pack2(bf16 lo, bf16 hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }
// two values rounded to nearest even in one instruction, the first in the low half
__device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 r = __builtin_convertvector((f2){lo, hi}, b2);
  uint32_t u;
  memcpy(&u, &r, 4);
  return u;
}
__device__ __forceinline__ floatx4 mfma(uint4 a, uint4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf8(a), as_bf8(b), c, 0, 0, 0);
}
__device__ __forceinline__ uint4 row8(const bf16* p) { return *reinterpret_cast<const uint4*>(p); }
// a relu's output is positive (it is never negative; -0 counts as zero)
__device__ __forceinline__ bool on(uint32_t b) { return (b & 0x7FFFu) != 0u; }
constexpr uint4 ZERO4 = {0u, 0u, 0u, 0u};

// ------------------------------------------------------------------ encoder
// h0 = relu(X W + b): the weights as the first operand, so that a lane ends with four consecutive
// features of one node (8-byte stores)
__global__ __launch_bounds__(256) void k_enc(int64_t N, const bf16* __restrict__ X, const bf16* __restrict__ Wt,
                                              const float* __restrict__ bias, bf16* __restrict__ h) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int64_t i = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + r;
  uint4 x = row8(X + min(i, N - 1) * XP);
  if (g != 0) x = ZERO4;  // columns 8 .. 31 are zero
#pragma unroll
  for (int cb = 0; cb < 4; cb++) {
    const floatx4 b = *reinterpret_cast<const floatx4*>(bias + cb * 16 + 4 * g);
    const floatx4 v = mfma(row8(Wt + (cb * 16 + r) * KX + 8 * g), x, b);
    if (i < N)
      *reinterpret_cast<uint2*>(h + i * H + cb * 16 + 4 * g) =
          make_uint2(cvt2(fmaxf(v[0], 0.f), fmaxf(v[1], 0.f)), cvt2(fmaxf(v[2], 0.f), fmaxf(v[3], 0.f)));
  }
}

// ------------------------------------------------------------------ one layer, forward
// messages m_e = relu([h_recv, h_send, F] Wm + bm), their sums, u = relu([h, agg] Wu + bu) and
// h + u, for the 16 nodes of each wavefront; LAST: also the decoder and the contact flags.
// 32 edges at a time: the message product leaves lane l with edges 4*(l/16) + q (of both halves)
// of feature l mod 16, which is the operand of the segmented sum: a product with the 0/1 matrix
// of edges and receivers, exact but for the order of an FP32 sum (the 0/1 operand comes from the
// row offsets). A message that is not finite spreads over the wavefront's nodes there (0 * inf):
// where a sum is not finite, the wavefront's edges are gone through again and summed one by one.
// Bound by the chain of a chunk (end points, rows, 40 + 4 products, 20 LDS reads of weights) at three
// wavefronts per SIMD: 120,000 nodes and 840,000 edges take 60 us a layer; the message product, the
// sum and the update as kernels of their own took 67 + 23 + 15. Four wavefronts per SIMD spill
// (78 us). Both weight images (39 KB, rows padded for the banks) are staged once per workgroup,
// three of which fit a compute unit: 768 workgroups walk the tiles (1,024: 14% slower).
struct LayerArgs {
  int64_t N;
  const int32_t *rowOff, *recv, *send;
  const bf16 *h, *ef, *x, *Wm, *Wu;
  const float *bm, *bu, *Wd, *bd;
  bf16 *hOut, *agg;
  uint64_t *mMask, *uMask;
  float* out;
  uint8_t* flag;
};
constexpr int LY_BS = 256;
constexpr int WMP = KM + 8, WUP = KU + 8;  // padded LDS rows
template <bool STORE, bool LAST>
__global__ __launch_bounds__(LY_BS, 3) void k_layer(LayerArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 Wm[H * WMP];
  __shared__ __attribute__((aligned(16))) bf16 Wu[H * WUP];
  __shared__ float Wd[H * NOUT];
  // (every load in flight before the first store)
  {
    constexpr int QM = H * KM / 8 / LY_BS, QU = H * KU / 8 / LY_BS;
    static_assert(QM * LY_BS * 8 == H * KM && QU * LY_BS * 8 == H * KU, "whole passes over the images");
    uint4 v[QM + QU];
#pragma unroll
    for (int q = 0; q < QM; q++) v[q] = row8(a.Wm + (q * LY_BS + threadIdx.x) * 8);
#pragma unroll
    for (int q = 0; q < QU; q++) v[QM + q] = row8(a.Wu + (q * LY_BS + threadIdx.x) * 8);
#pragma unroll
    for (int q = 0; q < QM; q++) {
      const int i = q * LY_BS + threadIdx.x;
      *reinterpret_cast<uint4*>(&Wm[i / (KM / 8) * WMP + i % (KM / 8) * 8]) = v[q];
    }
#pragma unroll
    for (int q = 0; q < QU; q++) {
      const int i = q * LY_BS + threadIdx.x;
      *reinterpret_cast<uint4*>(&Wu[i / (KU / 8) * WUP + i % (KU / 8) * 8]) = v[QM + q];
    }
  }
  if (LAST && threadIdx.x < H * NOUT) Wd[threadIdx.x] = a.Wd[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  float bm[4];
#pragma unroll
  for (int cb = 0; cb < 4; cb++) bm[cb] = a.bm[cb * 16 + r];
  const int64_t nt = (a.N + 15) / 16;
  for (int64_t t = (int64_t)xcd_block(blockIdx.x, gridDim.x) * (LY_BS / 64) + (threadIdx.x >> 6); t < nt;
       t += (int64_t)gridDim.x * (LY_BS / 64)) {
    const bool node = t * 16 + r < a.N;
    const int64_t i = node ? t * 16 + r : a.N - 1;
    const int32_t b0 = a.rowOff[node ? i : a.N], b1 = a.rowOff[i + 1];
    const int32_t e0 = __shfl(b0, 0), e1 = __shfl(b1, 15);
    floatx4 agg[4];
    bool touch = false;
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll
      for (int cb = 0; cb < 4; cb++) agg[cb] = floatx4{0, 0, 0, 0};
      int32_t rc[2], sd[2];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const int32_t e = max(min(e0 + 16 * q + r, e1 - 1), 0);
        rc[q] = e0 < e1 ? a.recv[e] : 0;
        sd[q] = e0 < e1 ? a.send[e] : 0;
      }
      for (int32_t eb = e0; eb < e1; eb += 32) {
        uint4 z[2][5];
#pragma unroll
        for (int q = 0; q < 2; q++) {
          // past the last edge: that edge again (it counts for no node below, and no load is
          // conditional)
          const int32_t e = min(eb + 16 * q + r, e1 - 1);
          const int64_t er = rc[q], es = sd[q];
          const int32_t en = min(eb + 32 + 16 * q + r, e1 - 1);  // the next ends, a chunk ahead
          rc[q] = a.recv[en];
          sd[q] = a.send[en];
          z[q][4] = row8(a.ef + (int64_t)e * EP + 8 * (g & 1));
          if (g >= 2) z[q][4] = ZERO4;  // columns 16 .. 31 are zero
          z[q][0] = row8(a.h + er * H + 8 * g);
          z[q][1] = row8(a.h + er * H + 32 + 8 * g);
          z[q][2] = row8(a.h + es * H + 8 * g);
          z[q][3] = row8(a.h + es * H + 32 + 8 * g);
          if (LAST) {
            // overlap inputs (column 3, in the lanes of group 0) of this half's edges, against the
            // lane's node's range of them
            const uint64_t pos = __ballot(bf2f((bf16)(z[q][4].y >> 16)) > 0.f) & 0xFFFFull;
            const int lo = min(max(b0 - (eb + 16 * q), 0), 16), hi = min(max(b1 - (eb + 16 * q), 0), 16);
            touch = touch || ((uint32_t)pos & ((1u << hi) - 1u) & ~((1u << lo) - 1u)) != 0u;
          }
        }
        // (the weights stay in LDS: held in registers over the loop they would be spilled)
        int wo = r * WMP + 8 * g;
        asm volatile("" : "+v"(wo));
        floatx4 acc[2][4];
#pragma unroll
        for (int cb = 0; cb < 4; cb++) acc[0][cb] = acc[1][cb] = floatx4{bm[cb], bm[cb], bm[cb], bm[cb]};
#pragma unroll
        for (int ks = 0; ks < 5; ks++) {
          asm volatile("" ::: "memory");  // a step's weights at a time
#pragma unroll
          for (int cb = 0; cb < 4; cb++) {
            const uint4 w = row8(&Wm[cb * 16 * WMP + ks * 32 + wo]);
            acc[0][cb] = mfma(z[0][ks], w, acc[0][cb]);
            acc[1][cb] = mfma(z[1][ks], w, acc[1][cb]);
          }
        }
        // relu, rounded once
        uint4 mv[4];
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; j++) v[j] = fmaxf(acc[j >> 2][cb][j & 3], 0.f);
          mv[cb] = make_uint4(cvt2(v[0], v[1]), cvt2(v[2], v[3]), cvt2(v[4], v[5]), cvt2(v[6], v[7]));
        }
        if (STORE) {
          // sign words: bit 16 * cb + feature of edge 4 * (lane / 16) + q
#pragma unroll
          for (int q = 0; q < 2; q++) {
            uint64_t word = 0;
#pragma unroll
            for (int cb = 0; cb < 4; cb++) {
              const uint32_t w0 = q ? mv[cb].z : mv[cb].x, w1 = q ? mv[cb].w : mv[cb].y;
              const uint64_t s0 = __ballot(on(w0)), s1 = __ballot(on(w0 >> 16)), s2 = __ballot(on(w1)),
                             s3 = __ballot(on(w1 >> 16));
              const uint64_t sq = (r & 2) ? ((r & 1) ? s3 : s2) : ((r & 1) ? s1 : s0);
              word |= ((sq >> (16 * (r >> 2))) & 0xFFFFull) << (16 * cb);
            }
            const int32_t e = eb + 16 * q + r;
            if (g == 0 && e < e1) a.mMask[e] = word;
          }
        }
        // the 0/1 operand: node r against edges eb + 16 * (j / 4) + 4 * g + j % 4
        const int lo = min(max(b0 - eb, 0), 32), hi = min(max(b1 - eb, 0), 32);
        const uint32_t in = (uint32_t)((1ull << hi) - 1ull) & ~(uint32_t)((1ull << lo) - 1ull);
        const uint32_t i0 = in >> (4 * g), i1 = i0 >> 16;
        if (pass == 0) {
          const uint4 sw = make_uint4((i0 & 1u) * 0x3F80u | (i0 >> 1 & 1u) * 0x3F800000u,
                                      (i0 >> 2 & 1u) * 0x3F80u | (i0 >> 3 & 1u) * 0x3F800000u,
                                      (i1 & 1u) * 0x3F80u | (i1 >> 1 & 1u) * 0x3F800000u,
                                      (i1 >> 2 & 1u) * 0x3F80u | (i1 >> 3 & 1u) * 0x3F800000u);
#pragma unroll
          for (int cb = 0; cb < 4; cb++) agg[cb] = mfma(mv[cb], sw, agg[cb]);
        } else {
          for (int k = 0; k < 32; k++) {
            // edge eb + k: group (k % 16) / 4, value 4 * (k / 16) + k % 4 of its lanes
            const int kg = (k & 15) >> 2, j = 2 * (k >> 4) + ((k & 3) >> 1);
            const bool mine = (in >> k) & 1u;
#pragma unroll
            for (int cb = 0; cb < 4; cb++) {
              const uint32_t w = j == 0 ? mv[cb].x : (j == 1 ? mv[cb].y : (j == 2 ? mv[cb].z : mv[cb].w));
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const uint32_t o = __shfl(w, 16 * kg + 4 * g + q);
                const float v = bf2f((bf16)((k & 1) ? o >> 16 : o & 0xFFFFu));
                agg[cb][q] += mine ? v : 0.f;
              }
            }
          }
        }
      }
      bool fin = true;
#pragma unroll
      for (int cb = 0; cb < 4; cb++)
#pragma unroll
        for (int q = 0; q < 4; q++) fin = fin && fabsf(agg[cb][q]) <= 3.402823466e38f;
      if (__all(fin)) break;
    }
    // agg: features 16 * cb + 4 * g + q of node r, rounded once
    uint2 ag[4];
#pragma unroll
    for (int cb = 0; cb < 4; cb++) ag[cb] = make_uint2(cvt2(agg[cb][0], agg[cb][1]), cvt2(agg[cb][2], agg[cb][3]));
    if (STORE && node)
#pragma unroll
      for (int cb = 0; cb < 4; cb++) *reinterpret_cast<uint2*>(a.agg + i * H + cb * 16 + 4 * g) = ag[cb];
    // update: the weights' columns in the order of the operand's features
    uint4 hz[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) hz[ks] = row8(a.h + i * H + ks * 32 + 8 * g);
    int uo = r * WUP + 4 * g;
    asm volatile("" : "+v"(uo));
    floatx4 up[4];
#pragma unroll
    for (int cb = 0; cb < 4; cb++) {
      const bf16* w = &Wu[cb * 16 * WUP + uo];
      floatx4 u = *reinterpret_cast<const floatx4*>(a.bu + cb * 16 + 4 * g);
#pragma unroll
      for (int ks = 0; ks < 2; ks++) u = mfma(row8(w + ks * 32 + 4 * g), hz[ks], u);
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const uint2 w0 = *reinterpret_cast<const uint2*>(w + H + ks * 32),
                    w1 = *reinterpret_cast<const uint2*>(w + H + ks * 32 + 16);
        u = mfma(make_uint4(w0.x, w0.y, w1.x, w1.y), make_uint4(ag[2 * ks].x, ag[2 * ks].y, ag[2 * ks + 1].x, ag[2 * ks + 1].y), u);
      }
      up[cb] = u;
    }
    uint64_t um = 0;
    float o[NOUT] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int cb = 0; cb < 4; cb++) {
      const int f0 = cb * 16 + 4 * g;
      const uint2 hw = *reinterpret_cast<const uint2*>(a.h + i * H + f0);
      const bf16 hh[4] = {(bf16)(hw.x & 0xFFFFu), (bf16)(hw.x >> 16), (bf16)(hw.y & 0xFFFFu), (bf16)(hw.y >> 16)};
      bf16 hn[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const bf16 u = f2bf(fmaxf(up[cb][q], 0.f));
        um |= (uint64_t)(on(u) ? 1u : 0u) << (f0 + q);
        hn[q] = f2bf(bf2f(hh[q]) + bf2f(u));
        if (LAST)
#pragma unroll
          for (int c = 0; c < NOUT; c++) o[c] += bf2f(hn[q]) * Wd[(f0 + q) * NOUT + c];
      }
      if (node && (STORE || !LAST))
        *reinterpret_cast<uint2*>(a.hOut + i * H + f0) = make_uint2(pack2(hn[0], hn[1]), pack2(hn[2], hn[3]));
    }
    if (STORE) {
      um |= (uint64_t)__shfl_xor((unsigned long long)um, 16);
      um |= (uint64_t)__shfl_xor((unsigned long long)um, 32);
      if (node && g == 0) a.uMask[i] = um;
    }
    if (LAST) {
#pragma unroll
      for (int c = 0; c < NOUT; c++) {
        o[c] += __shfl_xor(o[c], 16);
        o[c] += __shfl_xor(o[c], 32);
      }
      // a node is in contact when its floor overlap input or the overlap input of one of its edges
      // is positive. Nodes not in contact move in free flight (the network's output is not used for
      // them), so they carry no loss.
      if (node && g == 0) {
#pragma unroll
        for (int c = 0; c < NOUT; c++) a.out[i * NOUT + c] = a.bd[c] + o[c];
        a.flag[i] = touch || bf2f(a.x[i * XP + 4]) > 0.f ? 1 : 0;
      }
    }
  }
}

// ------------------------------------------------------------------ loss and decoder, backward
// loss = mean over nodes of |a - t|^2, dA = 2 (a - t) / N, dh = dA W^T, partials of dW (H x 3) and
// db (3): DEC_ROWS nodes per workgroup, a feature per lane, DEC_ROWS / 4 nodes per wavefront
// (25,000 nodes: 9 us; a reduction of the workgroup per feature took 68)
constexpr int DEC_ROWS = 64, DECW = (H + 1) * NOUT;
__global__ __launch_bounds__(256) void k_loss_dec(int64_t N, const float* __restrict__ a, const float* __restrict__ t,
                                                   const uint8_t* __restrict__ flag, const bf16* __restrict__ h,
                                                   const float* __restrict__ W, float* __restrict__ dh,
                                                   float* __restrict__ part, float* __restrict__ partLoss) {
  __shared__ float G[DEC_ROWS][NOUT + 1];
  __shared__ float sm[4][H][NOUT];
  const int64_t i0 = (int64_t)blockIdx.x * DEC_ROWS;
  const int k = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (wv == 0) {
    const int64_t i = i0 + k;
    float l = 0.f;
#pragma unroll
    for (int c = 0; c < NOUT; c++) {
      const float x = a[min(i, N - 1) * NOUT + c] - t[min(i, N - 1) * NOUT + c];
      const float d = i < N && flag[min(i, N - 1)] ? x : 0.f;
      l += d * d;
      G[k][c] = 2.f * d / (float)N;
    }
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
    if (k == 0) partLoss[blockIdx.x] = l;
  }
  const float w[NOUT] = {W[k * NOUT], W[k * NOUT + 1], W[k * NOUT + 2]};
  __syncthreads();
  float s[NOUT] = {0.f, 0.f, 0.f};
#pragma unroll 4
  for (int q = 0; q < DEC_ROWS / 4; q++) {
    const int row = wv * (DEC_ROWS / 4) + q;
    const int64_t i = i0 + row;
    if (i >= N) break;
    const float g[NOUT] = {G[row][0], G[row][1], G[row][2]};
    const float x = bf2f(h[i * H + k]);
    dh[i * H + k] = (g[0] * w[0] + g[1] * w[1]) + g[2] * w[2];
#pragma unroll
    for (int c = 0; c < NOUT; c++) s[c] += x * g[c];
  }
#pragma unroll
  for (int c = 0; c < NOUT; c++) sm[wv][k][c] = s[c];
  __syncthreads();
  float* P = part + (int64_t)blockIdx.x * DECW;
  if (threadIdx.x < H * NOUT) {
    const int kk = threadIdx.x / NOUT, c = threadIdx.x % NOUT;
    P[threadIdx.x] = ((sm[0][kk][c] + sm[1][kk][c]) + sm[2][kk][c]) + sm[3][kk][c];
  } else if (threadIdx.x < DECW) {
    const int c = threadIdx.x - H * NOUT;
    float b = 0.f;
    for (int q = 0; q < DEC_ROWS; q++) b += G[q][c];
    P[threadIdx.x] = b;
  }
}

// ------------------------------------------------------------------ update, backward
// dUb = BF16(dh * (u > 0)); [dhp | dagg] = [dh | 0] + dUb Wu^T: dhp FP32, dagg BF16 (g, the gradient
// of every message of the node before its relu mask)
__global__ __launch_bounds__(256) void k_bwd_update(int64_t N, const float* __restrict__ dh,
                                                     const uint64_t* __restrict__ uMask, const bf16* __restrict__ Wr,
                                                     bf16* __restrict__ dUb, float* __restrict__ dhp,
                                                     bf16* __restrict__ gOut) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t * 16 >= N) return;
  const bool node = t * 16 + r < N;
  const int64_t i = node ? t * 16 + r : N - 1;
  const uint64_t um = uMask[i];
  uint4 d[2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const int f0 = ks * 32 + 8 * g;
    const float4 x = *reinterpret_cast<const float4*>(dh + i * H + f0), y = *reinterpret_cast<const float4*>(dh + i * H + f0 + 4);
    const uint32_t m = (uint32_t)(um >> f0);
    const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
    bf16 b[8];
#pragma unroll
    for (int q = 0; q < 8; q++) b[q] = f2bf((m >> q) & 1u ? v[q] : 0.f);
    d[ks] = make_uint4(pack2(b[0], b[1]), pack2(b[2], b[3]), pack2(b[4], b[5]), pack2(b[6], b[7]));
    if (node) *reinterpret_cast<uint4*>(dUb + i * H + f0) = d[ks];
  }
#pragma unroll
  for (int cb = 0; cb < 8; cb++) {
    floatx4 acc = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 2; ks++) acc = mfma(row8(Wr + (cb * 16 + r) * H + ks * 32 + 8 * g), d[ks], acc);
    if (cb < 4) {
      const int64_t o = i * H + cb * 16 + 4 * g;
      const float4 x = *reinterpret_cast<const float4*>(dh + o);
      if (node) *reinterpret_cast<float4*>(dhp + o) = make_float4(x.x + acc[0], x.y + acc[1], x.z + acc[2], x.w + acc[3]);
    } else if (node) {
      *reinterpret_cast<uint2*>(gOut + i * H + (cb - 4) * 16 + 4 * g) =
          make_uint2(pack2(f2bf(acc[0]), f2bf(acc[1])), pack2(f2bf(acc[2]), f2bf(acc[3])));
    }
  }
}

// ------------------------------------------------------------------ messages, backward
// an FP32 value as three BF16 terms of 8 bits each, by truncation: their sum is the value itself
// (a value that is not finite is its first term)
// (two values at a time, each term of both packed in one word)
__device__ __forceinline__ uint32_t top16(float& x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  const bool fin = (u & 0x7F800000u) != 0x7F800000u;
  const uint32_t b = fin ? u >> 16 : (uint32_t)f2bf(x);
  x = fin ? x - bf2f((bf16)b) : 0.f;
  return b;
}
__device__ __forceinline__ void split3_8(const float (&x)[8], uint4 (&o)[3]) {
  float y[8];
#pragma unroll
  for (int q = 0; q < 8; q++) y[q] = x[q];
#pragma unroll
  for (int p = 0; p < 3; p++) {
    uint32_t b[8];
#pragma unroll
    for (int q = 0; q < 8; q++) b[q] = top16(y[q]);
    o[p] = make_uint4(b[0] | b[1] << 16, b[2] | b[3] << 16, b[4] | b[5] << 16, b[6] | b[7] << 16);
  }
}
// s += g masked by 8 bits
__device__ __forceinline__ void add_masked(float (&s)[8], uint4 v, uint32_t m) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    s[2 * q] += (m >> (2 * q)) & 1u ? bf2f((bf16)(w[q] & 0xFFFFu)) : 0.f;
    s[2 * q + 1] += (m >> (2 * q + 1)) & 1u ? bf2f((bf16)(w[q] >> 16)) : 0.f;
  }
}
// S1 and S2 of the wavefront's 16 nodes (four lanes per node, 16 features each), and
// dh = dhp + S1 Wrecv^T + S2 Wsend^T. OPPOSITE: rev[e] is the opposite edge throughout, so the edges
// that a node sends are the opposites of those it receives; else the edges by sender give S2.
struct MsgArgs {
  int64_t N;
  const int32_t *rowOff, *recv, *send, *rev, *sOff, *sEdge;
  const uint64_t* mask;
  const bf16 *g, *Wm;
  const float* dhp;
  float *dh, *S1, *S2;
};
template <bool OPPOSITE>
__global__ __launch_bounds__(256) void k_bwd_message(MsgArgs a) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t * 16 >= a.N) return;
  const bool node = t * 16 + r < a.N;
  const int64_t i = node ? t * 16 + r : a.N - 1;
  float s1[2][8], s2[2][8];
#pragma unroll
  for (int ks = 0; ks < 2; ks++)
#pragma unroll
    for (int q = 0; q < 8; q++) s1[ks][q] = s2[ks][q] = 0.f;
  const uint4 gi[2] = {row8(a.g + i * H + 8 * g), row8(a.g + i * H + 32 + 8 * g)};
  const int32_t e0 = a.rowOff[i], e1 = a.rowOff[i + 1];
  // 16 edges at a time: lane g of a node fetches the words of four of them, all in flight together
  // (two waits on memory per batch, the second one also for the neighbours' rows)
  for (int32_t eb = e0; eb < e1; eb += 16) {
    int32_t nb[4];
    uint64_t m1[4], m2[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int32_t e = min(eb + 4 * k + g, e1 - 1);
      const int32_t o = a.rev[e];
      nb[k] = OPPOSITE ? a.send[e] : a.recv[o];
      m1[k] = a.mask[e];
      m2[k] = a.mask[o];
      if (eb + 4 * k + g >= e1) m1[k] = m2[k] = 0;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (eb + 4 * k >= e1) break;
      uint4 v[4][2];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int64_t j = __shfl(nb[k], r + 16 * q);
#pragma unroll
        for (int ks = 0; ks < 2; ks++) v[q][ks] = row8(a.g + j * H + ks * 32 + 8 * g);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint64_t x1 = (uint64_t)__shfl((unsigned long long)m1[k], r + 16 * q),
                       x2 = (uint64_t)__shfl((unsigned long long)m2[k], r + 16 * q);
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          add_masked(s1[ks], gi[ks], (uint32_t)(x1 >> (ks * 32 + 8 * g)));
          add_masked(s2[ks], v[q][ks], (uint32_t)(x2 >> (ks * 32 + 8 * g)));
        }
      }
    }
  }
  uint4 p1[2][3], p2[2][3];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    split3_8(s1[ks], p1[ks]);
    split3_8(s2[ks], p2[ks]);
  }
#pragma unroll
  for (int cb = 0; cb < 4; cb++) {
    floatx4 acc = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const uint4 w1 = row8(a.Wm + (cb * 16 + r) * H + ks * 32 + 8 * g),
                  w2 = row8(a.Wm + (H + cb * 16 + r) * H + ks * 32 + 8 * g);
#pragma unroll
      for (int p = 2; p >= 0; p--) {
        acc = mfma(w1, p1[ks][p], acc);
        acc = mfma(w2, p2[ks][p], acc);
      }
    }
    const int64_t o = i * H + cb * 16 + 4 * g;
    const float4 x = *reinterpret_cast<const float4*>(a.dhp + o);
    if (node)
      *reinterpret_cast<float4*>(a.dh + o) = make_float4(x.x + acc[0], x.y + acc[1], x.z + acc[2], x.w + acc[3]);
  }
  if (!node) return;
  if (!OPPOSITE) {
    // the weight gradient takes the edges that the node sends
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int q = 0; q < 8; q++) s2[ks][q] = 0.f;
    for (int32_t k = a.sOff[i]; k < a.sOff[i + 1]; k++) {
      const int32_t e = a.sEdge[k];
      const int64_t j = a.recv[e];
      const uint64_t m = a.mask[e];
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
        add_masked(s2[ks], row8(a.g + j * H + ks * 32 + 8 * g), (uint32_t)(m >> (ks * 32 + 8 * g)));
    }
  }
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const int64_t o = i * H + ks * 32 + 8 * g;
    *reinterpret_cast<float4*>(a.S1 + o) = make_float4(s1[ks][0], s1[ks][1], s1[ks][2], s1[ks][3]);
    *reinterpret_cast<float4*>(a.S1 + o + 4) = make_float4(s1[ks][4], s1[ks][5], s1[ks][6], s1[ks][7]);
    *reinterpret_cast<float4*>(a.S2 + o) = make_float4(s2[ks][0], s2[ks][1], s2[ks][2], s2[ks][3]);
    *reinterpret_cast<float4*>(a.S2 + o + 4) = make_float4(s2[ks][4], s2[ks][5], s2[ks][6], s2[ks][7]);
  }
}

// ------------------------------------------------------------------ weight gradients over nodes
// One partial per workgroup: [h, agg]^T dUb (KU x H), the column sums of dUb (H), h^T S1 and h^T S2
// (2H x H). Chunks of 32 nodes are staged in LDS transposed, so that the operands are 16-byte
// reads; wavefront w forms output features 16 w .. 16 w + 15 (16 accumulators). A workgroup per
// compute unit at most: more would write and read more partials (66 KB each) than they save.
constexpr int DWN = KU * H + H + 2 * H * H;
__global__ __launch_bounds__(256) void k_dw_node(int64_t N, const bf16* __restrict__ h, const bf16* __restrict__ agg,
                                                  const bf16* __restrict__ dUb, const float* __restrict__ S1,
                                                  const float* __restrict__ S2, float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) bf16 At[KU][32 + 8];
  __shared__ __attribute__((aligned(16))) bf16 Dt[7][H][32 + 8];  // dUb, the terms of S1, those of S2
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  floatx4 au[8], am[8];
#pragma unroll
  for (int cb = 0; cb < 8; cb++) au[cb] = am[cb] = floatx4{0, 0, 0, 0};
  float bias = 0.f;
  const int64_t nch = (N + 31) / 32;
  const int rr = threadIdx.x & 31, c8 = (threadIdx.x >> 5) * 8;
  auto put = [&](bf16 (*T)[32 + 8], uint4 v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; q++) {
      T[c8 + 2 * q][rr] = (bf16)(w[q] & 0xFFFFu);
      T[c8 + 2 * q + 1][rr] = (bf16)(w[q] >> 16);
    }
  };
  // a chunk's rows (zero past the last), loaded while the products of the chunk before run
  uint4 vh, va, vd;
  float x1[8], x2[8];
  auto fetch = [&](int64_t ch) {
    const bool live = ch * 32 + rr < N;
    const int64_t o = (live ? ch * 32 + rr : N - 1) * H + c8;
    vh = row8(h + o);
    va = row8(agg + o);
    vd = row8(dUb + o);
#pragma unroll
    for (int q = 0; q < 8; q += 4) {
      const float4 y1 = *reinterpret_cast<const float4*>(S1 + o + q), y2 = *reinterpret_cast<const float4*>(S2 + o + q);
      x1[q] = y1.x; x1[q + 1] = y1.y; x1[q + 2] = y1.z; x1[q + 3] = y1.w;
      x2[q] = y2.x; x2[q + 1] = y2.y; x2[q + 2] = y2.z; x2[q + 3] = y2.w;
    }
    if (!live) {
      vh = va = vd = ZERO4;
#pragma unroll
      for (int q = 0; q < 8; q++) x1[q] = x2[q] = 0.f;
    }
  };
  if (blockIdx.x < nch) fetch(blockIdx.x);
  for (int64_t ch = blockIdx.x; ch < nch; ch += gridDim.x) {
    put(At, vh);
    put(At + H, va);
    put(Dt[0], vd);
    uint4 t3[3];
    split3_8(x1, t3);
#pragma unroll
    for (int p = 0; p < 3; p++) put(Dt[1 + p], t3[p]);
    split3_8(x2, t3);
#pragma unroll
    for (int p = 0; p < 3; p++) put(Dt[4 + p], t3[p]);
    __syncthreads();
    if (ch + gridDim.x < nch) fetch(ch + gridDim.x);
    uint4 d[7];
#pragma unroll
    for (int p = 0; p < 7; p++) d[p] = row8(&Dt[p][wv * 16 + r][8 * g]);
    {
      const uint32_t w[4] = {d[0].x, d[0].y, d[0].z, d[0].w};
#pragma unroll
      for (int q = 0; q < 4; q++) bias += bf2f((bf16)(w[q] & 0xFFFFu)) + bf2f((bf16)(w[q] >> 16));
    }
#pragma unroll
    for (int cb = 0; cb < 8; cb++) {
      const uint4 x = row8(&At[cb * 16 + r][8 * g]);
      au[cb] = mfma(x, d[0], au[cb]);
      if (cb < 4) {
#pragma unroll
        for (int p = 2; p >= 0; p--) {
          am[cb] = mfma(x, d[1 + p], am[cb]);
          am[4 + cb] = mfma(x, d[4 + p], am[4 + cb]);
        }
      }
    }
    __syncthreads();
  }
  float* P = part + (int64_t)blockIdx.x * DWN;
  float* Pm = P + KU * H + H;
#pragma unroll
  for (int cb = 0; cb < 8; cb++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int o = (cb * 16 + 4 * g + q) * H + wv * 16 + r;
      P[o] = au[cb][q];
      Pm[o] = am[cb][q];  // rows 0 .. 63: S1, 64 .. 127: S2
    }
  bias += __shfl_xor(bias, 16);
  bias += __shfl_xor(bias, 32);
  if (g == 0) P[KU * H + wv * 16 + r] = bias;
}

// ------------------------------------------------------------------ weight gradients over input rows
// in^T D over M rows of inputs, row ONE of the operand set to one (its output row is the bias
// gradient). EDGE: edge inputs, D_e = mask_e applied to g of the receiver; else node inputs,
// D_i = BF16(dh_i * (h0_i > 0)). Each wavefront walks chunks of 32 rows; one partial per workgroup.
struct RowArgs {
  int64_t M;
  const bf16* in;
  const int32_t* recv;
  const uint64_t* mask;
  const bf16* g;
  const float* dh;
  const bf16* h0;
};
constexpr int DWR = 16 * H;
template <bool EDGE>
__global__ __launch_bounds__(256) void k_dw_rows(RowArgs a, float* __restrict__ part) {
  __shared__ float sm[4][DWR];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  floatx4 acc[4];
#pragma unroll
  for (int cb = 0; cb < 4; cb++) acc[cb] = floatx4{0, 0, 0, 0};
  const int64_t nch = (a.M + 31) / 32;
  for (int64_t ch = (int64_t)blockIdx.x * 4 + wv; ch < nch; ch += (int64_t)gridDim.x * 4) {
    const int64_t m0 = ch * 32 + 8 * g;
    // (rows past the last: the last one again, zeroed after the loads)
    bf16 x[8], d[4][8];
    uint64_t w[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int64_t m = min(m0 + j, a.M - 1);
      x[j] = a.in[m * (EDGE ? EP : XP) + (EDGE ? r : (r & (XP - 1)))];
      if (EDGE) {
        w[j] = a.mask[m];
        const int64_t i = a.recv[m];
#pragma unroll
        for (int cb = 0; cb < 4; cb++) d[cb][j] = a.g[i * H + cb * 16 + r];
      } else {
        w[j] = 0;
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
          d[cb][j] = f2bf(a.dh[m * H + cb * 16 + r]);
          w[j] |= (uint64_t)(on(a.h0[m * H + cb * 16 + r]) ? 1u : 0u) << (cb * 16 + r);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const bool live = m0 + j < a.M;
      if (!live || (!EDGE && r >= XP)) x[j] = 0;
      if (live && r == ONE) x[j] = (bf16)0x3F80;
#pragma unroll
      for (int cb = 0; cb < 4; cb++)
        if (!live || !((w[j] >> (cb * 16 + r)) & 1ull)) d[cb][j] = 0;
    }
    const uint4 xv = make_uint4(pack2(x[0], x[1]), pack2(x[2], x[3]), pack2(x[4], x[5]), pack2(x[6], x[7]));
#pragma unroll
    for (int cb = 0; cb < 4; cb++)
      acc[cb] = mfma(xv, make_uint4(pack2(d[cb][0], d[cb][1]), pack2(d[cb][2], d[cb][3]), pack2(d[cb][4], d[cb][5]),
                                    pack2(d[cb][6], d[cb][7])), acc[cb]);
  }
#pragma unroll
  for (int cb = 0; cb < 4; cb++)
#pragma unroll
    for (int q = 0; q < 4; q++) sm[wv][(4 * g + q) * H + cb * 16 + r] = acc[cb][q];
  __syncthreads();
  for (int q = threadIdx.x; q < DWR; q += 256)
    part[(int64_t)blockIdx.x * DWR + q] = ((sm[0][q] + sm[1][q]) + sm[2][q]) + sm[3][q];
}

// ------------------------------------------------------------------ sums of the partials
// every region of the gradient in one launch: 64 columns per workgroup, the partials of a column
// over 16 wavefronts, then those in order. The last workgroup adds the loss up (in FP64).
// 25,000 nodes, 175,000 edges: 9 us; one thread per column and eleven
// launches took 257.
struct SumArgs {
  struct Region {
    const float* src;
    int64_t stride;
    int nblk, n;
    float* dst;
    int blk0;
  };
  Region r[14];
  int n, blocks;
};
__global__ __launch_bounds__(1024) void k_sum_partials(SumArgs a, int64_t nLoss, const float* __restrict__ partLoss,
                                                        double* loss) {
  if ((int)blockIdx.x == a.blocks) {
    __shared__ double sd[1024];
    double l = 0.;
    for (int64_t b = threadIdx.x; b < nLoss; b += 1024) l += (double)partLoss[b];
    sd[threadIdx.x] = l;
    __syncthreads();
    for (int st = 512; st > 0; st >>= 1) {
      if ((int)threadIdx.x < st) sd[threadIdx.x] += sd[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = sd[0];
    return;
  }
  int q = 0;
  while (q + 1 < a.n && (int)blockIdx.x >= a.r[q + 1].blk0) q++;
  const SumArgs::Region R = a.r[q];
  __shared__ float sm[16][64];
  const int col = ((int)blockIdx.x - R.blk0) * 64 + (threadIdx.x & 63), wv = threadIdx.x >> 6;
  float s = 0.f;
  if (col < R.n) {
#pragma unroll 8
    for (int b = wv; b < R.nblk; b += 16) s += R.src[(int64_t)b * R.stride + col];
  }
  sm[wv][threadIdx.x & 63] = s;
  __syncthreads();
  if (wv == 0 && col < R.n) {
#pragma unroll
    for (int k = 1; k < 16; k++) s += sm[k][threadIdx.x];
    R.dst[col] = s;
  }
}

// ------------------------------------------------------------------ optimizer and images
// BF16 images of the weights (K x 64 each): transposed [64 x K] and row-major [K x 64]
struct ImgArgs {
  int64_t src[5];
  int K[5];
  int64_t t[5], r[5];
  bf16* img;
};
__device__ __forceinline__ void image_write(const ImgArgs& g, int64_t i, float w) {
#pragma unroll
  for (int q = 0; q < 5; q++) {
    const int64_t t = i - g.src[q];
    if (t >= 0 && t < (int64_t)g.K[q] * H) {
      const bf16 b = f2bf(w);
      g.img[g.r[q] + t] = b;
      g.img[g.t[q] + (t % H) * g.K[q] + t / H] = b;
    }
  }
}
__global__ void k_adam(int64_t n, float* p, const float* __restrict__ g, float* m, float* v, float lr, float b1,
                       float b2, float eps, float c1, float c2, ImgArgs im) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float w = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = w;
  image_write(im, i, w);
}
__global__ void k_images(int64_t n, const float* __restrict__ p, ImgArgs im) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) image_write(im, i, p[i]);
}

// ------------------------------------------------------------------ state
struct Mpnn {
  int device = 0;
  hipStream_t stream = nullptr;
  PLayout L;
  DBuf<float> P, G, Am, Av;   // parameters, gradients, Adam moments
  DBuf<bf16> img;             // BF16 images (per weight: transposed then row-major)
  size_t imgT[2 + 4], imgR[2 + 4];  // offsets: enc, m0, u0, m1, u1
  int64_t adamStep = 0;
  // graph
  int64_t N = 0, E = 0;
  DBuf<int32_t> rowOff, recv, send, rev;
  // edges by sender, for a caller's graph in which rev is not the opposite edge throughout
  DBuf<int32_t> sOff, sEdge;
  bool opposite = true;
  DBuf<bf16> X, EF;
  DBuf<float> T;  // targets
  DBuf<int32_t> deg, slotSide, edgeOfSlot;
  // graph from an engine context: the host row of each node in the output (spheres in user-id
  // order); empty for graphs given by the caller
  std::vector<int64_t> outRow;
  DBuf<int64_t> rowDev;  // outRow on the device
  DBuf<float> ordered;   // outputs, and targets as given, in output order
  Ctx* fromCtx = nullptr;  // the engine context of the current graph (storage order of its nodes)
  DBuf<uint32_t> degScan;
  DBuf<uint32_t> nodeUid;  // user id of each node of a graph from an engine context
  uint64_t uidCtx = 0;  // the context (serial), refresh and upload count nodeUid was taken at
  int64_t uidRefresh = -1, uidN = -1;
  uint64_t uidUploads = 0;
  // activations
  DBuf<bf16> h[3], agg[2];
  DBuf<uint64_t> mMask[2], uMask[2];  // relu signs of the messages and of the updates, a bit per feature
  DBuf<float> out, dhA, dhB, S1, S2, part, partLoss;
  DBuf<bf16> dUb, g;          // gradients at the relus of the updates, and of the summed messages
  double *hres = nullptr, *hresDev = nullptr;  // the loss, in pinned host memory
  DBuf<uint8_t> cflag;  // node in contact (else in free flight)
  hipEvent_t done = nullptr;  // orders the network's stream and an engine context's stream
  // the last learned step, which reads out and cflag on the stream of this context: a forward pass that
  // follows it without a new graph from there (which orders the streams) waits for it
  hipEvent_t moved = nullptr;
  const Ctx* movedCtx = nullptr;
  // graphs kept on the device (training sets): inputs, structure and targets
  struct Kept {
    int64_t N = -1, E = 0;
    DBuf<int32_t> rowOff, recv, send, rev, sOff, sEdge;
    bool opposite = true;
    DBuf<bf16> X, EF;
    DBuf<float> T;
    void release() {
      rowOff.release(); recv.release(); send.release(); rev.release(); X.release(); EF.release(); T.release();
      sOff.release(); sEdge.release();
      N = -1;
    }
  };
  std::vector<Kept> kept;
};

// output row of each node: its own index for graphs given by the caller, the rank of its user
// id among the spheres for a graph from an engine context
static void out_rows(Mpnn& s) {
  if (!s.fromCtx || !s.outRow.empty() || s.N == 0) return;
  // the user ids of the nodes as they were when the graph was built (the context may have
  // re-sorted its particles since)
  std::vector<uint32_t> uid((size_t)s.N);
  WDG_HIP(hipMemcpyAsync(uid.data(), s.nodeUid.p, s.N * 4, hipMemcpyDeviceToHost, s.stream));
  WDG_HIP(hipStreamSynchronize(s.stream));
  // the rank of each user id among the nodes', by counting (ids are distinct and below the number of
  // particles)
  std::vector<int64_t> rank((size_t)*std::max_element(uid.begin(), uid.end()) + 1, 0);
  for (const uint32_t u : uid) rank[u] = 1;
  int64_t r = 0;
  for (int64_t& q : rank) {
    const int64_t here = q;
    q = r;
    r += here;
  }
  s.outRow.resize((size_t)s.N);
  for (int64_t t = 0; t < s.N; t++) s.outRow[t] = rank[uid[t]];
  s.rowDev.ensure((size_t)s.N);
  WDG_HIP(hipMemcpyAsync(s.rowDev.p, s.outRow.data(), s.N * sizeof(int64_t), hipMemcpyHostToDevice, s.stream));
  WDG_HIP(hipStreamSynchronize(s.stream));
}
// rows of NOUT floats between node order and output order
__global__ __launch_bounds__(256) void k_rows(int64_t n, const int64_t* __restrict__ row, const float* __restrict__ in,
                                               float* __restrict__ out, int toOutput) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * NOUT) return;
  const int64_t o = row[t / NOUT] * NOUT + t % NOUT;
  if (toOutput) out[o] = in[t];
  else out[t] = in[o];
}

template <class T>
static void copy_buf(DBuf<T>& dst, const DBuf<T>& src, size_t n, hipStream_t st) {
  dst.ensure(std::max<size_t>(n, 1));
  if (n) WDG_HIP(hipMemcpyAsync(dst.p, src.p, n * sizeof(T), hipMemcpyDeviceToDevice, st));
}

static ImgArgs img_args(Mpnn& s) {
  ImgArgs g{};
  const int Ks[5] = {KX, KM, KU, KM, KU};
  const size_t src[5] = {s.L.encW, s.L.mW[0], s.L.uW[0], s.L.mW[1], s.L.uW[1]};
  size_t o = 0;
  for (int q = 0; q < 5; q++) {
    s.imgT[q] = o; o += (size_t)Ks[q] * H;
    s.imgR[q] = o; o += (size_t)Ks[q] * H;
    g.src[q] = (int64_t)src[q]; g.K[q] = Ks[q];
    g.t[q] = (int64_t)s.imgT[q]; g.r[q] = (int64_t)s.imgR[q];
  }
  s.img.ensure(o);
  g.img = s.img.p;
  return g;
}
static void images(Mpnn& s) {
  const ImgArgs g = img_args(s);
  hipLaunchKernelGGL(k_images, dim3(nblocks((int64_t)s.L.total, 256)), dim3(256), 0, s.stream, (int64_t)s.L.total,
                     (const float*)s.P.p, g);
  WDG_LAUNCH_CHECK();
}

// store: also what the backward pass reads (relu signs, summed messages)
static void forward(Mpnn& s, bool store) {
  const int64_t N = s.N, E = s.E;
  const size_t n = (size_t)std::max<int64_t>(N, 1);
  for (auto& b : s.h) b.ensure(n * H);
  s.out.ensure(n * NOUT);
  s.cflag.ensure(n);
  if (store)
    for (int l = 0; l < 2; l++) {
      s.agg[l].ensure(n * H);
      s.uMask[l].ensure(n);
      s.mMask[l].ensure((size_t)std::max<int64_t>(E, 1));
    }
  if (N == 0) return;
  if (s.movedCtx) WDG_HIP(hipStreamWaitEvent(s.stream, s.moved, 0));
  s.movedCtx = nullptr;
  const int64_t nt = (N + 15) / 16;
  hipLaunchKernelGGL(k_enc, dim3(nblocks(nt, 4)), dim3(256), 0, s.stream, N, (const bf16*)s.X.p,
                     (const bf16*)(s.img.p + s.imgT[0]), (const float*)(s.P.p + s.L.encB), s.h[0].p);
  WDG_LAUNCH_CHECK();
  for (int l = 0; l < 2; l++) {
    LayerArgs a{};
    a.N = N;
    a.rowOff = s.rowOff.p; a.recv = s.recv.p; a.send = s.send.p;
    a.h = s.h[l].p; a.ef = s.EF.p; a.x = s.X.p;
    a.Wm = s.img.p + s.imgT[1 + 2 * l]; a.Wu = s.img.p + s.imgT[2 + 2 * l];
    a.bm = s.P.p + s.L.mB[l]; a.bu = s.P.p + s.L.uB[l];
    a.Wd = s.P.p + s.L.decW; a.bd = s.P.p + s.L.decB;
    a.hOut = s.h[l + 1].p; a.agg = s.agg[l].p; a.mMask = s.mMask[l].p; a.uMask = s.uMask[l].p;
    a.out = s.out.p; a.flag = s.cflag.p;
    auto* k = store ? (l ? k_layer<true, true> : k_layer<true, false>) : (l ? k_layer<false, true> : k_layer<false, false>);
    hipLaunchKernelGGL(k, dim3((unsigned)std::min<int64_t>(nblocks(nt, LY_BS / 64), 768)), dim3(LY_BS), 0, s.stream, a);
    WDG_LAUNCH_CHECK();
  }
}

// gradients of the loss (mean squared error against s.T) into s.G; returns the loss
static double backward(Mpnn& s) {
  const int64_t N = s.N, E = s.E;
  const int64_t nt = (N + 15) / 16;
  const size_t n = (size_t)N;
  s.dhA.ensure(n * H); s.dhB.ensure(n * H);
  s.S1.ensure(n * H); s.S2.ensure(n * H);
  s.dUb.ensure(n * H); s.g.ensure(n * H);
  // workgroups of the weight gradients (each leaves one partial): one per compute unit for the
  // products over nodes, more for those over edges, whose partials are small
  const int64_t bN = std::min<int64_t>((N + 31) / 32, 256), bE = std::min<int64_t>((E + 127) / 128, 512),
                bX = std::min<int64_t>((N + 127) / 128, 512), bD = (N + DEC_ROWS - 1) / DEC_ROWS;
  const int64_t oN = 0, oE = oN + 2 * bN * DWN, oX = oE + 2 * bE * DWR, oD = oX + bX * DWR;
  s.part.ensure((size_t)(oD + bD * DECW));
  s.partLoss.ensure((size_t)bD);
  SumArgs sum{};
  auto region = [&](const float* src, int64_t stride, int64_t nblk, int cnt, size_t dst) {
    SumArgs::Region& r = sum.r[sum.n++];
    r = {src, stride, (int)nblk, cnt, s.G.p + dst, sum.blocks};
    sum.blocks += (cnt + 63) / 64;
  };
  hipLaunchKernelGGL(k_loss_dec, dim3((unsigned)bD), dim3(256), 0, s.stream, N, (const float*)s.out.p,
                     (const float*)s.T.p, (const uint8_t*)s.cflag.p, (const bf16*)s.h[2].p,
                     (const float*)(s.P.p + s.L.decW), s.dhA.p, s.part.p + oD, s.partLoss.p);
  WDG_LAUNCH_CHECK();
  region(s.part.p + oD, DECW, bD, DECW, s.L.decW);  // decW then decB are adjacent
  for (int l = 1; l >= 0; l--) {
    hipLaunchKernelGGL(k_bwd_update, dim3(nblocks(nt, 4)), dim3(256), 0, s.stream, N, (const float*)s.dhA.p,
                       (const uint64_t*)s.uMask[l].p, (const bf16*)(s.img.p + s.imgR[2 + 2 * l]), s.dUb.p, s.dhB.p,
                       s.g.p);
    WDG_LAUNCH_CHECK();
    MsgArgs a{};
    a.N = N;
    a.rowOff = s.rowOff.p; a.recv = s.recv.p; a.send = s.send.p; a.rev = s.rev.p;
    a.sOff = s.sOff.p; a.sEdge = s.sEdge.p;
    a.mask = s.mMask[l].p; a.g = s.g.p; a.Wm = s.img.p + s.imgR[1 + 2 * l];
    a.dhp = s.dhB.p; a.dh = s.dhA.p; a.S1 = s.S1.p; a.S2 = s.S2.p;
    hipLaunchKernelGGL(s.opposite ? k_bwd_message<true> : k_bwd_message<false>, dim3(nblocks(nt, 4)), dim3(256), 0,
                       s.stream, a);
    WDG_LAUNCH_CHECK();
    float *pN = s.part.p + oN + l * bN * DWN, *pE = s.part.p + oE + l * bE * DWR;
    hipLaunchKernelGGL(k_dw_node, dim3((unsigned)bN), dim3(256), 0, s.stream, N, (const bf16*)s.h[l].p,
                       (const bf16*)s.agg[l].p, (const bf16*)s.dUb.p, (const float*)s.S1.p, (const float*)s.S2.p, pN);
    WDG_LAUNCH_CHECK();
    if (E > 0) {
      RowArgs r{};
      r.M = E; r.in = s.EF.p; r.recv = s.recv.p; r.mask = s.mMask[l].p; r.g = s.g.p;
      hipLaunchKernelGGL(k_dw_rows<true>, dim3((unsigned)bE), dim3(256), 0, s.stream, r, pE);
      WDG_LAUNCH_CHECK();
    }
    region(pN, DWN, bN, KU * H + H, s.L.uW[l]);  // uW then uB are adjacent
    region(pN + KU * H + H, DWN, bN, 2 * H * H, s.L.mW[l]);
    region(pE, DWR, E > 0 ? bE : 0, NEI * H, s.L.mW[l] + 2 * H * H);
    region(nullptr, 0, 0, (KE - NEI) * H, s.L.mW[l] + (size_t)(2 * H + NEI) * H);
    region(pE + ONE * H, DWR, E > 0 ? bE : 0, H, s.L.mB[l]);
  }
  RowArgs r{};
  r.M = N; r.in = s.X.p; r.dh = s.dhA.p; r.h0 = s.h[0].p;
  hipLaunchKernelGGL(k_dw_rows<false>, dim3((unsigned)bX), dim3(256), 0, s.stream, r, s.part.p + oX);
  WDG_LAUNCH_CHECK();
  region(s.part.p + oX, DWR, bX, NIN * H, s.L.encW);
  region(nullptr, 0, 0, (KX - NIN) * H, s.L.encW + (size_t)NIN * H);
  region(s.part.p + oX + ONE * H, DWR, bX, H, s.L.encB);
  hipLaunchKernelGGL(k_sum_partials, dim3((unsigned)sum.blocks + 1), dim3(1024), 0, s.stream, sum, bD,
                     (const float*)s.partLoss.p, s.hresDev);
  WDG_LAUNCH_CHECK();
  WDG_HIP(hipStreamSynchronize(s.stream));
  return *s.hres / (double)N;
}

// ------------------------------------------------------------------ graph from an engine context
// Edges between spheres closer than cutoff (ri + rj), from the context's slot list (which must
// hold every such pair: its Verlet distance is at least 0.05 (ri + rj) plus the largest
// displacement since its last rebuild); each sphere's edges in its adjacency order.
// Node n = storage index - nW (spheres only).
struct GraphArgs {
  int64_t nW, nSph;
  const uint32_t *adj, *adjOff, *A, *B, *info;
  const double *px, *py, *pz, *vx, *vy, *vz, *rad;
  double cutoff, floorZ;
  int32_t *deg, *rowOff, *recv, *send, *rev, *slotSide;
  int32_t* edgeOfSlot;  // [2 * nslots]
  bf16 *X, *EF;
};
// a row of K inputs as BF16, in 16-byte stores
template <int K>
__device__ __forceinline__ void store_row(bf16* o, const float* f) {
#pragma unroll
  for (int c = 0; c < K; c += 8) {
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = (uint32_t)f2bf(f[c + 2 * q]) | ((uint32_t)f2bf(f[c + 2 * q + 1]) << 16);
    *reinterpret_cast<uint4*>(o + c) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}
__device__ __forceinline__ bool edge_keep(const GraphArgs& g, uint32_t s, uint32_t slot, uint32_t& other) {
  if ((g.info[slot] & CI_TYPE_MASK) != CT_SS) return false;
  const uint32_t a = g.A[slot], b = g.B[slot];
  other = a == s ? b : a;
  const double dx = g.px[other] - g.px[s], dy = g.py[other] - g.py[s], dz = g.pz[other] - g.pz[s];
  const double rs = g.rad[s] + g.rad[other];
  return (dx * dx + dy * dy) + dz * dz < (g.cutoff * rs) * (g.cutoff * rs);
}
__global__ void k_mg_count(GraphArgs g) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.nSph) return;
  const uint32_t s = (uint32_t)(g.nW + t);
  int32_t c = 0;
  uint32_t other;
  for (uint32_t k = g.adjOff[s]; k < g.adjOff[s + 1]; k++) c += edge_keep(g, s, g.adj[k] & ~ADJ_PA, other) ? 1 : 0;
  g.deg[t] = c;
}
// the structure of the graph: each sphere's kept edges in its adjacency order
__global__ void k_mg_fill(GraphArgs g) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.nSph) return;
  const uint32_t s = (uint32_t)(g.nW + t);
  int32_t e = g.rowOff[t];
  uint32_t other;
  for (uint32_t k = g.adjOff[s]; k < g.adjOff[s + 1]; k++) {
    const uint32_t slot = g.adj[k] & ~ADJ_PA;
    if (!edge_keep(g, s, slot, other)) continue;
    g.send[e] = (int32_t)(other - g.nW);
    g.recv[e] = (int32_t)t;
    const int side = g.A[slot] == s ? 0 : 1;
    g.slotSide[e] = (int32_t)(2 * slot + side);
    g.edgeOfSlot[2 * slot + side] = e;
    e++;
  }
}
// inputs of every edge (threads [0, E)) and node (threads [E, E + nSph)), and the opposite
// edge of each edge; one thread per row, so that the double-precision input arithmetic runs
// on full wavefronts
__global__ __launch_bounds__(256) void k_mg_inputs(GraphArgs g, int64_t E) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < E) {
    const int64_t i = g.nW + g.recv[q], j = g.nW + g.send[q];
    g.rev[q] = g.edgeOfSlot[g.slotSide[q] ^ 1];
    float f[EP];
    for (int c = NEI; c < EP; c++) f[c] = 0.f;
    edge_inputs(g.px[i], g.py[i], g.pz[i], g.px[j], g.py[j], g.pz[j], g.vx[i], g.vy[i], g.vz[i], g.vx[j], g.vy[j],
                g.vz[j], g.rad[i], g.rad[j], f);
    store_row<EP>(g.EF + q * EP, f);
  } else if (q < E + g.nSph) {
    const int64_t t = q - E, s = g.nW + t;
    float x[XP];
    for (int c = NIN; c < XP; c++) x[c] = 0.f;
    node_inputs(g.vx[s], g.vy[s], g.vz[s], g.rad[s], g.pz[s] - g.floorZ, x);
    store_row<XP>(g.X + t * XP, x);
  }
}
// coarse step: v += a dT, x += v dT for the spheres; a is the network's output (in units of
// unit) for a sphere in contact, the field's gravity for one in free flight
__global__ void k_mg_advance(int64_t nW, int64_t nSph, const float* __restrict__ a, const uint8_t* __restrict__ inContact,
                             double dT, double unit, double gx, double gy, double gz, double* px, double* py,
                             double* pz, double* vx, double* vy, double* vz, const uint32_t* flags) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nSph) return;
  const int64_t s = nW + t;
  if (!(flags[s] & F_INTEGRATED)) return;
  const bool c = inContact[t] != 0;
  const double ax = c ? unit * a[t * NOUT] : gx, ay = c ? unit * a[t * NOUT + 1] : gy,
               az = c ? unit * a[t * NOUT + 2] : gz;
  const double v[3] = {vx[s] + ax * dT, vy[s] + ay * dT, vz[s] + az * dT};
  vx[s] = v[0]; vy[s] = v[1]; vz[s] = v[2];
  px[s] = px[s] + v[0] * dT; py[s] = py[s] + v[1] * dT; pz[s] = pz[s] + v[2] * dT;
}
// largest squared displacement since the last rebuild, as ordered bits (non-negative doubles)
__global__ __launch_bounds__(256) void k_mg_disp(int64_t n, const double* __restrict__ px, const double* __restrict__ py,
                                                  const double* __restrict__ pz, const double* __restrict__ lx,
                                                  const double* __restrict__ ly, const double* __restrict__ lz,
                                                  unsigned long long* out) {
  __shared__ double wm[4];
  double m = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double dx = px[i] - lx[i], dy = py[i] - ly[i], dz = pz[i] - lz[i];
    m = fmax(m, (dx * dx + dy * dy) + dz * dz);
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  // one device-wide atomic per workgroup
  if (threadIdx.x == 0)
    atomicMax(out, (unsigned long long)__double_as_longlong(fmax(fmax(wm[0], wm[1]), fmax(wm[2], wm[3]))));
}

}  // namespace wdg

using namespace wdg;

struct wdg_mpnn {
  Mpnn s;
};

extern thread_local std::string wdg_mpnn_err;
thread_local std::string wdg_mpnn_err;

template <class F>
static int mguard(F&& f) {
  try {
    f();
    return WDG_OK;
  } catch (const Error& e) {
    wdg_mpnn_err = e.what();
    return e.code;
  } catch (const std::exception& e) {
    wdg_mpnn_err = e.what();
    return WDG_E_STATE;
  }
}

// splitmix64 stream for the initial weights
static uint64_t smix(uint64_t& x) {
  uint64_t z = (x += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

extern "C" {

const char* wdg_mpnn_last_error(void) { return wdg_mpnn_err.c_str(); }

int wdg_mpnn_create(int device, uint64_t seed, wdg_mpnn** out) {
  if (!out) return WDG_E_ARG;
  *out = nullptr;
  auto* m = new wdg_mpnn();
  int rc = mguard([&] {
    Mpnn& s = m->s;
    s.device = device;
    WDG_HIP(hipSetDevice(device));
    WDG_HIP(hipStreamCreate(&s.stream));
    WDG_HIP(hipEventCreateWithFlags(&s.done, hipEventDisableTiming));
    WDG_HIP(hipEventCreateWithFlags(&s.moved, hipEventDisableTiming));
    WDG_HIP(hipHostMalloc((void**)&s.hres, sizeof(double), hipHostMallocDefault));
    WDG_HIP(hipHostGetDevicePointer((void**)&s.hresDev, s.hres, 0));
    const size_t n = s.L.total;
    s.P.ensure(n); s.G.ensure(n); s.Am.ensure(n); s.Av.ensure(n);
    // Glorot-uniform weights over the used input rows, zero biases and padding rows (the
    // decoder below)
    std::vector<float> p(n, 0.f);
    uint64_t st = seed;
    auto fill = [&](size_t off, int K, int Kused, int O) {
      const float lim = std::sqrt(6.f / (float)(Kused + O));
      for (int k = 0; k < K; k++)
        for (int o = 0; o < O; o++) {
          const double u = (double)(smix(st) >> 11) * (1.0 / 9007199254740992.0);
          p[off + (size_t)k * O + o] = k < Kused ? (float)((2 * u - 1) * lim) : 0.f;
        }
    };
    fill(s.L.encW, KX, NIN, H);
    for (int l = 0; l < 2; l++) {
      fill(s.L.mW[l], KM, 2 * H + NEI, H);
      // rows of the unused edge-input columns are zero
      for (int k = 2 * H + NEI; k < KM; k++)
        for (int o = 0; o < H; o++) p[s.L.mW[l] + (size_t)k * H + o] = 0.f;
      fill(s.L.uW[l], KU, KU, H);
    }
    // the decoder starts at zero weights and a bias of free fall: the untrained network is the
    // ballistic coarse step, and training learns the contact accelerations on top of it
    p[s.L.decB + 2] = (float)(-9.81 / MPNN_A0);
    WDG_HIP(hipMemcpy(s.P.p, p.data(), n * 4, hipMemcpyHostToDevice));
    WDG_HIP(hipMemset(s.Am.p, 0, n * 4));
    WDG_HIP(hipMemset(s.Av.p, 0, n * 4));
    WDG_HIP(hipMemset(s.G.p, 0, n * 4));
    images(s);
    WDG_HIP(hipStreamSynchronize(s.stream));
  });
  if (rc) {
    delete m;
    return rc;
  }
  *out = m;
  return WDG_OK;
}

int wdg_mpnn_destroy(wdg_mpnn* m) {
  if (!m) return WDG_OK;
  Mpnn& s = m->s;
  DBuf<float>* fb[] = {&s.P, &s.G, &s.Am, &s.Av, &s.T, &s.out, &s.dhA, &s.dhB, &s.S1, &s.S2, &s.part, &s.partLoss, &s.ordered};
  for (auto* b : fb) b->release();
  DBuf<bf16>* bb[] = {&s.img, &s.X, &s.EF, &s.h[0], &s.h[1], &s.h[2], &s.agg[0], &s.agg[1],
                      &s.dUb, &s.g};
  for (auto* b : bb) b->release();
  for (int l = 0; l < 2; l++) { s.mMask[l].release(); s.uMask[l].release(); }
  s.sOff.release(); s.sEdge.release(); s.rowDev.release();
  s.cflag.release();
  s.rowOff.release(); s.recv.release(); s.send.release(); s.rev.release();
  s.deg.release(); s.slotSide.release(); s.edgeOfSlot.release(); s.degScan.release(); s.nodeUid.release();
  for (auto& k : s.kept) k.release();
  if (s.stream) (void)hipStreamSynchronize(s.stream);
  if (s.done) (void)hipEventDestroy(s.done);
  if (s.moved) (void)hipEventDestroy(s.moved);
  if (s.stream) (void)hipStreamDestroy(s.stream);
  if (s.hres) (void)hipHostFree(s.hres);
  delete m;
  return WDG_OK;
}

int wdg_mpnn_num_params(wdg_mpnn* m, int64_t* n) {
  if (!m || !n) return WDG_E_ARG;
  *n = (int64_t)m->s.L.total;
  return WDG_OK;
}

int wdg_mpnn_get_params(wdg_mpnn* m, float* p, float* g) {
  if (!m) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    WDG_HIP(hipStreamSynchronize(s.stream));
    if (p) WDG_HIP(hipMemcpy(p, s.P.p, s.L.total * 4, hipMemcpyDeviceToHost));
    if (g) WDG_HIP(hipMemcpy(g, s.G.p, s.L.total * 4, hipMemcpyDeviceToHost));
  });
}

int wdg_mpnn_set_params(wdg_mpnn* m, const float* p) {
  if (!m || !p) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    WDG_HIP(hipMemcpy(s.P.p, p, s.L.total * 4, hipMemcpyHostToDevice));
    images(s);
    WDG_HIP(hipStreamSynchronize(s.stream));
  });
}

/* graph from host arrays: x [N x 7] node inputs, CSR by receiver rowOff[N+1], send[E], rev[E],
 * ef [E x 15] edge inputs, targets t [N x 3] (may be NULL) */
int wdg_mpnn_set_graph(wdg_mpnn* m, int64_t N, int64_t E, const float* x, const int32_t* rowOff,
                       const int32_t* send, const int32_t* rev, const float* ef, const float* t) {
  if (!m || N < 0 || E < 0 || (N > 0 && (!x || !rowOff)) || (E > 0 && (!send || !rev || !ef))) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    if (rowOff[0] != 0 || rowOff[N] != E) throw Error(WDG_E_ARG, "rowOff must run from 0 to E");
    std::vector<bf16> X((size_t)std::max<int64_t>(N, 1) * XP, 0), F((size_t)std::max<int64_t>(E, 1) * EP, 0);
    std::vector<int32_t> recv((size_t)std::max<int64_t>(E, 1));
    for (int64_t i = 0; i < N; i++) {
      if (rowOff[i + 1] < rowOff[i]) throw Error(WDG_E_ARG, "rowOff must not decrease");
      for (int c = 0; c < NIN; c++) X[i * XP + c] = f2bf(x[i * NIN + c]);
      for (int32_t e = rowOff[i]; e < rowOff[i + 1]; e++) recv[e] = (int32_t)i;
    }
    for (int64_t e = 0; e < E; e++) {
      if (send[e] < 0 || send[e] >= N || rev[e] < 0 || rev[e] >= E) throw Error(WDG_E_ARG, "edge index out of range");
      for (int c = 0; c < NEI; c++) F[e * EP + c] = f2bf(ef[e * NEI + c]);
    }
    bool opposite = true;
    for (int64_t e = 0; e < E && opposite; e++)
      opposite = rev[rev[e]] == e && send[rev[e]] == recv[e] && recv[rev[e]] == send[e];
    std::vector<int32_t> sOff, sEdge;
    if (!opposite) {
      sOff.assign((size_t)N + 1, 0);
      for (int64_t e = 0; e < E; e++) sOff[send[e] + 1]++;
      for (int64_t i = 0; i < N; i++) sOff[i + 1] += sOff[i];
      std::vector<int32_t> at(sOff.begin(), sOff.end() - 1);
      sEdge.resize((size_t)E);
      for (int64_t e = 0; e < E; e++) sEdge[at[send[e]]++] = (int32_t)e;
    }
    s.opposite = opposite;
    s.N = N;
    s.E = E;
    s.outRow.clear();
    s.fromCtx = nullptr;
    s.X.ensure(X.size()); s.EF.ensure(F.size());
    s.rowOff.ensure((size_t)N + 1); s.recv.ensure(recv.size()); s.send.ensure(recv.size()); s.rev.ensure(recv.size());
    s.T.ensure((size_t)std::max<int64_t>(N, 1) * NOUT);
    WDG_HIP(hipMemcpy(s.X.p, X.data(), X.size() * 2, hipMemcpyHostToDevice));
    WDG_HIP(hipMemcpy(s.EF.p, F.data(), F.size() * 2, hipMemcpyHostToDevice));
    WDG_HIP(hipMemcpy(s.rowOff.p, rowOff, ((size_t)N + 1) * 4, hipMemcpyHostToDevice));
    if (E > 0) {
      WDG_HIP(hipMemcpy(s.recv.p, recv.data(), E * 4, hipMemcpyHostToDevice));
      WDG_HIP(hipMemcpy(s.send.p, send, E * 4, hipMemcpyHostToDevice));
      WDG_HIP(hipMemcpy(s.rev.p, rev, E * 4, hipMemcpyHostToDevice));
    }
    if (!opposite) {
      s.sOff.ensure(sOff.size()); s.sEdge.ensure(sEdge.size());
      WDG_HIP(hipMemcpy(s.sOff.p, sOff.data(), sOff.size() * 4, hipMemcpyHostToDevice));
      WDG_HIP(hipMemcpy(s.sEdge.p, sEdge.data(), sEdge.size() * 4, hipMemcpyHostToDevice));
    }
    if (t) WDG_HIP(hipMemcpy(s.T.p, t, (size_t)N * NOUT * 4, hipMemcpyHostToDevice));
  });
}

/* forward pass; out [N x 3] (may be NULL) */
int wdg_mpnn_forward(wdg_mpnn* m, float* out) {
  if (!m) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    forward(s, false);
    if (out) out_rows(s);
    if (out && s.N > 0) {
      const float* o = s.out.p;
      if (!s.outRow.empty()) {
        s.ordered.ensure((size_t)s.N * NOUT);
        hipLaunchKernelGGL(k_rows, dim3(nblocks(s.N * NOUT, 256)), dim3(256), 0, s.stream, s.N,
                           (const int64_t*)s.rowDev.p, (const float*)s.out.p, s.ordered.p, 1);
        WDG_LAUNCH_CHECK();
        o = s.ordered.p;
      }
      WDG_HIP(hipMemcpyAsync(out, o, (size_t)s.N * NOUT * 4, hipMemcpyDeviceToHost, s.stream));
      WDG_HIP(hipStreamSynchronize(s.stream));
    }
    // without an output the pass stays queued: wdg_mpnn_advance orders the engine's stream after it
    if (!s.fromCtx) WDG_HIP(hipStreamSynchronize(s.stream));
  });
}

/* targets t [N x 3] of the current graph, in its output order */
int wdg_mpnn_set_targets(wdg_mpnn* m, const float* t) {
  if (!m || !t) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    out_rows(s);
    const size_t nt = (size_t)s.N * NOUT;
    s.T.ensure(std::max<size_t>(nt, 1));
    if (!nt) return;
    if (s.outRow.empty()) {
      WDG_HIP(hipMemcpyAsync(s.T.p, t, nt * 4, hipMemcpyHostToDevice, s.stream));
    } else {
      s.ordered.ensure(nt);
      WDG_HIP(hipMemcpyAsync(s.ordered.p, t, nt * 4, hipMemcpyHostToDevice, s.stream));
      hipLaunchKernelGGL(k_rows, dim3(nblocks(s.N * NOUT, 256)), dim3(256), 0, s.stream, s.N,
                         (const int64_t*)s.rowDev.p, (const float*)s.ordered.p, s.T.p, 0);
      WDG_LAUNCH_CHECK();
    }
    WDG_HIP(hipStreamSynchronize(s.stream));
  });
}

/* the current graph: sizes, and (each array may be NULL) its CSR, inputs as stored (BF16
 * widened to float) and the output row of each node */
int wdg_mpnn_get_graph(wdg_mpnn* m, int64_t* N, int64_t* E, int32_t* rowOff, int32_t* send, int32_t* rev, float* x,
                       float* ef, int64_t* nodeRow) {
  if (!m) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    WDG_HIP(hipStreamSynchronize(s.stream));
    if (N) *N = s.N;
    if (E) *E = s.E;
    if (rowOff) WDG_HIP(hipMemcpy(rowOff, s.rowOff.p, ((size_t)s.N + 1) * 4, hipMemcpyDeviceToHost));
    if (send && s.E) WDG_HIP(hipMemcpy(send, s.send.p, (size_t)s.E * 4, hipMemcpyDeviceToHost));
    if (rev && s.E) WDG_HIP(hipMemcpy(rev, s.rev.p, (size_t)s.E * 4, hipMemcpyDeviceToHost));
    auto widen = [&](const DBuf<bf16>& b, int64_t rows, int K, int used, float* out) {
      std::vector<bf16> h((size_t)rows * K);
      if (rows) WDG_HIP(hipMemcpy(h.data(), b.p, h.size() * 2, hipMemcpyDeviceToHost));
      for (int64_t r = 0; r < rows; r++)
        for (int c2 = 0; c2 < used; c2++) out[r * used + c2] = bf2f(h[(size_t)r * K + c2]);
    };
    if (x) widen(s.X, s.N, XP, NIN, x);
    if (ef) widen(s.EF, s.E, EP, NEI, ef);
    if (nodeRow) {
      out_rows(s);
      for (int64_t q = 0; q < s.N; q++) nodeRow[q] = s.outRow.empty() ? q : s.outRow[q];
    }
  });
}

/* keep the current graph (inputs, structure, targets) on the device under slot */
int wdg_mpnn_keep_graph(wdg_mpnn* m, int32_t slot) {
  if (!m || slot < 0) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    if ((size_t)slot >= s.kept.size()) s.kept.resize((size_t)slot + 1);
    Mpnn::Kept& k = s.kept[slot];
    copy_buf(k.rowOff, s.rowOff, (size_t)s.N + 1, s.stream);
    copy_buf(k.recv, s.recv, (size_t)s.E, s.stream);
    copy_buf(k.send, s.send, (size_t)s.E, s.stream);
    copy_buf(k.rev, s.rev, (size_t)s.E, s.stream);
    k.opposite = s.opposite;
    if (!s.opposite) {
      copy_buf(k.sOff, s.sOff, (size_t)s.N + 1, s.stream);
      copy_buf(k.sEdge, s.sEdge, (size_t)s.E, s.stream);
    }
    copy_buf(k.X, s.X, (size_t)s.N * XP, s.stream);
    copy_buf(k.EF, s.EF, (size_t)s.E * EP, s.stream);
    copy_buf(k.T, s.T, (size_t)s.N * NOUT, s.stream);
    k.N = s.N;
    k.E = s.E;
    WDG_HIP(hipStreamSynchronize(s.stream));
  });
}

/* make a kept graph current (outputs in its node order) */
int wdg_mpnn_use_graph(wdg_mpnn* m, int32_t slot) {
  if (!m || slot < 0) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    if ((size_t)slot >= s.kept.size() || s.kept[slot].N < 0) throw Error(WDG_E_ARG, "no graph kept in this slot");
    Mpnn::Kept& k = s.kept[slot];
    s.N = k.N;
    s.E = k.E;
    copy_buf(s.rowOff, k.rowOff, (size_t)s.N + 1, s.stream);
    copy_buf(s.recv, k.recv, (size_t)s.E, s.stream);
    copy_buf(s.send, k.send, (size_t)s.E, s.stream);
    copy_buf(s.rev, k.rev, (size_t)s.E, s.stream);
    s.opposite = k.opposite;
    if (!s.opposite) {
      copy_buf(s.sOff, k.sOff, (size_t)s.N + 1, s.stream);
      copy_buf(s.sEdge, k.sEdge, (size_t)s.E, s.stream);
    }
    copy_buf(s.X, k.X, (size_t)s.N * XP, s.stream);
    copy_buf(s.EF, k.EF, (size_t)s.E * EP, s.stream);
    copy_buf(s.T, k.T, (size_t)s.N * NOUT, s.stream);
    s.outRow.clear();
    s.fromCtx = nullptr;
  });
}

/* forward + backward against the targets of the graph: loss, gradients (wdg_mpnn_get_params) */
int wdg_mpnn_grad(wdg_mpnn* m, double* loss) {
  if (!m) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    if (s.N == 0) throw Error(WDG_E_STATE, "empty graph");
    forward(s, true);
    const double l = backward(s);
    if (loss) *loss = l;
  });
}

/* one Adam step (lr, beta1, beta2, eps) with the current gradients */
int wdg_mpnn_adam(wdg_mpnn* m, double lr, double b1, double b2, double eps) {
  if (!m) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    s.adamStep++;
    const double c1 = 1 - std::pow(b1, (double)s.adamStep), c2 = 1 - std::pow(b2, (double)s.adamStep);
    hipLaunchKernelGGL(k_adam, dim3(nblocks((int64_t)s.L.total, 256)), dim3(256), 0, s.stream, (int64_t)s.L.total,
                       s.P.p, (const float*)s.G.p, s.Am.p, s.Av.p, (float)lr, (float)b1, (float)b2, (float)eps,
                       (float)c1, (float)c2, img_args(s));
    WDG_LAUNCH_CHECK();
    WDG_HIP(hipStreamSynchronize(s.stream));
  });
}

int wdg_mpnn_graph_from_ctx(wdg_mpnn* m, wdg_ctx* ctx, double cutoff, double floorZ, double maxDisp, int force,
                            int64_t* nNodes, int64_t* nEdges, int* rebuilt) {
  if (!m || !ctx || !(cutoff > 0)) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    Ctx& c = ctx_of(ctx);
    if (c.field.periodic) throw Error(WDG_E_ARG, "the learned step supports aperiodic scenes");
    if (c.forcesPending) flush_forces(c);
    const int64_t nSph = c.n - c.nW;
    // the network's kernels of the previous graph (on its own stream) end before the graph changes
    WDG_HIP(hipEventRecord(s.done, s.stream));
    WDG_HIP(hipStreamWaitEvent(c.stream, s.done, 0));
    s.deg.ensure((size_t)nSph + 1);
    s.rowOff.ensure((size_t)nSph + 1);
    GraphArgs g{};
    g.nW = c.nW; g.nSph = nSph;
    g.cutoff = cutoff; g.floorZ = floorZ;
    g.deg = s.deg.p; g.rowOff = s.rowOff.p;
    // the context's arrays as they are now: a refresh permutes the particles into buffers of its
    // own, so these are bound again after every collider call
    auto bind = [&]() {
      Contacts& C = c.con();
      g.adj = C.adj.p; g.adjOff = C.adjOff.p; g.A = C.A.p; g.B = C.B.p; g.info = C.info.p;
      g.px = c.pos[0].p; g.py = c.pos[1].p; g.pz = c.pos[2].p;
      g.vx = c.vel[0].p; g.vy = c.vel[1].p; g.vz = c.vel[2].p; g.rad = c.radius.p;
    };
    // edge counts over the current slot list, and in the same round trip the largest
    // displacement since its refresh (the slot list holds every edge while that stays below maxDisp)
    auto count = [&](bool disp, double& d2) -> int64_t {
      bind();
      unsigned long long* d = reinterpret_cast<unsigned long long*>(c.red.p);
      if (disp) {
        WDG_HIP(hipMemsetAsync(d, 0, 8, c.stream));
        hipLaunchKernelGGL(k_mg_disp, dim3((unsigned)std::min<int64_t>(nblocks(nSph, 256), 256)), dim3(256), 0,
                           c.stream, nSph, (const double*)(c.pos[0].p + c.nW), (const double*)(c.pos[1].p + c.nW),
                           (const double*)(c.pos[2].p + c.nW), (const double*)(c.lastPos[0].p + c.nW),
                           (const double*)(c.lastPos[1].p + c.nW), (const double*)(c.lastPos[2].p + c.nW), d);
        WDG_LAUNCH_CHECK();
      }
      hipLaunchKernelGGL(k_mg_count, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, g);
      WDG_LAUNCH_CHECK();
      scan_exclusive(c, reinterpret_cast<const uint32_t*>(s.deg.p), reinterpret_cast<uint32_t*>(s.rowOff.p), nSph,
                     reinterpret_cast<uint32_t*>(s.rowOff.p + nSph));
      uint32_t hE = 0;
      unsigned long long hb = 0;
      WDG_HIP(hipMemcpyAsync(&hE, s.rowOff.p + nSph, 4, hipMemcpyDeviceToHost, c.stream));
      if (disp) WDG_HIP(hipMemcpyAsync(&hb, d, 8, hipMemcpyDeviceToHost, c.stream));
      WDG_HIP(hipStreamSynchronize(c.stream));
      memcpy(&d2, &hb, 8);
      return (int64_t)hE;
    };
    if (std::isnan(c.verletDist)) throw Error(WDG_E_STATE, "run the collider once before building graphs");
    // the slot list holds every pair closer than r1 + r2 + 2 verletDist at its refresh, so it
    // holds every edge while no sphere has moved farther than verletDist - need since then
    const double need = 0.5 * (cutoff - 1.) * 2. * c.rmax;
    const double allow = c.verletDist - need;
    bool rb = force != 0 || !c.boundsValid || allow < 0;
    int64_t E = 0;
    if (!rb && nSph > 0) {
      double d2 = 0.;
      E = count(true, d2);
      rb = d2 > allow * allow;
    }
    if (rb) {
      // rebuild with room for maxDisp of motion before the next one
      c.verletDist = std::max(c.verletDist, need + std::max(maxDisp, 0.));
      wdg_collide_params p{c.verletDist, 1};
      collide(c, &p);
      double d2;
      if (nSph > 0) E = count(false, d2);
    }
    if (rebuilt) *rebuilt = rb ? 1 : 0;
    bind();
    Contacts& C = c.con();
    s.edgeOfSlot.ensure((size_t)std::max<int64_t>(2 * C.n, 2));
    s.recv.ensure((size_t)std::max<int64_t>(E, 1)); s.send.ensure((size_t)std::max<int64_t>(E, 1));
    s.rev.ensure((size_t)std::max<int64_t>(E, 1)); s.slotSide.ensure((size_t)std::max<int64_t>(E, 1));
    s.opposite = true;
    s.X.ensure((size_t)std::max<int64_t>(nSph, 1) * XP);
    s.EF.ensure((size_t)std::max<int64_t>(E, 1) * EP);
    s.T.ensure((size_t)std::max<int64_t>(nSph, 1) * NOUT);
    g.recv = s.recv.p; g.send = s.send.p; g.rev = s.rev.p; g.slotSide = s.slotSide.p; g.edgeOfSlot = s.edgeOfSlot.p;
    g.X = s.X.p; g.EF = s.EF.p;
    if (nSph > 0) {
      hipLaunchKernelGGL(k_mg_fill, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, g);
      WDG_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_mg_inputs, dim3(nblocks(E + nSph, 256)), dim3(256), 0, c.stream, g, E);
      WDG_LAUNCH_CHECK();
    }
    // the user ids of the nodes change only with a refresh (or an upload) of the context
    if (s.uidCtx != c.serial || s.uidRefresh != c.nRefresh || s.uidUploads != c.uploads || s.uidN != nSph) {
      s.nodeUid.ensure((size_t)std::max<int64_t>(nSph, 1));
      if (nSph > 0)
        WDG_HIP(hipMemcpyAsync(s.nodeUid.p, c.uid.p + c.nW, nSph * 4, hipMemcpyDeviceToDevice, c.stream));
      s.uidCtx = c.serial;
      s.uidRefresh = c.nRefresh;
      s.uidUploads = c.uploads;
      s.uidN = nSph;
    }
    // the network's next kernels (its own stream) start after the graph is built, and so after a learned
    // step queued before it on the same stream
    WDG_HIP(hipEventRecord(s.done, c.stream));
    WDG_HIP(hipStreamWaitEvent(s.stream, s.done, 0));
    if (s.movedCtx == &c) s.movedCtx = nullptr;
    // output rows (spheres in user-id order) are found when an output is asked for
    s.outRow.clear();
    s.fromCtx = &c;
    s.N = nSph;
    s.E = E;
    if (nNodes) *nNodes = nSph;
    if (nEdges) *nEdges = E;
  });
}

int wdg_mpnn_advance(wdg_mpnn* m, wdg_ctx* ctx, double dT) {
  if (!m || !ctx) return WDG_E_ARG;
  return mguard([&] {
    Mpnn& s = m->s;
    Ctx& c = ctx_of(ctx);
    const int64_t nSph = c.n - c.nW;
    if (s.N != nSph) throw Error(WDG_E_STATE, "the network's graph is not of this context");
    if (s.fromCtx != &c) throw Error(WDG_E_STATE, "the network's graph was not built from this context");
    // the forward pass (network stream) ends before the engine's stream moves the spheres
    WDG_HIP(hipEventRecord(s.done, s.stream));
    WDG_HIP(hipStreamWaitEvent(c.stream, s.done, 0));
    if (c.forcesPending) flush_forces(c);
    // the contact history describes the state before the coarse step, which the network
    // replaces: the next contact loop starts it afresh
    clear_history(c);
    if (nSph > 0) {
      hipLaunchKernelGGL(k_mg_advance, dim3(nblocks(nSph, 256)), dim3(256), 0, c.stream, c.nW, nSph,
                         (const float*)s.out.p, (const uint8_t*)s.cflag.p, dT, MPNN_A0, c.field.gravity[0],
                         c.field.gravity[1], c.field.gravity[2], c.pos[0].p, c.pos[1].p, c.pos[2].p, c.vel[0].p, c.vel[1].p,
                         c.vel[2].p, (const uint32_t*)c.flags.p);
      WDG_LAUNCH_CHECK();
      WDG_HIP(hipEventRecord(s.moved, c.stream));
      s.movedCtx = &c;
    }
    c.dirtyKnown = false;
  });
}

}  // extern "C"
