// crm_mlp.hip -- the pointwise network that stands in for the bulk microphysics, trained and
// evaluated on the matrix cores: BF16 operands, FP32 accumulation (v_mfma_f32_16x16x16_bf16 and
// 16x16x32), FP32 master weights and Adam moments.
//
// A training step is two launches: k_train takes a tile of rows per workgroup through the forward
// and backward passes and leaves its share of the loss and of every gradient in memory; k_reduce
// adds the shares in a fixed order, applies Adam and writes the new weights in the orders in
// which the kernels read them.  As one GEMM launch per layer and direction, with column sums,
// clears, Adam and two repacking kernels (21 launches, gradients by atomics), a step of 16,384
// rows took 292 us.
//
// The 9 inputs are padded to 16 and the 6 outputs to 16, with zero weights in the padding; rows
// past the batch have zero inputs and zero output gradients, so they contribute nothing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/crm_mlp.h"
#include "crm_index.hpp"
#include "crm_mlp_dev.hpp"

namespace crm_mlp_ns {

// Offsets (bf16 elements) of the weights in the fragment order of the fused inference (F).
constexpr int F_L1 = 0;                    // layer 1: 8 output blocks x 64 lanes x 4 (K = 16)
constexpr int F_L2 = F_L1 + 8 * 64 * 4;    // layer 2: (8 output x 4 K blocks) x 64 lanes x 8
constexpr int F_L3 = F_L2 + 32 * 64 * 8;   // layer 3: as layer 2
constexpr int F_L4 = F_L3 + 32 * 64 * 8;   // layer 4: 4 K blocks x 64 lanes x 8 (16 outputs)
constexpr int F_SIZE = F_L4 + 4 * 64 * 8;
constexpr int B_SIZE = 3 * NH + NP;        // biases b1 b2 b3 b4

// The training orders: blocks of 64 lanes x 4, an A operand of v_mfma_f32_16x16x16_bf16 each.
// Forward (rows = outputs of the layer), block ob * (K blocks) + kb; backward (rows = inputs),
// block ib * (output blocks) + nb, for layers 4, 3 and 2.
constexpr int FRAG = 64 * 4;
constexpr int T_L1 = 0, T_L2 = T_L1 + 8 * FRAG, T_L3 = T_L2 + 64 * FRAG, T_L4 = T_L3 + 64 * FRAG;
constexpr int T_B4 = T_L4 + 8 * FRAG, T_B3 = T_B4 + 8 * FRAG, T_B2 = T_B3 + 64 * FRAG;
constexpr int T_SIZE = T_B2 + 64 * FRAG;

typedef unsigned u4 __attribute__((ext_vector_type(4)));  // 8 bf16, element 0 in the low half
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bh2 __attribute__((ext_vector_type(2)));
typedef short sh2 __attribute__((ext_vector_type(2)));

// The copies of the parameters that the kernels read (device memory).
struct Weights {
  bf16 *F, *T;                // weights in inference and training order
  float *b1, *b2, *b3, *b4;   // biases (b4 padded to 16)
};

// Packed parameter idx of value w into every copy.  Element (k, n) of a layer is lane
// n % 16 + 16 (k % 16 / 4), slot k % 4 of its forward block; in a 32-wide K block of the inference
// order the slots of a lane are k % 4 and 4 + k % 4 (its two 16-wide halves).
__device__ __forceinline__ void place(const Weights& o, int idx, float w) {
  auto layer = [&](int off, int nout, int f, int t, int tb, bool wide) {
    const int e = idx - off, k = e / nout, n = e % nout;
    const bf16 h = to_bf16(w);
    const int ob = n / 16, kb = k / 16, lane = n % 16 + 16 * (k % 16 / 4), i = k % 4;
    const int kbs = wide ? 8 : 1;
    o.T[t + (ob * kbs + kb) * FRAG + lane * 4 + i] = h;
    o.F[f + (wide ? ((ob * 4 + k / 32) * 64 + lane) * 8 + 4 * (kb & 1) + i : (ob * 64 + lane) * 4 + i)] = h;
    if (tb >= 0) {
      const int nbs = nout == NH ? 8 : 1;
      o.T[tb + (kb * nbs + ob) * FRAG + (k % 16 + 16 * (n % 16 / 4)) * 4 + n % 4] = h;
    }
  };
  if (idx < OFF_B1) {
    layer(OFF_W1, NH, F_L1, T_L1, -1, false);
  } else if (idx < OFF_W2) {
    o.b1[idx - OFF_B1] = w;
  } else if (idx < OFF_B2) {
    layer(OFF_W2, NH, F_L2, T_L2, T_B2, true);
  } else if (idx < OFF_W3) {
    o.b2[idx - OFF_B2] = w;
  } else if (idx < OFF_B3) {
    layer(OFF_W3, NH, F_L3, T_L3, T_B3, true);
  } else if (idx < OFF_W4) {
    o.b3[idx - OFF_B3] = w;
  } else if (idx < OFF_B4) {
    layer(OFF_W4, CRM_MLP_NOUT, F_L4, T_L4, T_B4, true);
  } else {
    o.b4[idx - OFF_B4] = w;
  }
}
// (one thread per parameter; the padding of every copy stays zero from its allocation)
__global__ void k_place(const float* p, Weights o) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < CRM_MLP_NPARAM) place(o, idx, p[idx]);
}

// ---- training --------------------------------------------------------------------------------
constexpr int TROWS = 64;     // rows of a tile, 16 per wave
constexpr int TLD = TROWS + 4;  // row stride of a [feature][row] tile in LDS: 8-byte reads of 16 features spread over the banks
constexpr int PSTRIDE = (CRM_MLP_NPARAM + 1 + 63) / 64 * 64;  // a workgroup's shares: gradients, squared error

__device__ __forceinline__ f4 mfma16(s4 a, s4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
__device__ __forceinline__ s4 pack4(const float (&v)[4]) {
  s4 r;
#pragma unroll
  for (int j = 0; j < 4; j++) r[j] = (short)to_bf16(v[j]);
  return r;
}

// acc[ob] = sum over kb of W block (ob, kb) times in[kb]; the K blocks in order, so that each sum
// has one order, and the output blocks inside, so that eight products are in flight.  The weights
// of the whole layer are read before its first product (128 registers of the 512 a wave has
// here): left to itself the compiler reads eight blocks at a time and waits out the L2's latency
// eight times a layer (91 us a launch at 16,384 rows).
template <int OB, int KB>
__device__ __forceinline__ void blocks(const bf16* W, const s4 (&in)[KB], f4 (&acc)[OB], int lane) {
  s4 w[KB][OB];
#pragma unroll
  for (int kb = 0; kb < KB; kb++)
#pragma unroll
    for (int ob = 0; ob < OB; ob++) w[kb][ob] = *(const s4*)&W[(ob * KB + kb) * FRAG + lane * 4];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ob = 0; ob < OB; ob++) acc[ob] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < KB; kb++)
#pragma unroll
    for (int ob = 0; ob < OB; ob++) acc[ob] = mfma16(w[kb][ob], in[kb], acc[ob]);
}

// Loss and gradients of the rows of this workgroup's tiles (64 at a time) into part[blockIdx.x].
// The layers run transposed, as in the fused inference below: the weights are the A operand and
// the rows the B operand, so one layer's D fragment -- lane (r, q) holds features 4q..4q+3 of row
// r -- is the next one's B fragment, forward and backward, and a wave takes its 16 rows through
// both passes in registers.  The weight gradients contract over the rows, which lie across the
// lanes: every wave leaves its activations and pre-activation gradients in LDS as [feature][row]
// tiles, and the four waves share the 144 16 x 16 gradient blocks, whose accumulators stay in
// registers over the workgroup's tiles.  109 KB of LDS: one workgroup per CU, and a grid of at
// most one per CU.  Bound by latency: 424 MFMAs per wave and tile are 3 us at the matrix rate; the
// shares (141 KB per workgroup) are 36 MB at 256 workgroups, written here and read by k_reduce.
__global__ void __launch_bounds__(256) k_train(const float* X, const float* T, int n, Weights w, const float* norm,
                                               float* part) {
  __shared__ __attribute__((aligned(16))) bf16 sX[KP][TLD], sH[3][NH][TLD], sY[NP][TLD], sD[3][NH][TLD];
  __shared__ float red[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, r = lane & 15, q = lane >> 4;
  float mean[4], rs[4], osc[4], b4[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    mean[j] = norm[NORM_MEAN + 4 * q + j];
    rs[j] = norm[NORM_RSCALE + 4 * q + j];
    osc[j] = norm[NORM_OSCALE + 4 * q + j];
    b4[j] = w.b4[4 * q + j];
  }
  f4 g1[2], g2[2][8], g3[2][8], g4[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    g1[i] = g4[i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int o = 0; o < 8; o++) g2[i][o] = g3[i][o] = f4{0.f, 0.f, 0.f, 0.f};
  }
  float gb[3] = {0.f, 0.f, 0.f}, gb4 = 0.f, e2 = 0.f;
  const int row = 16 * wave + r;
  for (Strided tile = tiles_of(n, TROWS, blockIdx.x, gridDim.x); tile.more(); tile.next()) {
    const long m = tile.at * TROWS + row;
    const bool have = m < n;
    // an offset the compiler cannot see through, so that the weight reads stay inside the loop
    // (hoisted out of it, the network would be held in registers and spill)
    int fo = 0;
    asm volatile("" : "+v"(fo));
    const bf16* W = w.T + fo;
    s4 x[1], h[3][8], d[8], y[1];
    f4 acc[8];
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int c = 4 * q + j;
      v[j] = have && c < CRM_MLP_NIN ? (X[m * CRM_MLP_NIN + c] - mean[j]) * rs[j] : 0.f;
    }
    x[0] = pack4(v);
#pragma unroll
    for (int j = 0; j < 4; j++) sX[4 * q + j][row] = (bf16)x[0][j];
    // bias and ReLU of a layer's sums, to registers and LDS
    auto activate = [&](const float* bias, int l) {
#pragma unroll
      for (int ob = 0; ob < 8; ob++) {
        const f4 b = *(const f4*)&bias[16 * ob + 4 * q];
        float a[4];
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = fmaxf(acc[ob][j] + b[j], 0.f);
        h[l][ob] = pack4(a);
#pragma unroll
        for (int j = 0; j < 4; j++) sH[l][16 * ob + 4 * q + j][row] = (bf16)h[l][ob][j];
      }
    };
    blocks<8, 1>(W + T_L1, x, acc, lane);
    activate(w.b1, 0);
    blocks<8, 8>(W + T_L2, h[0], acc, lane);
    activate(w.b2, 1);
    blocks<8, 8>(W + T_L3, h[1], acc, lane);
    activate(w.b3, 2);
    f4 out[1];
    blocks<1, 8>(W + T_L4, h[2], out, lane);
    // loss of the normalised outputs and its gradient 2 (y - t') / (6 n)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int c = 4 * q + j;
      v[j] = 0.f;
      if (have && c < CRM_MLP_NOUT) {
        const float e = (out[0][j] + b4[j]) - T[m * CRM_MLP_NOUT + c] / osc[j];
        e2 += e * e;
        v[j] = 2.f * e / (6.f * (float)n);
      }
    }
    y[0] = pack4(v);
#pragma unroll
    for (int j = 0; j < 4; j++) sY[4 * q + j][row] = (bf16)y[0][j];
    // the ReLU mask of a layer's back-propagated sums, to registers and LDS
    auto mask = [&](int l) {
#pragma unroll
      for (int ib = 0; ib < 8; ib++) {
        float a[4];
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = from_bf16((bf16)h[l][ib][j]) > 0.f ? acc[ib][j] : 0.f;
        d[ib] = pack4(a);
#pragma unroll
        for (int j = 0; j < 4; j++) sD[l][16 * ib + 4 * q + j][row] = (bf16)d[ib][j];
      }
    };
    blocks<8, 1>(W + T_B4, y, acc, lane);
    mask(2);
    blocks<8, 8>(W + T_B3, d, acc, lane);
    mask(1);
    blocks<8, 8>(W + T_B2, d, acc, lane);
    mask(0);
    __syncthreads();
    // weight gradients: this wave's input blocks 2 wave and 2 wave + 1 (layer 1: output blocks)
#pragma unroll
    for (int ks = 0; ks < TROWS / 16; ks++) {
      const int c = 16 * ks + 4 * q;
      auto at = [&](const bf16* p) { return *(const s4*)p; };
      const s4 xa = at(&sX[r][c]), ya = at(&sY[r][c]);
      s4 a1[2], a2[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int f = 16 * (2 * wave + i) + r;
        a1[i] = at(&sH[0][f][c]);
        a2[i] = at(&sH[1][f][c]);
        g1[i] = mfma16(xa, at(&sD[0][f][c]), g1[i]);
        g4[i] = mfma16(at(&sH[2][f][c]), ya, g4[i]);
      }
#pragma unroll
      for (int o = 0; o < 8; o++) {
        const s4 d2 = at(&sD[1][16 * o + r][c]), d3 = at(&sD[2][16 * o + r][c]);
#pragma unroll
        for (int i = 0; i < 2; i++) {
          g2[i][o] = mfma16(a1[i], d2, g2[i][o]);
          g3[i][o] = mfma16(a2[i], d3, g3[i][o]);
        }
      }
    }
    // bias gradients: sums over the rows
    if (t < NH) {
#pragma unroll
      for (int l = 0; l < 3; l++)
        for (int c = 0; c < TROWS; c += 4) {
          const s4 a = *(const s4*)&sD[l][t][c];
#pragma unroll
          for (int j = 0; j < 4; j++) gb[l] += from_bf16((bf16)a[j]);
        }
      if (t < NP)
        for (int c = 0; c < TROWS; c++) gb4 += from_bf16(sY[t][c]);
    }
    __syncthreads();
  }
  float* o = part + (size_t)blockIdx.x * PSTRIDE;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int b = 2 * wave + i;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int k = 4 * q + j, f = 16 * b + k;
      if (k < CRM_MLP_NIN) o[OFF_W1 + k * NH + 16 * b + r] = g1[i][j];
      if (r < CRM_MLP_NOUT) o[OFF_W4 + f * CRM_MLP_NOUT + r] = g4[i][j];
#pragma unroll
      for (int ob = 0; ob < 8; ob++) {
        o[OFF_W2 + f * NH + 16 * ob + r] = g2[i][ob][j];
        o[OFF_W3 + f * NH + 16 * ob + r] = g3[i][ob][j];
      }
    }
  }
  if (t < NH) {
    o[OFF_B1 + t] = gb[0];
    o[OFF_B2 + t] = gb[1];
    o[OFF_B3 + t] = gb[2];
    if (t < CRM_MLP_NOUT) o[OFF_B4 + t] = gb4;
  }
  for (int k = 32; k >= 1; k >>= 1) e2 += __shfl_xor(e2, k, 64);
  if (lane == 0) red[wave] = e2;
  __syncthreads();
  if (t == 0) o[CRM_MLP_NPARAM] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Sums of the np workgroups' shares, 64 parameters per workgroup and a quarter of the shares per
// wave.  ADAM: the update of the parameters and of every copy of the weights; otherwise the
// gradient to g.  The loss goes to `loss` (host memory the device can write).
template <bool ADAM>
__global__ void __launch_bounds__(256) k_reduce(const float* part, int np, int n, float* g, float* p, float* m, float* v,
                                                float lr, float c1, float c2, Weights w, float* loss) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, idx = blockIdx.x * 64 + lane;
  float s = 0.f;
#pragma unroll 8
  for (int k = wave; k < np; k += 4) s += part[(size_t)k * PSTRIDE + idx];
  red[wave][lane] = s;
  __syncthreads();
  if (wave > 0 || idx > CRM_MLP_NPARAM) return;
  const float gi = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
  if (idx == CRM_MLP_NPARAM) {
    *loss = gi / (6.f * (float)n);
    return;
  }
  if constexpr (ADAM) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float mi = b1 * m[idx] + (1.f - b1) * gi;
    float vi = b2 * v[idx] + (1.f - b2) * gi * gi;
    m[idx] = mi;
    v[idx] = vi;
    const float pn = p[idx] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[idx] = pn;
    place(w, idx, pn);
  } else {
    g[idx] = gi;
  }
}

// Fused inference, the whole network in registers.  The layers run transposed, H^T = W^T A^T:
// the weights are the A operand (rows = output features) and the points the B operand
// (columns), so the D fragment of one layer -- lane (r, q) holds features 4q..4q+3 of point r
// -- is the B fragment of the next one, and activations never leave the registers.  The
// 128-wide layers use v_mfma_f32_16x16x32_bf16, whose 32 K slots a lane fills with eight
// values; the K order inside a 32-feature block is a free choice as long as A and B agree,
// and we take slot (q, i) = feature 4q + i (i < 4) or 16 + 4q + (i - 4) (i >= 4), which is
// exactly the two D fragments of output blocks 2kb and 2kb + 1.  The weights are stored in that
// fragment order (place: each lane's operand is 8 or 16 contiguous bytes) and copied into LDS by every workgroup; a wave owns 64 points (4 blocks of 16) per
// tile and reads each weight fragment once for the 4 blocks.  The grid is persistent: two
// workgroups per CU (the weights take 74 KiB of LDS) loop over the tiles.
__device__ __forceinline__ f4 mfma32(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// relu of two values rounded to BF16 (nearest, ties to even: v_cvt_pk_bf16_f32), packed.  The
// rounding keeps the sign, so relu after it equals relu before it, and on BF16 bit patterns
// relu is the signed 16-bit max with 0 (negative values and -0 have the sign bit set).
__device__ __forceinline__ unsigned relu_pk(float a, float b) {
  const bh2 h = __builtin_convertvector((f2){a, b}, bh2);
  return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(sh2, h), (sh2){0, 0}));
}

// D fragment of output block ob -> its half of the next layer's B fragment of block ob / 2.
__device__ __forceinline__ void relu_store(const f4& acc, u4& dst, int half) {
  dst[2 * half] = relu_pk(acc[0], acc[1]);
  dst[2 * half + 1] = relu_pk(acc[2], acc[3]);
}

// A 128 -> 128 hidden layer for the wave's four point blocks.  The epilogue of output block
// ob - 1 is written after the products of block ob, so it runs under them.
__device__ __forceinline__ void hidden128(const bf16* fr, const float* bias, const u4 (&in)[4][4], u4 (&out)[4][4],
                                          int lane) {
  const int q = lane >> 4;
  f4 acc[2][4];
#pragma unroll
  for (int ob = 0; ob < 8; ob++) {
    const f4 b = *(const f4*)&bias[16 * ob + 4 * q];
    f4(&a)[4] = acc[ob & 1];
#pragma unroll
    for (int pb = 0; pb < 4; pb++) a[pb] = b;
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      const u4 w = *(const u4*)&fr[((ob * 4 + kb) * 64 + lane) * 8];
#pragma unroll
      for (int pb = 0; pb < 4; pb++) a[pb] = mfma32(w, in[pb][kb], a[pb]);
    }
    if (ob > 0) {
#pragma unroll
      for (int pb = 0; pb < 4; pb++) relu_store(acc[(ob - 1) & 1][pb], out[pb][(ob - 1) >> 1], (ob - 1) & 1);
    }
  }
#pragma unroll
  for (int pb = 0; pb < 4; pb++) relu_store(acc[1][pb], out[pb][3], 1);
}

// X[n][9] raw inputs.  MODE 0 (the CRM): Y[n][8] = the 6 de-normalised rates, then 1 where
// the inputs lie inside the training envelope (else 0), then 0.  MODE 1: Y[n][6], the rates.
template <int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_infer(const float* X, long n, MlpView v,
                                                                                       float* Y) {
  __shared__ __attribute__((aligned(16))) bf16 fl[F_SIZE];
  __shared__ __attribute__((aligned(16))) float bl[B_SIZE];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int i = t; i < F_SIZE / 8; i += 256) ((uint4*)fl)[i] = ((const uint4*)v.F)[i];
  for (int i = t; i < NH; i += 256) {
    bl[i] = v.b1[i];
    bl[NH + i] = v.b2[i];
    bl[2 * NH + i] = v.b3[i];
  }
  if (t < NP) bl[3 * NH + t] = v.b4[t];
  __syncthreads();

  const int r = lane & 15, q = lane >> 4;
  const float* nm = v.norm;
  float mean[4], rs[4], lo[4], hi[4], osc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int f = 4 * q + i;
    const bool ok = f < CRM_MLP_NIN;
    mean[i] = ok ? nm[NORM_MEAN + f] : 0.f;
    rs[i] = ok ? nm[NORM_RSCALE + f] : 1.f;
    lo[i] = ok ? nm[NORM_LO + f] : -INFINITY;
    hi[i] = ok ? nm[NORM_HI + f] : INFINITY;
    osc[i] = f < CRM_MLP_NOUT ? nm[NORM_OSCALE + f] : 0.f;
  }
  const long ntiles = (n + 63) / 64, stride = (long)gridDim.x * 4;
  // raw inputs of the tile: every lane loads its 16 slots unconditionally from clamped (valid)
  // addresses, so the loads issue together; slots past the 9 features or past n are masked
  float xr[4][4];
  auto load_tile = [&](long tile) {
#pragma unroll
    for (int pb = 0; pb < 4; pb++) {
      const long pt = min(tile * 64 + 16 * pb + r, n - 1);
#pragma unroll
      for (int i = 0; i < 4; i++) xr[pb][i] = X[pt * CRM_MLP_NIN + min(4 * q + i, CRM_MLP_NIN - 1)];
    }
  };
  long tile = (long)blockIdx.x * 4 + wave;
  if (tile < ntiles) load_tile(tile);
  for (; tile < ntiles; tile += stride) {
    const long p0 = tile * 64;
    // an offset the compiler cannot see through, so the weight reads stay inside the loop
    // (hoisted out of it, the whole network would be held in registers and spill)
    int fo = 0;
    asm volatile("" : "+v"(fo));
    const bf16* fw = fl + fo;
    s4 x0[4];
    int in[4];
#pragma unroll
    for (int pb = 0; pb < 4; pb++) {
      const bool live = p0 + 16 * pb + r < n;
      float xn[4];
      in[pb] = 1;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool have = 4 * q + i < CRM_MLP_NIN && live;
        const float xv = xr[pb][i];
        if (have) in[pb] &= (xv >= lo[i] && xv <= hi[i]);
        xn[i] = have ? (xv - mean[i]) * rs[i] : 0.f;
      }
      const bh2 h0 = __builtin_convertvector((f2){xn[0], xn[1]}, bh2);
      const bh2 h1 = __builtin_convertvector((f2){xn[2], xn[3]}, bh2);
      x0[pb] = __builtin_bit_cast(s4, (u2){__builtin_bit_cast(unsigned, h0), __builtin_bit_cast(unsigned, h1)});
    }
    // the next tile's inputs load under this tile's products
    if (tile + stride < ntiles) load_tile(tile + stride);
    u4 ha[4][4], hb[4][4];
    // layer 1 (K = 16: the 9 inputs, padded)
#pragma unroll
    for (int ob = 0; ob < 8; ob++) {
      const f4 b = *(const f4*)&bl[16 * ob + 4 * q];
      const s4 w = *(const s4*)&fw[F_L1 + (ob * 64 + lane) * 4];
#pragma unroll
      for (int pb = 0; pb < 4; pb++)
        relu_store(__builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, x0[pb], b, 0, 0, 0), ha[pb][ob >> 1], ob & 1);
    }
    hidden128(fw + F_L2, bl + NH, ha, hb, lane);
    hidden128(fw + F_L3, bl + 2 * NH, hb, ha, lane);
    // layer 4: outputs 4q..4q+3 of point r (q < 2 hold the 6 rates and padding)
    const f4 b4 = *(const f4*)&bl[3 * NH + 4 * q];
    f4 acc[4] = {b4, b4, b4, b4};
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      const u4 w = *(const u4*)&fw[F_L4 + (kb * 64 + lane) * 8];
#pragma unroll
      for (int pb = 0; pb < 4; pb++) acc[pb] = mfma32(w, ha[pb][kb], acc[pb]);
    }
#pragma unroll
    for (int pb = 0; pb < 4; pb++) {
      const long pt = p0 + 16 * pb + r;
      if constexpr (MODE == 0) {
        // the point's envelope flag: all four lane quarters agree
        int a = in[pb] & __shfl_xor(in[pb], 16);
        a &= __shfl_xor(a, 32);
        if (q < 2 && pt < n) {
          f4 o;
          o[0] = acc[pb][0] * osc[0];
          o[1] = acc[pb][1] * osc[1];
          o[2] = q == 0 ? acc[pb][2] * osc[2] : (a ? 1.f : 0.f);
          o[3] = q == 0 ? acc[pb][3] * osc[3] : 0.f;
          *(f4*)&Y[pt * 8 + 4 * q] = o;
        }
      } else {
        if (q < 2 && pt < n) {
#pragma unroll
          for (int j = 0; j < 4; j++)
            if (4 * q + j < CRM_MLP_NOUT) Y[pt * CRM_MLP_NOUT + 4 * q + j] = acc[pb][j] * osc[j];
        }
      }
    }
  }
}

}  // namespace crm_mlp_ns

using namespace crm_mlp_ns;

struct crm_mlp {
  int device = 0;
  hipStream_t s = nullptr;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // packed FP32
  Weights w{};
  int ncu = 0;            // compute units of the device (persistent grids)
  float* norm = nullptr;  // [NORM_SIZE]
  float host_norm[NORM_SIZE] = {};
  float* loss = nullptr;  // pinned host memory, written by k_reduce
  int cap = 0;            // workgroups' shares in part
  float* part = nullptr;
  long step = 0;
};

namespace {
// Persistent grid of the fused inference: two workgroups per CU, fewer for small batches.
template <int MODE>
void launch_infer(hipStream_t s, const crm_mlp* m, const float* X, long n, float* Y) {
  const long tiles = (n + 63) / 64;
  const long grid = std::min<long>((tiles + 3) / 4, 2L * m->ncu);
  if (n > 0) k_infer<MODE><<<dim3((unsigned)grid), dim3(256), 0, s>>>(X, n, mlp_view(m), Y);
}

#define MLPCHECK(x)                                   \
  do {                                                \
    if ((x) != hipSuccess) return CRM_ERR_DEVICE;     \
  } while (0)

// the forward and backward pass of n rows of X and T (device), and the sums of its shares
template <bool ADAM>
int step(crm_mlp* m, const float* X, const float* T, int n, float lr, float c1, float c2) {
  const int np = (int)std::min<long>(((long)n + TROWS - 1) / TROWS, m->ncu);
  if (np > m->cap) {
    if (m->part) (void)hipFree(m->part);
    m->part = nullptr;
    m->cap = 0;
    MLPCHECK(hipMalloc(&m->part, (size_t)np * PSTRIDE * sizeof(float)));
    m->cap = np;
  }
  k_train<<<dim3((unsigned)np), dim3(256), 0, m->s>>>(X, T, n, m->w, m->norm, m->part);
  k_reduce<ADAM><<<dim3(PSTRIDE / 64), dim3(256), 0, m->s>>>(m->part, np, n, m->g, m->p, m->m, m->v, lr, c1, c2, m->w,
                                                            m->loss);
  MLPCHECK(hipGetLastError());
  return CRM_OK;
}

void place_params(crm_mlp* m) {
  k_place<<<dim3((CRM_MLP_NPARAM + 255) / 256), dim3(256), 0, m->s>>>(m->p, m->w);
}
}  // namespace

extern "C" {

int crm_mlp_create(crm_mlp** out, int device) {
  if (!out) return CRM_ERR_ARG;
  *out = nullptr;
  auto* m = new crm_mlp();
  m->device = device;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&m->s) != hipSuccess) {
    delete m;
    return CRM_ERR_DEVICE;
  }
  bool ok = hipMalloc(&m->p, CRM_MLP_NPARAM * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->g, CRM_MLP_NPARAM * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->m, CRM_MLP_NPARAM * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->v, CRM_MLP_NPARAM * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->w.F, F_SIZE * sizeof(bf16)) == hipSuccess &&
            hipMalloc(&m->w.T, T_SIZE * sizeof(bf16)) == hipSuccess &&
            hipMalloc(&m->w.b1, NH * sizeof(float)) == hipSuccess && hipMalloc(&m->w.b2, NH * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->w.b3, NH * sizeof(float)) == hipSuccess && hipMalloc(&m->w.b4, NP * sizeof(float)) == hipSuccess &&
            hipMalloc(&m->norm, NORM_SIZE * sizeof(float)) == hipSuccess &&
            hipHostMalloc(&m->loss, sizeof(float), hipHostMallocDefault) == hipSuccess;
  if (!ok) {
    crm_mlp_destroy(m);
    return CRM_ERR_NOMEM;
  }
  if (hipDeviceGetAttribute(&m->ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || m->ncu < 1) {
    crm_mlp_destroy(m);
    return CRM_ERR_DEVICE;
  }
  (void)hipMemset(m->p, 0, CRM_MLP_NPARAM * sizeof(float));
  (void)hipMemset(m->w.F, 0, F_SIZE * sizeof(bf16));
  (void)hipMemset(m->w.T, 0, T_SIZE * sizeof(bf16));
  (void)hipMemset(m->w.b4, 0, NP * sizeof(float));
  (void)hipMemset(m->m, 0, CRM_MLP_NPARAM * sizeof(float));
  (void)hipMemset(m->v, 0, CRM_MLP_NPARAM * sizeof(float));
  for (int c = 0; c < 16; c++) {
    m->host_norm[NORM_SCALE + c] = 1.f;
    m->host_norm[NORM_RSCALE + c] = 1.f;
    m->host_norm[NORM_OSCALE + c] = 1.f;
    m->host_norm[NORM_LO + c] = -INFINITY;
    m->host_norm[NORM_HI + c] = INFINITY;
  }
  (void)hipMemcpy(m->norm, m->host_norm, sizeof(m->host_norm), hipMemcpyHostToDevice);
  place_params(m);
  (void)hipStreamSynchronize(m->s);
  *out = m;
  return CRM_OK;
}

int crm_mlp_destroy(crm_mlp* m) {
  if (!m) return CRM_ERR_ARG;
  (void)hipSetDevice(m->device);
  void* bufs[] = {m->p, m->g, m->m, m->v, m->w.F, m->w.T, m->w.b1, m->w.b2, m->w.b3, m->w.b4, m->norm, m->part};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (m->loss) (void)hipHostFree(m->loss);
  if (m->s) (void)hipStreamDestroy(m->s);
  delete m;
  return CRM_OK;
}

int crm_mlp_set_params(crm_mlp* m, const float* params) {
  if (!m || !params) return CRM_ERR_ARG;
  MLPCHECK(hipMemcpyAsync(m->p, params, CRM_MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice, m->s));
  MLPCHECK(hipMemsetAsync(m->m, 0, CRM_MLP_NPARAM * sizeof(float), m->s));
  MLPCHECK(hipMemsetAsync(m->v, 0, CRM_MLP_NPARAM * sizeof(float), m->s));
  m->step = 0;
  place_params(m);
  MLPCHECK(hipStreamSynchronize(m->s));
  return CRM_OK;
}

int crm_mlp_get_params(const crm_mlp* m, float* params) {
  if (!m || !params) return CRM_ERR_ARG;
  MLPCHECK(hipMemcpyAsync(params, m->p, CRM_MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, m->s));
  MLPCHECK(hipStreamSynchronize(m->s));
  return CRM_OK;
}

int crm_mlp_set_norm(crm_mlp* m, const float* mean, const float* scale, const float* oscale, const float* lo,
                     const float* hi) {
  if (!m) return CRM_ERR_ARG;
  for (int c = 0; c < CRM_MLP_NIN; c++) {
    if (mean) m->host_norm[NORM_MEAN + c] = mean[c];
    if (scale) {
      if (!(scale[c] > 0.f)) return CRM_ERR_ARG;
      m->host_norm[NORM_SCALE + c] = scale[c];
      m->host_norm[NORM_RSCALE + c] = 1.f / scale[c];
    }
    if (lo) m->host_norm[NORM_LO + c] = lo[c];
    if (hi) m->host_norm[NORM_HI + c] = hi[c];
  }
  for (int c = 0; c < CRM_MLP_NOUT; c++)
    if (oscale) {
      if (!(oscale[c] > 0.f)) return CRM_ERR_ARG;
      m->host_norm[NORM_OSCALE + c] = oscale[c];
    }
  MLPCHECK(hipMemcpyAsync(m->norm, m->host_norm, sizeof(m->host_norm), hipMemcpyHostToDevice, m->s));
  MLPCHECK(hipStreamSynchronize(m->s));
  return CRM_OK;
}

int crm_mlp_forward(crm_mlp* m, const float* X, int n, float* Y) {
  if (!m || !X || !Y || n < 0) return CRM_ERR_ARG;
  launch_infer<1>(m->s, m, X, n, Y);
  MLPCHECK(hipGetLastError());
  MLPCHECK(hipStreamSynchronize(m->s));
  return CRM_OK;
}

int crm_mlp_grad(crm_mlp* m, const float* X, const float* T, int n, float* grad, float* loss) {
  if (!m || !X || !T || n < 1) return CRM_ERR_ARG;
  int rc = step<false>(m, X, T, n, 0.f, 1.f, 1.f);
  if (rc) return rc;
  if (grad) MLPCHECK(hipMemcpyAsync(grad, m->g, CRM_MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, m->s));
  MLPCHECK(hipStreamSynchronize(m->s));
  if (loss) *loss = *m->loss;
  return CRM_OK;
}

int crm_mlp_train_step(crm_mlp* m, const float* X, const float* T, int n, float lr, float* loss) {
  if (!m || !X || !T || n < 1 || !(lr > 0.f)) return CRM_ERR_ARG;
  const float k = (float)(m->step + 1), c1 = 1.f - std::pow(0.9f, k), c2 = 1.f - std::pow(0.999f, k);
  int rc = step<true>(m, X, T, n, lr, c1, c2);
  if (rc) return rc;
  m->step++;
  MLPCHECK(hipStreamSynchronize(m->s));
  if (loss) *loss = *m->loss;
  return CRM_OK;
}

}  // extern "C"

// for the CRM engines (crm_driver.hpp): the device-side view of a network
namespace crm_mlp_ns {
MlpView mlp_view(const crm_mlp* m) {
  MlpView v;
  v.F = m->w.F;
  v.b1 = m->w.b1;
  v.b2 = m->w.b2;
  v.b3 = m->w.b3;
  v.b4 = m->w.b4;
  v.norm = m->norm;
  return v;
}
int mlp_device(const crm_mlp* m) { return m->device; }
void mlp_infer(hipStream_t s, const crm_mlp* m, const float* X, long n, float* Y) { launch_infer<0>(s, m, X, n, Y); }
}  // namespace crm_mlp_ns
