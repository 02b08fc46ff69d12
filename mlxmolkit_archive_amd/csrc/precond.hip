// Learned per-atom initial inverse Hessian for the BFGS minimizer, gfx950.
//
// A small MLP maps per-atom features (MMFF type one-hot, degree, ring flags, summed bond
// and angle force constants; MLP_IN = 104) through two hidden layers of width 64 (ReLU)
// to 6 numbers, the Cholesky factor L of a 3x3 SPD block:
//   L = [[sp(o0), 0, 0], [o1, sp(o2), 0], [o3, o4, sp(o5)]],  sp(v) = softplus(v) + 1e-3,
//   block = L L^T.
// Weights are row-major fp32 [out][in] (W1 64x104, W2 64x64, W3 6x64) plus biases.
//
// Kernels:
//   k_mlp_infer_bf16  inference on MFMA (v_mfma_f32_32x32x8_bf16, FP32 accumulation): one
//                     wave per 32 atoms; activations are re-laid out through LDS between
//                     layers; writes the 9 floats of each block
//   k_mlp_train       training: forward, backward and weight gradients of a tile of atoms in LDS,
//                     layers on FP32 MFMA, weight gradients on FP64 MFMA
//   k_mlp_train_sum   the workgroups' partial gradients summed in a fixed order (deterministic)
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "mmff_hip.h"

namespace {

constexpr int MLP_IN = 104;
constexpr int MLP_KPAD = 112;  // MLP_IN rounded up to the MFMA k-step of 8
constexpr int MLP_H = 64;
constexpr int MLP_OUT = 6;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float softplus_eps(float v) {
  return (v > 20.f ? v : log1pf(expf(v))) + 1e-3f;
}
__device__ __forceinline__ float sigmoidf(float v) { return 1.f / (1.f + expf(-v)); }

// 3x3 block L L^T from the 6 outputs
__device__ __forceinline__ void chol_block(const float* o, float* blk) {
  const float l00 = softplus_eps(o[0]), l10 = o[1], l11 = softplus_eps(o[2]);
  const float l20 = o[3], l21 = o[4], l22 = softplus_eps(o[5]);
  const float b00 = l00 * l00, b01 = l00 * l10, b02 = l00 * l20;
  const float b11 = l10 * l10 + l11 * l11, b12 = l10 * l20 + l11 * l21;
  const float b22 = l20 * l20 + l21 * l21 + l22 * l22;
  blk[0] = b00; blk[1] = b01; blk[2] = b02;
  blk[3] = b01; blk[4] = b11; blk[5] = b12;
  blk[6] = b02; blk[7] = b12; blk[8] = b22;
}

struct MlpW {
  const float *w1, *b1, *w2, *b2, *w3, *b3;
};

// ------------------------------------------------------------------------------------
// Inference on MFMA, bound by reading the features (416 bytes per atom). A wave takes 32 atoms
// at a time; the next tile's features (13 x 16 bytes per lane) are loaded into registers while
// this one is computed. The products are formed transposed (A = weights, B = activations), so a
// lane ends up with four consecutive units of one atom per register quad: one packed conversion
// per two values and one 8-byte LDS write per four, where units in lanes took a rounding sequence
// and a 2-byte write each. The first layer's weights stay in registers, the others in LDS. Row
// strides of 58 and 34 words put the 32 rows of an 8-byte operand read in 32 different bank pairs.
// v_mfma_f32_32x32x8_bf16 operand layout (wave64): lane l supplies A[l%32][4*(l/32)+0..3]
// and B[4*(l/32)+0..3][l%32]; it receives D[8*(r/4) + 4*(l/32) + r%4][l%32], r = 0..15.
// The weights and the first tile are loaded all at once before anything waits: 32 atoms take 5.9 us
// from one launch to the next, 12.6 us with the weights laid out a word at a time.
// 500,003 atoms, launches back to back: 51 us (4.4 TB/s of features and blocks; a copy reaches 4.8),
// 62 us with the weights a word at a time. One call: 326 us with 4-byte feature loads and units in
// lanes, 134 us with 16-byte loads and units in lanes, 69 us with the weights a word at a time, 50 us now.
constexpr int INF_WAVES = 4;
constexpr int INF_LDX = 116, INF_LDH = 68;  // row strides (bf16) of features and hidden units
constexpr int INF_WAVE_SHORTS = 32 * INF_LDX + 32 * INF_LDH + 2 * 32 * 9;  // features, hidden, blocks (f32)
constexpr int INF_W23_SHORTS = 64 * INF_LDH + 32 * INF_LDH + 2 * 160;      // W2, W3, biases (f32)
// W1 is staged where the waves' tiles go afterwards
static_assert(64 * INF_LDX <= INF_WAVES * INF_WAVE_SHORTS, "staging area");
constexpr size_t INF_LDS = 2 * (size_t)(INF_W23_SHORTS + INF_WAVES * INF_WAVE_SHORTS);
constexpr int INF_GRID = 512;  // two workgroups per CU (registers), each taking tiles in turn
static_assert(INF_LDS <= 65536, "no raised LDS limit needed");
constexpr int INF_VEC = 32 * MLP_IN / 4 / 64;  // 16-byte feature loads per lane and tile (13)

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// two floats as bf16, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  const bf2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// D[unit][atom] (32 x 32) = W (32 rows x 8 KS) times the transpose of the activations (rows of act)
template <int KS, class WOP>
__device__ __forceinline__ f32x16 mfma_tile(const WOP& w, const short* act, int act_ld, int lane) {
  f32x16 acc = {0.f};
  const short* p = act + (lane & 31) * act_ld + (lane >> 5) * 4;
#pragma unroll
  for (int k = 0; k < KS; k++)
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(w(k), *(const bf16x4*)(p + 8 * k), acc, 0, 0, 0);
  return acc;
}

// bias + ReLU, then store the tile as bf16 activations at units n0.. of the atoms' rows of hid
__device__ __forceinline__ void store_relu(const f32x16& acc, const float* bias, int n0, short* hid, int lane) {
  short* row = hid + (lane & 31) * INF_LDH + n0 + 4 * (lane >> 5);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float4 b = *(const float4*)(bias + n0 + 8 * q + 4 * (lane >> 5));
    uint2 v;
    v.x = pack_bf16(fmaxf(acc[4 * q] + b.x, 0.f), fmaxf(acc[4 * q + 1] + b.y, 0.f));
    v.y = pack_bf16(fmaxf(acc[4 * q + 2] + b.z, 0.f), fmaxf(acc[4 * q + 3] + b.w, 0.f));
    *(uint2*)(row + 8 * q) = v;
  }
}

// VEC: the features are 16-byte aligned (rows are 26 x 16 bytes), so a tile is read in 16-byte
// words; otherwise in 4-byte ones
template <bool VEC>
__global__ void __launch_bounds__(64 * INF_WAVES, 2)
    k_mlp_infer_bf16(MlpW W, const float* __restrict__ feat, int n_atoms, float* __restrict__ blocks) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c32 = lane & 31;
  short* s2 = (short*)smem;                  // W2 [64][INF_LDH]
  short* s3 = s2 + 64 * INF_LDH;             // W3 [32][INF_LDH], rows 6..31 zero
  float* bias = (float*)(s3 + 32 * INF_LDH); // b1, b2, b3 padded to 32
  short* tiles = (short*)(bias + 160);
  const int n_tiles = (n_atoms + 31) / 32, step = gridDim.x * INF_WAVES;
  int t = blockIdx.x * INF_WAVES + wv;
  float4 f[INF_VEC];
  // Lanes past the last atom read the last word again: a row only reaches its own atom's outputs,
  // and those past n_atoms are not stored. (A load under a condition of its own is waited for.)
  auto fetch = [&](int tile) {
    const int last = min(32, n_atoms - tile * 32) * (MLP_IN / 4) - 1;
    const float4* src = (const float4*)feat + (size_t)tile * (32 * MLP_IN / 4);
#pragma unroll
    for (int v = 0; v < INF_VEC; v++) {
      const int i = min(v * 64 + lane, last);
      if (VEC) {
        f[v] = src[i];
      } else {
        const float* p = (const float*)src + 4 * i;
        f[v] = make_float4(p[0], p[1], p[2], p[3]);
      }
    }
  };
  if (t < n_tiles) fetch(t);  // in flight while the weights are laid out
  bf16x4 w1a[MLP_KPAD / 8], w1b[MLP_KPAD / 8];
  {
    short* s1 = tiles;
    // all loads first: one latency instead of one per few words (the launch's fixed cost)
    constexpr int N1 = 64 * MLP_IN / 4, V1 = (N1 + 64 * INF_WAVES - 1) / (64 * INF_WAVES), V2 = 64 * 64 / 4 / (64 * INF_WAVES);
    auto word = [](const float* w, int i) { return make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]); };
    auto put = [](short* d, float4 v) { *(uint2*)d = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)); };
    float4 u1[V1], u2[V2];
#pragma unroll
    for (int v = 0; v < V1; v++) u1[v] = word(W.w1, min(v * 64 * INF_WAVES + tid, N1 - 1));
#pragma unroll
    for (int v = 0; v < V2; v++) u2[v] = word(W.w2, v * 64 * INF_WAVES + tid);
    const float4 u3 = word(W.w3, min(tid, MLP_OUT * 16 - 1));
#pragma unroll
    for (int v = 0; v < V1; v++) {
      const int i = min(v * 64 * INF_WAVES + tid, N1 - 1), o = i / (MLP_IN / 4);
      put(s1 + o * INF_LDX + 4 * (i - o * (MLP_IN / 4)), u1[v]);
    }
    if (tid < 128) put(s1 + (tid >> 1) * INF_LDX + MLP_IN + 4 * (tid & 1), make_float4(0.f, 0.f, 0.f, 0.f));
#pragma unroll
    for (int v = 0; v < V2; v++) {
      const int i = v * 64 * INF_WAVES + tid;
      put(s2 + (i >> 4) * INF_LDH + 4 * (i & 15), u2[v]);
    }
    for (int i = tid; i < 32 * 16; i += 64 * INF_WAVES)
      put(s3 + (i >> 4) * INF_LDH + 4 * (i & 15), i < MLP_OUT * 16 ? u3 : make_float4(0.f, 0.f, 0.f, 0.f));
    if (tid < 160) bias[tid] = tid < 64 ? W.b1[tid] : tid < 128 ? W.b2[tid - 64] : tid < 128 + MLP_OUT ? W.b3[tid - 128] : 0.f;
    __syncthreads();
    const short* p = s1 + c32 * INF_LDX + (lane >> 5) * 4;
#pragma unroll
    for (int k = 0; k < MLP_KPAD / 8; k++) {
      w1a[k] = *(const bf16x4*)(p + 8 * k);
      w1b[k] = *(const bf16x4*)(p + 32 * INF_LDX + 8 * k);
    }
    __syncthreads();  // the tiles below reuse the LDS
  }
  auto op1a = [&](int k) { return w1a[k]; };
  auto op1b = [&](int k) { return w1b[k]; };
  const short* p2 = s2 + c32 * INF_LDH + (lane >> 5) * 4;
  auto op2a = [&](int k) { return *(const bf16x4*)(p2 + 8 * k); };
  auto op2b = [&](int k) { return *(const bf16x4*)(p2 + 32 * INF_LDH + 8 * k); };
  const short* p3 = s3 + c32 * INF_LDH + (lane >> 5) * 4;
  auto op3 = [&](int k) { return *(const bf16x4*)(p3 + 8 * k); };
  short* act = tiles + wv * INF_WAVE_SHORTS;  // bf16 [32][INF_LDX]
  short* hid = act + 32 * INF_LDX;            // bf16 [32][INF_LDH]
  float* blk = (float*)(hid + 32 * INF_LDH);  // outputs [32][8], then blocks [32][9]
  for (int i = lane; i < 32 * (MLP_KPAD - MLP_IN); i += 64)
    act[(i >> 3) * INF_LDX + MLP_IN + (i & 7)] = 0;  // the padding columns of the first layer
  for (; t < n_tiles; t += step) {
    const int a0 = t * 32;
    // features of 32 atoms -> bf16 tile
#pragma unroll
    for (int v = 0; v < INF_VEC; v++) {
      const int i = v * 64 + lane, r = i / (MLP_IN / 4), k = 4 * (i - r * (MLP_IN / 4));
      uint2 b;
      b.x = pack_bf16(f[v].x, f[v].y);
      b.y = pack_bf16(f[v].z, f[v].w);
      *(uint2*)(act + r * INF_LDX + k) = b;
    }
    if (t + step < n_tiles) fetch(t + step);
    wave_lds_fence();
    // layer 1: [32 x 112] x W1^T -> [32 x 64]
    f32x16 h0 = mfma_tile<MLP_KPAD / 8>(op1a, act, INF_LDX, lane), h1 = mfma_tile<MLP_KPAD / 8>(op1b, act, INF_LDX, lane);
    store_relu(h0, bias, 0, hid, lane);
    store_relu(h1, bias, 32, hid, lane);
    wave_lds_fence();
    // layer 2: [32 x 64] x W2^T -> [32 x 64], over the same rows once both products have read them
    h0 = mfma_tile<8>(op2a, hid, INF_LDH, lane);
    h1 = mfma_tile<8>(op2b, hid, INF_LDH, lane);
    wave_lds_fence();
    store_relu(h0, bias + 64, 0, hid, lane);
    store_relu(h1, bias + 64, 32, hid, lane);
    wave_lds_fence();
    // layer 3: [32 x 64] x W3^T -> [32 x 32], units 0..5 used: 0-3 in the lower half's first
    // quad, 4 and 5 in the upper half's
    const f32x16 o = mfma_tile<8>(op3, hid, INF_LDH, lane);
    if (lane < 32)
      *(float4*)(blk + c32 * 8) = make_float4(o[0] + bias[128], o[1] + bias[129], o[2] + bias[130], o[3] + bias[131]);
    else
      *(float2*)(blk + c32 * 8 + 4) = make_float2(o[0] + bias[132], o[1] + bias[133]);
    wave_lds_fence();
    float b[9];
    if (lane < 32) chol_block(blk + lane * 8, b);
    wave_lds_fence();
    if (lane < 32) {
#pragma unroll
      for (int q = 0; q < 9; q++) blk[lane * 9 + q] = b[q];
    }
    wave_lds_fence();
    const int n_out = 9 * min(32, n_atoms - a0);
    float* dst = blocks + (size_t)a0 * 9;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      const int i = v * 64 + lane;
      if (i < n_out) dst[i] = blk[i];
    }
    wave_lds_fence();
  }
}

// ------------------------------------------------------------------------------------
// Training: loss, blocks and the gradient of sum_a w_a ||P_a - T_a||^2.
//
// k_mlp_train takes tiles of 64 atoms through the network forwards and backwards and into the
// weight gradients, all in one workgroup's LDS (149 KB, one workgroup of 8 waves per CU), so no
// activation or delta goes through memory. The layers run on FP32 MFMA (16x16x4, a wave takes 16
// atoms and half the outputs of a layer); the weight gradients delta^T x input run on FP64 MFMA
// (16x16x4), which multiplies FP32 values exactly and sums over the atoms in FP64, six 16x16
// tiles per wave held in registers over all tiles of the workgroup. Each workgroup leaves one
// FP64 partial sum per parameter and k_mlp_train_sum adds them in a fixed order, so the gradient
// is deterministic. Row strides are 4 x odd words, so the operand reads (16 rows x 4 columns)
// touch 64 different banks.
//
// Measured at 8,192 atoms: 32 us a step, launches and allocations included (38 us with the weights
// and features brought into LDS a word at a time: most workgroups take one tile, so that latency is
// theirs in full), against 2.90 ms with
// one lane per atom in the layers and one lane per parameter in the weight gradients (2.53 ms
// of it a serial walk over the atoms on 44 of 256 CUs). 64-atom tiles put the 8,192-atom
// mini-batch on 128 CUs; 32-atom ones would use all 256 but double the partial sums (11 MB).
constexpr int NP_W1 = 64 * MLP_IN, NP_B1 = 64, NP_W2 = 64 * 64, NP_B2 = 64, NP_W3 = MLP_OUT * 64, NP_B3 = MLP_OUT;
constexpr int OFF_B1 = NP_W1, OFF_W2 = OFF_B1 + NP_B1, OFF_B2 = OFF_W2 + NP_W2, OFF_W3 = OFF_B2 + NP_B2,
              OFF_B3 = OFF_W3 + NP_W3;
constexpr int MLP_NPARAM = OFF_B3 + NP_B3;

constexpr int TR_ATOMS = 64, TR_NT = 512, TR_MAX_GRID = 256;
constexpr int LDX = 108, LDH = 68, LDO = 12;  // row strides of features, hidden units, outputs
constexpr int TR_LDS_FLOATS = TR_ATOMS * (LDX + 4 * LDH + 2 * LDO) + 64 * LDX + 64 * LDH + 16 * LDH;
constexpr size_t TR_LDS = (size_t)TR_LDS_FLOATS * 4;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

inline int train_tiles(int n_atoms) { return n_atoms / TR_ATOMS + (n_atoms % TR_ATOMS > 0); }
// Workgroups of the training kernel: at most one per CU's worth, with tiles shared out evenly.
inline int train_grid(int n_atoms) {
  const int tiles = train_tiles(n_atoms);
  const int rounds = (tiles + TR_MAX_GRID - 1) / TR_MAX_GRID;
  return rounds > 0 ? (tiles + rounds - 1) / rounds : 0;
}
// Their partial sums, with room to start them at a 256-byte boundary
inline size_t train_ws_bytes(int workgroups) { return (size_t)workgroups * MLP_NPARAM * sizeof(double) + 256; }

// One 16 x 16 tile of A (rows of `a`, stride lda) times the transpose of B (rows of `b`, stride
// ldb) over K columns, added to acc. v_mfma_f32_16x16x4: lane l supplies A[l%16][l/16] and
// B[l/16][l%16] of each 4-column step and holds D[4 (l/16) + r][l%16], r = 0..3.
template <int K, bool RELU>
__device__ __forceinline__ f32x4 mfma16(const float* a, int lda, const float* b, int ldb, f32x4 acc, int lane) {
  const float* pa = a + (lane & 15) * lda + (lane >> 4);
  const float* pb = b + (lane & 15) * ldb + (lane >> 4);
#pragma unroll 8
  for (int k = 0; k < K; k += 4) {
    const float av = RELU ? fmaxf(pa[k], 0.f) : pa[k];
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, pb[k], acc, 0, 0, 0);
  }
  return acc;
}

// The same with B given by its rows: D += A (16 x K) * b (K x 16 at column offset folded into b).
template <int K>
__device__ __forceinline__ f32x4 mfma16_nn(const float* a, int lda, const float* b, int ldb, f32x4 acc, int lane) {
  const float* pa = a + (lane & 15) * lda + (lane >> 4);
  const float* pb = b + (lane >> 4) * ldb + (lane & 15);
#pragma unroll 8
  for (int k = 0; k < K; k += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[k], pb[k * ldb], acc, 0, 0, 0);
  return acc;
}

__global__ void __launch_bounds__(TR_NT) k_mlp_train(MlpW W, const float* __restrict__ feat, int n_atoms,
                                                     const float* __restrict__ target,
                                                     const float* __restrict__ weight, float* __restrict__ blocks,
                                                     float* __restrict__ loss_out, double* __restrict__ part) {
  extern __shared__ __align__(16) float sm[];
  float* xs = sm;                       // features [64][LDX]
  float* z1 = xs + TR_ATOMS * LDX;      // pre-activations [64][LDH]
  float* z2 = z1 + TR_ATOMS * LDH;
  float* d1 = z2 + TR_ATOMS * LDH;      // deltas [64][LDH]
  float* d2 = d1 + TR_ATOMS * LDH;
  float* os = d2 + TR_ATOMS * LDH;      // outputs [64][LDO]
  float* dos = os + TR_ATOMS * LDO;     // output deltas [64][LDO], columns 6, 7 zero
  float* w1 = dos + TR_ATOMS * LDO;     // weights, rows as in memory
  float* w2 = w1 + 64 * LDX;
  float* w3 = w2 + 64 * LDH;            // rows 6..15 zero
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int tiles = (n_atoms + TR_ATOMS - 1) / TR_ATOMS;
  // All of a thread's weight and feature words are loaded before the first is stored: one latency
  // instead of one per few words. Features past the last atom read its last word again and become
  // zeros on the way into LDS.
  auto word = [](const float* p, int i) { return make_float4(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]); };
  constexpr int NX = TR_ATOMS * MLP_IN / 4, VX = (NX + TR_NT - 1) / TR_NT;  // words of a tile's features (and of W1)
  static_assert(TR_ATOMS == 64 && NP_W1 == TR_ATOMS * MLP_IN && NP_W2 == 8 * TR_NT, "word counts");
  float4 fx[VX];
  auto fetch = [&](int t) {
    const int last = min(TR_ATOMS, n_atoms - t * TR_ATOMS) * (MLP_IN / 4) - 1;
    const float* src = feat + (size_t)t * TR_ATOMS * MLP_IN;
#pragma unroll
    for (int v = 0; v < VX; v++) fx[v] = word(src, min(v * TR_NT + tid, last));
  };
  {
    float4 u1[VX], u2[2], u3;
#pragma unroll
    for (int v = 0; v < VX; v++) u1[v] = word(W.w1, min(v * TR_NT + tid, NX - 1));
#pragma unroll
    for (int v = 0; v < 2; v++) u2[v] = word(W.w2, v * TR_NT + tid);
    u3 = word(W.w3, min(tid, NP_W3 / 4 - 1));
    if (blockIdx.x < tiles) fetch(blockIdx.x);
#pragma unroll
    for (int v = 0; v < VX; v++) {
      const int i = min(v * TR_NT + tid, NX - 1), o = i / (MLP_IN / 4);
      *(float4*)(w1 + o * LDX + 4 * (i - o * (MLP_IN / 4))) = u1[v];
    }
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const int i = v * TR_NT + tid;
      *(float4*)(w2 + (i >> 4) * LDH + 4 * (i & 15)) = u2[v];
    }
    if (tid < 16 * 16) *(float4*)(w3 + (tid >> 4) * LDH + 4 * (tid & 15)) = tid < NP_W3 / 4 ? u3 : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const int rt = wv & 3, half = wv >> 2;      // 16-atom row tile and column half of a layer
  const int row = rt * 16, c16 = lane & 15, q = lane >> 4;
  f64x4 g[6];                                 // weight-gradient tiles of this wave
#pragma unroll
  for (int i = 0; i < 6; i++) g[i] = f64x4{0.0, 0.0, 0.0, 0.0};
  double gb = 0.0;                            // bias gradient of thread tid (b1, b2, b3)
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    const int a0 = t * TR_ATOMS, na = min(TR_ATOMS, n_atoms - a0);
#pragma unroll
    for (int v = 0; v < VX; v++) {
      const int i = v * TR_NT + tid, r = i / (MLP_IN / 4);
      if (i < NX)
        *(float4*)(xs + r * LDX + 4 * (i - r * (MLP_IN / 4))) = r < na ? fx[v] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (t + gridDim.x < tiles) fetch(t + gridDim.x);
    __syncthreads();
    // forward; a layer's output tile has its biases as the start of the sums
    auto layer_out = [&](f32x4 acc, float* z, int ld, int n0) {
#pragma unroll
      for (int r = 0; r < 4; r++) z[(row + 4 * q + r) * ld + n0 + c16] = acc[r];
    };
    auto biased = [&](const float* bias, int n0) {
      const float v = bias[n0 + c16];
      return f32x4{v, v, v, v};
    };
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int n0 = 32 * half + 16 * h;
      layer_out(mfma16<MLP_IN, false>(xs + row * LDX, LDX, w1 + n0 * LDX, LDX, biased(W.b1, n0), lane), z1, LDH, n0);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int n0 = 32 * half + 16 * h;
      layer_out(mfma16<64, true>(z1 + row * LDH, LDH, w2 + n0 * LDH, LDH, biased(W.b2, n0), lane), z2, LDH, n0);
    }
    __syncthreads();
    if (half == 0) {
      const float v = c16 < MLP_OUT ? W.b3[c16] : 0.f;
      const f32x4 o = mfma16<64, true>(z2 + row * LDH, LDH, w3, LDH, f32x4{v, v, v, v}, lane);
      if (c16 < MLP_OUT) layer_out(o, os, LDO, 0);
    }
    __syncthreads();
    // per atom: block, loss and the delta of the six outputs
    if (tid < TR_ATOMS) {
      float dout[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      const int a = a0 + tid;
      if (tid < na) {
        float o[MLP_OUT], blk[9], G[9];
        for (int j = 0; j < MLP_OUT; j++) o[j] = os[tid * LDO + j];
        chol_block(o, blk);
        const float w = weight ? weight[a] : 1.f;
        float l = 0.f;
        for (int k = 0; k < 9; k++) {
          const float d = blk[k] - target[(size_t)a * 9 + k];
          l = fmaf(d, d, l);
          G[k] = 2.f * w * d;  // dLoss/dP
          if (blocks) blocks[(size_t)a * 9 + k] = blk[k];
        }
        if (loss_out) loss_out[a] = l;
        // P = L L^T: dLoss/dL = (G + G^T) L
        const float L[9] = {softplus_eps(o[0]), 0.f, 0.f, o[1], softplus_eps(o[2]), 0.f, o[3], o[4], softplus_eps(o[5])};
        float dL[9];
        for (int i = 0; i < 3; i++)
          for (int j = 0; j < 3; j++) {
            float v = 0.f;
            for (int k = 0; k < 3; k++) v = fmaf(G[i * 3 + k] + G[k * 3 + i], L[k * 3 + j], v);
            dL[i * 3 + j] = v;
          }
        dout[0] = dL[0] * sigmoidf(o[0]);
        dout[1] = dL[3];
        dout[2] = dL[4] * sigmoidf(o[2]);
        dout[3] = dL[6];
        dout[4] = dL[7];
        dout[5] = dL[8] * sigmoidf(o[5]);
      }
      for (int j = 0; j < 8; j++) dos[tid * LDO + j] = dout[j];
    }
    if (!part) {
      __syncthreads();
      continue;  // loss and blocks only
    }
    __syncthreads();
    // backward; rows past the last atom are zero whatever the weights hold
    auto delta_out = [&](f32x4 acc, const float* z, float* d, int n0) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = row + 4 * q + r;
        d[i * LDH + n0 + c16] = (i < na && z[i * LDH + n0 + c16] > 0.f) ? acc[r] : 0.f;
      }
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int n0 = 32 * half + 16 * h;
      delta_out(mfma16_nn<8>(dos + row * LDO, LDO, w3 + n0, LDH, zero, lane), z2, d2, n0);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int n0 = 32 * half + 16 * h;
      delta_out(mfma16_nn<64>(d2 + row * LDH, LDH, w2 + n0, LDH, zero, lane), z1, d1, n0);
    }
    __syncthreads();
    // weight gradients: rows 16 rt.. of W1 (input tiles 0-3 or 4-6) and W2 (0-1 or 2-3), and one
    // tile of W3 for the upper waves. v_mfma_f64_16x16x4: lane l supplies A[l%16][l/16] and
    // B[l/16][l%16] and holds D[l/16 + 4 r][l%16].
#pragma unroll 2
    for (int a = q; a < TR_ATOMS; a += 4) {
      const double v1 = d1[a * LDH + row + c16], v2 = d2[a * LDH + row + c16];
      const float *x = xs + a * LDX + 64 * half + c16, *h = z1 + a * LDH + 32 * half + c16;
      g[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, (double)x[0], g[0], 0, 0, 0);
      g[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, (double)x[16], g[1], 0, 0, 0);
      if (half == 0) {
        g[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, (double)x[32], g[2], 0, 0, 0);
        g[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, (double)x[48], g[3], 0, 0, 0);
      } else {
        const float xv = c16 < MLP_IN - 96 ? x[32] : 0.f;  // inputs 96..103
        g[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, (double)xv, g[2], 0, 0, 0);
        const float v3 = c16 < MLP_OUT ? dos[a * LDO + c16] : 0.f;
        g[3] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)v3, (double)fmaxf(z2[a * LDH + row + c16], 0.f), g[3], 0, 0, 0);
      }
      g[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(v2, (double)fmaxf(h[0], 0.f), g[4], 0, 0, 0);
      g[5] = __builtin_amdgcn_mfma_f64_16x16x4f64(v2, (double)fmaxf(h[16], 0.f), g[5], 0, 0, 0);
    }
    if (tid < 128 + MLP_OUT) {
      const float* col = tid < 64 ? d1 + tid : tid < 128 ? d2 + tid - 64 : dos + tid - 128;
      const int ld = tid < 128 ? LDH : LDO;
      for (int a = 0; a < TR_ATOMS; a++) gb += (double)col[a * ld];
    }
    __syncthreads();  // the next tile overwrites the LDS
  }
  if (!part) return;
  double* out = part + (size_t)blockIdx.x * MLP_NPARAM;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int m = row + q + 4 * r;
    double* o1 = out + m * MLP_IN + 64 * half + c16;
    o1[0] = g[0][r];
    o1[16] = g[1][r];
    if (half == 0) {
      o1[32] = g[2][r];
      o1[48] = g[3][r];
    } else {
      if (c16 < MLP_IN - 96) o1[32] = g[2][r];
      const int j = q + 4 * r;
      if (j < MLP_OUT) out[OFF_W3 + j * 64 + row + c16] = g[3][r];
    }
    double* o2 = out + OFF_W2 + m * 64 + 32 * half + c16;
    o2[0] = g[4][r];
    o2[16] = g[5][r];
  }
  if (tid < 128 + MLP_OUT) out[tid < 64 ? OFF_B1 + tid : tid < 128 ? OFF_B2 + tid - 64 : OFF_B3 + tid - 128] = gb;
}

// grad[p] = sum over the workgroups' partial sums in a fixed order: 32 parameters per workgroup,
// eight groups of lanes each take every eighth partial sum.
__global__ void __launch_bounds__(256) k_mlp_train_sum(const double* __restrict__ part, int n_part,
                                                       float* __restrict__ grad) {
  __shared__ double s[8][32];
  const int j = threadIdx.x & 31, k = threadIdx.x >> 5, p = blockIdx.x * 32 + j;
  double v = 0.0;
  if (p < MLP_NPARAM) {
#pragma unroll 8
    for (int b = k; b < n_part; b += 8) v += part[(size_t)b * MLP_NPARAM + p];
  }
  s[k][j] = v;
  __syncthreads();
  if (k == 0 && p < MLP_NPARAM) {
    for (int i = 1; i < 8; i++) v += s[i][j];
    grad[p] = (float)v;
  }
}

MlpW mlp_weights(const float* params) {
  MlpW W;
  W.w1 = params;
  W.b1 = W.w1 + NP_W1;
  W.w2 = W.b1 + NP_B1;
  W.b2 = W.w2 + NP_W2;
  W.w3 = W.b2 + NP_B2;
  W.b3 = W.w3 + NP_W3;
  return W;
}

}  // namespace

// defined with the rest of the error state in mmff_hip.hip
int mmffhip_set_error(int code, const char* msg);
#define perr mmffhip_set_error

extern "C" {

int mmffhip_mlp_dims(int32_t* n_in, int32_t* n_hidden, int32_t* n_out, int32_t* n_params) {
  if (n_in) *n_in = MLP_IN;
  if (n_hidden) *n_hidden = MLP_H;
  if (n_out) *n_out = MLP_OUT;
  if (n_params) *n_params = MLP_NPARAM;
  return MMFFHIP_OK;
}

int mmffhip_mlp_infer(const float* params, const float* feat, int32_t n_atoms, float* blocks, void* stream) {
  if (n_atoms < 0) return perr(MMFFHIP_ERR_ARG, "n_atoms < 0");
  if (n_atoms == 0) return MMFFHIP_OK;
  if (!params || !feat || !blocks) return perr(MMFFHIP_ERR_ARG, "params, feat and blocks are required");
  const MlpW W = mlp_weights(params);
  const int tiles = (n_atoms + 31) / 32, need = (tiles + INF_WAVES - 1) / INF_WAVES;
  const int grid = need < INF_GRID ? need : INF_GRID;
  const bool vec = ((uintptr_t)feat & 15) == 0;
  if (vec)
    hipLaunchKernelGGL(k_mlp_infer_bf16<true>, dim3(grid), dim3(64 * INF_WAVES), INF_LDS, (hipStream_t)stream, W, feat,
                       n_atoms, blocks);
  else
    hipLaunchKernelGGL(k_mlp_infer_bf16<false>, dim3(grid), dim3(64 * INF_WAVES), INF_LDS, (hipStream_t)stream, W, feat,
                       n_atoms, blocks);
  return hipGetLastError() == hipSuccess ? MMFFHIP_OK : perr(MMFFHIP_ERR_HIP, "launch failed");
}

int mmffhip_mlp_workspace(int32_t n_atoms, size_t* bytes) {
  if (!bytes || n_atoms < 0) return perr(MMFFHIP_ERR_ARG, "bad arguments");
  // The tiles are shared out evenly, so more atoms can take fewer workgroups (16,384: 256, 16,385:
  // 129). The size asked for does not follow: room for n_atoms is room for every smaller batch.
  const int tiles = train_tiles(n_atoms);
  *bytes = train_ws_bytes(tiles < TR_MAX_GRID ? tiles : TR_MAX_GRID);
  return MMFFHIP_OK;
}

int mmffhip_mlp_forward_backward(const float* params, const float* feat, int32_t n_atoms, const float* target,
                                 const float* weight, float* blocks, float* loss, float* grad, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  if (n_atoms <= 0) return perr(MMFFHIP_ERR_ARG, "n_atoms must be positive");
  if (!params || !feat || !target || !workspace) return perr(MMFFHIP_ERR_ARG, "params, feat, target, workspace required");
  const int grid = train_grid(n_atoms);
  if (workspace_bytes < train_ws_bytes(grid)) return perr(MMFFHIP_ERR_SIZE, "workspace too small");
  if (hipFuncSetAttribute((const void*)&k_mlp_train, hipFuncAttributeMaxDynamicSharedMemorySize, (int)TR_LDS) !=
      hipSuccess)
    return perr(MMFFHIP_ERR_HIP, "hipFuncSetAttribute failed");
  const MlpW W = mlp_weights(params);
  double* part = grad ? (double*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255) : nullptr;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_train, dim3(grid), dim3(TR_NT), TR_LDS, s, W, feat, n_atoms, target, weight, blocks, loss,
                     part);
  if (grad)
    hipLaunchKernelGGL(k_mlp_train_sum, dim3((MLP_NPARAM + 31) / 32), dim3(256), 0, s, (const double*)part, grid, grad);
  return hipGetLastError() == hipSuccess ? MMFFHIP_OK : perr(MMFFHIP_ERR_HIP, "launch failed");
}

}  // extern "C"
