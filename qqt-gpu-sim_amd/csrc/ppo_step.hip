// One PPO minibatch of the mlp ActorCritic above its first layer, with every
// weight gradient formed in the kernel (train/ppo.py:401-421 on
// train/model.py:140-153, 192-196, 215-256): qqt_ppo_step.
//
// Per row, from z1 = x W0^T + b0: LayerNorm 1 + ReLU -> Linear(128,128) ->
// LayerNorm 2 + ReLU -> three Linear(128,64) + ReLU -> 5 move logits, 2 bomb
// logits, value; masked log-softmax, log-probabilities, entropies; the
// clipped surrogate, the clipped value loss and the entropy bonus with
// torch's gradient rules (min / max ties split the gradient in halves, clamp
// passes it at its bounds); then the backward down to dz1.  Out come dz1, the
// gradients of all parameters above W0 (b0 included) and the statistics.
//
// Bound: the matrix cores, the row phases' VALU work and the operand reads
// between barriers; bytes are small (z1 in, dz1 out: 1 KB per row).  122,880
// multiply-adds per row (forward, input gradients, weight gradients), as six
// bfloat16 products each (below): 0.74 M per row.
//
// Shape: persistent workgroups (one per CU, 8 wavefronts) walk 32-row tiles.
// The activations of a tile live in LDS, the weight-gradient accumulators
// (128 x 128 and 192 x 128 float32 per workgroup, 80 registers per lane) stay
// in registers for the whole launch, so no activation or row gradient but dz1
// goes to HBM; a row-output kernel followed by batched products moved 4.2 KB
// per row out and 3.5 KB back in.  Partial sums go to the workspace once per
// workgroup and ppo_finish_kernel adds them in workgroup order
// (deterministic).  Measured on a 180,224-row minibatch: 347 us with 18 us of
// packing and reduction beside it, where the row-output kernel (float32 MFMA),
// its batched products, reductions and copies took 860 us; 36 k cycles per
// 32-row tile: the two backward product phases 9.1 k (MFMA-bound), the two
// LayerNorms at the tile's ends 4.2 k, loss and dhy 3.2 k each, the others 2.1
// to 2.5 k, waiting at the nine barriers 7.5 k.
//
// Products: v_mfma_f32_16x16x32_bf16 on three bfloat16 pieces of each operand,
// x = x0 + x1 + x2, which hold float32's 24 bits at any magnitude: a row or a
// weight keeps its precision whatever stands beside or before it, with no
// scales.  The sum takes x0 y0, x0 y1, x1 y0, x1 y1, x0 y2 and x2 y0; the three
// left out are below 2^-25 of x y.  In the data products the leading product
// has an accumulator of its own (one rounding of the whole sum per 32
// features).  (float16 pairs under running power-of-two scales, four products,
// took 305 us and held 22 bits of each workgroup's largest row: rows of 1e-9
// of it lost all of dz1, and the bias and LayerNorm sums of 8,192 rows were 1.3
// to 1.6 times as far from float64 as the float32 kernel's.)  Errors against
// float64 from the same z1, geometric means over three kinds of data, the
// row-output float32 kernel -> this one: 1 to 1,021 rows dW1 1.8e-7 -> 1.1e-7,
// dWh 1.5-2.4e-7 -> 0.9-1.6e-7, bias and LayerNorm sums 0.6-1.9e-7 -> 0.4-1.3e-7;
// 1 to 180,224 rows dW1 1.4e-7 -> 0.7e-7, dWh 1.1-2.2e-7 -> 0.6-1.3e-7, sums
// 0.5-1.3e-7 -> 0.3-1.1e-7; the worst dz1 row of 40,001 that span nine orders of
// magnitude 8.7e-7 -> 6.7e-7.
//
// Data products contract over features (8 consecutive features of a row per
// lane); weight gradients contract over the tile's 32 rows, the same LDS rows
// read through the transposing ds_read_b64_tr_b16.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include "mlp_common.h"
#include "pipeline.h"
#include "qqt_common.h"
#include "qqt_hip.h"
#include "qqt_learn.h"

namespace qqt {

extern thread_local char g_err[512];

namespace pstep {

constexpr int R = 32;         // rows per tile
constexpr int T = 512;        // threads: 8 wavefronts; 16 threads per row in the row phases
constexpr int H = 128, HY = 192;
constexpr int MAX_WGS = 256;  // one workgroup per CU
// LDS row strides (halves): 8 banks apart per row, so both the 16-byte operand
// reads (8 rows per cycle) and the transposing reads (4 rows of 32 bytes) are
// conflict-free
constexpr int HS = H + 16, YS = HY + 16;
// float rows; a head's hidden units (and an output's weights) are 68 apart, so
// that the eight outputs of a row read distinct banks (64 apart they took
// turns: 5.2 k of 38 k cycles of a tile in the loss phase, 3.6 k of 36 k now)
constexpr int XS = H + 4, HP = 64 + 4, HYS = 3 * HP;
constexpr float LN_EPS = 1e-5f;

// weight fragments of the workspace (values): [tile][K step][piece][lane][8]
constexpr int FRAG = 512;                    // values of one (tile, step, piece)
constexpr int F_Z2 = 0;                      // W1,   8 tiles x 4 steps: z2 = W1 h1
constexpr int F_HY = F_Z2 + 8 * 4 * 3 * FRAG;    // Wh,  12 x 4: hy = Wh h2
constexpr int F_DH2 = F_HY + 12 * 4 * 3 * FRAG;  // Wh^T, 8 x 6: dh2 = Wh^T dhy
constexpr int F_DH1 = F_DH2 + 8 * 6 * 3 * FRAG;  // W1^T, 8 x 4: dh1 = W1^T dz2
constexpr int F_END = F_DH1 + 8 * 4 * 3 * FRAG;
constexpr int N_FRAGS = F_END / (3 * FRAG) * 64;   // (tile, step, lane) items of the pack kernel

// one workgroup's partial sums (floats)
constexpr int P_W1 = 0, P_WH = P_W1 + H * H, P_WF = P_WH + HY * H, P_G1 = P_WF + 8 * 64,
              P_B1 = P_G1 + H, P_G2 = P_B1 + H, P_B2 = P_G2 + H, P_DB0 = P_B2 + H,
              P_DB1 = P_DB0 + H, P_DBH = P_DB1 + H, P_DBF = P_DBH + HY, P_ST = P_DBF + 8,
              P_MX = P_ST + 5, P_N = P_MX + 1;
constexpr int P_PAD = (P_N + 63) / 64 * 64;

// workspace: fragments | partials
constexpr size_t WS_PART = (size_t)F_END * 2;

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float float8v __attribute__((ext_vector_type(8)));

struct __align__(16) Lds {
  uint16_t h1[3][R][HS], h2[3][R][HS];      // pieces of h1, h2
  union {                                   // ... of dhy, then of dz2
    uint16_t dy[3][R][YS], dz[3][R][HS];
  };
  float ex[R][XS];                          // z2, dh2, dh1 on their way to the row phases
  float hy[R][HYS];
  float dl[R][8];
  uint32_t in[R][16];                       // loss inputs (fetch_loss)
  float sum[3][R][16];                      // each thread's running output-gradient sum, statistic, max |dz1|
  float ln[4][H];                           // gamma1, beta1, gamma2, beta2
  float b1[H], bh[HY], wf[8][HP], bf[8];
  float mx[8];                              // per wavefront: max |dz1|
};

// 2^e for a clamped exponent
__device__ __forceinline__ float pow2(int e) { return ldexpf(1.0f, max(-100, min(100, e))); }
// power of two that brings magnitude m into (2^13, 2^14]
__device__ __forceinline__ float scale_for(float m) {
  return m > 0.0f ? pow2(13 - ilogbf(m)) : 1.0f;
}

// a value that is the same in every lane, as a scalar register
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// v + v rotated by N lanes within each row of 16
template <int N>
__device__ __forceinline__ float ror16(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float v) {
  v += ror16<8>(v);
  v += ror16<4>(v);
  v += ror16<2>(v);
  return v + ror16<1>(v);
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, ror16<8>(v));
  v = fmaxf(v, ror16<4>(v));
  v = fmaxf(v, ror16<2>(v));
  return fmaxf(v, ror16<1>(v));
}
// largest value of the wavefront, in every lane
__device__ __forceinline__ float max64(float v) {
  v = max16(v);
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}

__device__ __forceinline__ bf8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf8*>(p); }

// The three bfloat16 pieces of eight values, v = p[0] + p[1] + p[2] (each the
// nearest to what the ones before leave).
__device__ __forceinline__ void split8(const float (&v)[8], bf8 (&p)[3]) {
  float8v r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = v[i];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    p[k] = __builtin_convertvector(r, bf8);
    if (k < 2) r -= __builtin_convertvector(p[k], float8v);
  }
}
// ... to an LDS plane each
template <int S>
__device__ __forceinline__ void put8(const float (&v)[8], uint16_t (&plane)[3][R][S], int row, int at) {
  bf8 p[3];
  split8(v, p);
#pragma unroll
  for (int k = 0; k < 3; ++k) *reinterpret_cast<bf8*>(&plane[k][row][at]) = p[k];
}

// The six products of two operands' pieces, smallest first; the three left out
// are below 2^-25 of the whole.
constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ floatx4 mfma_bf(bf8 a, bf8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// c[i] += a[i] b for N tiles, product by product (N independent accumulators
// between two uses of one)
template <int N, int M>
__device__ __forceinline__ void add_products(const bf8 (&a)[N][3], const bf8 (&b)[3], floatx4 (&c)[N][M], int n) {
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < N; ++i) c[i][n] = mfma_bf(a[i][PA[k]], b[PB[k]], c[i][n]);
}

// The pieces of eight consecutive features of a row.
template <int S>
__device__ __forceinline__ void ld_pieces(bf8 (&f)[3], const uint16_t (&plane)[3][R][S], int row, int at) {
#pragma unroll
  for (int n = 0; n < 3; ++n) f[n] = ld8(&plane[n][row][at]);
}

// One K step of a data product: c[u] += a[u's tile] b[u's rows], the leading
// product into c[u][0] and the others into c[u][1] (one rounding of the whole
// sum per step of 32 instead of six).
__device__ __forceinline__ void data_step(const bf8 (&a)[3], const bf8 (&b)[2][3], floatx4 (&c)[2][2]) {
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      floatx4& t = c[rt][k == 5 ? 0 : 1];
      t = mfma_bf(a[PA[k]], b[rt][PB[k]], t);
    }
}

// Sum of each of the eight values over the wavefront's four 16-lane rows;
// lane group g = lane / 16 keeps values 2 (g & 1) + 4 (g >> 1) + {0, 1}.
__device__ __forceinline__ void add_rows(const float (&v)[8], float (&acc)[2]) {
  float b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 4]),
                                                    false, false);
    b[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(b[i]), __float_as_uint(b[i + 2]),
                                                    false, false);
    acc[i] += __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// LayerNorm of a row over its 16 threads (8 values each): xh and 1/std, and
// the ReLU output.
__device__ __forceinline__ void ln_forward(float (&z)[8], const float* gam, const float* bet,
                                           float& rstd, float (&h)[8]) {
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) s += z[i];
  const float mean = sum16(s) * (1.0f / H);
  float d2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    z[i] -= mean;
    d2 = __builtin_fmaf(z[i], z[i], d2);
  }
  rstd = 1.0f / sqrtf(sum16(d2) * (1.0f / H) + LN_EPS);
  float g[8], b[8];
  load8(gam, g);
  load8(bet, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    z[i] *= rstd;
    h[i] = fmaxf(__builtin_fmaf(z[i], g[i], b[i]), 0.0f);
  }
}

// Backward of LayerNorm + ReLU for a row's 16 threads: d = gradient of the
// ReLU output on entry, of the LayerNorm's input on exit; dg, db = this
// thread's terms of the affine gradients.
__device__ __forceinline__ void ln_backward(float (&d)[8], const float (&x)[8], const float* gam,
                                            const float* bet, float rstd, float (&dg)[8],
                                            float (&db)[8]) {
  float g[8], b[8];
  load8(gam, g);
  load8(bet, b);
  float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    db[i] = __builtin_fmaf(x[i], g[i], b[i]) > 0.0f ? d[i] : 0.0f;
    dg[i] = db[i] * x[i];
    d[i] = db[i] * g[i];
    s1 += d[i];
    s2 = __builtin_fmaf(d[i], x[i], s2);
  }
  const float m1 = sum16(s1) * (1.0f / H), m2 = sum16(s2) * (1.0f / H);
#pragma unroll
  for (int i = 0; i < 8; ++i) d[i] = rstd * ((d[i] - m1) - x[i] * m2);
}

__device__ __forceinline__ float tree8(const float (&u)[8]) {
  return ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
}

// Weights -> the pieces of their MFMA A fragments (element i of lane (r16, q) in K
// step s of tile m: M[16 m + r16][32 s + 8 q + i], M = W1, Wh, Wh^T, W1^T).
__global__ __launch_bounds__(256) void ppo_pack_kernel(const qqt_ppo_step_args a) {
  uint16_t* const F = static_cast<uint16_t*>(a.workspace);
  const int item = blockIdx.x * 256 + threadIdx.x;  // (fragment, lane)
  if (item >= N_FRAGS) return;
  const int f = item >> 6, lane = item & 63, r16 = lane & 15, q = lane >> 4;
  // fragments in workspace order: W1 (32), Wh (48), Wh^T (48), W1^T (32)
  const int part = f < 32 ? 0 : f < 80 ? 1 : f < 128 ? 2 : 3;
  const int g = f - (part == 0 ? 0 : part == 1 ? 32 : part == 2 ? 80 : 128);
  const int ks = part == 2 ? 6 : 4, m = 16 * (g / ks) + r16, k = 32 * (g % ks) + 8 * q;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (part == 0) v[i] = a.w1[m * H + k + i];
    else if (part == 1) v[i] = a.wh[m >> 6][(m & 63) * H + k + i];
    else if (part == 2) v[i] = a.wh[(k + i) >> 6][((k + i) & 63) * H + m];
    else v[i] = a.w1[(k + i) * H + m];
  }
  bf8 p[3];
  split8(v, p);
#pragma unroll
  for (int n = 0; n < 3; ++n) *reinterpret_cast<bf8*>(F + (size_t)(3 * f + n) * FRAG + lane * 8) = p[n];
}

__global__ __launch_bounds__(T) void ppo_step_kernel(const qqt_ppo_step_args a, int tiles) {
  __shared__ Lds s;
  int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  // positions derived from the thread index; set again in each tile from an
  // opaque copy, so that the compiler forms addresses where they are used
  // instead of holding dozens of them (and spilling) across the loop
  int lane, r16, q, row, j, o, part, grp, lane16;
  auto place = [&]() {
    lane = t & 63;
    r16 = lane & 15, q = lane >> 4;
    row = t >> 4, j = t & 15;                   // row phases: features 8j .. 8j + 7 of `row`
    o = j >> 1, part = j & 1;                   // output o of the row, half of its 64 inputs
    grp = o < 5 ? 0 : o < 7 ? 1 : 2;
    lane16 = lane * 16;
  };
  place();
  // weight fragments: one lane offset for all of them, the rest is scalar
  const Rsrc F = rsrc(a.workspace, F_END * 2);
  auto frag = [&](bf8 (&f)[3], int base, int ks, int tile, int step) {
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const int at = 2 * (base + ((tile * ks + step) * 3 + n) * FRAG);
      f[n] = __builtin_bit_cast(bf8, __builtin_amdgcn_raw_buffer_load_b128(F, lane16, at, 0));
    }
  };

  // ---- parameters -> LDS
  if (t < H) {
    s.ln[0][t] = a.ln1_w[t];
    s.ln[1][t] = a.ln1_b[t];
    s.ln[2][t] = a.ln2_w[t];
    s.ln[3][t] = a.ln2_b[t];
    s.b1[t] = a.b1[t];
  }
  if (t < HY) s.bh[t] = a.bh[t >> 6][t & 63];
  {
    const int o = t >> 6, k = t & 63;
    s.wf[o][k] = o < 5 ? a.wf[0][o * 64 + k] : o < 7 ? a.wf[1][(o - 5) * 64 + k] : a.wf[2][k];
  }
  if (t < 8) s.bf[t] = t < 5 ? a.bf[0][t] : t < 7 ? a.bf[1][t - 5] : a.bf[2][0];
  __syncthreads();
  const float gmin = uniform(-1.0f / (float)a.batch);                          // d loss / d min_i
  const float gmax = uniform(a.value_coef * 0.5f / (float)a.batch);            // ... / d max_i
  const float gh = uniform(-a.entropy_coef / (float)a.batch);                  // ... / d entropy_i

  // ---- accumulators of the whole launch
  floatx4 dwh[3][4], dw1[2][4];                  // feature tiles (3a + i | 2a + i) x (4b + n)
  const int ta = w >> 1, tb = w & 1;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
#pragma unroll
    for (int i = 0; i < 3; ++i) dwh[i][n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i) dw1[i][n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  float dwf[8], dbh[3];
#pragma unroll
  for (int o = 0; o < 8; ++o) dwf[o] = 0.0f;
  dbh[0] = dbh[1] = dbh[2] = 0.0f;
  float g1[2] = {0.0f, 0.0f}, be1[2] = {0.0f, 0.0f}, g2[2] = {0.0f, 0.0f}, be2[2] = {0.0f, 0.0f};
  float db0[2] = {0.0f, 0.0f}, db1[2] = {0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < 3; ++k) s.sum[k][row][j] = 0.0f;

  float zn[8];                                   // next tile's z1
  auto fetch = [&](int tile) {
    const int g = tile * R + row;
#pragma unroll
    for (int i = 0; i < 8; ++i) zn[i] = 0.0f;
    if (tile < tiles && g < a.batch) load8(a.z1 + (size_t)tile * R * H + (row * H + 8 * j), zn);
  };
  // The loss inputs of a row come from anywhere in the buffer: lane j of the
  // row's 16 brings one of them (4 floats, 2 actions, 7 mask bytes), its index
  // fetched a tile ahead and itself at the end of the tile before, and leaves
  // it in LDS, so neither the loss nor the weight fragments queued behind
  // these loads wait for HBM.
  int64_t gnext = 0;
  auto fetch_index = [&](int tile) {
    const int gl = min(tile * R + row, a.batch - 1);
    gnext = a.row_index ? a.row_index[gl] : (int64_t)gl;
  };
  uint32_t lin = 0;
  auto fetch_loss = [&]() {
    const bool byte_in = j >= 6 && j < 13;
    const char* const lbase =
        j == 0 ? (const char*)a.old_logp : j == 1 ? (const char*)a.adv : j == 2 ? (const char*)a.ret
      : j == 3 ? (const char*)a.old_val : j < 6 ? (const char*)(a.actions + (j - 4))
      : j < 11 ? (const char*)(a.move_mask + (j - 6)) : j < 13 ? (const char*)(a.bomb_mask + (j - 11))
               : (const char*)a.old_logp;
    const int lstep = j < 4 ? 4 : j < 6 ? 16 : j < 11 ? 5 : j < 13 ? 2 : 4;
    if (a.row_index) gnext = min(max(gnext, (int64_t)0), a.src_rows - 1);
    const char* const p = lbase + gnext * lstep;
    if (byte_in) lin = *reinterpret_cast<const uint8_t*>(p);
    else lin = *reinterpret_cast<const uint32_t*>(p);
  };
  bf8 wz[4][3];
  auto load_wz = [&]() {
#pragma unroll
    for (int k = 0; k < 4; ++k) frag(wz[k], F_Z2, 4, w, k);
  };
  fetch(blockIdx.x);
  fetch_index(blockIdx.x);
  load_wz();
  fetch_loss();

  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    asm volatile("" : "+v"(t));
    place();
    const int g = tile * R + row;
    const bool live = g < a.batch;
    // ---- LayerNorm 1 (rows past the batch: z1 = 0; their gradients are 0)
    float x1[8], rs1, hv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x1[i] = zn[i];
    ln_forward(x1, s.ln[0] + 8 * j, s.ln[1] + 8 * j, rs1, hv);
    put8(hv, s.h1, row, 8 * j);
    fetch_index(tile + gridDim.x);
    __syncthreads();

    // ---- z2 = W1 h1 + b1: wavefront w, features 16w .. 16w + 15 of both row tiles
    {
      floatx4 c[2][2] = {};                     // [row tile][leading | others]
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        bf8 b[2][3];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) ld_pieces(b[rt], s.h1, 16 * rt + r16, 32 * k + 8 * q);
        data_step(wz[k], b, c);
      }
      const floatx4 b = *reinterpret_cast<const floatx4*>(&s.b1[16 * w + 4 * q]);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        *reinterpret_cast<floatx4*>(&s.ex[16 * rt + r16][16 * w + 4 * q]) = (c[rt][1] + c[rt][0]) + b;
    }
    // head tiles w and 8 + w / 2: half before LayerNorm 2, half during it
    bf8 wy[4][2][3];
    auto load_wy = [&](int k) {
#pragma unroll
      for (int u = 0; u < 2; ++u) frag(wy[k][u], F_HY, 4, u ? 8 + (w >> 1) : w, k);
    };
    load_wy(0);
    load_wy(1);
    __syncthreads();

    // ---- LayerNorm 2
    load_wy(2);
    load_wy(3);
    float x2[8], rs2;
    load8(&s.ex[row][8 * j], x2);
    ln_forward(x2, s.ln[2] + 8 * j, s.ln[3] + 8 * j, rs2, hv);
    put8(hv, s.h2, row, 8 * j);
    __syncthreads();

    // ---- heads' hidden layers: tile w for both row tiles (w & 1 first), tile
    // 8 + w / 2 for row tile w & 1
    {
      floatx4 c[3][2] = {};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        bf8 b[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u) ld_pieces(b[u], s.h2, 16 * (tb ^ u) + r16, 32 * k + 8 * q);
#pragma unroll
        for (int n = 0; n < 6; ++n)
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            floatx4& t = c[u][n == 5 ? 0 : 1];
            t = mfma_bf(wy[k][u >> 1][PA[n]], b[u & 1][PB[n]], t);
          }
      }
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const int ft = u < 2 ? w : 8 + ta, rt = u == 1 ? tb ^ 1 : tb;
        const floatx4 b = *reinterpret_cast<const floatx4*>(&s.bh[16 * ft + 4 * q]);
        floatx4 v = (c[u][1] + c[u][0]) + b;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaxf(v[i], 0.0f);
        *reinterpret_cast<floatx4*>(&s.hy[16 * rt + r16][16 * ft + 4 * q + (HP - 64) * (ft >> 2)]) = v;
      }
      s.in[row][j] = lin;
    }
    __syncthreads();

    // ---- outputs and loss: lanes 2o, 2o + 1 of a row's 16 hold output o
    {
      const float* y = &s.hy[row][HP * grp + 32 * part];
      const float* wo = &s.wf[o][32 * part];
      floatx4 part4 = {0.0f, 0.0f, 0.0f, 0.0f};          // four short chains round less
#pragma unroll
      for (int k = 0; k < 32; k += 4) {
        const floatx4 yv = *reinterpret_cast<const floatx4*>(y + k), wv = *reinterpret_cast<const floatx4*>(wo + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) part4[i] = __builtin_fmaf(yv[i], wv[i], part4[i]);
      }
      float acc = (part4[0] + part4[1]) + (part4[2] + part4[3]);
      acc += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc), 0xB1, 0xf, 0xf, true));
      const float logit = acc + s.bf[o];
      const float old_logp = __uint_as_float(s.in[row][0]), adv = __uint_as_float(s.in[row][1]);
      const float ret = __uint_as_float(s.in[row][2]), old_val = __uint_as_float(s.in[row][3]);
      const int taken = (int)s.in[row][grp == 1 ? 5 : 4];
      const uint32_t mask = s.in[row][min(o, 6) + 6];
      const float NEG = -3.4028234663852886e38f;
      const bool first = part == 0;
      const bool mv = grp == 0, bo = grp == 1;
      const float z = mask ? logit : NEG;
      const float mm = max16(mv ? z : NEG), mb = max16(bo ? z : NEG);
      const float m = mv ? mm : mb;
      const float e = grp < 2 ? expf(z - m) : 0.0f;
      const float sm = sum16(mv && first ? e : 0.0f), sb = sum16(bo && first ? e : 0.0f);
      const float lse = m + logf(mv ? sm : sb);
      const float lp = grp < 2 ? fmaxf(z - lse, NEG) : 0.0f;
      const float p = grp < 2 ? expf(z - lse) : 0.0f;
      const float hm = -sum16(mv && first ? lp * p : 0.0f), hb = -sum16(bo && first ? lp * p : 0.0f);
      const bool mine = grp < 2 && o == taken + (bo ? 5 : 0);
      const float logp = sum16(mine && first ? lp : 0.0f);
      const float v = sum16(grp == 2 && first ? logit : 0.0f);
      // policy term
      const float ratio = expf(logp - old_logp);
      const float cr = fminf(fmaxf(ratio, a.ratio_lo), a.ratio_hi);
      const float s1 = ratio * adv, s2 = cr * adv;
      const float w1 = s1 < s2 ? 1.0f : s1 == s2 ? 0.5f : 0.0f;
      const float w2 = 1.0f - w1;
      const float pass = (ratio >= a.ratio_lo && ratio <= a.ratio_hi) ? 1.0f : 0.0f;
      const float glogp = gmin * (w1 * adv + w2 * adv * pass) * ratio;
      // value term
      const float dvc = v - old_val;
      const float vc = old_val + fminf(fmaxf(dvc, -a.clip_eps), a.clip_eps);
      const float e1 = (v - ret) * (v - ret), e2 = (vc - ret) * (vc - ret);
      const float u1 = e1 > e2 ? 1.0f : e1 == e2 ? 0.5f : 0.0f;
      const float u2 = 1.0f - u1;
      const float vpass = (dvc >= -a.clip_eps && dvc <= a.clip_eps) ? 1.0f : 0.0f;
      float d;
      if (grp == 2) d = gmax * (u1 * 2.0f * (v - ret) + u2 * 2.0f * (vc - ret) * vpass);
      else d = mask ? glogp * ((mine ? 1.0f : 0.0f) - p) - gh * p * (lp + (mv ? hm : hb)) : 0.0f;
      if (!live) d = 0.0f;
      if (first) s.dl[row][o] = d;
      s.sum[0][row][j] += d;
      if (live)
        s.sum[1][row][j] += j == 0 ? -fminf(s1, s2) : j == 1 ? 0.5f * fmaxf(e1, e2) : j == 2 ? hm + hb
            : j == 3 ? old_logp - logp : fabsf(ratio - 1.0f) > a.clip_eps ? 1.0f : 0.0f;
    }
    bf8 wd[6][3];
    auto load_wd = [&](int k) { frag(wd[k], F_DH2, 6, w, k); };
#pragma unroll
    for (int k = 0; k < 3; ++k) load_wd(k);
    __syncthreads();

    // ---- dhy = (Wf^T dl) [hy > 0], and the output layer's gradient: wavefront
    // w takes rows 4w .. 4w + 3, lane l hidden unit l of each head
#pragma unroll
    for (int k = 3; k < 6; ++k) load_wd(k);
    {
      float wfr[8];                              // output layer's column `lane` of each row
#pragma unroll
      for (int k = 0; k < 8; ++k) wfr[k] = s.wf[k][lane];
#pragma unroll 1
      for (int rr = 0; rr < 4; ++rr) {
        const int r = 4 * w + rr;
        float dl[8];
        load8(&s.dl[r][0], dl);
        const float y0 = s.hy[r][lane], y1 = s.hy[r][HP + lane], y2 = s.hy[r][2 * HP + lane];
        float d0 = 0.0f;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          d0 = __builtin_fmaf(dl[k], wfr[k], d0);
          dwf[k] = __builtin_fmaf(dl[k], y0, dwf[k]);
        }
        float d1 = __builtin_fmaf(dl[6], wfr[6], dl[5] * wfr[5]);
        float d2 = dl[7] * wfr[7];
        dwf[5] = __builtin_fmaf(dl[5], y1, dwf[5]);
        dwf[6] = __builtin_fmaf(dl[6], y1, dwf[6]);
        dwf[7] = __builtin_fmaf(dl[7], y2, dwf[7]);
        d0 = y0 > 0.0f ? d0 : 0.0f;
        d1 = y1 > 0.0f ? d1 : 0.0f;
        d2 = y2 > 0.0f ? d2 : 0.0f;
        dbh[0] += d0;
        dbh[1] += d1;
        dbh[2] += d2;
        auto put = [&](float v, int c) {
#pragma unroll
          for (int n = 0; n < 3; ++n) {
            const __bf16 p = (__bf16)v;
            s.dy[n][r][c] = __builtin_bit_cast(uint16_t, p);
            v -= (float)p;
          }
        };
        put(d0, lane);
        put(d1, 64 + lane);
        put(d2, 128 + lane);
      }
    }
    __syncthreads();

    // ---- dh2 = Wh^T dhy (features 16w .. of both row tiles); dWh += dhy^T h2
    {
      floatx4 c[2][2] = {};                     // [row tile][leading | others]
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        bf8 b[2][3];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) ld_pieces(b[rt], s.dy, 16 * rt + r16, 32 * k + 8 * q);
        data_step(wd[k], b, c);
      }
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        *reinterpret_cast<floatx4*>(&s.ex[16 * rt + r16][16 * w + 4 * q]) = c[rt][1] + c[rt][0];
      bf8 av[3][3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int n = 0; n < 3; ++n) av[i][n] = ld_rows<bf8, YS>(s.dy[n][0], 3 * ta + i, lane);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bf8 b[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) b[m] = ld_rows<bf8, HS>(s.h2[m][0], 4 * tb + n, lane);
        add_products(av, b, dwh, n);
        if (n & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    fetch(tile + gridDim.x);
    __syncthreads();

    // ---- LayerNorm 2 backward -> dz2
    float dv[8], tg[8], tb8[8];
    load8(&s.ex[row][8 * j], dv);
    ln_backward(dv, x2, s.ln[2] + 8 * j, s.ln[3] + 8 * j, rs2, tg, tb8);
    put8(dv, s.dz, row, 8 * j);           // (dhy's planes: read before the barrier above)
    add_rows(tg, g2);
    add_rows(tb8, be2);
    add_rows(dv, db1);
    bf8 wu[4][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) frag(wu[k], F_DH1, 4, w, k);
    __syncthreads();

    // ---- dh1 = W1^T dz2; dW1 += dz2^T h1
    {
      floatx4 c[2][2] = {};                     // [row tile][leading | others]
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        bf8 b[2][3];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) ld_pieces(b[rt], s.dz, 16 * rt + r16, 32 * k + 8 * q);
        data_step(wu[k], b, c);
      }
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        *reinterpret_cast<floatx4*>(&s.ex[16 * rt + r16][16 * w + 4 * q]) = c[rt][1] + c[rt][0];
      bf8 av[2][3];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int n = 0; n < 3; ++n) av[i][n] = ld_rows<bf8, HS>(s.dz[n][0], 2 * ta + i, lane);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bf8 b[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) b[m] = ld_rows<bf8, HS>(s.h1[m][0], 4 * tb + n, lane);
        add_products(av, b, dw1, n);
        if (n & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();

    // ---- LayerNorm 1 backward -> dz1
    load_wz();
    fetch_loss();
    load8(&s.ex[row][8 * j], dv);
    ln_backward(dv, x1, s.ln[0] + 8 * j, s.ln[1] + 8 * j, rs1, tg, tb8);
    add_rows(tg, g1);
    add_rows(tb8, be1);
    add_rows(dv, db0);
    if (live) {
      float m = s.sum[2][row][j];
#pragma unroll
      for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(dv[i]));
      s.sum[2][row][j] = m;
      float4* out = reinterpret_cast<float4*>(a.dz1 + (size_t)tile * R * H + (row * H + 8 * j));
      out[0] = make_float4(dv[0], dv[1], dv[2], dv[3]);
      out[1] = make_float4(dv[4], dv[5], dv[6], dv[7]);
    }
  }
  __syncthreads();   // the last tile's reads of ex are done: LDS is scratch from here

  // ---- this workgroup's partial sums
  float* const P = reinterpret_cast<float*>(static_cast<char*>(a.workspace) + WS_PART) +
                   (size_t)blockIdx.x * P_PAD;
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 16 * (4 * tb + n) + r16;
#pragma unroll
      for (int u = 0; u < 3; ++u) P[P_WH + (16 * (3 * ta + u) + 4 * q + i) * H + col] = dwh[u][n][i];
#pragma unroll
      for (int u = 0; u < 2; ++u) P[P_W1 + (16 * (2 * ta + u) + 4 * q + i) * H + col] = dw1[u][n][i];
    }
  // per-wavefront sums meet in LDS: columns (6 kinds), output layer, biases
  float* const cs = &s.hy[0][0];                 // [8 wavefronts][6][128] = 24.6 KB
  float* const fs = &s.ex[0][0];                 // [8][8][64] = 16 KB
  float* const hs = reinterpret_cast<float*>(&s.dy[0][0][0]);    // [8][192]
  {
    const int c = 8 * j + 2 * (q & 1) + 4 * (q >> 1);
    float* p = cs + w * 6 * H + c;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      p[0 * H + i] = g1[i];
      p[1 * H + i] = be1[i];
      p[2 * H + i] = g2[i];
      p[3 * H + i] = be2[i];
      p[4 * H + i] = db0[i];
      p[5 * H + i] = db1[i];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) fs[(w * 8 + k) * 64 + lane] = dwf[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) hs[w * HY + 64 * k + lane] = dbh[k];
    const float m = max64(s.sum[2][row][j]);
    if (lane == 0) s.mx[w] = m;
  }
  __syncthreads();
  for (int i = t; i < 6 * H; i += T) {
    float u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = cs[k * 6 * H + i];
    P[P_G1 + i] = tree8(u);                             // G1, B1, G2, B2, DB0, DB1 in order
  }
  {
    float u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = fs[k * 512 + t];
    P[P_WF + t] = tree8(u);
  }
  if (t < HY) {
    float u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) u[k] = hs[k * HY + t];
    P[P_DBH + t] = tree8(u);
  } else if (t < HY + 13) {                            // output biases, statistics
    const int k = t - HY;
    const float(*const rows)[16] = k < 8 ? s.sum[0] : s.sum[1];
    const int c = k < 8 ? 2 * k : k - 8;
    float u[8];
#pragma unroll
    for (int n = 0; n < 8; ++n)
      u[n] = (rows[4 * n][c] + rows[4 * n + 1][c]) + (rows[4 * n + 2][c] + rows[4 * n + 3][c]);
    P[P_DBF + k] = tree8(u);                            // DBF, ST in order
  } else if (t == HY + 13) {
    float v = 0.0f;
    for (int k = 0; k < 8; ++k) v = fmaxf(v, s.mx[k]);
    P[P_MX] = v;
  }
}

// Partial sums of the workgroups -> gradients, statistics and dz1's scale.
// 64 outputs per workgroup, FP threads each (a share of the workgroups each).
constexpr int FP = 8;        // (tree8)
__global__ __launch_bounds__(64 * FP) void ppo_finish_kernel(const qqt_ppo_step_args a, int wgs) {
  __shared__ float red[FP][64];
  const int c = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + c;
  const float* P = reinterpret_cast<const float*>(static_cast<const char*>(a.workspace) + WS_PART) + i;
  const int per = (wgs + FP - 1) / FP, k0 = part * per, k1 = min(wgs, k0 + per);
  float v = 0.0f;
  if (i == P_MX) {
    for (int k = k0; k < k1; ++k) v = fmaxf(v, P[(size_t)k * P_PAD]);
  } else if (i < P_N) {       // eight chains, then a tree: short chains round less
    float u[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    int k = k0;
    for (; k + 8 <= k1; k += 8)
#pragma unroll
      for (int n = 0; n < 8; ++n) u[n] += P[(size_t)(k + n) * P_PAD];
    for (; k < k1; ++k) u[0] += P[(size_t)k * P_PAD];
    v = tree8(u);
  }
  red[part][c] = v;
  __syncthreads();
  if (part != 0 || i >= P_N) return;
  if (i == P_MX) {
    float m = 1e-30f;
#pragma unroll
    for (int k = 0; k < FP; ++k) m = fmaxf(m, red[k][c]);
    *a.dz_scale = scale_for(m);
    return;
  }
  float u[8];
#pragma unroll
  for (int k = 0; k < FP; ++k) u[k] = red[k][c];
  v = tree8(u);
  if (i < P_WH) a.dw1[i] = v;
  else if (i < P_WF) a.dwh[(i - P_WH) >> 13][(i - P_WH) & 8191] = v;
  else if (i < P_G1) {
    const int k = i - P_WF;
    if (k < 320) a.dwf[0][k] = v;
    else if (k < 448) a.dwf[1][k - 320] = v;
    else a.dwf[2][k - 448] = v;
  }
  else if (i < P_B1) a.dln1_w[i - P_G1] = v;
  else if (i < P_G2) a.dln1_b[i - P_B1] = v;
  else if (i < P_B2) a.dln2_w[i - P_G2] = v;
  else if (i < P_DB0) a.dln2_b[i - P_B2] = v;
  else if (i < P_DB1) a.db0[i - P_DB0] = v;
  else if (i < P_DBH) a.db1[i - P_DB1] = v;
  else if (i < P_DBF) a.dbh[(i - P_DBH) >> 6][(i - P_DBH) & 63] = v;
  else if (i < P_ST) {
    const int k = i - P_DBF;
    if (k < 5) a.dbf[0][k] = v;
    else if (k < 7) a.dbf[1][k - 5] = v;
    else a.dbf[2][0] = v;
  }
  else a.stats[i - P_ST] = v / (float)a.batch;
}

__host__ inline int tiles_of(int batch) { return (batch + R - 1) / R; }
__host__ inline int wgs_of(int batch) { return tiles_of(batch) < MAX_WGS ? tiles_of(batch) : MAX_WGS; }

}  // namespace pstep
}  // namespace qqt

extern "C" {

int64_t qqt_ppo_step_workspace_bytes(int32_t batch) {
  using namespace qqt::pstep;
  if (batch <= 0) return -1;
  return (int64_t)WS_PART + (int64_t)wgs_of(batch) * P_PAD * 4;
}

int qqt_ppo_step(const qqt_ppo_step_args* a, void* stream) {
  using namespace qqt;
  using namespace qqt::pstep;
  g_err[0] = 0;
  bool ok = a && a->z1 && a->ln1_w && a->ln1_b && a->w1 && a->b1 && a->ln2_w && a->ln2_b &&
            a->actions && a->move_mask && a->bomb_mask && a->old_logp && a->adv && a->ret &&
            a->old_val && a->dz1 && a->dz_scale && a->stats && a->db0 && a->dln1_w && a->dln1_b &&
            a->dw1 && a->db1 && a->dln2_w && a->dln2_b && a->workspace;
  for (int h = 0; ok && h < 3; ++h)
    ok = a->wh[h] && a->bh[h] && a->wf[h] && a->bf[h] && a->dwh[h] && a->dbh[h] && a->dwf[h] &&
         a->dbf[h];
  if (!ok) {
    snprintf(g_err, sizeof(g_err), "qqt_ppo_step: null argument");
    return QQT_E_ARG;
  }
  uintptr_t al = (uintptr_t)a->z1 | (uintptr_t)a->dz1 | (uintptr_t)a->w1 | (uintptr_t)a->workspace;
  for (int h = 0; h < 3; ++h) al |= (uintptr_t)a->wh[h];
  if (a->batch <= 0 || (al & 15) || !(a->clip_eps >= 0.0f)) {
    snprintf(g_err, sizeof(g_err), "qqt_ppo_step: bad batch, clip or 16-byte alignment");
    return QQT_E_ARG;
  }
  if (a->workspace_bytes < qqt_ppo_step_workspace_bytes(a->batch)) {
    snprintf(g_err, sizeof(g_err), "qqt_ppo_step: workspace too small");
    return QQT_E_ARG;
  }
  if (a->row_index && (a->src_rows <= 0 || (((uintptr_t)a->row_index) & 7))) {
    snprintf(g_err, sizeof(g_err), "qqt_ppo_step: row_index needs src_rows > 0 and 8-byte alignment");
    return QQT_E_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  const int tiles = tiles_of(a->batch), wgs = wgs_of(a->batch);
  hipLaunchKernelGGL(ppo_pack_kernel, dim3((N_FRAGS + 255) / 256), dim3(256), 0, st, *a);
  QQT_LAUNCH(QQT_KERNEL_PPO, ppo_step_kernel, dim3(wgs), dim3(T), st, *a, tiles);
  hipLaunchKernelGGL(ppo_finish_kernel, dim3(P_PAD / 64), dim3(64 * FP), 0, st, *a, wgs);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "ppo step launch failed: %s", hipGetErrorString(err));
    return QQT_E_LAUNCH;
  }
  return QQT_OK;
}

}  // extern "C"
