// The recurrent part of the lstm learner's update over whole sequences: an
// LSTM of 128 hidden units over T frames of m envs (train/ppo.py:463-490),
// forward and backward, one launch each.
//
// Forward: z[t] = zx[t] + W_hh h[t-1], gates i, f, o = sigmoid, g = tanh,
// c = f c + i g, h = o tanh(c), then both carried on multiplied by keep[t]
// (0 where the episode ended).  Backward: the same chain from t = T-1 down,
// giving dz[t], from which the caller forms every weight gradient as one
// product over all frames.
//
// What bounds it: the chain.  A frame needs the whole previous h of its env
// but no other env's, so a workgroup owns 16 envs (one MFMA tile of rows)
// for all T frames and nothing crosses workgroups.  Its eight wavefronts
// hold W_hh in registers for the whole launch (128 per lane: 64 KB of LDS
// reads or an L2 round trip per frame otherwise); a frame is one exchange
// of h (forward) or dz (backward) through double-buffered LDS with one
// barrier, and what a frame loads from memory is in flight during the
// products before its use.  Products are float32 MFMA (v_mfma_f32_16x16x4_f32): 8,192
// matrix-core cycles per frame and CU.  Operands are read from LDS as 16
// bytes per lane, so a group of four K steps takes k = 16 s + 4 q + i at
// step i on both sides.
//
// Measured, 32 frames x 256 envs (16 workgroups): forward 204 us, backward
// 167 us, against 110 us of matrix-core time each; the rest is the chain's
// own latency (gate functions, the exchange, the first loads).  Frame by
// frame through nn.LSTM the same minibatch is about 1,500 launches and 14 ms
// of host time: a whole update of that size 16.5 -> 4.6 ms.  The error of h
// against float64 is that of nn.LSTM's kernels (1.05e-7 and 1.06e-7).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include "qqt_common.h"
#include "qqt_hip.h"
#include "qqt_learn.h"

namespace qqt {

extern thread_local char g_err[512];

namespace lseq {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int HID = 128, G4 = 4 * HID;
constexpr int R = 16;                 // envs per workgroup: one MFMA tile of rows
constexpr int NTHR = 512;             // wavefront w: hidden units 16 w .. + 15
// LDS row pitches: 4 modulo 64 floats, so the 16 rows of one 16-byte read
// and the four row groups of one store land in distinct banks
constexpr int PH = HID + 4, PZ = G4 + 4;

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }

__global__ __launch_bounds__(NTHR) void lstm_seq_fwd_kernel(const qqt_lstm_seq_args a) {
  __shared__ __align__(16) float hb[2][R][PH];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4, e0 = blockIdx.x * R, u = 16 * w + r;
  const size_t m = (size_t)a.rows;
  floatx4 wr[4][8];                   // B: W_hh rows (gate, unit u), k = 16 s + 4 q + i
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int s = 0; s < 8; ++s)
      wr[g][s] = *reinterpret_cast<const floatx4*>(a.w_hh + (size_t)(g * HID + u) * HID + 16 * s + 4 * q);
  for (int i = threadIdx.x; i < R * PH; i += NTHR) (&hb[0][0][0])[i] = 0.0f;
  // this lane's envs 4 q + j; rows past the batch repeat the last one and store nothing
  size_t row[4];
  bool ok[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = e0 + 4 * q + j;
    ok[j] = e < a.rows;
    row[j] = (size_t)min(e, a.rows - 1);
  }
  floatx4 zn[4], kn, c = {0.0f, 0.0f, 0.0f, 0.0f};
  auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t o = (size_t)t * m + row[j];
      kn[j] = a.keep[o];
#pragma unroll
      for (int g = 0; g < 4; ++g) zn[g][j] = a.zx[o * G4 + g * HID + u];
    }
  };
  __syncthreads();
  for (int t = 0; t < a.steps; ++t) {
    load(t);                          // used after the products
    floatx4 acc[2][4];                // (two half-length sums per gate, from zero)
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[0][g] = acc[1][g] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const floatx4 av = *reinterpret_cast<const floatx4*>(&hb[t & 1][r][16 * s + 4 * q]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[s & 1][g] = mfma4(av[i], wr[g][s][i], acc[s & 1][g]);
    }
    floatx4 z[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) z[g][j] = zn[g][j] + (acc[0][g][j] + acc[1][g][j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float gi = sigm(z[0][j]), gf = sigm(z[1][j]), gg = tanhf(z[2][j]), go = sigm(z[3][j]);
      const float cn = gf * c[j] + gi * gg, h = go * tanhf(cn);
      if (ok[j]) {
        const size_t o = (size_t)t * m + row[j];
        float* gp = a.gates + o * G4 + u;
        gp[0] = gi;
        gp[HID] = gf;
        gp[2 * HID] = gg;
        gp[3 * HID] = go;
        a.c[o * HID + u] = cn;
        a.h[o * HID + u] = h;
      }
      c[j] = cn * kn[j];
      hb[(t + 1) & 1][4 * q + j][u] = h * kn[j];
    }
    __syncthreads();                  // h of this frame is whole; the other buffer is free
  }
}

__global__ __launch_bounds__(NTHR) void lstm_seq_bwd_kernel(const qqt_lstm_seq_args a) {
  __shared__ __align__(16) float zb[2][R][PZ];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4, e0 = blockIdx.x * R, u = 16 * w + r;
  const size_t m = (size_t)a.rows;
  floatx4 wr[32];                     // B: W_hh column u, k = 16 s + 4 q + i
#pragma unroll
  for (int s = 0; s < 32; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) wr[s][i] = a.w_hh[(size_t)(16 * s + 4 * q + i) * HID + u];
  size_t row[4];
  bool ok[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = e0 + 4 * q + j;
    ok[j] = e < a.rows;
    row[j] = (size_t)min(e, a.rows - 1);
  }
  // one frame's operands: gates, dh of the frame's own output, and c and
  // keep of the frame before it
  floatx4 gn[4], dn, cp, kp;
  auto load = [&](int t) __attribute__((always_inline)) {
    const int tp = max(t - 1, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t o = (size_t)t * m + row[j], op = (size_t)tp * m + row[j];
#pragma unroll
      for (int g = 0; g < 4; ++g) gn[g][j] = a.gates[o * G4 + g * HID + u];
      dn[j] = a.dh[o * HID + u];
      cp[j] = a.c[op * HID + u];
      kp[j] = a.keep[op];
    }
  };
  floatx4 ct, ch = {0.0f, 0.0f, 0.0f, 0.0f}, cc = ch;   // c[t]; carried dh, dc
#pragma unroll
  for (int j = 0; j < 4; ++j) ct[j] = a.c[((size_t)(a.steps - 1) * m + row[j]) * HID + u];
  load(a.steps - 1);
  for (int t = a.steps - 1; t >= 0; --t) {
    // the carried gradients stop at the sequence's start and where the
    // state was detached
    const bool cut = t == 0 || (a.window > 0 && t % a.window == 0);
    floatx4 (*const zrow)[PZ / 4] = reinterpret_cast<floatx4(*)[PZ / 4]>(&zb[t & 1][0][0]);
    const floatx4 kprev = kp, cprev = cp;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float gi = gn[0][j], gf = gn[1][j], gg = gn[2][j], go = gn[3][j];
      const float tc = tanhf(ct[j]);
      const float dh = dn[j] + ch[j];
      const float dc = cc[j] + (dh * go) * (1.0f - tc * tc);
      const float c0 = t == 0 ? 0.0f : cprev[j] * kprev[j];
      const float dzi = (dc * gg) * (gi * (1.0f - gi)), dzf = (dc * c0) * (gf * (1.0f - gf)),
                  dzg = (dc * gi) * (1.0f - gg * gg), dzo = (dh * tc) * (go * (1.0f - go));
      float* zl = &zb[t & 1][4 * q + j][u];
      zl[0] = dzi;
      zl[HID] = dzf;
      zl[2 * HID] = dzg;
      zl[3 * HID] = dzo;
      if (ok[j]) {
        float* zp = a.dz + ((size_t)t * m + row[j]) * G4 + u;
        zp[0] = dzi;
        zp[HID] = dzf;
        zp[2 * HID] = dzg;
        zp[3 * HID] = dzo;
      }
      cc[j] = cut ? 0.0f : (dc * gf) * kprev[j];
      ct[j] = cprev[j];
    }
    load(max(t - 1, 0));
    __syncthreads();                  // dz of this frame is whole
    if (cut) {                        // (uniform)
      ch = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      continue;
    }
    floatx4 acc[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[g] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const floatx4 av = zrow[r][4 * s + q];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[s >> 3] = mfma4(av[i], wr[s][i], acc[s >> 3]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      ch[j] = ((acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j])) * kprev[j];
  }
}

// 0 when the arguments both directions share are usable.
static int check_args(const char* fn, const qqt_lstm_seq_args* a, bool backward) {
  const void* own = !a ? nullptr : backward ? (const void*)a->dh : (const void*)a->zx;
  if (!a || !a->w_hh || !a->keep || !a->gates || !a->c || !own || (backward ? !a->dz : !a->h)) {
    snprintf(g_err, sizeof(g_err), "%s: null argument", fn);
    return QQT_E_ARG;
  }
  if (a->steps <= 0 || a->rows <= 0 || a->window < 0 || (((uintptr_t)a->w_hh) & 15)) {
    snprintf(g_err, sizeof(g_err), "%s: bad steps, rows, window or w_hh alignment", fn);
    return QQT_E_ARG;
  }
  return QQT_OK;
}

static int check_launch(const char* fn) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "%s launch failed: %s", fn, hipGetErrorString(err));
    return QQT_E_LAUNCH;
  }
  return QQT_OK;
}

}  // namespace lseq
}  // namespace qqt

extern "C" {

int qqt_lstm_seq_forward(const qqt_lstm_seq_args* a, void* stream) {
  using namespace qqt;
  g_err[0] = 0;
  const int rc = lseq::check_args("qqt_lstm_seq_forward", a, false);
  if (rc != QQT_OK) return rc;
  hipLaunchKernelGGL(lseq::lstm_seq_fwd_kernel, dim3((a->rows - 1) / lseq::R + 1), dim3(lseq::NTHR),
                     0, (hipStream_t)stream, *a);
  return lseq::check_launch("lstm sequence forward");
}

int qqt_lstm_seq_backward(const qqt_lstm_seq_args* a, void* stream) {
  using namespace qqt;
  g_err[0] = 0;
  const int rc = lseq::check_args("qqt_lstm_seq_backward", a, true);
  if (rc != QQT_OK) return rc;
  hipLaunchKernelGGL(lseq::lstm_seq_bwd_kernel, dim3((a->rows - 1) / lseq::R + 1), dim3(lseq::NTHR),
                     0, (hipStream_t)stream, *a);
  return lseq::check_launch("lstm sequence backward");
}

}  // extern "C"
