/*
 * qqt_learn.h - C ABI of the training kernels that work on whole parameter
 * tensors (libqqt_hip.so, beside qqt_hip.h; same conventions: plain device
 * pointers, asynchronous on the caller's stream, no allocation, 0 or a
 * negative QQT_E_* code with qqt_last_error()).
 */
#ifndef QQT_LEARN_H
#define QQT_LEARN_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* One PPO minibatch of the mlp ActorCritic above its first layer
 * (train/ppo.py:401-421 on train/model.py:140-153, 192-196, 215-256): from
 * z1 = x W0^T + b0 to the gradient of every parameter but W0, and dz1 for
 * W0's (qqt_l1_grad).  The parameters are the module's own float32 tensors
 * (contiguous); heads in the order move, bomb, critic with 5, 2 and 1
 * outputs. */
typedef struct qqt_ppo_step_args {
  int32_t batch;              /* rows B (the means' divisor) */
  float clip_eps;             /* float32(clip_eps): value clip and clip fraction */
  float ratio_lo, ratio_hi;   /* float32(1 - clip_eps), float32(1 + clip_eps) */
  float value_coef, entropy_coef;
  int64_t workspace_bytes;
  int64_t src_rows;           /* rows of the per-row inputs when row_index is set */
  const int64_t* row_index;   /* [B] or NULL: actions, masks, old_logp, adv, ret and old_val
                                 of row b are their row row_index[b], clamped into
                                 [0, src_rows); z1 and dz1 stay in minibatch order */
  const float* z1;            /* [B][128], 16-byte aligned */
  const float *ln1_w, *ln1_b; /* [128] */
  const float *w1, *b1;       /* [128][128], [128] */
  const float *ln2_w, *ln2_b; /* [128] */
  const float* wh[3];         /* [64][128] each */
  const float* bh[3];         /* [64] each */
  const float* wf[3];         /* [5][64], [2][64], [1][64] */
  const float* bf[3];         /* [5], [2], [1] */
  const int64_t* actions;     /* [.][2] */
  const uint8_t* move_mask;   /* [.][5] */
  const uint8_t* bomb_mask;   /* [.][2] */
  const float *old_logp, *adv, *ret, *old_val;   /* [.] */
  float* dz1;                 /* [B][128], 16-byte aligned */
  float* dz_scale;            /* [1]: power of two that brings max |dz1| to about 2^14 */
  float* stats;               /* [5]: pg, vf, entropy, old_logp - logp, clip fraction (means) */
  float* db0;                 /* [128] column sums of dz1 */
  float *dln1_w, *dln1_b, *dw1, *db1, *dln2_w, *dln2_b;
  float* dwh[3];
  float* dbh[3];
  float* dwf[3];
  float* dbf[3];
  void* workspace;            /* qqt_ppo_step_workspace_bytes(B) bytes, 16-byte aligned */
} qqt_ppo_step_args;

/* Workspace of qqt_ppo_step for a batch (-1 for a bad batch). */
int64_t qqt_ppo_step_workspace_bytes(int32_t batch);

int qqt_ppo_step(const qqt_ppo_step_args* args, void* stream);

/* Workspace (floats; at least qqt_l1_grad_workspace_floats) that holds the
 * partials of every chunk of 512 rows or more, so that each chunk of a small
 * batch gets its own workgroups; in a smaller one they walk up to four chunks
 * each.  The result is the same, bit for bit, in any workspace that
 * qqt_l1_grad accepts. */
int64_t qqt_l1_grad_preferred_floats(int32_t batch, int32_t k0);

/* qqt_l1_grad for an observation whose columns are a permutation of the
 * weight's: column k of the product is written to column cols[k] of dw0
 * (cols: [k0] on the device, every value of [0, k0) once). */
int qqt_l1_grad_columns(const qqt_l1_grad_args* args, const int64_t* cols, void* stream);

/* The first layer's weight (w: [128][k0] float32, contiguous) as the float16
 * fragments of qqt_mlp_act's w0, its columns taken in the order cols ([k0] on
 * the device).  out: 128 * 64 * kblocks halves, 16-byte aligned, kblocks the
 * 64-column blocks that hold k0. */
int qqt_w0_pack(const float* w, const int64_t* cols, int32_t k0, int32_t kblocks, void* out,
                void* stream);

/* The recurrent part of the lstm learner over whole sequences (train/ppo.py:
 * 463-490): gate order i, f, g, o, hidden width 128, the state entering frame
 * 0 zero, the state after frame t multiplied by keep[t].  All arrays are
 * contiguous float32; T = steps, M = rows (envs). */
typedef struct qqt_lstm_seq_args {
  int32_t steps, rows;
  int32_t window;             /* backward: no gradient passes into frame t from frame t + 1's
                                 state when t + 1 is a multiple of it (0: never cut) */
  int32_t pad;
  const float* w_hh;          /* [512][128], 16-byte aligned */
  const float* keep;          /* [T][M] */
  const float* zx;            /* [T][M][512] W_ih x + both biases (forward) */
  float* h;                   /* [T][M][128] out: h before keep (forward) */
  float* c;                   /* [T][M][128] c before keep: out of forward, in of backward */
  float* gates;               /* [T][M][512] gate values: out of forward, in of backward */
  const float* dh;            /* [T][M][128] gradient of h (backward) */
  float* dz;                  /* [T][M][512] out: gradient of z = zx + W_hh h (backward) */
} qqt_lstm_seq_args;

int qqt_lstm_seq_forward(const qqt_lstm_seq_args* args, void* stream);
int qqt_lstm_seq_backward(const qqt_lstm_seq_args* args, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* QQT_LEARN_H */
