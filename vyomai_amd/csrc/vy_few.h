// Products of 1 to 4 rows (decode) that make their own operand rows: y = epilogue(norm(...) W^T).  See vy_few.hip.
#pragma once
#include "vy_common.h"

namespace vy_few {

enum { STORE, QKV, GATED };         // epilogues
enum { PLAIN, LAYER, STREAM, PARTS, RMS };   // operand rows: as they are; LayerNorm of bf16 rows; the residual stream's next norm; LayerNorm of a
                                             // sum; RMS norm of bf16 rows

struct Args {
  const bf16* x; int64_t ldx;                      // PLAIN, LAYER: rows of K; STREAM: the sublayer's output rows (nullable)
  const bf16 *ln_g, *ln_b;                         // LAYER, PARTS
  const float* parts; int n_parts;                 // PARTS: rows bf16(parts[0] + .. + x_bias + x), parts [n_parts][M][K]
  const bf16* x_bias;
  // RMS: rows x / rms(x over n columns) w_pre, zeros behind column n of x
  const bf16* kv; const float* w_kv; int n_kv, np_kv;   // beside it: rows kv (stride ldx) by the same norm into row start[slot] of a cache
  bf16* cache; int64_t k_ss, k_st; int cap, ring; const int* start;
  const float* s_in; float* s_out; int64_t lds;    // STREAM: s_out = s_in + norm(x) w_post (workgroup 0 writes it); operand = norm(s_out) w_pre
  const float *w_post, *w_pre; int n, rms;         //   norms over the first n columns; w_post NULL: plain sum; w_pre NULL: s_out itself
  float eps;
  bf16* h; int64_t ldh;                            // LAYER, STREAM: the operand rows (workgroup 0 writes them; nullable)
  int* advance; const int* slots; int n_adv;       // workgroup 0: advance[slots[i]] += 1, i < n_adv
  const bf16* w; int N, M;                         // W [N][K] (GATED: [2 N][K], gate rows first), M <= 4 rows
  int once;                                        // W is streamed past the caches
  const bf16* bias; int act; float act_arg;        // STORE: act(x W^T + bias) + residual
  const bf16* residual; int64_t ldr;
  bf16* y; int64_t ldy;
  bf16 *q, *k, *v; int64_t c_sb, c_sh, c_sl;       // QKV: heads of 64; rotary pairs (d, d + 32) where cos_tab is given
  const float *cos_tab, *sin_tab; const int* pos_dev; int pos, nq, nkv;
};

bool few_k(int epi, int pro, int64_t K);           // does a kernel for K columns exist?
int few_go(int epi, int pro, const Args& a, int64_t K, hipStream_t st);   // VY_ERR_UNSUPPORTED: no

}  // namespace vy_few
