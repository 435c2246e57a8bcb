// Products of up to 32 activation rows with a weight matrix (csrc/few_rows.hip).
#pragma once
#include "common.h"

namespace nxd {

enum FewEpi { FEW_STORE = 0, FEW_RESID = 1, FEW_GLU = 2, FEW_ROPE_KV = 3, FEW_F32 = 4, FEW_RELU2 = 5 };

constexpr int FEW_MAX_ROWS = 32;

struct FewRowsParams {
  const uint16_t* x;       // [M, K] bf16 (row stride ldx), or the table of the rows xidx
  int64_t ldx;
  const int64_t* xidx;     // nullable: input row m is x[xidx[m]] (zeros for an id outside [0, xrows))
  int64_t xrows;
  uint16_t* xcopy;         // nullable [M, K]: receives the gathered rows
  const uint16_t* norm_w;  // nullable [K]: RMSNorm of the input rows
  float eps;
  const void* w;           // [Nw, K] bf16 or int8 (row stride ldw elements)
  int64_t ldw;
  const float* wscale;     // int8: [Nw], or one for all (ws_stride 0)
  int ws_stride;
  uint16_t* y;             // [M, N] bf16 (RESID: updated in place)
  int64_t ldy;
  float* yf;               // FEW_F32: [M, N] fp32 (row stride ldy)
  int M, N, K;             // N = output columns (GLU: the up rows start at weight row N)
  float alpha, cap;        // FEW_F32: alpha y, with cap > 0 cap tanh(alpha y / cap)
  // ROPE_KV: y rows hold [nq | nkv | nkv] heads of D; k / v also go to the cache
  int nq, nkv, D;
  const float *cos_t, *sin_t;   // [max_pos, D / 2]
  const int64_t* pos;           // [M]
  int T;                        // rows per sequence
  uint16_t *kc, *vc;
  int64_t c_sb, c_sh, c_sl;
  const int* cache_idx;         // [M / T] (nullable: identity)
  int Lmax, max_pos;
  // Sums of a reduction split over workgroups (nullable: never split): few_rows_workspace() floats, and as many zeroed
  // counters as it says (left zeroed)
  float* ws;
  int* tickets;
  int splits, half;             // (the kernel's own)
};

// Floats of FewRowsParams::ws and the number of its tickets for a product that is better split (0: it is not)
int64_t few_rows_workspace(int M, int N, int K, int* tickets);

// Whether a product of M rows with a norm, of N weight rows, takes half of the rows a workgroup
bool few_rows_halved(int M, int N, int K);

// 0: launched; < 0: not a call this kernel takes; 1: launch error
int few_rows_launch(int epi, const FewRowsParams& p, hipStream_t stream);

}  // namespace nxd
