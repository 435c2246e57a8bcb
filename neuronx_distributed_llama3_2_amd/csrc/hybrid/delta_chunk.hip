// Gated delta rule over long runs of new tokens, 64 at a time, on the fp32 matrix instructions.
//
// Within a chunk, with G_t the running sum of the log decays, the writes u_t of all its tokens solve
//   (I + A) U = diag(beta) (V - diag(e^G) K S_0),   A[t][s] = beta_t e^(G_t - G_s) k_t . k_s   (s < t)
// which is linear in the state S_0 the chunk starts from:  U = Y - W S_0.  Then
//   O   = diag(e^G) Q S_0 + P U,      P[t][s] = e^(G_t - G_s) q_t . k_s   (s <= t)
//   S_1 = e^(G_C) S_0 + K^T diag(e^(G_C - G)) U
//
//   delta_chunk_prepare : Y, W, P of every chunk and head in parallel: products of the chunk's keys and
//                         queries, the four 16 x 16 diagonal blocks of I + A inverted by substitution,
//                         the rest by block substitution with the right-hand sides in registers;
//   delta_chunk_scan    : the chunks of one head one after another for 16 columns of the state.
//   delta_chunk_state, delta_chunk_out : the same in two launches, the chain of the states and then all outputs, where few columns leave CUs
//                         idle or the keys are long (delta_chunk_split_floats).
//
// Everything is fp32 (v_mfma_f32_16x16x4_f32); the sums of log decays are formed in fp64, because the
// differences of large sums are what is exponentiated.
//
// Fragments.  Of a 16 x 16 block, lane l holds the four elements [4 (l / 16) + i][l % 16], i < 4: the
// instruction's result layout.  Taken over k in the order 4 (l / 16) + i, the same registers are a B
// operand, so results feed the next product without moving; an A operand's lane holds four consecutive
// elements of row l % 16.  Everything the scan reads is stored block by block in the order of its lanes
// (1 KiB a block, element ((l / 16) 16 + l % 16) 4 + i): a block is one contiguous load.
#include "delta_rule.h"

#include <algorithm>
#include <type_traits>

namespace nxd {
bool delta_chunk_norm(const DeltaParams& p);
namespace hybrid {

constexpr int CH = 64;   // tokens of a chunk

__device__ __forceinline__ f32x4_t mma4(const f32x4_t& a, const f32x4_t& b, f32x4_t c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// NB = DP / 16 column blocks of the keys.  One workgroup of NW waves per (head, chunk, sequence): what a short
// prompt waits for is one chunk's chain of products (2 chunks of 16 heads 26 us with 4 waves, 15.7 with 16; 64 chunks 77, 74).
template <int NB, int NW>
__global__ void __launch_bounds__(64 * NW) delta_chunk_prepare_kernel(DeltaParams p) {
  constexpr int DP = NB * 16, KS = DP + 4, AS = CH + 4;   // LDS row strides (floats)
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* kt = sm;                       // [64][KS] keys
  float* am = kt + CH * KS;             // [64][AS] A, later the inverted diagonal blocks in place
  __shared__ double gd[CH];
  __shared__ float beta[CH], eg[CH];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
  const int h = blockIdx.x, ch = blockIdx.y, b = blockIdx.z, H = p.H, G = p.G, V = p.V, g = h / (H / G);
  const int len = p.lens ? min(p.lens[b], p.T) : p.T;
  const int n = min(CH, len - ch * CH);
  if (n <= 0) return;
  const int64_t m0 = (int64_t)b * p.T + ch * CH;
  const int64_t cell = ((int64_t)b * p.nch + ch) * H + h;

  const int64_t qkcell = (((int64_t)b * p.nch + ch) * G + g) * CH * DP;
  for (int i = tid; i < CH * (DP / 4); i += 64 * NW) {   // block (d / 16, t / 16), lane i % 64: column d, four tokens
    const int d = 16 * (i / 256) + (i & 15), t = 16 * ((i / 64) & 3) + 4 * ((i / 16) & 3);
    const f32x4_t v = ld4(p.kn + qkcell + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) kt[(t + e) * KS + d] = v[e];
  }
  if (w == 0) {
    double s = lane < n ? (double)p.lg[(m0 + lane) * H + h] : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double q = __shfl_up(s, o, 64);
      if (lane >= o) s += q;
    }
    gd[lane] = s;
    eg[lane] = expf((float)s);
    beta[lane] = lane < n ? p.beta[(m0 + lane) * H + h] : 0.f;
    const double last = __shfl(s, 63, 64);
    float* e = p.ceg + cell * (2 * CH);
    e[lane] = expf((float)s);                  // e^G
    e[CH + lane] = expf((float)(last - s));    // e^(G_C - G)
  }
  __syncthreads();

  // ---- the 10 lower blocks of K K^T and of Q K^T, a wave each in turn
  float* P = p.cp + cell * (CH * CH);
  for (int job = w; job < 20; job += NW) {
    const bool isq = job >= 10;
    int bi = 0, bj = isq ? job - 10 : job;
    while (bj > bi) bj -= ++bi;               // (0,0) (1,0) (1,1) (2,0) ...
    const int t = 16 * bi + lr;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f}, acc2 = acc;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) {
      f32x4_t a;
      if (isq) a = ld4(p.qn + qkcell + ((bi * NB + kb) * 64 + lane) * 4);
      else a = ld4(kt + t * KS + 16 * kb + 4 * lq);
      const f32x4_t bb = ld4(kt + (16 * bj + lr) * KS + 16 * kb + 4 * lq);
      if (kb & 1) acc2 = mma4(bb, a, acc2);   // (transposed: a lane has four columns of row lr, as both are stored)
      else acc = mma4(bb, a, acc);
    }
    acc += acc2;
    const int row = 16 * bi + lr, col = 16 * bj + 4 * lq;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = isq ? col + i <= row : col + i < row;
      acc[i] = in ? acc[i] * expf((float)(gd[row] - gd[col + i])) : 0.f;
      if (!isq) acc[i] *= beta[row];
    }
    st4(isq ? P + ((bi * 4 + bj) * 64 + lane) * 4 : am + row * AS + col, acc);
  }
  __syncthreads();

  // ---- diagonal block w: (I + A_ww)^-1, column lr by the 16 lanes of the first quarter
  if (w < 4) {
    float x[16];
    const float* a = am + (16 * w) * AS + 16 * w;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = i == lr ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) s -= a[i * AS + j] * x[j];
      x[i] = s;
    }
    __builtin_amdgcn_wave_barrier();
    if (lq == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) am[(16 * w + i) * AS + 16 * w + lr] = x[i];
    }
  }
  __syncthreads();

  // ---- (I + A) [Y | W] = diag(beta) [V | e^G K], 16 columns at a time, a wave each in turn
  const int nv = (V + 15) / 16;
  for (int ct = w; ct < nv + NB; ct += NW) {
    const bool isv = ct < nv;
    const int col = (isv ? ct : ct - nv) * 16 + lr;
    f32x4_t y[4];
#pragma unroll
    for (int bi = 0; bi < 4; ++bi) {
      f32x4_t r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * bi + 4 * lq + i;
        float v;
        if (isv) v = t < n && col < V ? p.vn[((m0 + t) * H + h) * V + col] : 0.f;
        else v = kt[t * KS + col] * eg[t];
        r[i] = v * beta[t];
      }
      f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int bk = 0; bk < bi; ++bk) s = mma4(ld4(am + (16 * bi + lr) * AS + 16 * bk + 4 * lq), y[bk], s);
      r -= s;
      y[bi] = mma4(ld4(am + (16 * bi + lr) * AS + 16 * bi + 4 * lq), r, f32x4_t{0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int bi = 0; bi < 4; ++bi) {
      if (isv) {
        st4(p.cy + ((cell * nv + ct) * 4 + bi) * 256 + lane * 4, y[bi]);
      } else {
        float* o = p.cw + (cell * 4 + bi) * (NB * 256) + (ct - nv) * 256;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[((lr / 4) * 16 + 4 * lq + i) * 4 + (lr & 3)] = y[bi][i];
      }
    }
  }
}

// 16 state columns of one head, 8 waves.  Waves 0-3 (tokens 16 w .. of a chunk) compute U, waves 4-7 the
// outputs of the same tokens; the state's row blocks are spread over all of them.  So every SIMD has one
// wave on the chain state -> U -> state and one whose work fills its waits.  Operands are fetched two
// chunks ahead into two register sets.
template <typename T, int NB>
__global__ void __launch_bounds__(512, 2) delta_chunk_scan_kernel(DeltaParams p) {
  constexpr int DP = NB * 16, TPW = (NB + 7) / 8;
  __shared__ __attribute__((aligned(16))) f32x4_t ss[NB][64], us[4][64], ud[4][64];
  const int tid = threadIdx.x, lane = tid & 63, w8 = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lq = lane >> 4;
  const int w = w8 & 3;
  const bool outw = w8 >= 4;
  const int bh = blockIdx.x % (p.B * p.H), v0 = (blockIdx.x / (p.B * p.H)) * 16;   // a head's columns on one XCD
  const int b = bh / p.H, h = bh % p.H, H = p.H, G = p.G, V = p.V, g = h / (H / G);
  const int len = p.lens ? min(p.lens[b], p.T) : p.T;
  if (len <= 0) return;
  const int slot = slot_of(p.slots, b, p.nslots);
  const int64_t p0 = pos_of(p.pos, p.pos_stride, b);
  const int v = v0 + lr;
  const bool vok = v < V;
  float* state = p.state + (((int64_t)slot * H + h) * V + min(v, V - 1)) * DP;
  f32x4_t S[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int rt = w8 + 8 * i;
    S[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (rt < NB) {
      if (p0 > 0) S[i] = ld4(state + rt * 16 + 4 * lq);
      ss[rt][lane] = S[i];
    }
  }
  const int nch = (len + CH - 1) / CH;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  // one chunk's operands: rows of W (U waves) or of Q (output waves), K^T for the own state blocks, the
  // Y tile (U waves) or the P rows (output waves), e^G / e^(G_C - G) of the own rows and e^(G_C).  What a
  // padded token brings is zero.
  struct Ops {
    f32x4_t rowf[NB], kf[TPW][4], pf[4], eg;
    float ec;
  };
  Ops set[2];
  const int nv = (V + 15) / 16;
  // (past the last chunk the last one is read again: an unconditional fetch keeps the number of loads in
  // flight known, so a wait covers exactly one set)
  auto fetch = [&](int c, Ops& o) {
    c = min(c, nch - 1);
    const int64_t cell = ((int64_t)b * p.nch + c) * H + h, qkcell = (((int64_t)b * p.nch + c) * G + g) * CH * DP;
    const float* s = (outw ? p.qn + qkcell : p.cw + cell * CH * DP) + w * (NB * 256) + lane * 4;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) o.rowf[kb] = ld4(s + kb * 256);
    const float* e = p.ceg + cell * (2 * CH);
    o.eg = ld4(e + (outw ? 0 : CH) + 16 * w + 4 * lq);
    o.ec = e[CH - 1];
    // (output waves use the blocks up to the diagonal, the U waves the first)
    const float* q = outw ? p.cp + cell * (CH * CH) + w * 1024 + lane * 4 : p.cy + ((cell * nv + v0 / 16) * 4 + w) * 256 + lane * 4;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) o.pf[kb] = ld4(q + (outw ? kb * 256 : 0));
    const float* k = p.kn + qkcell + lane * 4;
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) o.kf[j][kb] = ld4(k + ((8 * j + 8 <= NB ? w8 + 8 * j : min(w8 + 8 * j, NB - 1)) * 4 + kb) * 256);
  };
  fetch(0, set[0]);
  asm volatile("" ::: "memory");   // (not interleaved: the loop's waits count on the order)
  fetch(1, set[1]);
  lds_barrier();
  auto chunk = [&](int c, Ops& o) {
    f32x4_t a0 = zero, a1 = zero, sb[NB];
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) sb[kb] = ss[kb][lane];
    __builtin_amdgcn_sched_barrier(0);   // all reads in flight before the first product
#pragma unroll
    for (int kb = 0; kb < NB; kb += 2) {   // NB is even
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.rowf[kb][i], sb[kb][i], a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.rowf[kb + 1][i], sb[kb + 1][i], a1, 0, 0, 0);
      }
    }
    f32x4_t r = a0 + a1;   // W S or Q S
    if (!outw) {
      r = o.pf[0] - r;
      us[w][lane] = r;
      ud[w][lane] = r * o.eg;
    }
    lds_barrier();
    f32x4_t ub[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) ub[kb] = ud[kb][lane];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if (8 * j + 8 <= NB || w8 + 8 * j < NB) {
        f32x4_t x = S[j] * o.ec, y = zero;
#pragma unroll
        for (int kb = 0; kb < 4; kb += 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kf[j][kb][i], ub[kb][i], x, 0, 0, 0);
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kf[j][kb + 1][i], ub[kb + 1][i], y, 0, 0, 0);
          }
        }
        S[j] = x + y;
        ss[w8 + 8 * j][lane] = S[j];
      }
    }
    if (outw) {
      r *= o.eg;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        if (kb <= w) r = mma4(o.pf[kb], us[kb][lane], r);
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // (a wave of padded tokens stores nothing)
        const int t = c * CH + 16 * w + 4 * lq + i;
        if (vok && t < len) p.o[(((int64_t)b * p.T + t) * H + h) * V + v] = r[i];
      }
    }
    fetch(c + 2, o);
    lds_barrier();
  };
  int c = 0;
  for (; c + 1 < nch; c += 2) {
    chunk(c, set[0]);
    chunk(c + 1, set[1]);
  }
  if (c < nch) chunk(c, set[0]);
  if (vok) {
#pragma unroll
    for (int i = 0; i < TPW; ++i)
      if (w8 + 8 * i < NB) st4(state + (w8 + 8 * i) * 16 + 4 * lq, S[i]);
  }
  if (v0 == 0 && h == 0) ring_write<T>(p, b, slot, p0, len, tid, 512);
}

// The scan in two launches, for few columns in all: what a chunk's columns need of the chunk before is the state alone, so the chain has U and the state
// only, and the outputs follow for all chunks side by side.  The sums are those of the kernel above, in its order.
//
// The chain.  Waves 0-3 compute U of 16 tokens each, all eight the state's blocks; the other four have nothing in a wave's way meanwhile.  Leaves the state each
// chunk starts from and U.
template <typename T, int NB>
__global__ void __launch_bounds__(512, 2) delta_chunk_state_kernel(DeltaParams p) {
  constexpr int DP = NB * 16, TPW = (NB + 7) / 8;
  __shared__ __attribute__((aligned(16))) f32x4_t ss[NB][64], ud[4][64];
  const int tid = threadIdx.x, lane = tid & 63, w8 = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lq = lane >> 4;
  const int w = w8 & 3;
  const int bh = blockIdx.x % (p.B * p.H), ct = blockIdx.x / (p.B * p.H), v0 = ct * 16;   // a head's columns on one XCD
  const int b = bh / p.H, h = bh % p.H, H = p.H, G = p.G, V = p.V, g = h / (H / G), nv = (V + 15) / 16;
  const int len = p.lens ? min(p.lens[b], p.T) : p.T;
  if (len <= 0) return;
  const int slot = slot_of(p.slots, b, p.nslots);
  const int64_t p0 = pos_of(p.pos, p.pos_stride, b);
  const int v = v0 + lr;
  const bool vok = v < V;
  float* state = p.state + (((int64_t)slot * H + h) * V + min(v, V - 1)) * DP;
  f32x4_t S[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int rt = w8 + 8 * i;
    S[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (rt < NB) {
      if (p0 > 0) S[i] = ld4(state + rt * 16 + 4 * lq);
      ss[rt][lane] = S[i];
    }
  }
  const int nch = (len + CH - 1) / CH;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  // the next chunk's operands to load, and where the present one's state and U go
  const int64_t cell = (int64_t)b * p.nch * H + h, qkcell = (int64_t)b * p.nch * G + g;
  const float* pw = p.cw + cell * CH * DP + w * (NB * 256);
  const float* py = p.cy + (cell * nv + ct) * 1024 + w * 256;
  const float *pe = p.ceg + cell * (2 * CH), *pc = pe;
  const float* pk = p.kn + qkcell * CH * DP;
  float* pu = p.cu + (cell * nv + ct) * 1024 + w * 256;
  float* ps = p.cs + (cell * nv + ct) * (NB * 256) + w8 * 256;
  const int64_t sw = (int64_t)H * CH * DP, sy = (int64_t)H * nv * 1024, sk = (int64_t)G * CH * DP, st = (int64_t)H * nv * (NB * 256);
  const auto loop = [&](auto uwave) __attribute__((always_inline)) {
    constexpr bool U = decltype(uwave)::value;
    // one chunk's operands: the own rows of W, of Y and of e^(G_C - G), K^T for the own state blocks and e^(G_C)
    struct Ops {
      f32x4_t rowf[U ? NB : 1], kf[TPW][4], y, eg;
      float ec;
    };
    Ops set[2];
    // Of the chunk's own set, W goes out for the next chunk but one as soon as it has been used; of the other set, K^T for the next one: neither stands
    // between the last product of a chunk and its barrier.  (Past the last chunk the last one is read again: the number of loads in flight stays known.)
    auto fetch_w = [&](Ops& o, int c) __attribute__((always_inline)) {
      if (U) {
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) o.rowf[U ? kb : 0] = ld4(pw + kb * 256 + lane * 4);
        o.y = ld4(py + lane * 4);
        o.eg = ld4(pe + CH + 16 * w + 4 * lq);
        if (c + 1 < nch) pw += sw, py += sy, pe += H * (2 * CH);
      }
    };
    auto fetch_k = [&](Ops& o, int c) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) o.kf[j][kb] = ld4(pk + ((8 * j + 8 <= NB ? w8 + 8 * j : min(w8 + 8 * j, NB - 1)) * 4 + kb) * 256 + lane * 4);
      o.ec = pc[CH - 1];
      if (c + 1 < nch) pk += sk, pc += H * (2 * CH);
    };
    fetch_w(set[0], 0);
    fetch_k(set[0], 0);
    asm volatile("" ::: "memory");   // (not interleaved: the loop's waits count on the order)
    fetch_w(set[1], 1);
    lds_barrier();
    auto chunk = [&](int c, Ops& o, Ops& other) __attribute__((always_inline)) {
      f32x4_t sb[U ? NB : 1];
      if (U) {
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) sb[U ? kb : 0] = ss[kb][lane];
      }
      __builtin_amdgcn_sched_barrier(0);   // all reads in flight before the first product
      fetch_k(other, c + 1);
      if (U) {
        f32x4_t a0 = zero, a1 = zero;
#pragma unroll
        for (int kb = 0; kb < NB; kb += 2) {   // NB is even
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.rowf[U ? kb : 0][i], sb[U ? kb : 0][i], a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(o.rowf[U ? kb + 1 : 0][i], sb[U ? kb + 1 : 0][i], a1, 0, 0, 0);
          }
        }
        f32x4_t r = a0 + a1;   // W S
        r = o.y - r;
        ud[w][lane] = r * o.eg;
        st4(pu + lane * 4, r);
      }
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        if (8 * j + 8 <= NB || w8 + 8 * j < NB) st4(ps + 8 * j * 256 + lane * 4, S[j]);
      pu += sy, ps += st;
      lds_barrier();
      f32x4_t ub[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) ub[kb] = ud[kb][lane];
      __builtin_amdgcn_sched_barrier(0);
      fetch_w(o, c + 2);
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        if (8 * j + 8 <= NB || w8 + 8 * j < NB) {
          f32x4_t x = S[j] * o.ec, y = zero;
#pragma unroll
          for (int kb = 0; kb < 4; kb += 2) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              x = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kf[j][kb][i], ub[kb][i], x, 0, 0, 0);
              y = __builtin_amdgcn_mfma_f32_16x16x4f32(o.kf[j][kb + 1][i], ub[kb + 1][i], y, 0, 0, 0);
            }
          }
          S[j] = x + y;
          ss[w8 + 8 * j][lane] = S[j];
        }
      }
      lds_barrier();
    };
    int c = 0;
    for (; c + 1 < nch; c += 2) {
      chunk(c, set[0], set[1]);
      chunk(c + 1, set[1], set[0]);
    }
    if (c < nch) chunk(c, set[0], set[1]);
  };
  if (w8 < 4) loop(std::true_type{});
  else loop(std::false_type{});
  if (vok) {
#pragma unroll
    for (int i = 0; i < TPW; ++i)
      if (w8 + 8 * i < NB) st4(state + (w8 + 8 * i) * 16 + 4 * lq, S[i]);
  }
  if (v0 == 0 && h == 0) ring_write<T>(p, b, slot, p0, len, tid, 512);
}

// The outputs of a chunk and head, a wave 16 tokens: its rows of Q and of P stay in registers for `per` blocks of 16 columns.
// NORM (65 to 128 columns, all of them in the workgroup): the wave's outputs go through LDS of its own to the order of delta_out4_kernel's lanes and take the
// gated norm there, the same sums in the same order: no fp32 outputs in memory, no launch after this one.
template <typename T, int NB, bool NORM>
__global__ void __launch_bounds__(256, NB <= 8 ? 4 : 2) delta_chunk_out_kernel(DeltaParams p, int per) {
  constexpr int DP = NB * 16, RS = 128 + 4;
  __shared__ __attribute__((aligned(16))) float rows[NORM ? 4 : 1][NORM ? 16 * RS : 4];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lq = lane >> 4;
  const int nv = (p.V + 15) / 16, groups = (nv + per - 1) / per;
  const int h = blockIdx.x / groups, ct0 = blockIdx.x % groups * per, c = blockIdx.y, b = blockIdx.z, H = p.H, G = p.G, V = p.V, g = h / (H / G);
  const int len = p.lens ? min(p.lens[b], p.T) : p.T;
  const int64_t m0 = (int64_t)b * p.T + c * CH + 16 * w;   // the wave's first row
  const int nrow = p.T - c * CH - 16 * w, live = len - c * CH - 16 * w;
  const int col = 4 * (lane & 31);
  T* y = static_cast<T*>(p.y) + m0 * p.ldy + h * V + col;
  if (live <= 0) {
    if (NORM && col < V)   // padding: a defined value for the projection
#pragma unroll
      for (int i = 0; i < 16; i += 2)
        if (i + (lane >> 5) < nrow) st4(y + (i + (lane >> 5)) * p.ldy, f32x4_t{0.f, 0.f, 0.f, 0.f});
    return;
  }
  const int64_t cell = ((int64_t)b * p.nch + c) * H + h, qkcell = (((int64_t)b * p.nch + c) * G + g) * CH * DP;
  f32x4_t q[NB], pf[4];
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) q[kb] = ld4(p.qn + qkcell + w * (NB * 256) + lane * 4 + kb * 256);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) pf[kb] = ld4(p.cp + cell * (CH * CH) + w * 1024 + lane * 4 + min(kb, w) * 256);   // (up to the diagonal)
  const f32x4_t eg = ld4(p.ceg + cell * (2 * CH) + 16 * w + 4 * lq);
  // (each register is loaded for the next block of columns as soon as it has been used)
  const float *ps = p.cs + (cell * nv + ct0) * (NB * 256) + lane * 4, *pu = p.cu + (cell * nv + ct0) * 1024 + lane * 4;
  f32x4_t s[NB], u[4];
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) s[kb] = ld4(ps + kb * 256);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) u[kb] = ld4(pu + min(kb, w) * 256);
  const int end = min(ct0 + per, nv);
#pragma unroll 1
  for (int ct = ct0; ct < end; ++ct) {
    if (ct + 1 < end) ps += NB * 256, pu += 1024;
    f32x4_t a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
    for (int kb = 0; kb < NB; kb += 2) {   // NB is even
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[kb][i], s[kb][i], a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[kb + 1][i], s[kb + 1][i], a1, 0, 0, 0);
      }
      s[kb] = ld4(ps + kb * 256);
      s[kb + 1] = ld4(ps + (kb + 1) * 256);
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x4_t r = a0 + a1;   // Q S
    r *= eg;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      if (kb <= w) r = mma4(pf[kb], u[kb], r);
      u[kb] = ld4(pu + min(kb, w) * 256);
    }
    const int v = ct * 16 + lr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (NORM) rows[NORM ? w : 0][(4 * lq + i) * RS + v] = r[i];
      else if (v < V && 4 * lq + i < live) p.o[((m0 + 4 * lq + i) * H + h) * V + v] = r[i];
    }
  }
  if (NORM) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the wave's own)
    const T* gate = static_cast<const T*>(p.proj) + m0 * p.ldp + p.C + h * V + col;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f}, nw = col < V ? ld4(p.norm_w + col) : zero;
    f32x4_t g[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = 2 * k + (lane >> 5);
      g[k] = zero;
      if (col < V && i < live) g[k] = ld4(gate + i * p.ldp);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = 2 * k + (lane >> 5);
      f32x4_t x = ld4(&rows[NORM ? w : 0][NORM ? i * RS + col : 0]);
      if (!(col < V && i < live)) x = zero;
      x = gated_norm4<32>(x, g[k], nw, V, p.eps);
      if (col < V && i < nrow) st4(y + i * p.ldy, x);
    }
  }
}

template <int NB, int NW>
static int run_prepare(const DeltaParams& p, hipStream_t s) {
  const size_t lds = (size_t)CH * (NB * 16 + 4 + CH + 4) * 4;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_prepare_kernel<NB, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return 2;
  hipLaunchKernelGGL((delta_chunk_prepare_kernel<NB, NW>), dim3((unsigned)p.H, (unsigned)p.nch, (unsigned)p.B), dim3(64 * NW), lds, s, p);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <typename T, int NB>
static int run_chunk(const DeltaParams& p, hipStream_t s) {
  const int rc = run_prepare<NB, NB <= 8 ? 16 : 8>(p, s);   // (16 waves have 128 registers each)
  if (rc) return rc;
  const int64_t grid = (int64_t)ceil_div(p.V, 16) * p.B * p.H;
  if (p.cs) {
    hipLaunchKernelGGL((delta_chunk_state_kernel<T, NB>), dim3((unsigned)grid), dim3(512), 0, s, p);
    // all columns of a chunk and head in one workgroup if there are enough of these
    const int nv = ceil_div(p.V, 16);
    if constexpr (NB <= 8)
      if (delta_chunk_norm(p)) {
        hipLaunchKernelGGL((delta_chunk_out_kernel<T, NB, true>), dim3((unsigned)p.H, (unsigned)p.nch, (unsigned)p.B), dim3(256), 0, s, p, nv);
        return hipGetLastError() == hipSuccess ? 0 : 1;
      }
    const int per = ceil_div(nv, (int)std::min<int64_t>(ceil_div64(1024, (int64_t)p.B * p.H * p.nch), nv));
    hipLaunchKernelGGL((delta_chunk_out_kernel<float, NB, false>), dim3((unsigned)(p.H * ceil_div(nv, per)), (unsigned)p.nch, (unsigned)p.B), dim3(256), 0, s, p, per);
    return hipGetLastError() == hipSuccess ? 0 : 1;
  }
  hipLaunchKernelGGL((delta_chunk_scan_kernel<T, NB>), dim3((unsigned)grid), dim3(512), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <typename T>
static int dispatch_chunk(const DeltaParams& p, hipStream_t s) {
  switch (p.DP / 32) {
    case 1: return run_chunk<T, 2>(p, s);
    case 2: return run_chunk<T, 4>(p, s);
    case 3: return run_chunk<T, 6>(p, s);
    case 4: return run_chunk<T, 8>(p, s);
    case 5: return run_chunk<T, 10>(p, s);
    case 6: return run_chunk<T, 12>(p, s);
    case 7: return run_chunk<T, 14>(p, s);
    case 8: return run_chunk<T, 16>(p, s);
  }
  return -1;
}

}  // namespace hybrid

// Floats for the scan in two launches, 0: in one.  The chain's part of a chunk takes 1.7 us instead of 3 (16 heads of 128 x 128, 64 chunks: 193 us -> 107
// and 43 for the outputs), the second launch and its 8 to 14 us of start are lost in longer runs, and with more columns than half of the CUs the
// one launch fills the chip as well.  The whole operation, us, one launch / two: 16 heads of 128 x 128 (128 blocks of columns), 512 tokens 75 / 78,
// 768 89 / 85, 1,024 104 / 94, 4,096 317 / 274; 8 of 64 x 64 (32 blocks) 256 tokens 35 / 34, 4,096 156 / 110; 4 of 128 x 128 256 tokens 44 / 43, 4,096 209 /
// 141, 4 x 128 x 72 in two sequences (40 blocks) 256 tokens 44 / 43, but with 64 blocks 4 to 10 chunks are no gain: 4 of 128 x 128 in two sequences 384 tokens 51 / 55, 16 of
// 96 x 64 512 tokens 54 / 57, 8 of 64 x 128 640 tokens 51 / 53, 896 62 / 60; 32 of 96 x 128 (256 blocks) 1,024 tokens 118 / 118, 4,096 392 / 406.  With keys of more than 128 the one launch has not the registers: 16 of 256 x 128, 128
// tokens 96 / 80, 4,096 903 / 544, two sequences of up to 2,000 542 / 356.  The states and U are 100 MB for 4,096 tokens of 16 heads of 128 x 128 beside 84 MB of the chunks' operands; not past
// 1 GiB, and the caller takes the one launch where there is no room for them.
int64_t delta_chunk_split_floats(const DeltaParams& p) {
  const int64_t nv = ceil_div(p.V, 16), blocks = nv * p.B * p.H, floats = blocks * p.nch * 16 * (64 + p.DP);
  const bool pays = p.DP > 128 ? blocks <= 256 && p.nch >= 2 : blocks <= 128 && p.nch >= (blocks <= 40 ? 4 : 12);
  return pays && floats <= (int64_t{1} << 28) ? floats : 0;
}

// Whether the launch of the outputs also norms them: the sizes that delta_out_launch gives 32 lanes a row, and workgroups for half of the CUs when each has all
// columns.  The outputs' fp32 writes and reads are what it saves.  The whole operation, us, with the norm's own launch / without: 16 heads of 128 x 128, 1,024 tokens 98.2 /
// 94.1, 2,048 150.9 / 145.5, 4,096 286 / 274, 8,192 605 / 575; 8 of 64 x 128 1,024 (128 workgroups) 60.8 / 60.5, 8,192 234 / 220; 4 of 128 x 72 2,048 (128) 90.3 / 90.3; 2 of 128 x
// 128 4,096 (128) 136.3 / 133.5; 16 of 64 x 100 800 66.9 / 64.3.
bool delta_chunk_norm(const DeltaParams& p) {
  return p.cs && p.DP <= 128 && p.V > 64 && p.V <= 128 && !(p.V % 4 || p.C % 4 || p.ldp % 4 || p.ldy % 4) && (int64_t)p.B * p.H * p.nch >= 128;
}

int delta_chunk_launch(bool f32, const DeltaParams& p, hipStream_t s) {
  return f32 ? hybrid::dispatch_chunk<float>(p, s) : hybrid::dispatch_chunk<uint16_t>(p, s);
}

}  // namespace nxd
