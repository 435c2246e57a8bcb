// Weight-gradient GEMM for the parallel linear layers on gfx950 MFMA:
//
//     main_grad[m, n] (fp32) += sum_t dy[t, m] * x[t, n]        (bf16 operands, fp32 accumulate)
//
// Both operands arrive token-major exactly as the forward / backward produced them (dy = output
// gradient [T, M], x = layer input [T, N], rows contiguous along the features): the reduction runs
// over their ROW index.  hipBLASLt needs both transposed to reach its TN speed (a separate tiled
// transpose per operand per layer, 2-5 % of the step) and runs the skinny tensor-parallel shards
// at 0.55-0.9 PF/s (profiles/r2_gemm_tp8_wgrad_layouts.jsonl); this kernel reads the token-major
// tiles with the hardware transpose read (ds_read_b64_tr_b16) instead, and splits the token range
// over workgroups when the output alone cannot fill the 256 CUs.
// Reference: the weight gradient of LinearWithAsyncCommunication.backward
// (src/neuronx_distributed/parallel_layers/layers.py:391-409) and GQAQKVLinearWithAsyncCommunication
// (src/neuronx_distributed/modules/qkv_linear.py:131-150), fp32 gradient accumulation as in the
// reference's use_fp32_grad_acc ZeRO-1 mode.
//
// Structure: the loop of gemm_tile.h (4 waves of 128 x 128 results, one workgroup per CU), both operands' images with contiguous
// features, read with the hardware's transposing read; a token count that is no multiple of 64 makes the first step a partial one.
//   * With one token split per tile the workgroup alone adds to its tile: it loads, adds and stores straight from the registers, the loads of 6 of 8
//     rounds on their way together.  Lanes exchange halves of their fragments so that 8 of them have a line, as lines can be read and written past the caches
//     only whole (half lines come twice, 4 to 8 % more): which gradients are, past_caches() says.  Through LDS, 512 bytes of a row each, 2 to 16 % more.  With S
//     splits the adds are S atomics in any order, through LDS so that they cover 256 contiguous bytes, issued without return and left in flight when the
//     workgroup exits.
//   * Against 8 waves of 128 x 64 in ping-pong: 1,000 tokens 4096 x 4096 54 -> 48 us, 16384 x 2048 97 -> 86; 3,000 128256 x 2048 1,708 -> 1,526; 8,192
//     6144 x 4096 406 -> 372; 8 experts' 14336 x 4096 over 32,768 3,903 -> 3,561.
//   * grouped (MoE expert weight gradients, dW[e] += x_e^T dy_e over expert-sorted rows): the grid covers (split, expert, tile); each
//     workgroup reads its expert's row range from the device offsets (no host sync).
#include "gemm_tile.h"

#include <algorithm>
#include <cstdlib>

namespace nxd {
namespace wg {

using tile::BK;
using tile::BM;
using tile::BN;
constexpr int NT = tile::THREADS;

struct Params {
  const uint16_t* dy;   // [T, M], row stride ld_dy
  const uint16_t* x;    // [T, N], row stride ld_x
  float* c;             // [M, N] fp32, row stride ldc
  int T, M, N;
  int64_t ld_dy, ld_x, ldc;
  int mt, nt;           // output tiles along M, N
  int splits;           // token splits per tile
  int t_per_split;      // tokens per split (multiple of BK)
  int band;             // row tiles per raster band
  int own;              // one split, aligned rows: a workgroup alone adds to its tile (load, add, store), else atomics
  // grouped mode: expert e owns rows offs[e] .. offs[e+1] of dy / x; c += e * c_es
  const int* offs;
  int E;
  int64_t c_es;
};

template <bool PAST>
__device__ __forceinline__ f32x4_t grad_load(const float* at) {
  const f32x4_t* v = reinterpret_cast<const f32x4_t*>(at);
  if constexpr (PAST) return __builtin_nontemporal_load(v);
  else return *v;
}
template <bool PAST>
__device__ __forceinline__ void grad_store(const f32x4_t& v, float* at) {
  if constexpr (PAST) __builtin_nontemporal_store(v, reinterpret_cast<f32x4_t*>(at));
  else *reinterpret_cast<f32x4_t*>(at) = v;
}

// TAIL: a split may have a partial step (the first one); PAST: the gradient past the caches; ZERO: the call itself has just cleared it, and it is not read (one split): 8 experts 4096 x 28672,
// with the clearing, 8,192 rows 3,167 -> 2,665 us, 1,024 2,011 -> 1,295; 14336 x 4096 8,192 rows 1,569 -> 1,283
template <bool GROUPED, bool TAIL, bool PAST, bool ZERO>
__global__ void __launch_bounds__(NT, 1) wgrad_kernel(Params p) {
  __shared__ __attribute__((aligned(16))) char smem[tile::LDS_BYTES];
  const int tiles = p.mt * p.nt;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int groups = GROUPED ? p.E : 1;
  const int split = id / (tiles * groups);   // splits outermost: a tile's partial sums land in different grid waves
  const int ge = GROUPED ? (id / tiles) % groups : 0;
  int rt, ct;
  {
    const int within = id % tiles;
    const int kb = p.band, bnd = within / (kb * p.nt), rem = within - bnd * kb * p.nt;
    const int h = min(kb, p.mt - bnd * kb);
    rt = bnd * kb + rem % h;
    ct = rem / h;
  }
  const int m0 = rt * BM, n0 = ct * BN;
  int t_begin, t_end;
  float* cbase = p.c;
  if constexpr (GROUPED) {
    const int g0 = p.offs[ge], g1 = p.offs[ge + 1];
    const int per = ceil_div(ceil_div(max(g1 - g0, 0), BK), p.splits) * BK;
    t_begin = g0 + split * per;
    t_end = min(g1, t_begin + per);
    if (t_begin >= t_end) return;      // empty group / split: nothing to add (workgroup-uniform)
    cbase += ge * p.c_es;
  } else {
    t_begin = split * p.t_per_split;
    t_end = min(p.T, t_begin + p.t_per_split);
  }
  t_begin = __builtin_amdgcn_readfirstlane(t_begin), t_end = __builtin_amdgcn_readfirstlane(t_end);
  tile::LoopTR loop(smem, p.dy + (int64_t)t_begin * p.ld_dy + m0, p.ld_dy, min(BM, p.M - m0),
                              p.x + (int64_t)t_begin * p.ld_x + n0, p.ld_x, min(BN, p.N - n0));
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int tokens = t_end - t_begin;
  loop.template run<TAIL>(acc, ceil_div(tokens, BK), (tokens - 1) % BK + 1);
  const int lane = loop.lane, wid = loop.wid, wm = loop.wm, wn = loop.wn;

  // 8 rounds of a wave's 16 rows x 128 columns through a padded LDS slab of its own
  constexpr int LD = 132;
  float* slab = reinterpret_cast<float*>(smem) + wid * (2 * 16 * LD);
  if (p.own) {
    // lanes r and r + 8 exchange halves of a pair of fragments: 128 contiguous bytes of 8 rows
    const bool up = lane & 8;
    const int row = m0 + 16 * wm + (lane & 7), col = n0 + tile::col<true>(wn, 0, lane) + (up ? 16 : 0);
    float* cp = cbase + (int64_t)row * p.ldc + col;
    constexpr int AHEAD = 6;
    f32x4_t cur[AHEAD][8];
    const bool whole = m0 + BM <= p.M && n0 + BN <= p.N;
    auto all = [&](auto ok) {
      auto at = [&](int i, int j) { return cp + (int64_t)(32 * i + 8 * (j & 1)) * p.ldc + 32 * (j >> 1); };
      auto load = [&](int i) {   // 16 rows
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (ok(i, j)) cur[i % AHEAD][j] = ZERO ? f32x4_t{0.f, 0.f, 0.f, 0.f} : grad_load<PAST>(at(i, j));
      };
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) load(i);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          f32x4_t lo, hi;
          asm volatile("" : "+a"(acc[i][j]), "+a"(acc[i][j + 1]));   // (or all exchanges are made before both branches: 256 spills)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float u = acc[i][j][e], v = acc[i][j + 1][e];
            const float o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(up ? u : v), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
            lo[e] = up ? o : u, hi[e] = up ? v : o;
          }
          if (ok(i, j)) grad_store<PAST>(cur[i % AHEAD][j] + lo, at(i, j));
          if (ok(i, j + 1)) grad_store<PAST>(cur[i % AHEAD][j + 1] + hi, at(i, j + 1));
        }
        if (i + AHEAD < 8) load(i + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (whole) all([](int, int) { return true; });
    else all([&](int i, int j) { return row + 32 * i + 8 * (j & 1) < p.M && col + 32 * (j >> 1) < p.N; });
    return;
  }
  __syncthreads();   // every wave is done with the ring
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<f32x4_t*>(slab + (lane & 15) * LD + tile::col<true>(0, j, lane)) = acc[i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll 8
    for (int rr = 0; rr < 32; ++rr) {
      const int row = m0 + 32 * i + 16 * wm + (rr >> 1), c = 64 * (rr & 1) + lane, col = n0 + 128 * wn + c;
      const float v = slab[(rr >> 1) * LD + c];
      if (row < p.M && col < p.N) unsafeAtomicAdd(cbase + (int64_t)row * p.ldc + col, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Few tokens, where most of the time goes into the gradient's reads and writes and into starting and ending a workgroup: 8 waves of
// 128 x 64 results with a load, an add and a store of 32 rows at a time, steps of 32 tokens in a ring of four, half the registers to fill and
// to empty.  us here / by the loop above:
//   * 8 experts' 4096 x 28672 and 14336 x 4096 gradients: 256 tokens each 1,505, 697 / 1,588, 807; 768 2,237, 1,056 / 2,300, 1,084; 1,024 2,644,
//     1,278 / 2,627, 1,308; 1,280 3,107, 1,507 / 3,032, 1,479; 1,536 3,505, 1,715 / 3,382, 1,646 (the gradient past the caches in both).  With one read,
//     address or load between two MFMAs of the loop above: 768 2,610, 1,265 / 2,623, 1,281; 1,024 2,845, 1,374 / 2,777, 1,366; 1,280 14336 x 4096 1,750 / 1,664; 2048 x 2816 768 147 /
//     146, 1,024 162 / 152; 128 experts' 2048 x 1536 1,024 1,130 / 1,092 (but 64 experts' 2048 x 1408 553 / 560): the line for groups is at 900;
//   * one gradient, whole steps of 32 tokens: 512 x 512 512 tokens 20 / 27, 1,024 32 / 37, 2,048 53 / 56, 3,072 75.3 / 74.9; 2048 x 2048 23 / 30, 34 /
//     39, 56 / 58, 78 / 78; 3072 x 4096 1,056 46.3 / 48.9, 2,048 68 / 69; 4096 x 4096 512 39 / 42, 1,056 54 / 56, 1,536 69 / 67; 16384 x 2048 1,024
//     102 / 109, 2,080 155 / 157, 3,072 205 / 199;
//     (through the caches)
//   * a partial last step (the loop's is its first): 4096 x 4096, 500 tokens 40 / 36, 700 45 / 40; 768 x 4096 or 128256 x 2048, 500 24, 560 / 28,
//     608, 700 29, 659 / 32, 668, 1,000 38, 794 / 38, 788.
//
// Ping-pong: each stage is two phases of 16 MFMAs per wave, every phase [LDS-DMA half-stage][fragment reads] barrier [16 MFMAs at raised
// priority] barrier, and wave group 1 (waves 4-7; every SIMD holds one wave of each group) runs one barrier behind group 0.  Ring
// safety, global barrier instances #n (group 0 passes #(4t+2h) and #(4t+2h+1) in phase (t, h); group 1 one later):
//   * stage S is read from #(4S-1) on (group 0, phase (S, 0)); both groups retire their pieces of S before arriving there (group 0 after
//     its MFMAs of (S-1, 1), group 1 before its reads of (S-1, 1));
//   * the last reads of stage S complete before #(4S+4) (group 1's MFMAs of (S, 1)); its slot is refilled with S+4 after that: group 1
//     in (S+1, 0/1), group 0 in (S+1, 1) and (S+2, 0);
//   * pieces issued after stage S's last: S+1 (4) and S+2's first half (2) -> vmcnt(6), less at the tail.
namespace few {

inline int most(bool past) { return past ? 900 : 1400; }   // tokens of a group
constexpr int BK = 32, STAGES = 4, NT = 512;
inline bool dense(int T, int tiles) {   // (one gradient, unsplit)
  if (T % BK) return T <= 450 || (T <= 700 && (tiles < 192 || tiles > 1024));
  return T <= 1056 || (T <= 2080 && (tiles < 160 || tiles > 256));
}
constexpr int IMG_BYTES = BK * 256 * 2;           // 16 KiB: one operand stage
constexpr int STAGE_BYTES = 2 * IMG_BYTES;        // A | B
constexpr int LDS_BYTES = STAGES * STAGE_BYTES;   // 128 KiB
constexpr int PIECES = IMG_BYTES / 1024 / (NT / 64);   // LDS-DMA pieces per wave per operand stage (2)
constexpr int DMA_PER_STAGE = 2 * PIECES;               // per thread per stage (A and B): 4

__device__ __attribute__((aligned(16))) uint32_t g_zero16[4];   // zero-initialised device global: the DMA
                                                                  // source of token rows past a group's end

__device__ __forceinline__ int swz(int t) { return 2 * ((t & 3) | (((t >> 3) & 1) << 2)); }
__device__ __forceinline__ int img_off(int t, int ch) { return t * 512 + 16 * (ch ^ swz(t)); }

typedef __attribute__((address_space(3))) char lds_char_t;
typedef __attribute__((address_space(3))) short4_t lds_short4_t;
__device__ __forceinline__ uint32_t lds_addr(const char* q) { return (uint32_t)(uintptr_t)(const lds_char_t*)q; }

// one 1 KiB LDS-DMA piece (16 B per lane) at the wave-uniform LDS address `lds_dst`
__device__ __forceinline__ void dma16(const void* src, uint32_t lds_dst) {
  uint32_t sv;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(sv) : "v"(src), "s"(lds_dst) : "memory");
}

// 16x16x32 operand fragment of features [c0, c0 + 16) from a token-major image: lane l holds
// feature c0 + (l & 15) at tokens 8 (l >> 4) + j, j = 0..7 -- two transposed reads, each a block
// of 4 token rows x 16 features per 16-lane group (lane 4q + p supplies row q, features 4p .. 4p+3).
__device__ __forceinline__ bf16x8_t frag(const char* img, int c0) {
  const int l = threadIdx.x & 63, g = l >> 4, i = l & 15, q = i >> 2, p = i & 3;
  const int col = c0 + 4 * p;
  const int t = 8 * g + q;
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(img + img_off(t, col >> 3) + 8 * (p & 1)));
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(img + img_off(t + 4, col >> 3) + 8 * (p & 1)));
  const short __attribute__((ext_vector_type(8))) a8 = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8_t, a8);
}

// TAIL: the last step may be a partial one (always with GROUPED).  The look at it costs every load a comparison and a selection:
// without them 1024 x 1024 over 512 tokens 22.9 -> 21.2 us, 800 30.0 -> 27.3, 16384 x 2048 over 800 97 -> 93.
template <bool GROUPED, bool TAIL, bool PAST, bool ZERO>
__global__ void __launch_bounds__(NT, 1) kernel(Params p) {
  __shared__ __attribute__((aligned(16))) char smem[LDS_BYTES];
  const int tiles = p.mt * p.nt;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int ge = GROUPED ? id / tiles : 0;
  int rt, ct;
  {
    const int within = GROUPED ? id % tiles : id;
    const int kb = p.band, bnd = within / (kb * p.nt), rem = within - bnd * kb * p.nt;
    const int h = min(kb, p.mt - bnd * kb);
    rt = bnd * kb + rem % h;
    ct = rem / h;
  }
  const int m0 = rt * BM, n0 = ct * BN;
  const int t_begin = GROUPED ? p.offs[ge] : 0, t_end = GROUPED ? p.offs[ge + 1] : p.T;
  if (t_begin >= t_end) return;      // empty group: nothing to add (workgroup-uniform)
  const int nk = ceil_div(t_end - t_begin, BK);
  float* cbase = p.c + ge * p.c_es;
  const int rows = t_end - t_begin;   // token rows >= rows of the last stage read zeros

  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = wid >> 2, wn = wid & 3;   // 2 x 4 waves: rows 128 wm.., cols 64 wn..

  f32x4_t acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const uint32_t lds0 = lds_addr(smem);
  // per-lane LDS-DMA source pointers of this tile's first token step (piece i of operand A / B);
  // a stage s reads them advanced by s * BK rows (one scalar 64-bit offset per operand)
  const uint16_t* src_a[PIECES];
  const uint16_t* src_b[PIECES];
  int tt_of[PIECES];
  {
    const int l = lane;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = wid * PIECES + i, tt = piece * 2 + (l >> 5), ch = (l & 31) ^ swz(tt);
      tt_of[i] = tt;
      src_a[i] = p.dy + (int64_t)(t_begin + tt) * p.ld_dy + min(m0 + 8 * ch, p.M - 8);
      src_b[i] = p.x + (int64_t)(t_begin + tt) * p.ld_x + min(n0 + 8 * ch, p.N - 8);
    }
  }
  const int grp = wm;
  auto issue_half = [&](int s, int hh) {
    if (s >= nk) return;
    const uint32_t img = lds0 + (s % STAGES) * STAGE_BYTES + wid * PIECES * 1024;
    const uint16_t* sa = src_a[hh] + (int64_t)s * BK * p.ld_dy;
    const uint16_t* sb = src_b[hh] + (int64_t)s * BK * p.ld_x;
    if (TAIL && s * BK + tt_of[hh] >= rows) sa = sb = reinterpret_cast<const uint16_t*>(g_zero16);
    dma16(sa, __builtin_amdgcn_readfirstlane(img + hh * 1024));
    dma16(sb, __builtin_amdgcn_readfirstlane(img + IMG_BYTES + hh * 1024));
  };
  auto wait_stage = [&](int S) {
    if (S + 2 < nk) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if (S + 1 < nk) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  auto barrier = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  issue_half(0, 0); issue_half(0, 1); issue_half(1, 0); issue_half(1, 1); issue_half(2, 0);
  wait_stage(0);
  if (grp == 1) issue_half(2, 1);
  barrier();
  if (grp == 1) barrier();   // the stagger
  bf16x8_t af[4], bf[4];
  for (int t = 0; t < nk; ++t) {
    const char* img = smem + (t % STAGES) * STAGE_BYTES;
    if (grp == 0) issue_half(t + 2, 1); else issue_half(t + 3, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[j] = frag(img + IMG_BYTES, wn * 64 + 16 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i) af[i] = frag(img, wm * 128 + 16 * i);
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    barrier();
    if (grp == 1) {
      if (t + 1 < nk) wait_stage(t + 1);
      issue_half(t + 3, 1);
    } else {
      issue_half(t + 3, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) af[i] = frag(img, wm * 128 + 16 * (4 + i));
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[4 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[4 + i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    if (grp == 0 && t + 1 < nk) wait_stage(t + 1);
    barrier();
  }
  if (grp == 0) barrier();

  // ---- epilogue: per wave, 4 rounds of 32 rows x 64 columns through a private padded LDS slab
  // ([32][68] fp32: the two row groups of a 32-lane store half are 4 rows apart -> 16 banks apart),
  // then 4 rows (of 256 contiguous bytes) per load and store.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  constexpr int LD = 68;
  float* slab = reinterpret_cast<float*>(smem) + wid * (32 * LD);
  const int ccol = lane & 15, crow = 4 * (lane >> 4);
  const int col = n0 + wn * 64 + 4 * ccol, row = m0 + wm * 128 + (lane >> 4);
  float* cp = cbase + (int64_t)row * p.ldc + col;
  const int left = col < p.N ? p.M - row : 0;   // rows of this lane that there are
  f32x4_t cur[8];
  auto load = [&](int rnd) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (32 * rnd + 4 * k < left) cur[k] = ZERO ? f32x4_t{0.f, 0.f, 0.f, 0.f} : grad_load<PAST>(cp + (int64_t)(32 * rnd + 4 * k) * p.ldc);
  };
  load(0);
  __syncthreads();   // every wave is done with the ring
#pragma unroll
  for (int rnd = 0; rnd < 4; ++rnd) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) slab[(16 * ii + crow + r) * LD + 16 * j + ccol] = acc[2 * rnd + ii][j][r];
    __builtin_amdgcn_wave_barrier();
    f32x4_t sum[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) sum[k] = cur[k] + *reinterpret_cast<const f32x4_t*>(slab + (4 * k + (lane >> 4)) * LD + 4 * ccol);
    if (rnd < 3) load(rnd + 1);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (32 * rnd + 4 * k < left) grad_store<PAST>(sum[k], cp + (int64_t)(32 * rnd + 4 * k) * p.ldc);
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace few

static int band_rows() {
  static const int b = [] {
    const char* e = getenv("NXD_WG_BAND");
    const int v = e ? atoi(e) : 4;
    return v > 0 ? v : 4;
  }();
  return b;
}

template <bool G, bool TAIL, bool ZERO = false>
void launch(const Params& p, int64_t nwg, bool past, hipStream_t stream) {
  hipLaunchKernelGGL((past ? &wgrad_kernel<G, TAIL, true, ZERO> : &wgrad_kernel<G, TAIL, false, ZERO>), dim3((unsigned)nwg), dim3(NT), 0, stream, p);
}
template <bool G, bool TAIL, bool ZERO = false>
void launch_few(const Params& p, int64_t nwg, bool past, hipStream_t stream) {
  hipLaunchKernelGGL((past ? &few::kernel<G, TAIL, true, ZERO> : &few::kernel<G, TAIL, false, ZERO>), dim3((unsigned)nwg), dim3(few::NT), 0, stream, p);
}

// Whether a gradient of so many bytes is read and written past the caches, which then keep the operands.  What a gradient costs depends on where it lies when it is
// added to, and in a training step it comes from memory once all gradients together are more than the memory-side cache (256 MB, 64 M parameters).  us, through the caches /
// past them:
//   * in a training step: 2048 x 2048 (16 MB), 256 tokens 21.4 / 21.5, 512 26.9 / 27.1, 960 36.8 / 36.8; 3072 x 2048 (24 MB) 23.9 / 22.8, 30.1 / 28.8, 40.2 /
//     38.7; 4096 x 4096, 256 tokens 36 / 34, 500 45 / 42, 1,000 58 / 55, 2,048 84 / 80, 8,192 239 / 240; 12288 x 4096 1,000 162 / 162; 16384 x 2048 3,000
//     201 / 201; 32000 x 4096 1,000 415 / 393; 128256 x 2048 3,000 1,605 / 1,581; 8 experts' 4096 x 28672 and 14336 x 4096, 2,048 rows 1,664 / 1,543 and
//     806 / 735, 4,096 rows 1,990 / 1,900 and 960 / 934, 8,192 rows 2,835 / 2,800 and 1,380 / 1,363;
//   * 3 GB of gradients in turn: 3840 x 2048 448 tokens 30.1 / 27.6, 15872 x 768 1,920 66.0 / 61.2; 8 experts' 768 x 1024 (24 MB) 9,216 rows 60.4 / 55.3, 12,000 64.4 /
//     62.5, 768 x 1408 9,216 62.0 / 60.0, 12,000 70.4 / 67.5;
//   * three gradients in turn, as where all of a small model's lie in that cache (given up for the steps above from 20 MB on): 3072 x 2048, 256 tokens 20.2 / 23.9, 1,024
//     36 / 41; 4096 x 4096 31 / 35, 51 / 55; 8 experts' 768 x 1024 1,024 rows 18.5 / 24.4; but 12288 x 4096 (192 MB) 101 / 94, 150 / 145, 8 experts' 14336 x 4096 775 /
//     682, 4096 x 28672 1,650 / 1,521, 8,192 rows 3,209 / 3,110.
bool past_caches(int64_t bytes) { return bytes >= (int64_t)20 << 20; }

}  // namespace wg

// Token splits per output tile.  Cost model in token steps (1.2 us) of one workgroup, times 256: grid waves of 256 workgroups x the steps
// per split, and the epilogues: 8 steps without a split; with splits 10 for one of them, and the atomics' rate bounds all workgroups together, 40
// steps for 256 tiles.  The smallest split count of minimal cost, of 4 steps at least, from 1,024 tokens on (below, unsplit products of few tiles take
// no longer than the shortest split ones and add in one order).  (A step takes 1.0 us since the loop has one read, address or load between two MFMAs; the choices are within 3 % of
// the best all the same.)  Unsplit / in the given splits, us, gradients from memory: 1,000 tokens 6144 x 4096 90 / 2: 196, 2048 x 2048 39 / 2: 41; 1,024 tokens 512 x 512 34 /
// 2: 27 / 4: 22, 1024 x 1024 35 / 2: 27 / 4: 24 / 8: 35, 768 x 4096 37 / 2: 35 / 3: 42; 3,000 tokens 3072 x 2048 74 / 2: 74 / 3: 106, 2048 x 2048 71 / 2: 58 / 4: 71; 4,096 tokens 512 x
// 512 84 / 8: 27 / 16: 24; 8,192 tokens 6144 x 4096 346 / 2: 409, 512 x 4096 157 / 4: 72 / 8: 80; 32,768 tokens 6144 x 4096 1,323 / 2: 1,163, 768 x 4096 579 / 5: 188 / 6: 270.
int wgrad_gemm_choose_splits(int T, int M, int N) {
  const int64_t tiles = (int64_t)ceil_div(M, wg::BM) * ceil_div(N, wg::BN);
  const int steps = ceil_div(T, wg::BK);
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int s = 1; s <= 32 && s <= steps; ++s) {
    if (s > 1 && (steps < 16 || steps / s < 4)) break;
    const int64_t cost = (tiles * s + 255) / 256 * 256 * ceil_div(steps, s) + (s == 1 ? 8 * 256 : std::max<int64_t>(10 * 256, 40 * tiles * s));
    if (cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

// Of a product into an aligned gradient: {splits, whether the kernel for few tokens takes it}
void wgrad_gemm_plan(int T, int M, int N, int splits, int* out) {
  const int steps = ceil_div(T, wg::BK);
  if (splits <= 0) splits = wgrad_gemm_choose_splits(T, M, N);
  splits = std::min(splits, steps);
  out[0] = ceil_div(steps, ceil_div(steps, splits));
  out[1] = out[0] == 1 && wg::few::dense(T, (int)std::min<int64_t>((int64_t)ceil_div(M, wg::BM) * ceil_div(N, wg::BN), INT32_MAX));
}

// c [M, N] fp32 += dy[T, M]^T x[T, N]; M % 8 == 0, N % 8 == 0, 16-B aligned rows.
int wgrad_gemm_launch(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, float* c, int64_t ldc, int T, int M,
                      int N, int splits, hipStream_t stream) {
  if (T <= 0 || M <= 0 || N <= 0) return 0;
  if (M % 8 || N % 8 || ld_dy % 8 || ld_x % 8) return -1;
  wg::Params p{};
  p.dy = static_cast<const uint16_t*>(dy);
  p.x = static_cast<const uint16_t*>(x);
  p.c = c;
  p.T = T; p.M = M; p.N = N;
  p.ld_dy = ld_dy; p.ld_x = ld_x; p.ldc = ldc;
  p.mt = ceil_div(M, wg::BM);
  p.nt = ceil_div(N, wg::BN);
  if (splits <= 0) splits = wgrad_gemm_choose_splits(T, M, N);
  const int steps = ceil_div(T, wg::BK);
  splits = splits < 1 ? 1 : (splits > steps ? steps : splits);
  p.t_per_split = ceil_div(steps, splits) * wg::BK;
  p.splits = ceil_div(T, p.t_per_split);
  p.own = p.splits == 1 && ldc % 4 == 0 && ldc >= N && (reinterpret_cast<uintptr_t>(c) & 15) == 0;
  p.band = wg::band_rows();
  const int64_t nwg = (int64_t)p.mt * p.nt * p.splits;
  if (nwg > INT32_MAX) return -2;
  const bool past = wg::past_caches((int64_t)M * N * 4);
  if (p.own && wg::few::dense(T, p.mt * p.nt)) {
    if (T % wg::few::BK) wg::launch_few<false, true>(p, nwg, past, stream);
    else wg::launch_few<false, false>(p, nwg, past, stream);
  } else if (T % wg::BK)
    wg::launch<false, true>(p, nwg, past, stream);
  else
    wg::launch<false, false>(p, nwg, past, stream);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// Grouped (zero: the caller has just cleared c, in this stream): c[e] [M, N] fp32 += dy[g0:g1]^T x[g0:g1] for every expert e, rows g0 = offs[e],
// g1 = offs[e+1] read on the device; splits per group chosen for the mean group size rows / E.
// M % 8 == 0, N % 8 == 0.
int wgrad_gemm_grouped_launch(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, float* c, int64_t ldc,
                              int64_t c_es, const int* offs, int E, int rows, int M, int N, bool zero, hipStream_t stream) {
  if (E <= 0 || M <= 0 || N <= 0 || rows <= 0) return 0;
  if (M % 8 || N % 8 || ld_dy % 8 || ld_x % 8) return -1;
  wg::Params p{};
  p.dy = static_cast<const uint16_t*>(dy);
  p.x = static_cast<const uint16_t*>(x);
  p.c = c;
  p.T = rows; p.M = M; p.N = N;
  p.ld_dy = ld_dy; p.ld_x = ld_x; p.ldc = ldc;
  p.mt = ceil_div(M, wg::BM);
  p.nt = ceil_div(N, wg::BN);
  p.offs = offs;
  p.E = E;
  p.c_es = c_es;
  // splits for a group half as long again as the mean one, as the longest is what a call waits for (all E groups' tiles share the grid).  16 experts
  // of 512 x 1024, 65,536 rows in groups of 0.5 to 1.5 of the mean 137 -> 91 us, 8 of 768 x 1024 16,384 78 -> 60 (even groups 60 -> 64); one group
  // of a third of all rows among 8 waits longer with few splits than even groups gain: 131,072 rows 655, even 223, by 8 splits each 271 and 300.
  const int mean = std::max(wg::BK, (rows / E) / wg::BK * wg::BK);
  p.splits = wgrad_gemm_choose_splits((int)std::min<int64_t>((int64_t)mean * 3 / 2, INT32_MAX), (int)std::min<int64_t>((int64_t)M * E, INT32_MAX), N);
  p.own = p.splits == 1 && ldc % 4 == 0 && ldc >= N && c_es % 4 == 0 && (E == 1 || c_es >= (int64_t)(M - 1) * ldc + N) && (reinterpret_cast<uintptr_t>(c) & 15) == 0;
  p.band = wg::band_rows();
  const int64_t nwg = (int64_t)p.mt * p.nt * E * p.splits;
  if (nwg > INT32_MAX) return -2;
  const bool past = wg::past_caches((int64_t)E * M * N * 4);
  if (p.own && rows / E <= wg::few::most(past)) {
    if (zero) wg::launch_few<true, true, true>(p, nwg, past, stream);
    else wg::launch_few<true, true>(p, nwg, past, stream);
  } else if (p.own && zero)
    wg::launch<true, true, true>(p, nwg, past, stream);
  else
    wg::launch<true, true>(p, nwg, past, stream);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace nxd
