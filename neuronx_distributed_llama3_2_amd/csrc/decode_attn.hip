// Decode attention on MFMA for small query groups (M = (Hq/Hkv) * T <= 16 rows per kv head):
// one workgroup of 4 or 8 waves (splits_of; FUSE: 8 at D 64) owns a (batch, kv head, key split); the keys per
// split (128-2,560) are sized so the grid reaches 256 to 512 workgroups; every wave runs an
// online-softmax flash-decoding loop over 32-key chunks (FUSE: 64) entirely in registers:
//
//   S^T[key][m] = K.Q^T   v_mfma_f32_16x16x32_bf16, K rows straight from the cache (16-B loads),
//                         Q^T fragments held for the whole loop (rows >= M are zero);
//   softmax             16 scores per lane (4 key tiles x 4), row max / sum over the 4 lanes of a
//                         query row with two xor-shuffles, exp2 with the scale folded in;
//   O[m][d] += P.V      P re-packed into the A operand with 16 lane shuffles per chunk, V staged
//                         through a per-wave LDS tile and read transposed (ds_read_b64_tr_b16);
//
// then the waves merge their (max, sum, O) through LDS once.  With one split the workgroup writes
// the final bf16 output; otherwise it writes the (m, l, o) partials that the last split of the head to
// finish (with tickets), inference.hip's merge kernel or, fused with o_proj, merge_oproj_kernel below combines.  Compared with the 128-key-chunk
// kernel there (four workgroup barriers per chunk and a merge launch at every length) this is one
// barrier per call.
//
// FUSE (attention + o_proj, one launch instead of two; caches up to NXD_DECODE_ATTN_OPROJ_MAXL =
// 1,024 keys): the grid is (batch, kv head, R row chunks
// of the o_proj output); every workgroup of a kv head recomputes that head group's attention (a
// few hundred L2-resident keys at decode lengths) and multiplies it by its Wo block [H/R rows x
// G*D columns], prefetched into registers before the attention starts, then adds the partial
// rows into an fp32 accumulator with float atomics (G*D columns of the o_proj reduction per
// workgroup).  No cross-workgroup wait: the next launch (the GLU projection's RMSNorm prologue and
// the down projection's residual epilogue, decode_fused.hip xadd / yadd) folds the accumulator into
// the residual stream with the rounding of the unfused o_proj epilogue and zeroes it.
#include "common.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace nxd {
namespace dattn {

constexpr int KB = 64;            // keys per chunk of a wave with FUSE; splits are multiples of it
constexpr int KPS = 1024;         // most keys per workgroup split (room for more than 64 K keys: more)
constexpr int WAVES = 4;          // without FUSE: waves of a workgroup where they are not 8,
constexpr int CHUNK = 32;         // keys per chunk of a wave

// Keys of a split (splits_of): those of a full cache, halved once for a sequence of at most a quarter of its room, again for an
// eighth, and so on (a few scalar instructions: with divisions, or 64-bit products in their place, every launch took 0.2 us more)
struct Splits {
  int room, full, least, most, waves;   // (waves of a workgroup)
  __host__ __device__ int keys(int slen) const {   // slen <= room
    const int n = slen > 1 ? slen : 1, a = __builtin_clz(n) - __builtin_clz(room), s = a - 1 - ((uint32_t)n << a > (uint32_t)room);
    const int k = ((s > 0 ? full >> s : full) + KB - 1) & -KB;
    return k < least ? least : (k > most ? most : k);
  }
};

struct Params {
  const uint16_t* q;
  int64_t q_sb, q_st, q_sh;
  const uint16_t* kc;
  const uint16_t* vc;
  int64_t c_sb, c_sh, c_sl;
  const int* cache_idx;
  const int* seq_len;
  uint16_t* out;
  int64_t o_sb, o_st, o_sh;
  float* po;   // [B*Hkv, nsplit, M, D] partials (nsplit > 1)
  float* pm;   // natural-log row max
  float* pl;
  int B, T, Hq, Hkv, nsplit;
  Splits sp;          // keys per split (FUSE: none)
  int kps;            // SYNC: keys per split (multiple of KB)
  float scale_log2;   // softmax scale * log2(e)
  // weight prefetch riding on the (tiny) attention grid: workgroups >= attn_wgs stream the two
  // byte ranges through the memory hierarchy so the next projections (o_proj, gate_up) find them
  // in the Infinity Cache instead of cold HBM; the attention itself leaves HBM idle
  const u32x4_t* pf[2];
  int64_t pf_n16[2];   // 16-byte chunks per range
  int attn_wgs;
  // FUSE: o_proj weight [Hout, Hq * D] (row stride ldwo), fp32 accumulator [B * T, Hout]
  const uint16_t* wo;
  int64_t ldwo;
  float* oacc;
  int Hout, R, NP;     // output rows, row chunks per kv head, Wo register passes (<= 4)
  // opt-in phase trace (decode_attn_set_trace): wave 0 of each workgroup stores s_memrealtime (100 MHz)
  // at entry and exit to trace[2 * blockIdx.x + {0, 1}]; null = off.  This is the trailing field whose
  // round-4 version aborted the decode tests: decode_attn2_launch built `Params p;` without value-
  // initialisation, so the field was stack garbage (non-null) there and the kernel stored through it
  // (profiles/r4_decode_attn_trace_abort.txt).  Every launcher now value-initialises its Params.
  uint64_t* trace;
  // SYNC (fused, long caches): per-(batch, kv head) arrival / done counters [2][kSyncHeads] (device
  // globals, zero at load, reset by the last workgroup of each head) and the bounded-spin error word
  unsigned* sync_cnt;
  int* sync_err;
  float* mo;          // SYNC: [B * Hkv, M, D] merged attention rows (the merger's hand-off)
  // key splits without FUSE: zeroed counters [B * Hkv] (left zeroed) with which the last split of a head to finish
  // merges them; null: a launch of its own does
  int* tickets;
};
static_assert(std::is_trivially_copyable<Params>::value && sizeof(Params) <= 4096, "kernel-argument struct");

static uint64_t* g_trace = nullptr;

constexpr int kSyncHeads = 4096;   // batch x kv heads covered by the SYNC counters
__device__ unsigned g_sync_cnt[3 * kSyncHeads];   // arrivals, done, merged-flag per head
__device__ int g_sync_err;

// Prefetch workgroup body: 4 independent 16-B loads in flight per lane, folded into one value that
// is stored only under a condition the host never creates (pf_n16[0] < 0), so the loads stay live.
__device__ __forceinline__ void prefetch_body(const Params& p, int wg, int nwg) {
  uint32_t acc = 0;
  const int64_t stride = (int64_t)nwg * blockDim.x;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const u32x4_t* base = p.pf[r];
    const int64_t n = p.pf_n16[r];
    int64_t i = (int64_t)wg * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
      const u32x4_t a = base[i], b = base[i + stride], c = base[i + 2 * stride], d = base[i + 3 * stride];
      acc ^= a[0] ^ b[1] ^ c[2] ^ d[3];
    }
    for (; i < n; i += stride) acc ^= base[i][0];
  }
  if (p.pf_n16[0] < 0) p.pm[threadIdx.x] = __uint_as_float(acc);
}

typedef __attribute__((address_space(3))) short4_t lds_s4_t;
typedef short short8_t __attribute__((ext_vector_type(8)));

// FUSE o_proj pieces: thread (row row0 + pass * rpp, 32-column segment) holds its Wo block in
// registers (<= 4 passes), then adds its rows' dot products with the attention output into oacc.
__device__ __forceinline__ void load_wo_regs(const Params& p, int row0, int col0, int rpp, u32x4_t (&wreg)[4][4]) {
  const uint16_t* wb = p.wo + (int64_t)row0 * p.ldwo + col0;
#pragma unroll
  for (int np = 0; np < 4; ++np) {
    if (np < p.NP) {
#pragma unroll
      for (int j = 0; j < 4; ++j) wreg[np][j] = *reinterpret_cast<const u32x4_t*>(wb + (int64_t)np * rpp * p.ldwo + 8 * j);
    }
  }
}

// out[t][row] += sum_c Wo[row][hkv*G*D + c] o[t][c] over this thread's 32 columns, reduced over the
// tpr threads of a row; of = [M][D] attention output (m = t * G + g)
template <int D>
__device__ __forceinline__ void oproj_tail(const Params& p, const float* of, const u32x4_t (&wreg)[4][4], int b, int row0,
                                           int rpp, int tpr, int seg, int G) {
  const int c0 = 32 * seg, gg = c0 / D, d0 = c0 % D;
#pragma unroll
  for (int np = 0; np < 4; ++np) {
    if (np >= p.NP) break;
    float w[32];
#pragma unroll
    for (int j = 0; j < 4; ++j) unpack8(wreg[np][j], w + 8 * j);
    const int row = row0 + np * rpp;
    for (int tt = 0; tt < p.T; ++tt) {
      const float* orow = of + (tt * G + gg) * D + d0;
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < 32; j += 4) {
        const f32x4_t o4 = *reinterpret_cast<const f32x4_t*>(orow + j);
        dot += w[j] * o4[0] + w[j + 1] * o4[1] + w[j + 2] * o4[2] + w[j + 3] * o4[3];
      }
      if (tpr > 32) dot = lanes_add<32>(dot);
      if (tpr > 16) dot = lanes_add<16>(dot);
      if (tpr > 8) dot = lanes_add<8>(dot);
      if (tpr > 4) dot = lanes_add<4>(dot);
      if (tpr > 2) dot = lanes_add<2>(dot);
      if (tpr > 1) dot = lanes_add<1>(dot);
      if (seg == 0) unsafeAtomicAdd(p.oacc + (int64_t)(b * p.T + tt) * p.Hout + row, dot);
    }
  }
}

// SYNC (with FUSE, caches past one pass): workgroup r of a kv head's R also computes key split r
// (kps keys; splits >= nsplit have none) and publishes its (m, l, o) partial with write-through (sc1)
// stores and an agent-scope arrival count; the split whose arrival completes the count merges the
// head once and publishes the merged rows (write-through) and a flag, which the head's other
// workgroups poll (bounded spin: every workgroup of the grid is resident, the host caps the grid at
// the CU count) before their o_proj slices: split-K attention + merge + o_proj in one launch, the KV
// cache read once.  The last workgroup of a head through the hand-off resets the head's counters.
// Measured SLOWER than the two launches it replaces at the notebook config (16.1 us per layer --
// 17.9 with every workgroup merging all partials itself -- vs 5.7 + 5.6 us; 0.759 vs 0.686
// ms/token; profiles/r6_decode/sync_ab.txt): the in-launch wait on the slowest split of a head costs
// more than a kernel boundary, so it is off by default (NXD_DECODE_ATTN_SYNC=1).
//
// Without FUSE the keys and values of a step are read once and the time is their way from memory plus what comes before
// and after it.  Measured per layer, before -> now (before: 8 waves at D 64, chunks of 64 keys, splits next to each other in
// the grid, a merge launch of 4.2 us):
//   4 sequences of 350-700 keys, 8 heads of 64       10.2 ->  7.6 us
//   6 of 512-1,024, 8 of 64                          12.0 ->  8.8
//   13 of 750-1,500, 8 of 128                        25.6 -> 19.5
//   32 of 1,024-2,048, 8 of 64 (100 MB)              32.2 -> 24.2 (4.2 TB/s; the loads alone 23.5)
// and with 8 waves again, now of chunks of 32, in parts that are a workgroup a CU (splits_of): 8.3, 17.6, 20.8 us for the last three.
// - chunks of 32 keys leave the registers for two to three workgroups a CU, so that one computes while the other's keys
//   are on their way (64 keys at D 128: one workgroup, 22.5 us instead of 18.5 at the same splits);
// - the first splits of all heads come first in the grid and the last, short or empty ones last: neighbours go to
//   different XCDs, and with an even number of splits next to each other half of the XCDs had the long ones;
// - values are read non-temporally (24.2 instead of 27.2 us at the largest), keys are not: a wave's read of 16 half lines
//   needs the cache for the other halves;
// - the sums of the waves lie over their V tiles, and the last split merges with 8 splits' sums in flight (one trip to
//   memory where weights first, sums then were two: 1 us).
template <int D, int NWV, bool FUSE, bool WO_LATE = true, bool SYNC = false>
__global__ void __launch_bounds__(64 * NWV) attn_kernel(Params p) {
  static_assert(!SYNC || FUSE, "SYNC is a FUSE form");
  constexpr int NS = D / 32;      // k-steps of the score MFMA
  constexpr int NDT = D / 16;     // 16-wide d tiles of the output
  constexpr int KC = FUSE ? KB : CHUNK;   // keys of a wave's chunk
  constexpr int KT = KC / 16;
  constexpr int VL = KC * D / 512;   // 16-B V loads per lane
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int mi = lane & 15, g = lane >> 4;
  uint16_t* vt = reinterpret_cast<uint16_t*>(smem) + wid * KC * D;              // this wave's V tile [KC][D]
  constexpr int RED = FUSE ? 16 * D : KC * D / 2;                               // floats from a wave's sums to the next one's
  float* red_o = reinterpret_cast<float*>(smem + (FUSE ? NWV * KC * D * 2 : 0));   // [NWV][16][D], or over the V tiles
  float* red_m = reinterpret_cast<float*>(smem + NWV * KC * D * 2) + (FUSE ? NWV * 16 * D : 0);   // [NWV][16]
  float* red_l = red_m + NWV * 16;

  if (!FUSE && (int)blockIdx.x >= p.attn_wgs) {
    prefetch_body(p, blockIdx.x - p.attn_wgs, gridDim.x - p.attn_wgs);
    return;
  }
  auto stamp = [&](int end) {
    if (p.trace != nullptr && tid == 0) p.trace[2 * blockIdx.x + end] = __builtin_amdgcn_s_memrealtime();
  };
  stamp(0);
  const int heads = p.B * p.Hkv;
  const int split = FUSE ? (SYNC ? (int)blockIdx.x % p.R : 0) : (int)blockIdx.x / heads;
  const int bh = FUSE ? (int)blockIdx.x / p.R : (int)blockIdx.x % heads;
  const int b = bh / p.Hkv, hkv = bh % p.Hkv;
  const int G = p.Hq / p.Hkv, M = G * p.T;
  // FUSE: this workgroup's Wo block (rows rc * NR .., columns of head group hkv) into registers,
  // in flight during the attention so its HBM latency hides behind it.  Thread (row r0 + pass * RPP,
  // 32-column segment seg).
  const int tpr = FUSE ? (G * D) / 32 : 1;
  const int seg = tid % tpr, r0 = tid / tpr, rpp = (64 * NWV) / tpr;
  const int nr = FUSE ? p.Hout / p.R : 0;
  const int row0 = FUSE ? ((int)blockIdx.x % p.R) * nr + r0 : 0;
  u32x4_t wreg[4][4];
  auto load_wo = [&]() { load_wo_regs(p, row0, hkv * G * D + 32 * seg, rpp, wreg); };
  if constexpr (FUSE && !WO_LATE) load_wo();   // round-3 order (A/B: NXD_DECODE_WO_LATE=0)
  const int cb = p.cache_idx ? p.cache_idx[b] : b;
  const int slen = FUSE ? p.seq_len[b] : min(p.seq_len[b], p.sp.room);
  const int kps = FUSE ? p.kps : p.sp.keys(slen);
  // splits that have keys; with tickets the others leave (a sequence without keys has one, which writes zeros)
  const int live = !FUSE && p.tickets ? max(1, min(p.nsplit, ceil_div(slen, kps))) : 0;
  if (!FUSE && p.tickets && split >= live) return stamp(1);
  const uint16_t* kbase = p.kc + (int64_t)cb * p.c_sb + (int64_t)hkv * p.c_sh;
  const uint16_t* vbase = p.vc + (int64_t)cb * p.c_sb + (int64_t)hkv * p.c_sh;

  // Q^T fragments: lane (mi, g) holds Q[mi][32 s + 8 g .. +7]
  bf16x8_t qf[NS];
  const int tt_q = mi / G, gg_q = mi % G;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    u32x4_t v = {0, 0, 0, 0};
    if (mi < M)
      v = *reinterpret_cast<const u32x4_t*>(p.q + (int64_t)b * p.q_sb + (int64_t)tt_q * p.q_st +
                                             (int64_t)(hkv * G + gg_q) * p.q_sh + 32 * s + 8 * g);
    qf[s] = __builtin_bit_cast(bf16x8_t, v);
  }
  const int lim = slen - (p.T - 1 - tt_q);        // keys visible to query row mi (causal over new tokens)

  float run_m = -INFINITY, run_l = 0.f;           // stats of query row mi (log2 domain)
  f32x4_t o[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // FUSE: the whole cache in one pass per workgroup (no key splits, no merge launch)
  const int kend = (FUSE && !SYNC) ? slen : min(slen, (split + 1) * kps);
  // K fragments and the V chunk of the NEXT chunk are loaded while this one runs its softmax and P.V
  u32x4_t kf[KT][NS], vv[VL];
  auto load_chunk = [&](int k0) {
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int idx = lane + 64 * i, key = idx / (D / 8), c = idx % (D / 8);
      const u32x4_t* a = reinterpret_cast<const u32x4_t*>(vbase + (int64_t)min(k0 + key, slen - 1) * p.c_sl + 8 * c);
      vv[i] = FUSE ? *a : __builtin_nontemporal_load(a);
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const uint16_t* kr = kbase + (int64_t)min(k0 + kt * 16 + mi, slen - 1) * p.c_sl + 8 * g;
#pragma unroll
      for (int s = 0; s < NS; ++s) kf[kt][s] = *reinterpret_cast<const u32x4_t*>(kr + 32 * s);
    }
  };
  int k0 = split * kps + wid * KC;
  if (k0 < kend) load_chunk(k0);
  // FUSE: the Wo block is issued AFTER the q and first K / V loads.  vmcnt retires in issue order:
  // issued first (round 3), the cold-HBM Wo loads had to land before the first score MFMA could
  // read its L2-resident K fragments, so their latency was added to the attention instead of
  // hidden behind it (attention + o_proj 7.16 -> 6.92 us, 0.619 -> 0.614 ms/token alternating, profiles/r4_decode_wo_late_ab.txt).
  if constexpr (FUSE && WO_LATE) load_wo();
  for (; k0 < kend; k0 += NWV * KC) {
    // ---- scores S^T[key][m] for key tiles of 16
    f32x4_t sc[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      sc[kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NS; ++s)
        sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[kt][s]), qf[s], sc[kt], 0, 0, 0);
    }
    // V tile -> LDS (row-major [key][D]) once the wave's previous transposed reads have retired
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int idx = lane + 64 * i, key = idx / (D / 8), c = idx % (D / 8);
      *reinterpret_cast<u32x4_t*>(vt + key * D + 8 * c) = vv[i];
    }
    if (k0 + NWV * KC < kend) load_chunk(k0 + NWV * KC);
    // ---- online softmax of query row mi over this chunk: lane holds keys k0 + 16 kt + 4 g + v
    float cm = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int key = k0 + kt * 16 + 4 * g + v;
        const float sv = key < lim ? sc[kt][v] * p.scale_log2 : -INFINITY;
        sc[kt][v] = sv;
        cm = fmaxf(cm, sv);
      }
    cm = lanes_max<32>(lanes_max<16>(cm));
    const float nm = fmaxf(run_m, cm);
    const float mu = nm == -INFINITY ? 0.f : nm;
    const float alpha = run_m == -INFINITY ? 0.f : exp2f(run_m - mu);
    float ls = 0.f;
    uint32_t p2[KT][2];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      float e[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        e[v] = exp2f(sc[kt][v] - mu);
        ls += e[v];
      }
      p2[kt][0] = pack2bf(e[0], e[1]);
      p2[kt][1] = pack2bf(e[2], e[3]);
    }
    ls = lanes_add<32>(lanes_add<16>(ls));
    run_l = run_l * alpha + ls;
    run_m = nm;
    // rescale O rows 4 g + v by their row's alpha (held by lane 4 g + v)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float a = __shfl(alpha, 4 * g + v, 64);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) o[dt][v] *= a;
    }
    // ---- P as the A operand: lane (mi, h) needs P[mi][32 ks + 8 h + j], j = 0..7
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int ks = 0; ks < KC / 32; ++ks) {
      const int src0 = (2 * (g & 1)) * 16 + mi, src1 = src0 + 16;
      const bool hi = (g >> 1) != 0;
      uint32_t w[4];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint32_t a0 = __shfl(p2[2 * ks][q], src0, 64), b0 = __shfl(p2[2 * ks + 1][q], src0, 64);
        const uint32_t a1 = __shfl(p2[2 * ks][q], src1, 64), b1 = __shfl(p2[2 * ks + 1][q], src1, 64);
        w[q] = hi ? b0 : a0;
        w[2 + q] = hi ? b1 : a1;
      }
      const u32x4_t pw = {w[0], w[1], w[2], w[3]};
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, pw);
      // V B-fragments: keys 32 ks + 8 g + (0..3 | 4..7), columns 16 dt + 4 p of the 16-lane group
      const int qrow = (lane & 15) >> 2, pc = lane & 3;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const uint16_t* a = vt + (32 * ks + 8 * g + qrow) * D + 16 * dt + 4 * pc;
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t*)a);
        const short4_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t*)(a + 4 * D));
        const short8_t v8 = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, __builtin_bit_cast(bf16x8_t, v8), o[dt], 0, 0, 0);
      }
    }
  }

  // ---- merge the 4 waves: stats of row mi from lanes g == 0, O rows 4 g + v, cols 16 dt + (lane & 15)
  if (g == 0) {
    red_m[wid * 16 + mi] = run_m;
    red_l[wid * 16 + mi] = run_l;
  }
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int v = 0; v < 4; ++v) red_o[wid * RED + (4 * g + v) * D + 16 * dt + (lane & 15)] = o[dt][v];
  __syncthreads();
  const int64_t pbase = ((int64_t)bh * p.nsplit + split) * M;
  for (int it = tid; it < M * D; it += 64 * NWV) {
    const int m = it / D, d = it % D;
    float gm = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWV; ++w) gm = fmaxf(gm, red_m[w * 16 + m]);
    float L = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float mw = red_m[w * 16 + m];
      const float wt = (mw == -INFINITY) ? 0.f : exp2f(mw - gm);
      L += wt * red_l[w * 16 + m];
      acc += wt * red_o[w * RED + m * D + d];
    }
    if (FUSE && !SYNC) {   // bf16-rounded as the unfused path's attention output, then o_proj below
      reinterpret_cast<float*>(smem)[m * D + d] = bf2f(f2bf(L > 0.f ? acc / L : 0.f));
    } else if (SYNC) {   // write-through partials (the merge reads them from other workgroups)
      if (split < p.nsplit) {
        __hip_atomic_store(p.po + (pbase + m) * D + d, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == 0) {
          __hip_atomic_store(p.pm + pbase + m, gm == -INFINITY ? -INFINITY : gm * 0.69314718056f, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(p.pl + pbase + m, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    } else if (p.nsplit == 1 || live == 1) {
      const int tt = m / G, gg = m % G;
      p.out[(int64_t)b * p.o_sb + (int64_t)tt * p.o_st + (int64_t)(hkv * G + gg) * p.o_sh + d] =
          f2bf(L > 0.f ? acc / L : 0.f);
    } else if (live > 1) {   // (through to memory: another workgroup reads them in this launch)
      __hip_atomic_store(p.po + (pbase + m) * D + d, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) {
        __hip_atomic_store(p.pm + pbase + m, gm == -INFINITY ? -INFINITY : gm * 0.69314718056f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p.pl + pbase + m, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      p.po[(pbase + m) * D + d] = acc;
      if (d == 0) {
        p.pm[pbase + m] = gm == -INFINITY ? -INFINITY : gm * 0.69314718056f;   // log2 -> natural-log domain
        p.pl[pbase + m] = L;
      }
    }
  }
  // ---- the last split of the head to come merges all of them (no split waits for another), in their order, so
  // the bits are the same whichever comes last
  if (!FUSE && live > 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* flg = reinterpret_cast<int*>(red_m);
    if (tid == 0) {
      flg[0] = __hip_atomic_fetch_add(p.tickets + bh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == live - 1;
      if (flg[0]) __hip_atomic_store(p.tickets + bh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!flg[0]) return stamp(1);
    // statistics and sums of 8 splits in flight together
    const int64_t pb = (int64_t)bh * p.nsplit * M;
    auto get = [](const float* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    for (int it = tid; it < M * D; it += 64 * NWV) {
      const int m = it / D, d = it % D, tt = m / G, gg = m % G;
      float gm = -INFINITY, L = 0.f, acc = 0.f;
      for (int s0 = 0; s0 < live; s0 += 8) {
        float ms[8], ls[8], os[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int64_t at = pb + (int64_t)min(s0 + i, live - 1) * M + m;
          ms[i] = get(p.pm + at);
          ls[i] = get(p.pl + at);
          os[i] = s0 + i < live ? get(p.po + at * D + d) : 0.f;
        }
        float nm = gm;
#pragma unroll
        for (int i = 0; i < 8; ++i) nm = fmaxf(nm, ms[i]);
        const float mu = nm == -INFINITY ? 0.f : nm, a = __expf(gm - mu);
        L *= a;
        acc *= a;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float w = __expf(ms[i] - mu);
          L += s0 + i < live ? w * ls[i] : 0.f;
          acc += w * os[i];
        }
        gm = nm;
      }
      p.out[(int64_t)b * p.o_sb + (int64_t)tt * p.o_st + (int64_t)(hkv * G + gg) * p.o_sh + d] = f2bf(L > 0.f ? acc / L : 0.f);
    }
    return stamp(1);
  }
  if constexpr (SYNC) {
    int* flg = reinterpret_cast<int*>(red_m);   // [0] lost, [1] merger: red_m is free once the waves are
                                                // merged (no static __shared__: it would shift the LDS base)
    float* of = reinterpret_cast<float*>(smem);   // [M][D] merged attention output
    float* wts = of + 16 * D;                     // [nsplit][16]
    const int ns = p.nsplit;
    const int64_t pb = (int64_t)bh * ns * M;
    float* mo = p.mo + (int64_t)bh * M * D;       // the head's merged output, handed to its other workgroups
    unsigned* cnt = p.sync_cnt + bh;
    unsigned* done = p.sync_cnt + kSyncHeads + bh;
    unsigned* flag = p.sync_cnt + 2 * kSyncHeads + bh;
    // publish: every storing wave drains its write-through partial stores, then one arrival per split;
    // the split whose arrival completes the count merges the head once
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      int merger = 0;
      if (split < ns) merger = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)ns - 1;
      flg[0] = 0;
      flg[1] = merger;
    }
    __syncthreads();
    if (flg[1]) {
      // every split's partial has arrived: merge (write-through / sc1 loads: no stale line from an
      // earlier launch), publish the merged rows write-through, then the head's flag
      for (int m = wid; m < M; m += NWV) {
        float gm = -INFINITY;
        for (int sp = lane; sp < ns; sp += 64)
          gm = fmaxf(gm, __hip_atomic_load(p.pm + pb + (int64_t)sp * M + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        gm = wave_max(gm);
        float L = 0.f;
        for (int sp = lane; sp < ns; sp += 64) {
          const float ms = __hip_atomic_load(p.pm + pb + (int64_t)sp * M + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const float w = ms == -INFINITY ? 0.f : __expf(ms - gm);
          wts[sp * 16 + m] = w;
          L += w * __hip_atomic_load(p.pl + pb + (int64_t)sp * M + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        L = wave_sum(L);
        const float inv = L > 0.f ? 1.f / L : 0.f;
        for (int sp = lane; sp < ns; sp += 64) wts[sp * 16 + m] *= inv;
      }
      __syncthreads();
      for (int it = tid; it < M * D; it += 64 * NWV) {
        const int m = it / D;
        const float* src = p.po + (pb + m) * D + it % D;
        const int64_t st = (int64_t)M * D;
        float acc = 0.f;
        int sp = 0;
        for (; sp + 3 < ns; sp += 4) {
          const float a0 = __hip_atomic_load(src + sp * st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const float a1 = __hip_atomic_load(src + (sp + 1) * st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const float a2 = __hip_atomic_load(src + (sp + 2) * st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const float a3 = __hip_atomic_load(src + (sp + 3) * st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          acc += wts[sp * 16 + m] * a0 + wts[(sp + 1) * 16 + m] * a1 + wts[(sp + 2) * 16 + m] * a2 + wts[(sp + 3) * 16 + m] * a3;
        }
        for (; sp < ns; ++sp) acc += wts[sp * 16 + m] * __hip_atomic_load(src + sp * st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const float v = bf2f(f2bf(acc));
        of[it] = v;
        __hip_atomic_store(mo + it, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      if (tid == 0) {
        for (unsigned spins = 0; __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u;) {
          __builtin_amdgcn_s_sleep(1);
          if (++spins > (1u << 24)) {   // ~0.5 s: the head's merge never arrived
            flg[0] = 1;
            __hip_atomic_store(p.sync_err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
        }
      }
      __syncthreads();
      const bool lost = flg[0] != 0;
      for (int it = tid; it < M * D; it += 64 * NWV)
        of[it] = lost ? __builtin_nanf("") : __hip_atomic_load(mo + it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();   // the merged rows are in LDS: this workgroup is done with the hand-off
    if (tid == 0) {
      const unsigned old = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old == (unsigned)p.R - 1) {   // the head's last workgroup: every peer has read the merged rows
        __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(flag, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if constexpr (FUSE) {
    __syncthreads();
    oproj_tail<D>(p, reinterpret_cast<const float*>(smem), wreg, b, row0, rpp, tpr, seg, G);
  }
  stamp(1);
}

// Keys of a split of a full cache: as many splits as bring the (batch, kv head, split) grid to ~NXD_DECODE_ATTN_WGS workgroups
// (default 512: two a CU, so that one's loads cover the other's arithmetic), of 128 keys (one pass of 4 waves; the caller's
// partial buffers hold Lmax / 128 splits) to 1,024.  Targets of 128 / 256 / 512 / 1,024: 11.4 / 9.9 / 8.8 / 9.8 us for 6 sequences of up
// to 1,024 keys of 8 heads of 64; 20.3 / 18.6 / 19.5 / 21.4 for 13 of up to 1,500 of 8 of 128; the same within 3 % for 1 and 4
// sequences; 24.2 / 25.3 at 512 / 1,024 for 32 of up to 2,048.
// Few heads of a long cache have fewer splits than that, since they have to be added up: 16, or where a head has no more than
// 256 sums 24 (merged by the last split) or 32.  8,000 keys of 8 heads in 64 / so many, us: 64 wide 18.3 / 12.2 with tickets, 12.6 /
// 11.9 without; 128 wide 27.5 / 16.0 and 17.8 / 15.8; four new tokens 40.6 / 15.9 and 68 / 20.9; with o_proj 128 wide 36.6 / 29.8,
// two new tokens 56.6 / 38.8.
// Short sequences in a large cache: 4 of 350-700 keys take 8.0 us with room for 1,024, 8,192 and 131,072 (9.9 by the share of a
// full cache), 13 of 750-1,500 19.9 / 20.6 with room for 1,792 / 8,192 (22.6), 8 of 2 heads of 750-1,500 9.1 in 16,384 (13.6).  Where the
// last split merges and 64 heads fill a quarter of the chip, 512 keys stay together: 16 of 250-500 8.4 us, in splits of 128 8.9.
static Splits splits_of(int Lmax, int B, int Hkv, int M, int D, bool tickets) {
  const int MD = M * D;
  if (tickets && Lmax <= 4608) {
    // 8 waves, one workgroup a CU: about 256 that have keys, at D 128 320 if all sequences were as long as the cache.  What such a call waits for
    // is the longest workgroup, and a merge costs 1-2 us: parts that are an eighth of a round too many cost more than parts that are
    // longer.  us by the rule below / here, sequences of 0.45 to 0.9 of the cache, 8 heads: D 64 4 of 2,304 keys 10.1 / 8.5, 6 of 1,280 9.3 / 8.2,
    // 8 of 2,304 11.2 / 10.3, 16 of 4,352 22.2 / 22.0, 32 of 640, 1,280, 2,304 11.0, 15.4, 23.0 / 8.9, 13.4, 20.8; D 128 1 of 4,352 11.8 / 9.6, 4 of
    // 1,756 13.0 / 10.5, 8 of 2,304 18.0 / 15.2, 13 of 1,756 20.1 / 17.6, 32 of 1,280 27.3 / 24.1; four new tokens, D 64, 16 of 1,280 14.9 / 12.5.
    // Not where two parts a head leave a sixth of the CUs idle and three are too many (D 64, 12 of 2,304 keys 13.1 / 13.7), nor where the call is
    // so short that 8 waves start later than 4 (1 of 640 6.7 / 7.3).  Whole heads of many keys only where the rule below gives a wave as many:
    // one long sequence among short ones is what the call waits for then (no more than 2,560 keys for 8 waves; D 128, 24 heads x 8 of 2,304 keys, all 36.0 / 32.5, one 18.5 / 26.8).
    // No more than about one workgroup a CU where all of them have keys, or a second round begins: with full parts of less than 320 keys (D 128, us in 320
    // workgroups / in 288 at most / by the rule below: 5 of 1,024 keys 13.0 / 9.8 / 11.7, 8 of 1,280 14.4 / 12.0 / 14.1, 13 of 768 14.2 / 12.5 / 13.8, 20
    // of 512 14.4 / 11.8 / 13.9; the last part half empty, 13 of 640 10.5 / 11.2 / 13.4), and where a launch of its own merges (more than 1,024 sums a head; four new tokens, 5 of 1,024 19.9 / 15.9 / 17.5, 8
    // of 1,280 22.4 / 18.5 / 20.2, 13 of 1,536 26.9 / 23.4 / 24.3; but two parts of 160 heads from 1,280 keys on, 20 of 1,756 29.9 / 31.3 by the rule
    // below).  There parts of 128 keys, half a chunk a wave, of more than 256 workgroups, or a last one that is mostly empty, are no better
    // than 4 waves: 7 of 640 17.5 / 16.4 by the rule below, 6 of 768 17.3 / 16.3, three new tokens 8 of 384 13.9 / 13.4.
    const int64_t heads = (int64_t)B * Hkv;
    const bool apart = MD > 1024;   // (merge_in_launch)
    const int least = D == 64 || heads >= 64 ? 256 : 128;
    auto parts = [&](int64_t wgs) { return D == 64 && Lmax <= 640 ? 1 : (int)std::min(std::max<int64_t>(1, wgs / heads), MD > 256 ? int64_t{16} : int64_t{24}); };
    auto keys = [&](int n) { return std::max(least, (ceil_div(Lmax, n) + KB - 1) / KB * KB); };
    int n = parts(D == 64 ? 270 : heads < 40 ? 256 : apart && (heads <= 144 || Lmax < 1280) ? 288 : 320), full = keys(n);
    if (n * heads > 288 && full < 320 && n * full < Lmax + full / 2) n = parts(288), full = keys(n);
    const bool idle = D == 64 && n == 2 && heads < 112, brief = D == 64 && heads < 32 && Lmax <= 1280;
    const bool uneven = n == 1 && heads < 224 && Lmax > (D == 64 ? 1280 : 640);
    const bool thin = apart && n > 1 && (full < 192 && n * heads > 256 || heads == 64 && Lmax <= 2 * full);
    if (full <= 2560 && !idle && !brief && !uneven && !thin) return {Lmax, full, std::min(full, heads >= 64 ? 512 : least), full, 8};
  }
  static const int target = [] {
    const char* e = getenv("NXD_DECODE_ATTN_WGS");
    const int v = e ? atoi(e) : 512;
    return v > 0 ? v : 512;
  }();
  const int64_t fill = ceil_div64((int64_t)Lmax * B * Hkv, target);
  const int n = (int)std::max<int64_t>(std::min<int64_t>(fill, Lmax), ceil_div(Lmax, MD > 256 ? 16 : tickets ? 24 : 32));
  const int full = std::max(128, (n + KB - 1) / KB * KB);
  return {Lmax, full, std::min(full, tickets && (int64_t)B * Hkv >= 64 ? 512 : 128), std::max(KPS, ceil_div(Lmax, KB * 64) * KB), WAVES};
}
static int most_splits(const Splits& sp) { return ceil_div(sp.room, std::min(sp.full, sp.most)); }

// Whether the last split merges: its trips to memory (8 splits at a time) come one after another, 0.7-1.2 us each, and a launch of
// its own takes about 4 us.  In the launch / apart, us: 2 trips 8.5 / 10.0, 3 trips 7.8 / 9.0, 4 trips 9.9 / 11.4 and 12.2 / 13.3, 6 trips
// 12.2 / 11.5, 8 trips 13.0 / 12.6 and 16.8 / 14.3, 12 trips 14.9 / 13.8, 64 trips (four tokens, 128 wide, 64 splits) 68 / 31.
// The trips counted are those of 4 waves, which these were; workgroups of 8 waves make half as many (few splits: 1-2 of them).
static bool merge_in_launch(int MD, const Splits& sp) { return ceil_div(MD, 64 * WAVES) * ceil_div(ceil_div(sp.room, sp.full), 8) <= 4; }

// Split attention's partials -> merged attention row block (bf16-rounded, as the merge kernel's
// output the o_proj GEMV would read) -> this workgroup's o_proj partial, fp32 atomics into oacc: the
// long-context form of FUSE (one launch instead of the merge + o_proj pair).  Grid (batch, kv head,
// R row chunks), the split weights of each query row in LDS.
// NP: passes over the workgroup's rows (p.NP; 0: read there).  Known, the loads of Wo behind the partials' are counted, and what comes first waits for the
// partials alone: the compiler's wait for an unknown number of loads was for all of them.
template <int D, int NWV, int NP>
__global__ void __launch_bounds__(64 * NWV) merge_oproj_kernel(Params p) {
  if (NP) p.NP = NP;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* of = reinterpret_cast<float*>(smem);   // [M][D] merged attention output
  float* wts = of + 16 * D;                     // [nsplit][16] normalised split weights
  const int tid = threadIdx.x;
  const int bh = (int)blockIdx.x / p.R, b = bh / p.Hkv, hkv = bh % p.Hkv;
  const int G = p.Hq / p.Hkv, M = G * p.T;
  const int tpr = (G * D) / 32, seg = tid % tpr, r0 = tid / tpr, rpp = (64 * NWV) / tpr;
  const int row0 = ((int)blockIdx.x % p.R) * (p.Hout / p.R) + r0;
  const int64_t pb = (int64_t)bh * p.nsplit * M;
  const int ns = p.nsplit, lane = tid & 63, wid = tid >> 6;
  // the splits are divided over H thread groups (partials summed through LDS); when a thread's share
  // fits in registers its partial-row loads are issued first, beside the stats loads below, so the
  // merge costs one memory round trip instead of two
  constexpr int PMAX = 16;
  const int elems = M * D, H = (64 * NWV) / elems >= 2 ? 2 : 1;
  const int64_t st = (int64_t)M * D;   // one split further
  const bool regs = elems * H <= 64 * NWV && (ns + H - 1) / H <= PMAX;
  const int e0 = tid % elems, h0 = tid / elems;
  const float* src0 = p.po + (pb + e0 / D) * D + e0 % D;
  float pv[PMAX];
  if (regs) {   // (past the last: the last again, not used)
#pragma unroll
    for (int c = 0; c < PMAX; c += 4)
      if (c * H < ns) {
#pragma unroll
        for (int i = c; i < c + 4; ++i) pv[i] = src0[(uint32_t)min(h0 + i * H, ns - 1) * (uint32_t)st];
      }
  }
  // split weights of query row m: one wave per row, one split per lane (all loads in parallel: a
  // serial walk over the splits was a chain of dependent L2 round trips, 7.8 us per launch).  The
  // stats are loaded before the Wo block, whose HBM latency then hides behind the merge (vmcnt
  // retires in issue order: issued first, Wo would gate the first use of the stats)
  constexpr int KM = (16 + NWV - 1) / NWV;   // rows per wave (M <= 16)
  const bool fast = regs && ns <= 64;
  float pmv[KM], plv[KM];
  if (fast) {
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const int m = wid + k * NWV;
      const bool ok = m < M && lane < ns;
      pmv[k] = ok ? p.pm[pb + (int64_t)lane * M + m] : -INFINITY;
      plv[k] = ok ? p.pl[pb + (int64_t)lane * M + m] : 0.f;
    }
  }
  u32x4_t wreg[4][4];
  load_wo_regs(p, row0, hkv * G * D + 32 * seg, rpp, wreg);
  if (fast) {
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const int m = wid + k * NWV;
      if (m >= M) break;   // wave-uniform
      float gm = pmv[k];
      gm = wave_max(gm);
      const float w = pmv[k] == -INFINITY ? 0.f : __expf(pmv[k] - gm);
      float L = w * plv[k];
      L = wave_sum(L);
      if (lane < ns) wts[lane * 16 + m] = L > 0.f ? w / L : 0.f;
    }
  } else for (int m = wid; m < M; m += NWV) {
    float gm = -INFINITY;
    for (int s = lane; s < ns; s += 64) gm = fmaxf(gm, p.pm[pb + (int64_t)s * M + m]);
    gm = wave_max(gm);
    float L = 0.f;
    for (int s = lane; s < ns; s += 64) {
      const float ms = p.pm[pb + (int64_t)s * M + m];
      const float w = ms == -INFINITY ? 0.f : __expf(ms - gm);
      wts[s * 16 + m] = w;
      L += w * p.pl[pb + (int64_t)s * M + m];
    }
    L = wave_sum(L);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    for (int s = lane; s < ns; s += 64) wts[s * 16 + m] *= inv;
  }
  __syncthreads();
  // weighted sum of the partial rows
  float* part = wts + ns * 16;   // [H][M * D]
  if (regs) {
    if (tid < elems * H) {
      const int m = e0 / D;
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < PMAX; ++i)
        if (h0 + i * H < ns) acc += wts[(h0 + i * H) * 16 + m] * pv[i];
      part[h0 * elems + e0] = acc;
    }
  } else for (int it = tid; it < elems * H; it += 64 * NWV) {   // four independent loads in flight per thread
    const int e = it % elems, h = it / elems, m = e / D, d = e % D;
    const float* src = p.po + (pb + m) * D + d;
    float acc = 0.f;
    int sp = h;
    for (; sp + 3 * H < ns; sp += 4 * H) {
      const float a0 = src[sp * st], a1 = src[(sp + H) * st], a2 = src[(sp + 2 * H) * st], a3 = src[(sp + 3 * H) * st];
      acc += wts[sp * 16 + m] * a0 + wts[(sp + H) * 16 + m] * a1 + wts[(sp + 2 * H) * 16 + m] * a2 +
             wts[(sp + 3 * H) * 16 + m] * a3;
    }
    for (; sp < ns; sp += H) acc += wts[sp * 16 + m] * src[sp * st];
    part[h * elems + e] = acc;
  }
  __syncthreads();
  for (int e = tid; e < elems; e += 64 * NWV) of[e] = bf2f(f2bf(H == 2 ? part[e] + part[elems + e] : part[e]));
  __syncthreads();
  oproj_tail<D>(p, of, wreg, b, row0, rpp, tpr, seg, G);
}

// Pending prefetch of the next decode_attn2 launch (set by decode_attn_set_prefetch, consumed by
// one launch: graph capture records the kernel arguments by value, so every captured layer keeps
// its own ranges).
static const void* g_pf[2] = {nullptr, nullptr};
static int64_t g_pf_bytes[2] = {0, 0};
static int g_pf_wgs = 0;

}  // namespace dattn

// Opt-in phase trace of the following decode attention launches (eager or captured: the pointer is
// recorded by value); null turns it off.  trace must hold 2 x (launch grid) uint64.
void decode_attn_set_trace(uint64_t* trace) { dattn::g_trace = trace; }

void decode_attn_set_prefetch(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes, int wgs) {
  dattn::g_pf[0] = a; dattn::g_pf_bytes[0] = a ? a_bytes : 0;
  dattn::g_pf[1] = b; dattn::g_pf_bytes[1] = b ? b_bytes : 0;
  dattn::g_pf_wgs = wgs;
}

// The plan of an attention without o_proj over a cache of Lmax keys: {splits, keys of a split of a sequence of len keys, whether
// the last split merges}
void decode_attn_plan(int Lmax, int B, int Hkv, int M, int D, int len, bool tickets, int* out) {
  const dattn::Splits sp = dattn::splits_of(Lmax, B, Hkv, M, D, tickets);
  out[0] = dattn::most_splits(sp);
  out[1] = sp.keys(len);
  out[2] = tickets && dattn::merge_in_launch(M * D, sp);
}

// Returns -1 when the shape is not covered (caller falls back to the 128-key-chunk kernel).
int decode_attn2_launch(const void* q, const int64_t* qs, const void* kc, const void* vc, const int64_t* cs,
                        const int* cache_idx, const int* seq_len, float* po, float* pm, float* pl, void* out,
                        const int64_t* os, int B, int T, int Hq, int Hkv, int D, int Lmax, float scale, int* nsplit_out,
                        hipStream_t stream, int* tickets = nullptr) {
  if (Hkv <= 0 || Hq % Hkv) return -1;
  const int M = (Hq / Hkv) * T;
  if (M > 16 || (D != 64 && D != 128)) return -1;
  dattn::Params p{};   // value-initialised: every field a launcher does not set is zero / null
  p.q = (const uint16_t*)q; p.q_sb = qs[0]; p.q_st = qs[1]; p.q_sh = qs[2];
  p.kc = (const uint16_t*)kc; p.vc = (const uint16_t*)vc;
  p.c_sb = cs[0]; p.c_sh = cs[1]; p.c_sl = cs[2];
  p.cache_idx = cache_idx; p.seq_len = seq_len;
  p.out = (uint16_t*)out; p.o_sb = os[0]; p.o_st = os[1]; p.o_sh = os[2];
  p.po = po; p.pm = pm; p.pl = pl;
  p.B = B; p.T = T; p.Hq = Hq; p.Hkv = Hkv;
  p.sp = dattn::splits_of(Lmax, B, Hkv, M, D, tickets != nullptr);
  p.nsplit = dattn::most_splits(p.sp);
  p.scale_log2 = scale * 1.4426950408889634f;
  *nsplit_out = p.nsplit;
  const int nwv = p.sp.waves;
  const size_t lds = (size_t)nwv * dattn::CHUNK * D * 2 + (size_t)2 * nwv * 16 * 4;
  p.tickets = dattn::merge_in_launch(M * D, p.sp) ? tickets : nullptr;
  if (p.tickets) *nsplit_out = 1;   // (nothing left to merge)
  p.attn_wgs = B * Hkv * p.nsplit;
  p.trace = dattn::g_trace;
  int pf_wgs = 0;
  for (int r = 0; r < 2; ++r) {
    // 16-B aligned start, whole chunks only (a prefetch never needs the ragged tail)
    const bool ok = dattn::g_pf[r] && (reinterpret_cast<uintptr_t>(dattn::g_pf[r]) & 15) == 0 && dattn::g_pf_bytes[r] >= 16;
    p.pf[r] = ok ? static_cast<const u32x4_t*>(dattn::g_pf[r]) : nullptr;
    p.pf_n16[r] = ok ? dattn::g_pf_bytes[r] / 16 : 0;
    if (ok) pf_wgs = dattn::g_pf_wgs > 0 ? dattn::g_pf_wgs : 256;
  }
  dattn::g_pf[0] = dattn::g_pf[1] = nullptr;
  dattn::g_pf_bytes[0] = dattn::g_pf_bytes[1] = 0;
  const dim3 grid(p.attn_wgs + pf_wgs), block(64 * nwv);
  auto* f = nwv == 8 ? (D == 64 ? &dattn::attn_kernel<64, 8, false> : &dattn::attn_kernel<128, 8, false>)
                     : (D == 64 ? &dattn::attn_kernel<64, dattn::WAVES, false> : &dattn::attn_kernel<128, dattn::WAVES, false>);
  (void)hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(f, grid, block, lds, stream, p);
  return (int)hipGetLastError();
}

namespace dattn {
int g_oproj_maxl = -1;   // NXD_DECODE_ATTN_OPROJ_MAXL, or decode_attn_set_oproj_maxl
int g_sync_on = -1;      // NXD_DECODE_ATTN_SYNC (default 0: measured slower), or decode_attn_set_sync
}
void decode_attn_set_sync(int v) { dattn::g_sync_on = v ? 1 : 0; }
void decode_attn_set_oproj_maxl(int v) { dattn::g_oproj_maxl = v; }

// Bounded-spin error word of the SYNC launches (a partial never arrived: that launch wrote NaN);
// reset clears it.  Synchronous (reads device memory).
int decode_attn_sync_error(bool reset) {
  int v = 0;
  (void)hipMemcpyFromSymbol(&v, HIP_SYMBOL(dattn::g_sync_err), sizeof(int), 0, hipMemcpyDeviceToHost);
  if (reset && v) {
    const int z = 0;
    (void)hipMemcpyToSymbol(HIP_SYMBOL(dattn::g_sync_err), &z, sizeof(int), 0, hipMemcpyHostToDevice);
  }
  return v;
}
int decode_attn_oproj_maxl() {
  if (dattn::g_oproj_maxl < 0) {
    const char* e = getenv("NXD_DECODE_ATTN_OPROJ_MAXL");
    dattn::g_oproj_maxl = e ? atoi(e) : 1024;
  }
  return dattn::g_oproj_maxl;
}

// Fused decode attention + o_proj (see FUSE above): oacc [B*T, Hout] fp32 must be zero on entry
// (the down projection's RESID epilogue re-zeroes it).  Returns -1 when the shape is not covered:
// cache capacity Lmax <= NXD_DECODE_ATTN_OPROJ_MAXL (default 1024: every workgroup of a kv head walks
// the whole cache; past that the split attention, whose keys per split fill the GPU, + merge + o_proj
// launches win -- 0.726 vs 0.774 ms/token at the notebook's 2,304-key cache,
// profiles/r6_decode/attn_split_ab.txt), M = G*T <= 16, D in {64, 128}, Wo blocks of <= 4 register
// passes.
int decode_attn_oproj_launch(const void* q, const int64_t* qs, const void* kc, const void* vc, const int64_t* cs,
                             const int* cache_idx, const int* seq_len, const void* wo, int64_t ldwo, int Hout, float* oacc,
                             float* po, float* pm, float* pl, float* mo, int B, int T, int Hq, int Hkv, int D, int Lmax,
                             float scale, hipStream_t stream) {
  if (Hkv <= 0 || Hq % Hkv) return -1;
  const int G = Hq / Hkv, M = G * T;
  const int maxl = decode_attn_oproj_maxl();
  // past maxl: split attention into the partials, then merge + o_proj (needs the partial buffers:
  // [B * Hkv * ceil(Lmax / 128) * M] rows of D, plus the two stats)
  const bool split = Lmax > maxl && po != nullptr && dattn::most_splits(dattn::splits_of(Lmax, B, Hkv, M, D, false)) > 1;
  if (M > 16 || (D != 64 && D != 128) || (Lmax > maxl && !split) || (G * D) % 32 || ldwo % 8) return -1;
  const int nwv = D == 64 ? 8 : 4;
  const int nt = 64 * nwv, tpr = (G * D) / 32;
  if (tpr > 64 || 64 % tpr || nt % tpr) return -1;
  const int rpp = nt / tpr;
  // row chunks per kv head: fill >= target workgroups (NXD_DECODE_OPROJ_WGS, default 256), at most 4
  // register passes per thread
  static const int target = [] {
    const char* e = getenv("NXD_DECODE_OPROJ_WGS");
    const int v = e ? atoi(e) : 256;
    return v > 0 ? v : 256;
  }();
  int R = 1;
  while ((int64_t)B * Hkv * R < target && Hout % (2 * R) == 0 && (Hout / (2 * R)) % rpp == 0) R *= 2;
  while (Hout % R == 0 && (Hout / R) % rpp == 0 && Hout / R / rpp > 4 && Hout % (2 * R) == 0 && (Hout / (2 * R)) % rpp == 0)
    R *= 2;
  if (Hout % R || (Hout / R) % rpp || Hout / R / rpp > 4 || Hout / R / rpp < 1) return -1;
  dattn::Params p{};
  p.q = (const uint16_t*)q; p.q_sb = qs[0]; p.q_st = qs[1]; p.q_sh = qs[2];
  p.kc = (const uint16_t*)kc; p.vc = (const uint16_t*)vc;
  p.c_sb = cs[0]; p.c_sh = cs[1]; p.c_sl = cs[2];
  p.cache_idx = cache_idx; p.seq_len = seq_len;
  p.B = B; p.T = T; p.Hq = Hq; p.Hkv = Hkv; p.nsplit = 1;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.wo = (const uint16_t*)wo; p.ldwo = ldwo; p.oacc = oacc; p.Hout = Hout; p.R = R; p.NP = Hout / R / rpp;
  p.attn_wgs = B * Hkv * R;
  p.trace = dattn::g_trace;
  const dim3 grid(p.attn_wgs), block(nt);
  if (dattn::g_sync_on < 0) {
    const char* e = getenv("NXD_DECODE_ATTN_SYNC");
    dattn::g_sync_on = e ? (atoi(e) != 0) : 0;
  }
  const bool sync_on = dattn::g_sync_on != 0;
  static const int n_cu = [] {
    int dev = 0, n = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    return n;
  }();
  if (split && sync_on && mo != nullptr && B * Hkv <= dattn::kSyncHeads && (int)grid.x <= n_cu) {
    // one launch: workgroup r of a head computes key split r (>= 128 keys, the partial buffers hold
    // Lmax / 128 splits), then merges the head's splits and runs its o_proj slice (SYNC above)
    int kps = (Lmax + R - 1) / R;
    kps = (kps + dattn::KB - 1) / dattn::KB * dattn::KB;
    kps = kps < 128 ? 128 : kps;
    const int ns = (Lmax + kps - 1) / kps;
    const size_t lds = (size_t)nwv * dattn::KB * D * 2 + (size_t)nwv * 16 * D * 4 + (size_t)2 * nwv * 16 * 4;
    if (ns <= R && (size_t)16 * D * 4 + (size_t)ns * 16 * 4 <= (size_t)nwv * dattn::KB * D * 2) {
      static unsigned* cnt = [] { void* a = nullptr; (void)hipGetSymbolAddress(&a, HIP_SYMBOL(dattn::g_sync_cnt)); return (unsigned*)a; }();
      static int* err = [] { void* a = nullptr; (void)hipGetSymbolAddress(&a, HIP_SYMBOL(dattn::g_sync_err)); return (int*)a; }();
      p.kps = kps; p.nsplit = ns; p.po = po; p.pm = pm; p.pl = pl; p.sync_cnt = cnt; p.sync_err = err;
      p.mo = mo;
      if (D == 64) {
        (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<64, 8, true, true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        hipLaunchKernelGGL((dattn::attn_kernel<64, 8, true, true, true>), grid, block, lds, stream, p);
      } else {
        (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<128, 4, true, true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        hipLaunchKernelGGL((dattn::attn_kernel<128, 4, true, true, true>), grid, block, lds, stream, p);
      }
      return (int)hipGetLastError();
    }
  }
  if (split) {
    const int ns = dattn::most_splits(dattn::splits_of(Lmax, B, Hkv, M, D, false));
    const size_t mlds = (size_t)16 * D * 4 + (size_t)ns * 16 * 4 + (size_t)2 * 16 * D * 4;
    if (mlds > 64 * 1024) return -1;
    int ns2 = 0;
    const int64_t no_out[3] = {0, 0, 0};
    const int rc = decode_attn2_launch(q, qs, kc, vc, cs, cache_idx, seq_len, po, pm, pl, nullptr, no_out, B, T, Hq, Hkv,
                                       D, Lmax, scale, &ns2, stream);
    if (rc != 0) return rc;
    if (ns2 != ns) return 3;   // the attention launch split differently: never write the output through null
    p.nsplit = ns; p.po = po; p.pm = pm; p.pl = pl;
    auto* f = D == 64 ? (p.NP == 1 ? &dattn::merge_oproj_kernel<64, 8, 1> : p.NP == 2 ? &dattn::merge_oproj_kernel<64, 8, 2>
                                     : p.NP == 4 ? &dattn::merge_oproj_kernel<64, 8, 4> : &dattn::merge_oproj_kernel<64, 8, 0>)
                      : (p.NP == 1 ? &dattn::merge_oproj_kernel<128, 4, 1> : p.NP == 2 ? &dattn::merge_oproj_kernel<128, 4, 2>
                                     : p.NP == 4 ? &dattn::merge_oproj_kernel<128, 4, 4> : &dattn::merge_oproj_kernel<128, 4, 0>);
    (void)hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mlds);
    hipLaunchKernelGGL(f, grid, block, mlds, stream, p);
    return (int)hipGetLastError();
  }
  const size_t lds = (size_t)nwv * dattn::KB * D * 2 + (size_t)nwv * 16 * D * 4 + (size_t)2 * nwv * 16 * 4;
  static const bool wo_late = [] {
    const char* e = getenv("NXD_DECODE_WO_LATE");
    return e ? atoi(e) != 0 : true;
  }();
  if (D == 64) {
    if (wo_late) {
      (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<64, 8, true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((dattn::attn_kernel<64, 8, true, true>), grid, block, lds, stream, p);
    } else {
      (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<64, 8, true, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((dattn::attn_kernel<64, 8, true, false>), grid, block, lds, stream, p);
    }
  } else {
    if (wo_late) {
      (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<128, 4, true, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((dattn::attn_kernel<128, 4, true, true>), grid, block, lds, stream, p);
    } else {
      (void)hipFuncSetAttribute((const void*)dattn::attn_kernel<128, 4, true, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((dattn::attn_kernel<128, 4, true, false>), grid, block, lds, stream, p);
    }
  }
  return (int)hipGetLastError();
}

}  // namespace nxd
