// y[M, N] = epilogue(x[M, K] w[N, K]^T) for 1 to 32 activation rows, bf16 or int8 weights: the projections of a decode
// step, each one launch with the element-wise work around it (RMSNorm of the input, residual add, SwiGLU, rotary
// positions and cache write, squared ReLU, capped fp32 logits).
//
// What bounds it is reading the weights once.  So weights go from memory straight to LDS (no registers
// held while they are on the way), 256 contiguous bytes (int8: 128) of a row at a time -- whole lines --, with several
// stages of every wave under way; the row pieces are stored rotated (XOR of the piece's number with the row's), so that
// the MFMA operands (16 rows x 16 bytes) are read back without bank conflicts.  A workgroup has tiles of R weight rows;
// its waves take 128 elements of the reduction in turn, and their sums meet in LDS, where a wave of its own finishes
// them (epilogue reads and stores never wait for weights, nor weights for them).  The activations are the other operand of
// v_mfma_f32_16x16x32_bf16.  What a CU gets from the caches is about what it gets from memory, so activations count
// like weights: they are read in operand order once a workgroup and kept in registers over its tiles where they fit.
// RMSNorm costs no pass over the rows: the products are those of bf16(x g), the sums of squares come from the same
// operands, and 1 / rms is a factor of the finished sums.  int8 weights are widened exactly (to bf16) on their way from LDS.
#include "few_rows.h"

#include <atomic>
#include <type_traits>

namespace nxd {
namespace few {

constexpr int KC = 128;   // reduction elements of a stage

// What a wave waits for.  Loads end in their order, so a wave that waits for its activations (in registers: the compiler places the wait) also waits for
// every load before them, and for as many after them as the compiler does not know of or, across a branch, is not sure of.  So weights are loaded by a
// builtin (as asm they were not counted: a streaming wave waited for all its stages whenever it came round to the first, 4096 x 4096 at 5 rows
// 8.7 -> 7.8 us, 2048 x 8192 at 4 rows 8.8 -> 8.1), a buffer load (global_load_lds counts as an access to both memories, after which the compiler
// waits for everything), in straight lines of whole rounds; and since the compiler lets an access to LDS that it sees wait for all such
// loads, the accesses of waves that stream weights are asm.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t base, uint32_t at, uint32_t lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(base, (__attribute__((address_space(3))) void*)(uintptr_t)lds, 16, (int)at, 0, 0, 2 /* nt */);
}
__device__ __forceinline__ void dma16_uncounted(const void* base, uint32_t at, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(at), "s"(base), "s"(lds)
               : "memory");
}
__device__ __forceinline__ void lds_read(u32x4_t (&v)[4], const uint32_t (&at)[4]) {
  asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
               : "memory");
}
__device__ __forceinline__ void lds_read(u32x4_t (&v)[2], const uint32_t (&at)[2]) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]), "=&v"(v[1]) : "v"(at[0]), "v"(at[1]) : "memory");
}
__device__ __forceinline__ void lds_write(uint32_t at, const f32x4_t& v) { asm volatile("ds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory"); }
// (the result of a matrix product: asm has to wait for it by itself, 8 wait states after 4 passes; these are 16)
__device__ __forceinline__ void lds_write_sum(uint32_t at, const f32x4_t& v) { asm volatile("s_nop 15\n\tds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_write(uint32_t at, float v) { asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory"); }
__device__ __forceinline__ uint32_t lds_at(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }

// int8 x 8 -> bf16 x 8 (exact)
__device__ __forceinline__ u32x4_t widen8(uint32_t lo, uint32_t hi) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = (float)(int8_t)(lo >> (8 * i));
    f[4 + i] = (float)(int8_t)(hi >> (8 * i));
  }
  return pack8(f);
}

// weight row r of a tile
template <int EPI, int R>
__device__ __forceinline__ int row_of(const FewRowsParams& p, int tile, int r) {
  constexpr int HR = R / 2;
  if (EPI == FEW_GLU) return min(tile * HR + (r & (HR - 1)), p.N - 1) + (r < HR ? 0 : p.N);
  if (EPI == FEW_ROPE_KV) {
    const int half = p.D / 2, qk = (p.nq + p.nkv) * (half / HR);
    if (tile < qk) return tile / (half / HR) * p.D + tile % (half / HR) * HR + (r & (HR - 1)) + (r < HR ? 0 : half);
    return min((p.nq + p.nkv) * p.D + (tile - qk) * R + r, p.N - 1);
  }
  return min(tile * R + r, p.N - 1);
}

// Geometry of a workgroup: NW waves that stream weights and FW that finish tiles; R weight rows a tile; MT tiles of 16
// activation rows (the grid's second dimension has the rest of M); D stages of a wave under way; CW chunks of the reduction a wave, their activations held in registers for
// all tiles (0: any number, activations streamed beside the weights)
template <int R, int MT, bool I8, int NW, int CW, int D>
struct Shape {
  static constexpr int GC = CW > 0 ? CW : 2;             // chunks of a wave with a norm
  static constexpr int ROWB = I8 ? KC : 2 * KC;          // bytes of a row in a stage
  static constexpr int STAGE = R * ROWB;                 // bytes of a stage of a wave
  static constexpr int DMAS = STAGE / 1024;              // loads of a stage
  static constexpr int RING = NW * D * STAGE;
  static constexpr int PART = NW * MT * 64 * 16;         // the waves' sums of a tile
  static constexpr int SQ = NW * MT * 16 * 4;            // the waves' sums of squares
  static constexpr int G = CW > 0 ? 0 : NW * GC * 256;   // the waves' parts of the norm's weight (CW > 0: in their parts of PART, where they wait for no more than one tile)
  static constexpr int FW = NW + MT > 12 ? 1 : MT;       // waves that finish tiles (12 waves leave each 168 registers)
};

// all loads but those of the newest n stages have come (OPS loads a stage, n < D)
template <int OPS, int D, int N = D - 1>
__device__ __forceinline__ void wait_stages(int n) {
  static_assert(OPS * (D - 1) < 64, "the counter has 6 bits");
  if constexpr (N > 0) {
    if (n >= N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OPS * N) : "memory");
    else wait_stages<OPS, D, N - 1>(n);
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

__device__ __forceinline__ void meet() {   // LDS writes are there; loads from memory stay under way
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The input rows: row m is x[m], or the table's row xidx[m] (as zeros for an id outside it)
template <bool XI>
__device__ __forceinline__ uint32_t input_row(const FewRowsParams& p, int m, bool& ok) {   // element offset
  ok = true;
  if constexpr (XI) {
    const int64_t id = p.xidx[m];
    ok = id >= 0 && id < p.xrows;
    return (uint32_t)((id < 0 ? 0 : id >= p.xrows ? p.xrows - 1 : id) * p.ldx);
  } else {
    return (uint32_t)(m * p.ldx);
  }
}

// The wave that finishes row tile t of every weight tile: sums of the streaming waves -> epilogue.  Lane (c, q) has
// activation row m = 16 t + c and weight rows 4 q .. 4 q + 3 of the tile (R == 8: q < 2, the rest are copies).
template <int EPI, bool NORM, int R, bool I8>
struct Finish {
  static constexpr int HR = R / 2;
  const FewRowsParams& p;
  const int lane, q, m, half;
  const bool live, wide, wide_c;   // a row that is there; its 4 values go out in one store (also to the cache)
  int row, tile, n;
  bool rot;
  float rstd;
  uint16_t y_pre[4];
  float cs[4], sn[4], scale[4];
  int64_t at, slot;

  __device__ __forceinline__ Finish(const FewRowsParams& p_, int lane_, int m0)
      : p(p_), lane(lane_), q(lane_ >> 4), m(min(m0 + (lane_ & 15), p_.M - 1)), half(p_.D / 2), live(m0 + (lane_ & 15) < p_.M),
        wide(p_.ldy % 4 == 0 && (EPI == FEW_F32 ? (uintptr_t)p_.yf % 16 : (uintptr_t)p_.y % 8) == 0),
        wide_c(EPI == FEW_ROPE_KV && (p_.c_sb | p_.c_sh | p_.c_sl) % 4 == 0 && ((uintptr_t)p_.kc | (uintptr_t)p_.vc) % 8 == 0) {
    if (EPI == FEW_ROPE_KV) {
      at = p.pos[m];
      slot = p.cache_idx ? p.cache_idx[m / p.T] : m / p.T;
    }
  }

  template <int NW>
  __device__ __forceinline__ void squares(const float* sq, int stride) {   // 1 / rms of the row
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) s += sq[i * stride];
    rstd = rsqrtf(s / (float)p.K + p.eps);
  }

  __device__ __forceinline__ void fetch(int tile_) {   // what the epilogue reads, before the sums are there
    tile = tile_;
    const int r = (4 * q) & (R - 1);
    row = row_of<EPI, R>(p, tile, r);
    rot = EPI == FEW_ROPE_KV && tile < (p.nq + p.nkv) * (half / HR);
    n = EPI == FEW_GLU ? tile * HR + (r & (HR - 1)) : EPI == FEW_ROPE_KV ? row : tile * R + r;
    if (I8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) scale[i] = p.wscale[row_of<EPI, R>(p, tile, r + i) * p.ws_stride];
    }
    if (EPI == FEW_RESID) {
      const uint16_t* y = p.y + (int64_t)m * p.ldy;
      if (wide && n + 4 <= p.N) {
        const u32x2_t v = *reinterpret_cast<const u32x2_t*>(y + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) y_pre[i] = (uint16_t)(v[i >> 1] >> (16 * (i & 1)));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) y_pre[i] = y[min(n + i, p.N - 1)];
      }
    }
    if (rot) {
      const int64_t a = (at < 0 ? 0 : at >= p.max_pos ? p.max_pos - 1 : at) * half + (row % p.D) % half;
      const f32x4_t cv = *reinterpret_cast<const f32x4_t*>(p.cos_t + a), sv = *reinterpret_cast<const f32x4_t*>(p.sin_t + a);
#pragma unroll
      for (int i = 0; i < 4; ++i) cs[i] = cv[i], sn[i] = sv[i];
    }
  }

  __device__ __forceinline__ void put(uint16_t* to, const uint16_t (&o)[4], int left, bool whole) const {   // `left` of the 4 values are there
    if (whole && left >= 4) {
      *reinterpret_cast<u32x2_t*>(to) = u32x2_t{(uint32_t)o[0] | (uint32_t)o[1] << 16, (uint32_t)o[2] | (uint32_t)o[3] << 16};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < left) to[i] = o[i];
    }
  }

  // A part of the reduction: its sums go through to memory (every part has a place of its own) ...
  __device__ __forceinline__ float* parts(int at) const { return p.ws + (int64_t)at * p.splits * 256 + lane; }
  __device__ __forceinline__ void leave(const f32x4_t& v, int at) const {
    float* ws = parts(at) + blockIdx.x % p.splits * 256;
#pragma unroll
    for (int i = 0; i < 4; ++i) __hip_atomic_store(ws + 64 * i, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // ... and are added up in the parts' order, whichever comes last
  __device__ __forceinline__ f32x4_t collect(int at) const {
    const float* ws = parts(at);
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < p.splits; j0 += 8) {   // 8 parts in flight together
      f32x4_t u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) u[j][i] = __hip_atomic_load(ws + min(j0 + j, p.splits - 1) * 256 + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j0 + j < p.splits) v += u[j];
    }
    return v;
  }

  __device__ __forceinline__ void finish(f32x4_t v) {
    if (NORM) v *= rstd;
    if (I8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] *= scale[i];
    }
    f32x4_t other;   // the pairs' other halves: HR rows away
    if (EPI == FEW_GLU || EPI == FEW_ROPE_KV) {
#pragma unroll
      for (int i = 0; i < 4; ++i) other[i] = __shfl_xor(v[i], 16 * (HR / 4), 64);
    }
    if (!live || 4 * q >= (EPI == FEW_GLU ? HR : R)) return;
    uint16_t o[4];
    if (EPI == FEW_F32) {
      float* y = p.yf + (int64_t)m * p.ldy + n;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float z = v[i] * p.alpha;
        v[i] = p.cap > 0.f ? p.cap * tanhf(z / p.cap) : z;
      }
      if (wide && n + 4 <= p.N) {
        *reinterpret_cast<f32x4_t*>(y) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < p.N) y[i] = v[i];
      }
      return;
    }
    const bool first = 4 * q < HR;   // of the pairs' halves
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (EPI == FEW_GLU) {
        o[i] = f2bf(v[i] / (1.f + __expf(-v[i])) * other[i]);
      } else if (EPI == FEW_RESID) {
        o[i] = f2bf(bf2f(y_pre[i]) + bf2f(f2bf(v[i])));
      } else if (EPI == FEW_RELU2) {
        o[i] = f2bf(fmaxf(v[i], 0.f) * fmaxf(v[i], 0.f));
      } else if (EPI == FEW_ROPE_KV && rot) {
        const float one = bf2f(f2bf(v[i])), two = bf2f(f2bf(other[i]));   // bf16 projection outputs
        o[i] = f2bf(first ? one * cs[i] - two * sn[i] : one * cs[i] + two * sn[i]);
      } else {
        o[i] = f2bf(v[i]);
      }
    }
    if (EPI == FEW_ROPE_KV) {
      const int qk_rows = (p.nq + p.nkv) * p.D;
      const int left = rot ? 4 : p.N - (qk_rows + (tile - (p.nq + p.nkv) * (half / HR)) * R + 4 * q);
      if (left <= 0) return;
      put(p.y + (int64_t)m * p.ldy + row, o, left, wide);
      const int vr = row - (rot ? p.nq * p.D : qk_rows);   // of the keys, or of the values
      if (vr < 0 || at < 0 || at >= p.Lmax) return;
      put((rot ? p.kc : p.vc) + slot * p.c_sb + (int64_t)(vr / p.D) * p.c_sh + at * p.c_sl + vr % p.D, o, left, wide_c);
    } else {
      if (n < p.N) put(p.y + (int64_t)m * p.ldy + n, o, p.N - n, wide);
    }
  }
};

// FULL: all that is loaded ahead is used: with CW > 0 a wave has D stages or more, with CW = 0 a workgroup has one tile and every wave whole rounds of D
// stages.  Then loads need no branch and are counted (above); else loads under a branch, which are not, are faster than some that nothing uses.  us, all
// counted and both ways in one kernel / apart: 32000 x 512 at 8 rows 9.6 / 9.0, 8192 x 512 at 16 5.6 / 4.9, 1024 x 1536 at 8 3.8 / 3.7, int8 8192 x
// 3072 at 6 11.2 / 9.7, with a norm 3072 x 1024 at 8 4.6 / 4.3
template <int EPI, bool NORM, bool XI, int R, int MT, bool I8, int NW, int CW, int D, bool SPLIT, bool HALF, bool FULL>
__global__ void __launch_bounds__((NW + Shape<R, MT, I8, NW, CW, D>::FW) * 64) kernel(FewRowsParams p, int tiles, int per, int step) {
  using S = Shape<R, MT, I8, NW, CW, D>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // (what the first loads need, asked for at once: asked for where it is used, it came in two or three trips one after the other: 1024 x 4096 at 4 rows 4.3
  // -> 4.2 us, 8192 x 4096 14.4 -> 14.0)
  asm volatile("" ::"s"(p.x), "s"(p.w), "s"(p.ldx), "s"(p.ldw), "s"(p.M), "s"(p.N), "s"(p.K), "s"(tiles), "s"(per), "s"(step));
  f32x4_t* part = reinterpret_cast<f32x4_t*>(smem + S::RING);       // [NW][MT][64]
  float* sq = reinterpret_cast<float*>(smem + S::RING + S::PART);   // [NW][16 MT]
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, q = lane >> 4, m0 = SPLIT ? 0 : blockIdx.y * (HALF ? p.half : 16 * MT);   // its first row
  if constexpr (HALF) p.M = min(p.M, m0 + p.half);
  static_assert(!SPLIT || (CW > 0 && !NORM), "split reductions hold their activations and need no norm");
  // its tiles: per of them next to each other, or (1) one of each round
  const int group = SPLIT ? blockIdx.x / p.splits : blockIdx.x, tile0 = group * per;
  tiles = min(tiles, per > 1 ? tile0 + per : tiles);

  // SPLIT: all waves of a workgroup share the tiles of which its part was the last to come
  auto finish_last = [&]() {
    meet();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");   // (keeps the loads below the tickets)
    int turn = 0;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      Finish<EPI, NORM, R, I8> f(p, lane, 16 * t);
      uint64_t todo = reinterpret_cast<const uint64_t*>(sq)[t];
      for (todo = (uint64_t)__builtin_amdgcn_readfirstlane((int)(todo >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)todo);
           todo; todo &= todo - 1, ++turn) {
        if (turn % (NW + S::FW) != w) continue;
        const int tile = tile0 + __builtin_ctzll(todo) * step;
        f.fetch(tile);
        f.finish(f.collect(tile * MT + t));
      }
    }
  };

  // Twice a tile all waves meet: when `part` is free, and when it is full
  if (w >= NW) {
    constexpr int T = MT / S::FW;
    Finish<EPI, NORM, R, I8> f0(p, lane, m0 + 16 * (w - NW) * T);
    Finish<EPI, NORM, R, I8> f1(p, lane, m0 + 16 * ((w - NW) * T + T - 1));
    for (int tile = tile0; tile < tiles; tile += step) {
      if (!SPLIT) {
        f0.fetch(tile);
        if (T > 1) f1.fetch(tile);
      }
      meet();
      meet();
      if (NORM && tile == tile0) {
        const float* mine = sq + (w - NW) * T * 16 + c;
        f0.template squares<NW>(mine, 16 * MT);
        if (T > 1) f1.template squares<NW>(mine + 16, 16 * MT);
      }
      const f32x4_t* mine = part + (w - NW) * T * 64 + lane;
      f32x4_t v = mine[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) v += mine[i * MT * 64];
      f32x4_t u;
      if (T > 1) {
        u = mine[64];
#pragma unroll
        for (int i = 1; i < NW; ++i) u += mine[(i * MT + 1) * 64];
      }
      if constexpr (SPLIT) {
        f0.leave(v, tile * MT + (w - NW) * T);
        if (T > 1) f1.leave(u, tile * MT + (w - NW) * T + 1);
      } else {
        f0.finish(v);
        if (T > 1) f1.finish(u);
      }
    }
    if constexpr (SPLIT) {   // lane j: a ticket of the j-th tile; the last part to take one finishes the tile
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int mt = (w - NW) * T + t, mine = (tile0 + lane * step) * MT + mt;
        int n = -1;
        if (tile0 + lane * step < tiles) n = __hip_atomic_fetch_add(p.tickets + mine, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = n == p.splits - 1;
        if (last) __hip_atomic_store(p.tickets + mine, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t todo = __ballot(last);
        if (lane == 0) reinterpret_cast<uint64_t*>(sq)[mt] = todo;
      }
      finish_last();
    }
    return;
  }

  const int nck = (p.K + KC - 1) / KC;
  int c0 = 0, c1 = nck;   // chunks of this workgroup
  if (SPLIT) {
    const int part = blockIdx.x % p.splits, n = (nck + p.splits - 1) / p.splits;
    c0 = min(part * n, nck), c1 = min(c0 + n, nck);
  }
  const int wc = c0 + w, cw = (c1 - wc + NW - 1) / NW;   // of this wave: wc, wc + NW, ...
  char* ring = smem + w * D * S::STAGE;
  const uint32_t ring_at = lds_at(ring);

  // ---- this lane's input rows (rows past M repeat the last one: their sums are not stored)
  uint32_t xrow[MT];   // (element offsets: the rows lie within 4 GB)
  bool xok[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xrow[t] = input_row<XI>(p, min(m0 + 16 * t + c, p.M - 1), xok[t]);
  // element of operand f of a chunk that this lane starts at
  auto kof = [&](int f) { return I8 ? 64 * (f >> 1) + 16 * q + 8 * (f & 1) : 32 * f + 8 * q; };
  auto load_x = [&](u32x4_t (&xv)[MT][4], int chunk) {
#pragma unroll
    for (int t = 0; t < MT; ++t)   // (both halves of a line one after the other)
#pragma unroll
      for (int f = 0; f < 4; ++f) xv[t][f] = *reinterpret_cast<const u32x4_t*>(p.x + (xrow[t] + (uint32_t)min(chunk * KC + kof(f), p.K - 8)));
  };
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) ss[t] = 0.f;
  // raw rows -> operands: zeros past the end; NORM: times the weight, with the squares summed the first time (1 / rms is
  // a factor of the sums)
  auto ready_x = [&](u32x4_t (&xv)[MT][4], const u32x4_t (&g)[4], int chunk, bool first) {
    const bool tail = (chunk + 1) * KC > p.K;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int k = chunk * KC + kof(f);
        u32x4_t v = xv[t][f];
        if (XI && !xok[t]) v = u32x4_t{0u, 0u, 0u, 0u};
        if (tail && k >= p.K) v = u32x4_t{0u, 0u, 0u, 0u};
        if (XI && first && p.xcopy && blockIdx.x == 0 && m0 + 16 * t + c < p.M && k < p.K)
          *reinterpret_cast<u32x4_t*>(p.xcopy + (int64_t)(m0 + 16 * t + c) * p.K + k) = v;
        if (NORM) {
          if (first) ss[t] = dot8_bf16(v, v, ss[t]);
          float a[8], b[8];
          unpack8(v, a);
          unpack8(g[f], b);
#pragma unroll
          for (int j = 0; j < 8; ++j) a[j] *= b[j];
          v = pack8(a);
        }
        xv[t][f] = v;
      }
  };

  // ---- weights: the next stage to issue
  uint32_t wrow[S::DMAS];   // (byte offsets: the weights take less than 4 GB)
  int it = tile0, ic = 0, is = 0, ahead = 0;   // its tile, chunk and place in the ring; stages under way
  // Every workgroup begins elsewhere in the reduction: rows lie a power of two apart, and the same piece of all of
  // them for all workgroups at a time is one channel's work
  const int rot = CW == 0 && cw > 0 ? blockIdx.x % cw : 0;
  auto order = [&](int i) {
    if (CW > 0) return i;
    const int j = i + rot;
    return j < cw ? j : j - cw;
  };
  auto start = [&](auto counted) {
    asm volatile("" ::: "memory");   // (in this order: waits count what came later)
    if (ic == 0) {
#pragma unroll
      for (int j = 0; j < S::DMAS; ++j) {
        const int r = I8 ? 8 * j + (lane >> 3) : 4 * j + (lane >> 4);
        wrow[j] = (uint32_t)row_of<EPI, R>(p, min(it, tiles - 1), r) * (uint32_t)p.ldw * (I8 ? 1 : 2);
      }
    }
    const int chunk = wc + order(ic) * NW;
    // (past the last stage, of a last workgroup or part: a range of nothing is not read)
    const __amdgpu_buffer_rsrc_t wbase = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.w), 0, CW > 0 && (it >= tiles || cw <= 0) ? 0 : -1, 0x00020000);
#pragma unroll
    for (int j = 0; j < S::DMAS; ++j) {
      int seg;   // the piece of the row that goes to this lane's place
      if (I8) {
        const int r = 8 * j + (lane >> 3);
        seg = (lane & 7) ^ ((r >> 1) & 7);
      } else {
        const int r = 4 * j + (lane >> 4);
        seg = (lane & 15) ^ (r & 15);
      }
      const uint32_t at = min(chunk * S::ROWB + 16 * seg, p.K * (I8 ? 1 : 2) - 16);
      const uint32_t to = __builtin_amdgcn_readfirstlane(ring_at + is * S::STAGE + j * 1024);
      if constexpr (counted.value) dma16(wbase, wrow[j] + at, to);
      else dma16_uncounted(p.w, wrow[j] + at, to);
    }
    asm volatile("" ::: "memory");
    ++ahead;
    if (++ic == cw) ic = 0, it += step;
    if (++is == D) is = 0;
  };
  auto issue = [&](auto counted) {
    if (it < tiles && cw > 0) start(counted);
  };

  f32x4_t acc[MT];
  int cs = 0;   // place in the ring of the stage to use
  uint32_t wat[I8 ? 2 : 4];   // its pieces, as this lane's operands, in the first place
#pragma unroll
  for (int i = 0; i < (I8 ? 2 : 4); ++i) {
    const int r = c & (R - 1);
    wat[i] = ring_at + r * S::ROWB + (((4 * i + q) ^ (I8 ? (r >> 1) & 7 : r & 15)) << 4);
  }
  auto take = [&](u32x4_t (&wf)[I8 ? 2 : 4]) {   // (the place may be filled again)
    uint32_t at[I8 ? 2 : 4];
#pragma unroll
    for (int i = 0; i < (I8 ? 2 : 4); ++i) at[i] = wat[i] + cs * S::STAGE;
    lds_read(wf, at);
    --ahead;
    if (++cs == D) cs = 0;
  };
  auto look = [&](u32x4_t (&wf)[I8 ? 2 : 4]) {   // the same, of loads that are not counted
#pragma unroll
    for (int i = 0; i < (I8 ? 2 : 4); ++i) wf[i] = *reinterpret_cast<const u32x4_t*>(ring + (wat[i] - ring_at) + cs * S::STAGE);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    --ahead;
    if (++cs == D) cs = 0;
  };
  auto multiply = [&](const u32x4_t (&wf)[I8 ? 2 : 4], const u32x4_t (&xv)[MT][4]) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      u32x4_t b;
      if constexpr (I8) b = widen8(wf[f >> 1][2 * (f & 1)], wf[f >> 1][2 * (f & 1) + 1]);
      else b = wf[f];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, xv[t][f]), acc[t], 0, 0, 0);
    }
  };
  auto clear = [&]() {
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  // NORM: the weight of this wave's chunks, 16 lanes a chunk, turned into operands through LDS of its own
  const uint32_t gs = CW > 0 ? lds_at(part + w * MT * 64) : lds_at(smem + S::RING + S::PART + S::SQ) + w * S::GC * 256;
  auto load_g = [&]() {
    u32x4_t v = {0u, 0u, 0u, 0u};
    if constexpr (NORM) v = *reinterpret_cast<const u32x4_t*>(p.norm_w + min((wc + min(q, S::GC - 1) * NW) * KC + 8 * c, p.K - 8));
    return v;
  };
  auto keep_g = [&](const u32x4_t& v) {
    static_assert(S::GC <= 4 && (CW == 0 || CW * 256 <= MT * 1024), "16 lanes a chunk");
    if (NORM && q < S::GC) lds_write(gs + 16 * lane, __builtin_bit_cast(f32x4_t, v));
  };
  auto read_g = [&](u32x4_t (&g)[4], int i) {   // of the wave's i-th chunk
    if constexpr (NORM) {
      uint32_t at[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) at[f] = gs + i * 256 + 2 * kof(f);
      lds_read(g, at);
    }
  };
  auto squares = [&]() {
    if (!NORM) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      float v = ss[t];
      v = lanes_add<32>(lanes_add<16>(v));
      if (q != 0) continue;
      if constexpr (FULL) lds_write(lds_at(sq + w * 16 * MT + 16 * t + c), v);
      else sq[w * 16 * MT + 16 * t + c] = v;
    }
  };
  auto publish = [&]() {
    meet();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if constexpr (FULL) lds_write_sum(lds_at(part + (w * MT + t) * 64 + lane), acc[t]);
      else part[(w * MT + t) * 64 + lane] = acc[t];
    }
    meet();
  };

  if constexpr (CW > 0) {
    u32x4_t x[CW][MT][4];
    const u32x4_t gl = load_g();
#pragma unroll
    for (int i = 0; i < CW; ++i) load_x(x[i], min(wc + i * NW, nck - 1));   // (chunks past the last one are not used)
    // FULL: the first D stages, without a branch, or the compiler would wait for them with the activations
    constexpr std::bool_constant<FULL> counted;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      if constexpr (FULL) start(counted);
      else issue(counted);
    }
    keep_g(gl);
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      u32x4_t g[4];
      read_g(g, i);
      ready_x(x[i], g, wc + i * NW, i < cw);
    }
    squares();
    for (int tile = tile0; tile < tiles; tile += step) {
      clear();
#pragma unroll
      for (int i = 0; i < CW; ++i) {
        if (i >= cw) break;
        u32x4_t wf[I8 ? 2 : 4];
        wait_stages<S::DMAS, D>(ahead - 1);
        if constexpr (FULL) take(wf);
        else look(wf);
        issue(counted);
        multiply(wf, x[i]);
      }
      publish();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (pieces that are not used)
    if constexpr (SPLIT) finish_last();
  } else {
    constexpr int XL = 4 * MT + (NORM && !FULL ? 4 : 0);   // loads of a stage beside the weights'
    u32x4_t x[D][MT][4];
    if constexpr (FULL) {   // no branch between the loads, so that the compiler knows what is under way
      const u32x4_t gl = load_g();
      u32x4_t g[4];
      clear();
      auto get = [&](int u) {
        load_x(x[u], wc + order(ic) * NW);
        start(std::true_type{});
      };
      auto use = [&](int u, int i, int later) {   // the stage of chunk i, `later` ones are under way
        u32x4_t wf[I8 ? 2 : 4];
        wait_stages<XL + S::DMAS, D>(later);
        take(wf);
        read_g(g, order(i));
        ready_x(x[u], g, wc + order(i) * NW, true);
        multiply(wf, x[u]);
      };
#pragma unroll
      for (int u = 0; u < D; ++u) get(u);
      keep_g(gl);
      int i = 0;
      for (; i + D < cw; i += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
          use(u, i + u, D - 1);
          get(u);
        }
      }
#pragma unroll
      for (int u = 0; u < D; ++u) use(u, i + u, D - 1 - u);
      squares();
      publish();
    } else {
      u32x4_t g[NORM ? D : 1][4];
      auto fetch = [&](u32x4_t (&xv)[MT][4], u32x4_t (&gv)[4]) {
        if (it < tiles && cw > 0) {
          const int chunk = wc + order(ic) * NW;
          load_x(xv, chunk);
#pragma unroll
          for (int f = 0; NORM && f < 4; ++f) gv[f] = *reinterpret_cast<const u32x4_t*>(p.norm_w + min(chunk * KC + kof(f), p.K - 8));
        }
        issue(std::false_type{});
      };
#pragma unroll
      for (int i = 0; i < D; ++i) fetch(x[i], g[NORM ? i : 0]);
      int tile = tile0, i = 0;
      bool first = true;
      clear();
      if (cw <= 0) squares();
      for (; cw <= 0 && tile < tiles; tile += step) publish();
      while (tile < tiles) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
          if (tile >= tiles) break;
          u32x4_t wf[I8 ? 2 : 4];
          wait_stages<XL, D>(ahead - 1);   // (of XL + DMAS loads a stage: the stage has come, and the next one's x nearly)
          look(wf);
          ready_x(x[u], g[NORM ? u : 0], wc + order(i) * NW, first);
          multiply(wf, x[u]);
          fetch(x[u], g[NORM ? u : 0]);
          if (++i == cw) {
            if (first) squares();
            first = false;
            publish();
            clear();
            i = 0, tile += step;
          }
        }
      }
    }
  }
}

template <int EPI, int R>
static int64_t tiles_of(const FewRowsParams& p) {
  if (EPI == FEW_GLU) return ceil_div64(p.N, R / 2);
  if (EPI == FEW_ROPE_KV) return (int64_t)(p.nq + p.nkv) * (p.D / 2 / (R / 2)) + ceil_div64((int64_t)p.nkv * p.D, R);
  return ceil_div64(p.N, R);
}


// HALF: two workgroups for the halves of the activation rows, one a CU
template <int EPI, bool NORM, bool XI, int R, int MT, bool I8, int NW, int CW, int D, bool SPLIT = false, bool HALF = false, bool FULL = false>
static int launch(FewRowsParams p, hipStream_t s, int splits = 1) {
  using S = Shape<R, MT, I8, NW, CW, D>;
  const int nck = ceil_div(p.K, KC);
  if ((CW > 0 || NORM) && ceil_div(nck, splits) > NW * S::GC) return -2;
  constexpr size_t lds = S::RING + S::PART + S::SQ + (NORM ? S::G : 0);
  static_assert(lds <= 160 * 1024, "LDS of a workgroup");
  const int64_t tiles = tiles_of<EPI, R>(p);
  auto* f = &kernel<EPI, NORM, XI, R, MT, I8, NW, CW, D, SPLIT, HALF, FULL>;
  // workgroups of a CU; the limit on LDS and what follows from it are set once on each device
  static std::atomic<int> known[16];
  int dev = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 1;
  if (dev < 16) per = known[dev].load(std::memory_order_relaxed);
  if (per < 1) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, (NW + S::FW) * 64, lds) != hipSuccess || per < 1) return 1;
    if (dev < 16) known[dev].store(per, std::memory_order_relaxed);
  }
  const int64_t room = (HALF ? 128 : 256 * (int64_t)per) / splits;   // workgroups side by side along the rows
  const int64_t rounds = FULL && CW == 0 ? 1 : ceil_div64(tiles, room < 1 ? 1 : room);
  if constexpr (!FULL)
    if (CW > 0 ? ceil_div(nck, splits) / NW * rounds >= D : rounds == 1 && nck % (NW * D) == 0)
      return launch<EPI, NORM, XI, R, MT, I8, NW, CW, D, SPLIT, HALF, true>(p, s, splits);
  int64_t groups = ceil_div64(tiles, rounds);
  // the two that read the same weights on one XCD (11008 x 4096 with SwiGLU, 17 rows, 126 groups 57.6 us, 128 35.2)
  if (HALF) groups = (groups + 7) / 8 * 8;
  if (SPLIT && rounds > 64) return -2;   // (a lane for every tile's ticket)
  p.splits = splits;
  if (HALF) p.half = (p.M + 1) / 2;
  // Tiles next to each other (a workgroup reads one stretch of the weights, and a line of the output is written on one XCD) where rows lie a power of
  // two apart, but not where the rows of a tile lie in two or three places, unless there are many tiles, nor parts of rows.  One of each round / next to
  // each other, us: 16 rows, 16384 x 2048 13.6 / 12.3, 32000 x 2048 23.5 / 22.1, 128256 x 2048 88.9 / 85.9, 128256 x 4096 167 / 159 (28 rows 26.3 / 23.3 for
  // 32000 x 2048); SwiGLU 8192 x 2048 13.3 / 13.5, 11008 x 2048 16.2 / 16.7, 8192 x 4096 25.1 / 26.2, 10240 x 4096 28.1 / 27.1, 14336 x 4096 40.4 / 39.3, 28 rows
  // 29.1 / 27.0 and 47.7 / 45.9; rotary 6144 x 4096 13.3 / 13.9; streamed 8192 x 8192 26.7 / 30.5; in parts 8192 x 8192 29.6 / 33.3, 4096 x 14336 24.3 / 25.3, but
  // 2048 x 12288 (long parts, four rounds) 14.1 / 13.8, 28 rows 15.7 / 15.1; rows no power of two apart, up to 16 rows 16384 x 3072 18.1 / 18.5, 32000 x 3072 31.8 / 32.5,
  // 32000 x 1536 17.5 / 17.8; few rounds of bf16 tiles of 11 waves 8192 x 4096 13.3 / 14.1, 16384 x 4096 23.0 / 23.5 (int8 at 32 rows 20.8 / 19.3)
  const bool pow2 = (p.ldw & (p.ldw - 1)) == 0;
  const int next = (SPLIT && (CW < 2 || rounds > 4)) || CW == 0 || EPI == FEW_ROPE_KV || (EPI == FEW_GLU && rounds < 7) ||
                   (!SPLIT && (!pow2 || (EPI != FEW_GLU && !I8 && CW > 2 && rounds <= 4))) ? 1 : (int)rounds;
  hipLaunchKernelGGL(f, dim3((unsigned)(groups * splits), (unsigned)(SPLIT ? 1 : HALF ? 2 : ceil_div(p.M, 16 * MT))), dim3((NW + S::FW) * 64), lds, s, p, (int)tiles, next, next > 1 ? 1 : (int)groups);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Which geometry (times in us at 4 / 16 / 32 rows, bf16, weights from memory; the choices were measured before the waits at the top of this file, what they
// take now: 16384 x 2048 with norm and SwiGLU 12.8 / 13.2 / 15.0, 128256 x 2048 79.7 / 82.0 / 86.6, 3072 x 2048 rotary 5.8 / 6.2 / 7.9, 28672 x 4096 36.7 / - /
// 44.1, 2048 x 8192 9.0 / 10.4 / 11.9, 4096 x 4096 at 4 / 13 rows 8.3 / 9.1):
//   K <= 2048: activations stay in 8 waves' registers and a workgroup goes over the tiles of 16 rows: 16384 x 2048 with
//     norm and SwiGLU 14.1 / 15.0 / 16.9 (activations streamed 15.8 / 19.0 / 71; int8 11.6 / 12.4 / 14.8),
//     128256 x 2048 86 / 92 / 98 (int8 46 / 50 / 54).
//     Up to 256 tiles there is a tile or less for a CU and streaming begins sooner: 3072 x 2048 6.1 / 6.8 against
//     6.6 / 7.9 (up to 16 rows: two tiles' operands of a streamed norm do not fit the registers, 19.9 against 10.5).
//   K <= 4224: 11 waves of 3 chunks: 28672 x 4096 40 / 43 / 55 (streamed 46 / 55 / 225; int8 25 / 27 / 40; below for 17 rows and more); without a norm and
//     up to 256 tiles streamed: 4096 x 4096 9.0 / 10.9 / 13.1 against 9.0 / 10.8 / 14.8.
//   longer: streamed, tiles of 16 rows for more than 2048 weight rows (4096 x 14336 23 / 28 / 38, of 8 rows 25 / 39 / 58),
//     else of 8, so that every CU has one (2048 x 8192 9.5 / 13.0 / 18.8, of 16 rows 11.5 / 15.4 / 20.8).  Streamed, a
//     workgroup reads all of the activations for its one tile: at 16 rows as much as the tile's weights, or twice that.
//     So with more rows the reduction is split (`parts`): a workgroup keeps the activations of its part for several tiles.
//     2048 x 8192 at 9 / 13 / 32 rows 10.7 / 12.2 / 18.9 streamed, 10.9 / 11.2 / 12.8 in parts of 1024 elements (up to 16
//     rows two workgroups a CU; of 1792, one a CU: 11.7 / 12.0 / 14.6); 2048 x 12288 at 9 / 16 / 32 16.0 / 18.9 / 27.3 -> 13.4 / 14.0 /
//     16.5 in parts of 1792 (of 1024 15.0 / 15.5 / 18.8: more parts to add up, more tiles a workgroup); 4096 x 14336 at 9 / 13 /
//     32 24.1 / 26.5 / 38.7 -> 24.4 / 24.5 / 29.2; 4096 x 11008 19.2 / 21.0 / 30.1 -> 21.0 / 21.3 / 25.6; 8192 x 8192 27.6 / 28.9 /
//     41.9 -> 28.8 / 29.0 / 33.5; 8192 x 28672 at 13 / 32 92 / 142 -> 88 / 102.
//     With a norm and above 16 rows a workgroup takes half of the rows, up to 512 tiles (K > 2048: 2,048): what the CU has to
//     read of the activations and to do for their norm counts more than the weights, which come from the XCD's cache the second time.  At 17 /
//     32 rows: 512 x 2048 7.8 / 9.2 -> 6.3 / 6.8, 3072 x 2048 8.5 / 9.9 -> 7.6 / 7.9 (4 stages under way 8.3 / 8.5), 8192 x 2048 11.5 / 12.3 -> 11.4 / 11.1
//     (12288 x 2048 13.5 / 15.2 -> 14.2 / 14.5); 1536 x 4096 15.9 / 18.5 -> 9.5 / 10.8, 6144 x 4096 20.5 / 23.0 -> 14.1 / 15.2, 28672 x 4096 with SwiGLU 50.5 / 53.4 ->
//     44.8 / 47.8 (int8 35.1 / 38.3 -> 30.6 / 32.0), 32000 x 4096 54 / 57 -> 50 / 54 (128256 x 4096 178 / 184 -> 194 / 215: halves that drift
//     apart read the weights twice).
//     Unsplit, up to 128 tiles and above 16 rows, a workgroup takes 16 of the rows only, so that every CU has one: 2048 x
//     2048 at 17 / 32 rows 5.8 / 7.1 -> 5.9 / 6.1 (int8 6.9 -> 5.3 at 32); with more tiles two would share a CU and its loads
//     (4096 x 4096 at 32 13.2 -> 18.7).
//     The parts' sums meet in memory; the last to come adds them up, its waves sharing its tiles (by one wave: 2.5 us more).
//     Streamed loads are waited for best where a wave has whole rounds of stages: two stages where it has two chunks (2048 x 2048 at 4 rows 4.3 ->
//     4.2 us, int8 4.25 -> 4.0), 7 or 11 waves where 8 leave a rest (4096 x 14336 at 4 / 9 rows 22.6 / 23.5 -> 21.4 / 22.3, 2048 x 5632 7.0 / 7.8 -> 6.6 /
//     7.5; 9 waves for 5120 x 13824 no better).  So fewer rows than before are worth splitting for: unsplit / in parts 2048 x 8192 at 14 / 16
//     rows 10.5 / 11.1 and 11.1 / 11.0, 2048 x 5632 at 12 / 16 8.0 / 9.7 and 8.9 / 10.0, 1024 x 8192 at 11 / 12 9.2 and 9.4 / 8.7.
constexpr int kLongPart = 72;   // chunks of the reduction from which parts are long

static int parts(int M, int N, int K) {   // of the reduction; 0: not split
  const int nck = ceil_div(K, KC), tiles = ceil_div(N, 16), per = nck > kLongPart ? 14 : 8;
  if (nck <= 33 || M > FEW_MAX_ROWS) return 0;
  if (tiles <= 128 ? M < (nck > kLongPart ? 9 : tiles <= 64 || nck > 64 ? 12 : nck <= 44 ? 17 : 15) : M <= 16 && (M < 12 || nck <= 96)) return 0;
  const int n = ceil_div(nck, per);
  return n > 32 || ceil_div(tiles, 256 / n) > 64 ? 0 : n;   // (a lane for every tile's ticket)
}

// Of 17 to 32 rows with a norm: whether a workgroup takes half of them
static bool halved(int nck, int64_t tiles) { return nck <= 16 ? tiles <= 512 : tiles <= 2048; }

template <int EPI, bool NORM, bool XI, int MT, bool I8>
static int pick(const FewRowsParams& p, hipStream_t s) {
  constexpr int DA = I8 ? (MT == 1 ? 6 : 4) : MT == 1 ? 4 : 3;   // (int8 stages have half the bytes)
  const int nck = ceil_div(p.K, KC);
  const int64_t tiles = tiles_of<EPI, 16>(p);
  if constexpr (NORM) {
    if (nck > 33) return -1;
    if (MT == 1 && tiles <= 256 && nck <= 16) return launch<EPI, true, XI, 16, 1, I8, 8, 0, 2>(p, s);
    if (MT == 2 && halved(nck, tiles)) {
      if (nck <= 16) return launch<EPI, true, XI, 16, 1, I8, 8, 2, 2, false, true>(p, s);
      return launch<EPI, true, XI, 16, 1, I8, 11, 3, 3, false, true>(p, s);
    }
    if (nck <= 16) return launch<EPI, true, XI, 16, MT, I8, 8, 2, DA>(p, s);
    return launch<EPI, true, XI, 16, MT, I8, 11, 3, 3>(p, s);
  } else {
    constexpr int D = MT == 1 ? 4 : 2;
    if (tiles > 256) {
      if (nck <= 16) return launch<EPI, false, false, 16, MT, I8, 8, 2, DA>(p, s);
      if (nck <= 33) return launch<EPI, false, false, 16, MT, I8, 11, 3, 3>(p, s);
    }
    if constexpr (EPI == FEW_STORE || EPI == FEW_RESID) {
      constexpr int X = I8 ? 2 : 1;
      const int n = p.ws ? parts(p.M, p.N, p.K) : 0;
      if (n && nck > kLongPart) return launch<EPI, false, false, 16, MT, I8, 7, 2, 4 * X, true>(p, s, n);
      if (n) return launch<EPI, false, false, 16, MT, I8, 8, 1, 2 * X, true>(p, s, n);
    }
    // (as many waves as give each whole rounds of stages, for one tile a workgroup; bf16 of 8192 x 7168 at 4 rows with 8 waves 20.9 us, with 7 21.6, int8 of 8192 x
    // 5632 at 8 rows 14.0, with 11 14.9, but 8192 x 14336 at 4 rows 38.6 and 37.3)
    if (MT == 1 && nck > 33 && nck % 32) {
      if (nck % 28 == 0 && (tiles <= (I8 ? 512 : 256) || nck > kLongPart)) return tiles > 128 ? launch<EPI, false, false, 16, 1, I8, 7, 0, 4>(p, s) : launch<EPI, false, false, 8, 1, I8, 7, 0, 4>(p, s);
      if (nck % 44 == 0 && tiles <= 256) return tiles > 128 ? launch<EPI, false, false, 16, 1, I8, 11, 0, 3>(p, s) : launch<EPI, false, false, 8, 1, I8, 11, 0, 4>(p, s);
    }
    if (tiles > 128) return launch<EPI, false, false, 16, MT, I8, 8, 0, D>(p, s);
    if (nck > 8 && nck <= 16) return MT == 2 ? launch<EPI, false, false, 16, 1, I8, 8, 0, 2>(p, s) : launch<EPI, false, false, 8, 1, I8, 8, 0, 2>(p, s);
    if (MT == 2) return launch<EPI, false, false, 16, 1, I8, 8, 0, 4>(p, s);
    return launch<EPI, false, false, 8, 1, I8, 8, 0, 4>(p, s);
  }
}

template <int EPI, bool NORM, bool XI>
static int rows(const FewRowsParams& p, hipStream_t s) {
  if constexpr (EPI != FEW_RELU2) {   // (the squared ReLU's model has no int8 weights)
    if (p.wscale) return p.M <= 16 ? pick<EPI, NORM, XI, 1, true>(p, s) : pick<EPI, NORM, XI, 2, true>(p, s);
  }
  if (p.wscale) return -1;
  return p.M <= 16 ? pick<EPI, NORM, XI, 1, false>(p, s) : pick<EPI, NORM, XI, 2, false>(p, s);
}

template <int EPI>
static int norms(const FewRowsParams& p, hipStream_t s) {
  return p.norm_w ? rows<EPI, true, false>(p, s) : rows<EPI, false, false>(p, s);
}

}  // namespace few

int64_t few_rows_workspace(int M, int N, int K, int* tickets) {
  const int n = few::parts(M, N, K);
  *tickets = n ? ceil_div(N, 16) * (M <= 16 ? 1 : 2) : 0;
  return (int64_t)*tickets * n * 256;
}

bool few_rows_halved(int M, int N, int K) { return M > 16 && M <= FEW_MAX_ROWS && ceil_div(K, few::KC) <= 33 && few::halved(ceil_div(K, few::KC), ceil_div64(N, 16)); }

int few_rows_launch(int epi, const FewRowsParams& p, hipStream_t s) {
  const int unit = p.wscale ? 16 : 8;   // elements of 16 bytes of weights
  if (p.M < 1 || p.M > FEW_MAX_ROWS || p.N < 1 || p.K < unit || p.K % unit || p.ldw % unit || p.ldx % 8) return -1;
  // 32-bit offsets, and their sums with a row's length
  const int64_t wrows = epi == FEW_GLU ? 2 * (int64_t)p.N : p.N;
  if ((wrows + 16) * p.ldw * (p.wscale ? 1 : 2) >= (1LL << 32) || ((p.xidx ? p.xrows : p.M) + 1) * p.ldx >= (1LL << 31)) return -1;
  if (p.xidx && (epi != FEW_ROPE_KV || !p.norm_w || p.xrows < 1)) return -4;
  if (epi == FEW_ROPE_KV && (p.D % 32 || !p.norm_w || ((uintptr_t)p.cos_t | (uintptr_t)p.sin_t) % 16)) return -1;
  switch (epi) {
    case FEW_STORE: return few::norms<FEW_STORE>(p, s);
    case FEW_RESID: return p.norm_w ? -1 : few::rows<FEW_RESID, false, false>(p, s);
    case FEW_GLU: return few::norms<FEW_GLU>(p, s);
    case FEW_ROPE_KV: return p.xidx ? few::rows<FEW_ROPE_KV, true, true>(p, s) : few::rows<FEW_ROPE_KV, true, false>(p, s);
    case FEW_F32: return few::norms<FEW_F32>(p, s);
    case FEW_RELU2: return p.norm_w ? -1 : few::rows<FEW_RELU2, false, false>(p, s);
  }
  return -1;
}

}  // namespace nxd
