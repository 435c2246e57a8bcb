// The main loop of the 256 x 256-tile products (grouped_rowgemm.hip, wgrad_gemm.hip, act_gemm.hip): C = A B over a reduction in steps of 64, bf16 operands, fp32 sums.
//
// What bounds it is the clock that the numbers allow (8192 x 8192 x 8192 with random ones 1.75 to 1.9 GHz, with zeros 2.36, counted as
// GRBM_GUI_ACTIVE over the kernel's time) and what stands between the MFMAs.
//   * 4 waves, one a SIMD, of 128 x 128 results each: 64 v_mfma_f32_16x16x32_bf16 for 16 fragments read from LDS, two thirds of what
//     8 waves of 128 x 64 read -- those read 192 KB a step where LDS gives 128 bytes a clock, as long as the MFMAs take.  The
//     256 sums of a lane are in AGPRs; the MFMAs are written in asm, because hipcc moves such sums between registers
//     (216 moves and 124 waits a step of 128 MFMAs: 0.22 PFLOP/s).
//   * A wave is alone on its SIMD, so the matrix cores wait for whatever it does beyond the 12 cycles that a MFMA leaves free: between two MFMAs
//     there is at most a read, an address or a load.  Above all no read stands behind the instruction that makes its address (5 cycles a
//     read): addresses move on by themselves once a step, between MFMAs that nothing else needs.  The word that says where a load goes in LDS (m0)
//     and the load have a MFMA between them.  Cycles a step of 2,048 for the MFMAs alone, A B^T / A B / A^T B: reads, addresses and loads four MFMAs apart 2,562 / 2,685 /
//     2,744, now 2,213 / 2,233 / 2,195 (without loads and the barrier 2,085 / 2,120 / 2,024).
//   * A step's operands are 64 KB of LDS.  Three steps of A are there and two of B (160 KB): during the MFMAs of one half of a step (32 of the reduction) the
//     next half is read; in the first half the loads of A go out, two steps ahead; after it a barrier
//     says that the step has been read and the next one is there, and B's loads go out with the first MFMAs of the second half.
//   * Loads go straight to LDS, 128 bytes of a row and more: whole lines (with 64 bytes of a row a CU gets 50 GB/s, with 128 it gets 90).
//   * Weight gradients, whose images can be cut in halves of whole lines, have a ring of half steps instead (LoopTR).
//   us, four MFMAs apart -> now, one card in turn: 8 experts, 8,192 rows uneven, 4096 -> 28672 1,638 / 1,817 (input gradient) -> 1,504 / 1,664; 8192 x 8192 x 8192 of
//   random numbers A B^T 745 -> 690, A B 756 -> 693, A^T B 835 -> 742 (a warmer card 776 -> 711, 787 -> 722, 874 -> 792: with random numbers what is saved in cycles
//   is partly given back in clock); SwiGLU of 8,192 columns, 2,048, 2,304 rows 134 -> 128.
//
// Images of a step in LDS, 16-byte chunks XORed so that 16 lanes of a read cover all banks once:
//   ROW  the reduction is contiguous: [256 rows][64], 128-byte rows
//   TR   the rows / columns are contiguous: [64][256], 512-byte rows, read with ds_read_b64_tr_b16
#pragma once
#include "common.h"

#include <type_traits>
#include <utility>

namespace nxd {
namespace tile {

constexpr int BM = 256, BN = 256, BK = 64, THREADS = 256;
constexpr int IMG_BYTES = 256 * BK * 2, B_BASE = 3 * IMG_BYTES, LDS_BYTES = 5 * IMG_BYTES;   // images: three of A, two of B

typedef __attribute__((address_space(3))) short4_t lds_short4_t;

__device__ __forceinline__ void load_lds(uint32_t at, const char* base, uint32_t lds) {   // 64 lanes x 16 B: base + at -> LDS lds + 16 lane
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory", "m0");
}
template <typename T>
__device__ __forceinline__ T* uniform(T* p) {   // one address for the wave
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<T*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)a));
}

// ROW images: chunk c of a row at c ^ row_swz.  Rows that are read together: 16 in a row, or 4 of every 8 (the columns of a B
// fragment, below); either way the last bit and row_swz differ in all 16.
__device__ __forceinline__ int row_swz(int row) { return (row >> 1 & 1) | (row >> 3 & 1) << 1 | ((row >> 2 ^ row >> 4) & 1) << 2; }
// TR images: chunk c of reduction row t at c ^ tr_swz
__device__ __forceinline__ int tr_swz(int t) { return 2 * ((t & 3) | (t >> 3 & 1) << 2); }

// Wave (wm, wn) has row fragments i at 32 i + 16 wm (all waves have as much of a tile with few rows) and the columns from 128 wn on.
// acc[i][j][e] is row 32 i + 16 wm + (lane & 15), column col(j, e): of B in ROW images 8 columns of a lane are contiguous over a pair
// of fragments, in TR images 4.
template <bool BT>
__device__ __forceinline__ int col(int wn, int j, int lane) {
  const int g = lane >> 4;
  return 128 * wn + (BT ? 16 * j + 4 * g : 32 * (j >> 1) + 8 * g + 4 * (j & 1));
}

// After the wait for the last sums: without this the compiler, which doesn't know what the asm of the MFMAs takes, may read them before the wait
template <int IM>
__device__ __forceinline__ void settled(f32x4_t (&acc)[8][8]) {
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
}

template <int... I, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {   // f(0), .. f(N - 1), each number a constant
  each(std::make_integer_sequence<int, N>{}, f);
}

// One product, and one with a load (64 lanes x 16 B: base + at -> LDS lds + MORE + 16 lane): it stands between m0 and the load that reads it.
// ZERO: the first product of a sum, whatever the registers hold.
template <bool ZERO = false>
__device__ __forceinline__ void mfma(f32x4_t& c, const bf16x8_t& b, const bf16x8_t& a) {
  if constexpr (ZERO) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(b), "v"(a));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a));
}
template <int MORE, bool ZERO = false>
__device__ __forceinline__ void mfma_load(f32x4_t& c, const bf16x8_t& b, const bf16x8_t& a, uint32_t at, const char* base, uint32_t lds) {
  if constexpr (ZERO)
    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0\n\tglobal_load_lds_dwordx4 %3, %4"
                 : "=&a"(c)
                 : "v"(b), "v"(a), "v"(at), "s"(base), "s"(lds), "n"(MORE)
                 : "memory", "m0", "scc");
  else
    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %4"
                 : "+a"(c)
                 : "v"(b), "v"(a), "v"(at), "s"(base), "s"(lds), "n"(MORE)
                 : "memory", "m0", "scc");
}
// An address for reads to come, made where nothing waits for it
__device__ __forceinline__ void move_to(int& at, int base, int by) { asm volatile("v_add_u32 %0, %1, %2" : "=v"(at) : "s"(by), "v"(base)); }
__device__ __forceinline__ void move_by(int& at, int by) { asm volatile("v_add_u32 %0, %1, %0" : "+v"(at) : "s"(by)); }
__device__ __forceinline__ void fixed() { __builtin_amdgcn_sched_barrier(0); }   // what stands before stays before
__device__ __forceinline__ void reads_done() { __builtin_amdgcn_s_waitcnt(0xC07F); }   // (lgkmcnt(0); the compiler knows of it)

template <bool BT>
struct Loop {
  char* smem;
  int lane, wid, wm, wn;
  uint32_t lds;
  uint32_t off[16];        // of this lane's pieces of A (0 .. 7) and B from a step's base
  const char *pa, *pb;     // the bases of the next step to load
  int64_t da, db;          // ... and from one step to the next
  uint32_t ld_a;           // for run_few: A's row, and how many there are
  int rows_a;
  uint32_t back;           // (reductions that end with half a step) pieces of the last step whose second half is past the end, a bit each

  // A: rows 0 .. rows - 1 from `a` on (ROW: a row is lda elements; TR: a reduction row), clamped to the last; B likewise
  __device__ __forceinline__ Loop(char* smem_, const uint16_t* a, int64_t lda, int rows, const uint16_t* b, int64_t ldb, int cols) : smem(smem_) {
    lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wid >> 1, wn = wid & 1;
    lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    set(a, lda, rows, b, ldb, cols);
  }
  __device__ __forceinline__ void set(const uint16_t* a, int64_t lda, int rows, const uint16_t* b, int64_t ldb, int cols) {   // the tile that is loaded from now on
    pa = uniform(reinterpret_cast<const char*>(a)), pb = uniform(reinterpret_cast<const char*>(b));
    da = BK * 2, db = BT ? (int64_t)BK * ldb * 2 : BK * 2;
    back = 0, ld_a = (uint32_t)lda, rows_a = rows;
    int lane = this->lane;
    asm volatile("" : "+v"(lane));   // (made anew for each tile: kept, what does not change takes the registers of a loop around this one)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const bool tr = i >= 8 && BT;
      const int piece = 8 * wid + (i & 7), n = i < 8 ? rows : cols;
      const uint32_t ld = (uint32_t)(i < 8 ? lda : ldb);   // (offsets have 32 bits)
      if (tr) {
        const int t = 2 * piece + (lane >> 5), c = (lane & 31) ^ tr_swz(t);
        off[i] = ((uint32_t)t * ld + (uint32_t)min(8 * c, n - 8)) * 2;
        if (t >= BK / 2) back |= 1u << i;
      } else {
        const int row = 8 * piece + (lane >> 3), c = (lane & 7) ^ row_swz(row);
        off[i] = ((uint32_t)min(row, n - 1) * ld + (uint32_t)(8 * c)) * 2;
        if (c >= 4) back |= 1u << i;
      }
    }
  }

  // fragment addresses: of A's first image by half, of A's images that are read now and of B's (ROW: [chunk bit 2], TR: [fragment])
  static constexpr int NB = BT ? 8 : 2;
  int base_a[2], ra[2], rb[NB];
  __device__ __forceinline__ void addresses(int b_base) {
    const int r = lane & 15, g = lane >> 4;
    const int row = 16 * wm + r;
    base_a[0] = row * 128 + 16 * (g ^ row_swz(row));
    base_a[1] = base_a[0] ^ 64;
    ra[0] = base_a[0], ra[1] = base_a[1];
    if constexpr (BT) {
#pragma unroll
      for (int j = 0; j < 8; ++j) rb[j] = b_base + tr_at(128 * wn + 16 * j);
    } else {
      const int c = 128 * wn + 8 * (r >> 2) + (r & 3);
      rb[0] = b_base + c * 128 + 16 * (g ^ row_swz(c));
      rb[1] = rb[0] ^ 64;   // (b_base is a multiple of 128)
    }
  }
  __device__ __forceinline__ int tr_at(int c0) const {   // lane 16 g + 4 q + p: 4 columns from c0 + 4 p on, of reduction rows 8 g + q (and + 4)
    const int t = 8 * (lane >> 4) + (lane >> 2 & 3), c = c0 + 4 * (lane & 3);
    return t * 512 + 16 * (c >> 3 ^ tr_swz(t)) + 8 * (c >> 2 & 1);
  }
  __device__ __forceinline__ bf16x8_t read_tr(int at) const {
    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + at));
    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + at + 4 * 512));
    const short __attribute__((ext_vector_type(8))) v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  }
  __device__ __forceinline__ bf16x8_t read_row(int at) const { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(smem + at)); }
  __device__ __forceinline__ bf16x8_t frag_a(int i, int h) const { return read_row(ra[h] + i * 4096); }
  __device__ __forceinline__ bf16x8_t frag_b(int j, int h) const {
    if constexpr (BT) return read_tr(rb[j] + h * (IMG_BYTES / 2));
    else return read_row(rb[h ^ (j & 1)] + (j & 1) * 512 + (j >> 1) * 4096);
  }

  template <bool HALF>
  __device__ __forceinline__ uint32_t from(int i, bool last) const {   // piece i (A: 0 .. 7) of the next step; HALF, last: its second half is past the end
    uint32_t at = off[i];
    if constexpr (HALF) {   // (the first half again: not used)
      const bool tr = i >= 8 && BT;
      if (last) at -= (back >> i & 1) * (tr ? (uint32_t)((i < 8 ? da : db) / 2) : 64u);
    }
    return at;
  }
  template <bool HALF>
  __device__ __forceinline__ void load(int i, int img, bool last) const {
    load_lds(from<HALF>(i, last), i < 8 ? pa : pb, lds + (i < 8 ? 0 : B_BASE) + img + (8 * wid + (i & 7)) * 1024);
  }

  // Fragments of the two halves of a step, and where its images lie: A's go round three places, B's take turns
  template <int IM>
  struct Frags {
    bf16x8_t a0[IM], b0[8], a1[IM], b1[8];
    int a_now = 0, a_next = IMG_BYTES, a_free = 2 * IMG_BYTES, b_now = 0;
  };
  __device__ __forceinline__ void advance_a(bool there) {   // towards the next step, if there is one
    if (there) pa += da;
  }
  __device__ __forceinline__ void advance_b(bool there) {
    if (there) pb += db;
  }
  // The loads of the first two of so many steps, and the first half's fragments
  template <bool HALF>
  __device__ __forceinline__ void begin(Frags<8>& f, int steps, bool end) {
#pragma unroll
    for (int i = 0; i < 16; ++i) load<HALF>(i, 0, end && steps == 1);
    advance_a(1 < steps), advance_b(1 < steps);
#pragma unroll
    for (int i = 0; i < 16; ++i) load<HALF>(i, IMG_BYTES, end && steps <= 2);   // (past the end: the last step again, not used)
    advance_a(2 < steps), advance_b(2 < steps);
    addresses(B_BASE);
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j) f.b0[j] = frag_b(j, 0), fixed();   // (in this order: the loop's waits count what came later)
#pragma unroll
    for (int i = 0; i < 8; ++i) f.a0[i] = frag_a(i, 0), fixed();
  }
  // One step: two halves, each its products, and between two of them at most a read of the next half's fragments (k: B's, then A's), an address or a load.  A
  // wave is alone on its SIMD: what stands between two products beyond the 12 cycles that the first leaves free, or waits for what stands just
  // before it, the matrix cores wait for.  ZERO: the first of its sums; last: what is loaded is the last step, of half the reduction; more: there is a step
  // after the one that is loaded; wait(): its turn's loads have come.
  template <bool HALF, bool ZERO, typename WAIT>
  __device__ __forceinline__ void step(f32x4_t (&acc)[8][8], Frags<8>& f, bool last, bool more, WAIT&& wait) {
    constexpr int M = 64, READS = 16, RD = 2, RD2 = 4, LD = 4;   // products; from one read (of the second half: RD2), or load, to the next
    constexpr int FREE = RD * READS, SP = (M - FREE) / NB;       // from there on the addresses of B move, their reads of a first half all out
    const uint32_t mine = lds + wid * 8192, to_a = mine + f.a_free, to_b = mine + f.b_now;
    const int b_by = f.b_now ? -IMG_BYTES : IMG_BYTES;
    each<M>([&](auto mc) __attribute__((always_inline)) {
      constexpr int m = mc, k = m / RD, l = m / LD;
      f32x4_t& c = acc[m >> 3][m & 7];
      if constexpr (m % RD == RD - 1 && k < READS) {   // (one of B's and one of A's in turn)
        if constexpr (k % 2 == 1) f.a1[k >> 1] = frag_a(k >> 1, 1);
        else f.b1[k >> 1] = frag_b(k >> 1, 1);
        fixed();
      }
      if constexpr (m >= FREE && (m - FREE) % SP == 0) move_by(rb[(m - FREE) / SP], b_by), fixed();
      if constexpr (m == M - 1) move_to(ra[0], base_a[0], f.a_next), fixed();
      if constexpr (m == 36) advance_a(more), fixed();
      if constexpr (m % LD == LD / 2 && l < 8) mfma_load<l * 1024, ZERO>(c, f.b0[m & 7], f.a0[m >> 3], from<HALF>(l, last), pa, to_a);
      else mfma<ZERO>(c, f.b0[m & 7], f.a0[m >> 3]);
      fixed();
    });
    reads_done();
    wait();
    __builtin_amdgcn_s_barrier();
    fixed();
    each<M>([&](auto mc) __attribute__((always_inline)) {
      constexpr int m = mc, k = m / RD2, l = m / LD;
      f32x4_t& c = acc[m >> 3][m & 7];
      if constexpr (m % RD2 == RD2 / 2) {
        if constexpr (k < 8) f.b0[k] = frag_b(k, 0);
        else f.a0[k - 8] = frag_a(k - 8, 0);
        fixed();
      }
      if constexpr (m == 0) move_to(ra[1], base_a[1], f.a_next), fixed();
      if constexpr (m == 36) advance_b(more), fixed();
      if constexpr (m % LD == LD - 1 && l < 8) mfma_load<B_BASE + l * 1024>(c, f.b1[m & 7], f.a1[m >> 3], from<HALF>(8 + l, last), pb, to_b);
      else mfma(c, f.b1[m & 7], f.a1[m >> 3]);
      fixed();
    });
    f.b_now ^= IMG_BYTES;
    const int freed = f.a_now;
    f.a_now = f.a_next, f.a_next = f.a_free, f.a_free = freed;
  }

  // Tiles of at most 32 IM rows: a step's products take a fourth of the time of a step's of 256 rows, or half, and its operands are 40 or 48 KB.  Four or three steps of both
  // operands are there, so that loads have two steps and more for their way; with the places above, B's had half a step, and a step took as long as a load.  What
  // bounds it now is the weights' bytes (from memory 5.2 TB/s, 16 rows of 8 experts).  us, before / now: 16 rows of each of 8 experts 4096 -> 28672 389 / 363, input gradient 369 / 360,
  // 100 rows 430 / 409 and 401 / 391; SwiGLU of 8,192 columns, reduction 2,048, 64 or 100 rows 25.3 / 21.3.
  // beside: other tiles with the same B run at the same time, and it is better to stay with them, so that the L2 has what it reads, than to run ahead: up to 64 rows wait for all loads of a
  // step (8,192 rows of 8 experts, about 1,024 each, 4096 -> 28672 1,526 before, 1,531 ahead, 1,523 beside; input gradient 1,526 / 1,544 / 1,512; 65 to 128 rows take as long as
  // the others if they wait so: input gradient 1,573 before, 1,660 with all of them, 1,530 with up to 64).
  template <int IM>
  struct Few {
    static constexpr int PLACES = IM == 2 ? 4 : 3, A_BYTES = IM * 4096, PLACE = A_BYTES + IMG_BYTES, LOADS = 8 + IM;
    static_assert(PLACES * PLACE <= LDS_BYTES, "LDS");
  };
  template <int IM>
  __device__ __forceinline__ void wait_few(int pieces, bool beside) const {   // all loads but those of the PLACES - 2 newest steps have come
    constexpr int S = Few<IM>::PLACES - 2;
    if (IM == 2 && beside) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else
    each<IM + 1>([&](auto n) __attribute__((always_inline)) {
      if (pieces == n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S * (8 + n)) : "memory");
    });
  }
  template <int IM, bool HALF>
  __device__ __forceinline__ void load_few(int i, int pieces, uint32_t place, bool last) const {   // (A: 0 .. IM - 1)
    if (i < IM && i >= pieces) return;
    if (i < IM) load_lds(from<HALF>(i, last), pa, place + (wid + 4 * i) * 1024);
    else load_lds(from<HALF>(8 + i - IM, last), pb, place + Few<IM>::A_BYTES + (8 * wid + i - IM) * 1024);
  }
  template <int IM, bool HALF>
  __device__ __forceinline__ void run_few(f32x4_t (&acc)[8][8], int steps, bool end, bool beside) {
    using F = Few<IM>;
    constexpr int M = 8 * IM, RD = IM == 2 ? 1 : 2;   // products; from one read to the next
    // of A, those with rows that there are; every fourth is this wave's
    const int pieces = min(((rows_a + 7) / 8 - wid + 3) / 4, IM);
    back &= ~((1u << IM) - 1);
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      const int row = 8 * (wid + 4 * i) + (lane >> 3), c = (lane & 7) ^ row_swz(row);
      off[i] = ((uint32_t)min(row, rows_a - 1) * ld_a + (uint32_t)(8 * c)) * 2;
      if (c >= 4) back |= 1u << i;
    }
#pragma unroll
    for (int s = 0; s < F::PLACES - 1; ++s) {   // (past the end: the last step again, not used)
#pragma unroll
      for (int i = 0; i < F::LOADS; ++i) load_few<IM, HALF>(i, pieces, lds + s * F::PLACE, end && s + 1 >= steps);
      advance_a(s + 1 < steps), advance_b(s + 1 < steps);
    }
    addresses(F::A_BYTES);
    Frags<IM> f;
    wait_few<IM>(pieces, false);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j) f.b0[j] = frag_b(j, 0), fixed();   // (in this order: the loop's waits count what came later)
#pragma unroll
    for (int i = 0; i < IM; ++i) f.a0[i] = frag_a(i, 0), fixed();
    int now = 0, free = (F::PLACES - 1) * F::PLACE;   // places of this step and of the one that is loaded
#pragma unroll 1
    for (int t = 0, whole = steps - (HALF && end); t < whole; ++t) {
      const int next = now == (F::PLACES - 1) * F::PLACE ? 0 : now + F::PLACE;
      const bool last = end && t + F::PLACES >= steps;
      asm volatile("s_nop 3");   // (after moves of the sums ahead of the loop)
      each<M>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = mc, k = m / RD, l = IM == 2 ? m - (M - F::LOADS) : m % 2 == 0 ? m / 2 - (M / 2 - F::LOADS) : -1;
        if constexpr (m % RD == RD - 1 && k < 8 + IM) {   // (one of B's and one of A's in turn)
          if constexpr (k < 2 * IM && k % 2 == 1) f.a1[k >> 1] = frag_a(k >> 1, 1);
          else f.b1[k < 2 * IM ? k >> 1 : k - IM] = frag_b(k < 2 * IM ? k >> 1 : k - IM, 1);
          fixed();
        }
        if constexpr (l >= 0) load_few<IM, HALF>(l, pieces, lds + free, last), fixed();
        mfma(acc[m >> 3][m & 7], f.b0[m & 7], f.a0[m >> 3]);
        fixed();
      });
      advance_a(t + F::PLACES < steps), advance_b(t + F::PLACES < steps);
#pragma unroll
      for (int j = 0; j < NB; ++j) move_by(rb[j], next - now);
      move_to(ra[0], base_a[0], next);
      reads_done();
      wait_few<IM>(pieces, beside);
      __builtin_amdgcn_s_barrier();
      fixed();
      each<M>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = mc, k = m / RD;
        if constexpr (m % RD == RD / 2 && k < 8 + IM) {
          if constexpr (k < 8) f.b0[k] = frag_b(k, 0);
          else f.a0[k - 8] = frag_a(k - 8, 0);
          fixed();
        }
        mfma(acc[m >> 3][m & 7], f.b1[m & 7], f.a1[m >> 3]);
        fixed();
      });
      move_to(ra[1], base_a[1], next);
      free = now, now = next;
      asm volatile("s_nop 7" ::: "memory");   // (the sums may move after the loop)
    }
    last_half<IM, HALF>(acc, f, end);
  }

  // acc += the products of so many steps.  IM: row fragments that have rows.  HALF, end: the last step has half the reduction.
  template <int IM, bool HALF>
  __device__ __forceinline__ void run(f32x4_t (&acc)[8][8], int steps, bool end, bool beside = false) {
    static_assert(IM == 8 || IM == 4 || IM == 2, "rows");
    if constexpr (IM < 8) {
      run_few<IM, HALF>(acc, steps, end, beside);
    } else {
      Frags<8> f;
      begin<HALF>(f, steps, end);
#pragma unroll 1
      for (int t = 0, whole = steps - (HALF && end); t < whole; ++t) {
        asm volatile("s_nop 3");   // (after moves of the sums ahead of the loop)
        step<HALF, false>(acc, f, end && t + 3 >= steps, t + 3 < steps, [&]() { asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); });   // (all but A's of the newest step)
        if (HALF) asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // (the sums may move after the loop)
      }
      last_half<8, HALF>(acc, f, end);
    }
  }
  template <int IM, bool HALF>
  __device__ __forceinline__ void last_half(f32x4_t (&acc)[8][8], Frags<IM>& f, bool end) {   // after the whole steps
    if (HALF && end) {   // (s_nop: the sums may have moved to other registers just before)
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("s_nop 3\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.b0[j]), "v"(f.a0[i]));
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");   // (loads that nothing reads; the last sums)
    settled<IM>(acc);
  }

  // acc = the products of one of several tiles, of so many whole steps each (2 or more), after begin() for the first one.  next(), if there is another one: the
  // loads go over to it, two steps before the end, so that it begins without a wait.  stored: every wave has made STORES vector stores since the last tile, no
  // fewer: the first step's loads came before them and are waited for alone (more stores, or other vector memory operations, would only be waited for too).
  template <int STORES, typename NEXT>
  __device__ __forceinline__ void run_tile(f32x4_t (&acc)[8][8], Frags<8>& f, int steps, bool stored, bool another, NEXT&& next) {
    static_assert(8 + STORES < 64, "vmcnt");
    const auto rest = [&](int t, int end) __attribute__((always_inline)) {   // towards step t + 3, or the next tile's t + 3 - steps
#pragma unroll 1
      for (; t < end; ++t)
        step<false, false>(acc, f, false, t + 3 < steps || (another && t + 3 > steps && t + 3 < 2 * steps), [&]() { asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); });
    };
    const int turn = steps - 2;
    if (turn == 0 && another) next();
    step<false, true>(acc, f, false, 3 < steps || (another && steps == 2), [&]() {
      if (stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + STORES) : "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    });
    rest(1, turn);
    if (turn > 0 && another) next();
    rest(max(1, turn), steps);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    settled<8>(acc);
  }
};

// Both operands' rows / columns contiguous (weight gradients): half steps of 32 of the reduction, 32 KB each, four of them there.  While the products of
// half step q run, the fragments of q + 1 are read, and q + 4 is loaded into the place of q, read during q - 1: a step to a step and a quarter
// for a load's way, where whole steps left half a step to one.  8 experts 4096 x 28672 over 12,288 rows 3,484 -> 3,397 us, 14336 x 4096 over 16,384
// 2,159 -> 2,069; one gradient of 8,192 or 3,000 tokens the same within 1 % (its reads and writes, and the clock).  Five half steps: 1 % less for
// 128256 x 2048, 2 % more for 1,344 to 4,096 tokens.
// The reads come in the first half of a half step and the loads in the second: the barrier waits for the reads, and spread over all of it, with the loads between them, the
// last ones were still on their way there (few tiles in splits took 2 to 4 % more than with whole steps: us, whole steps / half steps, spread / now: 2304 x 1280 over 4,224
// tokens 57.4 / 58.9 / 57.5, 3072 x 2048 4,608 86.8 / 88.8 / 86.5, 1280 x 512 4,800 30.9 / 32.0 / 31.3, unsplit 4864 x 1792 2,560 73.2 / 73.0 / 70.3; 8 experts' 4096 x
// 2048 over 12,552 rows 315 / 280 / 272).
struct LoopTR {
  static constexpr int HK = BK / 2, HALF_BYTES = HK * 256 * 2, PLACE_BYTES = 2 * HALF_BYTES, PLACES = 4, LOADS = 8;   // loads: of a wave, for a half step
  static_assert(PLACES * PLACE_BYTES <= LDS_BYTES, "LDS");
  char* smem;
  int lane, wid, wm, wn;
  uint32_t lds;
  uint32_t off[LOADS];   // of this lane's pieces of A (0 .. 3) and B from a half step's base
  const char *pa, *pb;
  int64_t da, db;    // bytes of 32 reduction rows

  __device__ __forceinline__ LoopTR(char* smem_, const uint16_t* a, int64_t lda, int rows, const uint16_t* b, int64_t ldb, int cols) : smem(smem_) {
    lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wid >> 1, wn = wid & 1;
    lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    pa = uniform(reinterpret_cast<const char*>(a)), pb = uniform(reinterpret_cast<const char*>(b));
    da = (int64_t)HK * lda * 2, db = (int64_t)HK * ldb * 2;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int t = 2 * (4 * wid + (i & 3)) + (lane >> 5), c = (lane & 31) ^ tr_swz(t);
      off[i] = (uint32_t)(t * (i < 4 ? lda : ldb) + min(8 * c, (i < 4 ? rows : cols) - 8)) * 2;
    }
  }
  __device__ __forceinline__ int tr_at(int c0) const {   // lane 16 g + 4 q + p: 4 columns from c0 + 4 p on, of reduction rows 8 g + q (and + 4)
    const int t = 8 * (lane >> 4) + (lane >> 2 & 3), c = c0 + 4 * (lane & 3);
    return t * 512 + 16 * (c >> 3 ^ tr_swz(t)) + 8 * (c >> 2 & 1);
  }
  __device__ __forceinline__ static bf16x8_t joined(const short4_t& lo, const short4_t& hi) {
    const short __attribute__((ext_vector_type(8))) v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  }
  __device__ __forceinline__ bf16x8_t read(int at) const {
    return joined(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + at)), __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + at + 4 * 512)));
  }
  __device__ __forceinline__ void load(int i, int place) const {
    load_lds(off[i], i < 4 ? pa : pb, lds + place + (i < 4 ? 0 : HALF_BYTES) + (4 * wid + (i & 3)) * 1024);
  }

  // acc += the products of so many steps (of two halves).  FIRST: the first step has `rows` of the reduction only (1 .. 64); nothing past them is read.
  template <bool FIRST>
  __device__ __forceinline__ void run(f32x4_t (&acc)[8][8], int steps, int rows = BK) {
    const int n = 2 * steps;
    if constexpr (FIRST) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {   // (rows past the last: that one again)
        const int have = max(min(rows - h * HK, HK), 1);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
          const int past = max(0, 2 * (4 * wid + (i & 3)) + (lane >> 5) - (have - 1));
          const uint32_t from = off[i] - past * (uint32_t)((i < 4 ? da : db) / HK);
          load_lds(from, i < 4 ? pa : pb, lds + h * PLACE_BYTES + (i < 4 ? 0 : HALF_BYTES) + (4 * wid + (i & 3)) * 1024);
          if (h == 1 && steps == 1) off[i] = from;   // (for the loads that nothing reads)
        }
        if (h == 0 ? rows > HK : steps > 1) {
          const int by = h == 0 ? HK : rows > HK ? rows - HK : rows;
          pa += da / HK * by, pb += db / HK * by;
        }
      }
    }
    auto advance = [&](int q) {   // towards half step q
      if (q < n) pa += da, pb += db;
    };
#pragma unroll
    for (int q = FIRST ? 2 : 0; q < PLACES; ++q) {   // (past the end: the last one again, not used)
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load(i, q * PLACE_BYTES);
      advance(q + 1);
    }
    int ra[8], rb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ra[i] = tr_at(32 * i + 16 * wm), rb[i] = HALF_BYTES + tr_at(128 * wn + 16 * i);
    auto there = [&]() {   // all loads but those of the two newest half steps have come, and all waves have read so far
      reads_done();
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    there();
    if constexpr (FIRST) {   // what was loaded twice counts nothing
      for (int i = threadIdx.x; i < 2 * (BK - rows) * 32; i += THREADS) {
        const int t = rows + (i >> 6);
        *reinterpret_cast<u32x4_t*>(smem + (t >> 5) * PLACE_BYTES + (i >> 5 & 1) * HALF_BYTES + (t & 31) * 512 + (i & 31) * 16) = u32x4_t{0u, 0u, 0u, 0u};
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    bf16x8_t a0[8], b0[8], a1[8], b1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) b0[j] = read(rb[j]);
#pragma unroll
    for (int i = 0; i < 8; ++i) a0[i] = read(ra[i]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();   // (half step 0 has been read)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) ra[i] += PLACE_BYTES, rb[i] += PLACE_BYTES;
    int now = 0;   // place of half step q
    auto after = [](int place) { return place == (PLACES - 1) * PLACE_BYTES ? 0 : place + PLACE_BYTES; };
    // a half step in `now`: its products, first with the reads of the next one's fragments between them, then with the loads and the addresses of the one after
    auto half = [&](const bf16x8_t (&a)[8], const bf16x8_t (&b)[8], bf16x8_t (&na)[8], bf16x8_t (&nb)[8]) {
      const int next = after(now), by = after(next) - next;
      const uint32_t to = lds + now + wid * 4096;
      short4_t part[2];
      each<64>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = mc, u = m >> 2, k = (m - 32) >> 1, l = (m - 32) >> 2;
        f32x4_t& c = acc[m >> 3][m & 7];
        if constexpr (m < 32) {
          part[m & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + (m & 2 ? ra[u] : rb[u]) + (m & 1) * 4 * 512));
          if constexpr (m & 1) (m & 2 ? na : nb)[u] = joined(part[0], part[1]);
          fixed();
        } else if constexpr (m & 1) {
          move_by(k < 8 ? rb[k & 7] : ra[k & 7], by), fixed();
        }
        if constexpr (m >= 32 && m % 4 == 2) mfma_load<(l < 4 ? 0 : HALF_BYTES) + (l & 3) * 1024>(c, b[m & 7], a[m >> 3], off[l], l < 4 ? pa : pb, to);
        else mfma(c, b[m & 7], a[m >> 3]);
        fixed();
      });
      now = next;
    };
#pragma unroll 1
    for (int q = 0; q < n; q += 2) {
      half(a0, b0, a1, b1);
      advance(q + PLACES + 1);
      there();
      half(a1, b1, a0, b0);
      advance(q + PLACES + 2);
      there();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (loads that nothing reads)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // (the last sums)
    settled<8>(acc);
  }
};

}  // namespace tile
}  // namespace nxd
