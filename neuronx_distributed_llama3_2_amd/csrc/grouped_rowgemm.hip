// Grouped (ragged-M) MoE expert GEMMs with 256 x 256 tiles on gfx950 MFMA: the forward and the
// input gradient of the expert MLPs over expert-sorted rows (expert e owns rows offs[e] ..
// offs[e+1], read on the device: no host sync, hipGraph-capturable).
//
//   FWD   y[m, n]  = sum_k x[m, k]  W[e][k, n]       A = x  [rows][K] , B = W[e] [K][N]  (k-major)
//   DGRAD dx[m, k] = sum_n dy[m, n] W[e][k, n]       A = dy [rows][N] , B = W[e] read as [k][n] rows
//
// Reference: the expert MLP of modules/moe/expert_mlps.py:169-265 (all-experts einsum / capacity
// drop); here only the chosen rows are computed.  The weight gradients of the same layer run on the
// token-major wgrad kernel (csrc/wgrad_gemm.hip, grouped mode).
//
// Structure: the loop of gemm_tile.h (4 waves, 256 x 256 tile, one workgroup per CU).  A and DGRAD's B are contiguous along the
// reduction (ROW images), FWD's B along the columns (TR).  Each workgroup finds its (expert, row tile) by a scan of the offsets;
// the tiles are numbered in an L2 band raster over (row tile, column tile).
// 8,192 rows of 8 experts, 4096 -> 28672 and 14336 -> 4096, us: FWD 2,170 -> 1,934 and 1,049 -> 943, DGRAD 2,263 -> 1,770 and
// 1,057 -> 832 (two ping-pong groups of 4 waves, grid of the worst case's tiles; the loop's ring since: gemm_tile.h).
// Few rows (bound by the weights' bytes): a tile of at most 128 rows loads and leaves in memory only the rows that there are.  16 rows of 8
// experts, FWD / DGRAD us, two groups of 4 waves -> here, and with all rows loaded and left: 4096 -> 28672 414 / 422 -> 414 / 387, 444 / 420; 14336 -> 4096
// 311 / 307 -> 214 / 217, 245 / 245; 4096 -> 1024 93 / 91 -> 55 / 52, 76 / 72.  Such tiles have a ring of three or four steps of both operands
// (run_few in gemm_tile.h), and split ones leave their sums past the L2: 4096 -> 28672 389 / 369 -> 318 / 350.
#include "gemm_tile.h"

#include <cstdlib>

namespace nxd {
namespace grg {

using tile::BK;
using tile::BM;
using tile::BN;
constexpr int NT = tile::THREADS;
enum Mode { FWD = 0, DGRAD = 1 };

struct Params {
  const uint16_t* a;    // [rows][lda]
  const uint16_t* b;    // W [E][K][N]
  uint16_t* c;          // [rows][ldc]
  const int* offs;      // [E + 1]
  int E, rows;
  int red;              // reduction length (FWD: K, DGRAD: N)
  int ncols;            // output columns (FWD: N, DGRAD: K)
  int64_t lda, ldb, ldc, b_es;
  int rt, nt;           // worst-case row tiles, column tiles
  int band;
  // Sums of the tiles left over from whole rounds of an XCD's CUs, their reductions in parts (nullable: never), and zeroed counters
  // (left zeroed): so many places an XCD, of so many fragments of 32 rows (room_for)
  float* ws;
  int* tickets;
  int slots, frags;
};

constexpr int XCDS = 8, XCD_CUS = 32;
// Parts of a tile at most; reduction steps of a part at least: writing a part's sums and reading them all back takes 15-30 us, 32
// steps take 35-55
constexpr int MAX_PARTS = 8, MIN_STEPS = 32;
constexpr int FRAG_FLOATS = 32 * BN;   // 32 rows of a tile

// Room for what may be split, by what is known of the rows: an expert's tile has no more rows than there are, and of the places one XCD's
// tiles need all (32 CUs) or, where there are few tiles, their parts.  8 experts, reduction 4096, columns 256 / 1,024 / 28,672: 16 rows 0.5, 2.1,
// 8.4 MB, 256 rows 8.4, 21, 67 MB (for a whole tile a CU always 67).
static void room_for(int red, int ncols, int rows, int E, int* slots, int* frags) {
  const int most = ceil_div(red, BK) / MIN_STEPS, parts = most < MAX_PARTS ? most : MAX_PARTS;
  const int64_t tiles = (int64_t)ceil_div(ncols, BN) * (rows / BM + (E < rows ? E : rows)), places = ceil_div64(tiles, XCDS) * parts;
  *slots = parts < 2 || rows <= 0 ? 0 : (int)(places < XCD_CUS ? places : XCD_CUS);
  *frags = rows > BM / 2 ? BM / 32 : ceil_div(rows, 32);
}

// HALF: the reduction ends with half a step
template <int MODE, bool HALF>
__global__ void __launch_bounds__(NT, 1) rowgemm_kernel(Params p) {
  __shared__ __attribute__((aligned(16))) char smem[tile::LDS_BYTES];
  // The tiles that there are (expert by expert), in equal shares for the XCDs (a grid of the worst case's left one with hardly any:
  // 36 of 40 row tiles x 16).  What is left of a share after whole rounds of 32 CUs is split along the reduction so that the
  // last round's CUs all have some: 72 tiles a share, 8192 rows of 8 experts x 4096 columns, take 2.25 rounds instead of 3.
  int real = 0;
  for (int i = 0; i < p.E; ++i) real += (max(p.offs[i + 1] - p.offs[i], 0) + BM - 1) / BM;
  const int total = real * p.nt, xcd = blockIdx.x % XCDS, idx = blockIdx.x / XCDS;
  const int share = total / XCDS + (xcd < total % XCDS), base = xcd * (total / XCDS) + min(xcd, total % XCDS);
  const int whole = share / XCD_CUS * XCD_CUS, tail = share - whole;
  const int steps = (p.red + BK - 1) / BK;
  int parts = 1, part = 0, id = base + idx;
  if (p.ws && tail > 0) parts = max(1, min(min(p.slots / tail, MAX_PARTS), steps / MIN_STEPS));
  if (idx >= whole) {
    const int j = idx - whole;
    if (j >= tail * parts) return;
    part = j % parts;
    id = base + whole + j / parts;
  } else {
    parts = 1;
  }
  int rt, ct;
  {
    const int kb = p.band, bnd = id / (kb * p.nt), rem = id - bnd * kb * p.nt;
    const int h = min(kb, real - bnd * kb);
    rt = bnd * kb + rem % h;
    ct = rem / h;
  }
  // (expert, row range) of row tile rt: tiles are numbered expert by expert
  int e = -1, r0 = 0, r1 = 0;
  {
    int acc = 0;
    for (int i = 0; i < p.E; ++i) {
      const int g0 = p.offs[i], g1 = p.offs[i + 1];
      const int nt_e = g1 > g0 ? (g1 - g0 + BM - 1) / BM : 0;
      if (rt < acc + nt_e) {
        e = i;
        r0 = g0 + (rt - acc) * BM;
        r1 = min(g1, r0 + BM);
        break;
      }
      acc += nt_e;
    }
  }
  if (e < 0) return;   // (not reached)
  const int n0 = ct * BN;
  // this part's reduction steps
  const int per = (steps + parts - 1) / parts, first = min(part * per, steps), nk = min(per, steps - first);
  e = __builtin_amdgcn_readfirstlane(e), r0 = __builtin_amdgcn_readfirstlane(r0), r1 = __builtin_amdgcn_readfirstlane(r1);
  const uint16_t* bw = p.b + (int64_t)e * p.b_es;
  tile::Loop<MODE == FWD> loop(smem, p.a + (int64_t)r0 * p.lda + first * BK, p.lda, r1 - r0,
                                      MODE == FWD ? bw + (int64_t)first * BK * p.ldb + n0 : bw + (int64_t)n0 * p.ldb + first * BK, p.ldb,
                                      min(BN, p.ncols - n0));
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // (an expert's last tile: with at most half the rows half the work, with a quarter a quarter: 8 experts of about 1,024 rows each, of which half have a
  // few rows more, 4096 -> 28672 1,744 -> 1,681 us)
  const bool end = HALF && part == parts - 1, beside = r0 > p.offs[e];   // (beside: run_few)
  if (nk > 0) {
    if (r1 - r0 > BM / 2) loop.template run<8, HALF>(acc, nk, end);
    else if (r1 - r0 > BM / 4) loop.template run<4, HALF>(acc, nk, end, beside);
    else loop.template run<2, HALF>(acc, nk, end, beside);
  }
  const int lane = loop.lane, wid = loop.wid, wm = loop.wm, wn = loop.wn;

  // ---- results through LDS, a wave's 128 x 128 in 32 KB of its own (16-byte chunks XORed with the row): 256 contiguous bytes of a row
  // a store
  char* own = smem + wid * (tile::LDS_BYTES / 4);
  auto put = [&](int i, const f32x4_t (&sums)[8]) __attribute__((always_inline)) {   // of row fragment i
#pragma unroll
    for (int j = 0; j < 8; j += MODE == FWD ? 1 : 2) {
      const int r = 16 * i + (lane & 15), c = tile::col<MODE == FWD>(0, j, lane);
      const u32x2_t lo = {pack2bf(sums[j][0], sums[j][1]), pack2bf(sums[j][2], sums[j][3])};
      char* to = own + r * 256 + 16 * ((c >> 3) ^ (r & 15));
      if (MODE == FWD) *reinterpret_cast<u32x2_t*>(to + 2 * (c & 7)) = lo;
      else *reinterpret_cast<u32x4_t*>(to) = u32x4_t{lo[0], lo[1], pack2bf(sums[j + 1][0], sums[j + 1][1]), pack2bf(sums[j + 1][2], sums[j + 1][3])};
    }
  };
  // ---- parts of a tile: sums to memory; the last part to come adds them up, in their order.  They are stored past the L2 (write-through) and waited for: a release
  // fence ahead of the ticket writes back all of an XCD's L2 for each part.  us, with the fence / now: 16 rows of each of 8 experts 4096 -> 28672 350 / 318, input gradient
  // 383 / 350, 100 rows 390 / 357 and 411 / 375; 8,192 rows 14336 -> 4096 791 / 766, 28672 -> 4096 (input gradient) 1,504 / 1,486.
  if (parts > 1) {
    const int slot = xcd * p.slots + idx - whole - part;   // of the tile's first part
    const int64_t place = (int64_t)p.frags * FRAG_FLOATS;
    float* sums = p.ws + slot * place;
    const int have = r1 - r0 > BM / 2 ? 8 : (r1 - r0 + 31) / 32;       // fragments with rows, or all
    // (each wave's sums lie together: a fragment's of all waves beside each other, 1,024 rows of 4 experts, 8192 -> 256, 99 -> 111 us)
    auto at = [&](int s, int i, int j) { return reinterpret_cast<uint64_t*>(sums + s * place) + ((wid * p.frags + i) * 8 + j) * 128 + lane; };
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < have) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x2_t two = {acc[i][j][2 * h], acc[i][j][2 * h + 1]};
            __hip_atomic_store(at(part, i, j) + 64 * h, __builtin_bit_cast(uint64_t, two), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (each wave's own, and the barrier: all of them are there before the ticket)
    __syncthreads();
    int* last = reinterpret_cast<int*>(smem);
    if (threadIdx.x == 0) {
      *last = __hip_atomic_fetch_add(p.tickets + slot, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
      if (*last) __hip_atomic_store(p.tickets + slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();   // (*last has been read by all)
    // Row fragment by row fragment, straight to the results, and four loads of a fragment (8 KB of a wave's) on their way at any time, over to the next one: with all
    // fragments of a part and then the next part, a part of 256 KB took 14 us.  Reduction x columns, us, so / now: 8,192 uneven rows of 8 experts 14336 x 4096 773 / 755, 28672 x
    // 4096 (input gradient) 1,499 / 1,478; one expert, 4,096 rows 12288 x 2048 171 / 162, 1,000 rows 16384 x 2048 (8 parts) 174 / 92, 512 rows 8192 x 2048 92 / 60.
    // P: parts, or more (the last one again, not used).
    auto add_up = [&](auto np) __attribute__((always_inline)) {
      constexpr int P = np, RING = 4, STEPS = P > RING ? P : RING;
      f32x4_t v[RING][8], row[8];
      auto fetch = [&](int u, int s, int i) __attribute__((always_inline)) {
        const uint64_t* from = at(min(s, parts - 1), min(i, have - 1), 0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const f32x2_t lo = __builtin_bit_cast(f32x2_t, from[128 * j]), hi = __builtin_bit_cast(f32x2_t, from[128 * j + 64]);
          v[u][j] = f32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
      };
#pragma unroll
      for (int u = 0; u < RING; ++u) fetch(u, u % P, u / P);
#pragma unroll 1
      for (int i = 0; i < have; i += STEPS / P) {
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
          const bool there = u % P < parts;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const f32x4_t sum = row[j] + v[u % RING][j];
            row[j] = u % P == 0 ? v[u % RING][j] : there ? sum : row[j];
          }
          fetch(u % RING, (u + RING) % P, i + (u + RING) / P);
          if (u % P == P - 1) put(i + u / P, row);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (parts == 2) add_up(std::integral_constant<int, 2>{});
    else if (parts <= 4) add_up(std::integral_constant<int, 4>{});
    else add_up(std::integral_constant<int, 8>{});
  } else {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) put(i, acc[i]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int c0 = 128 * wn + 8 * (lane & 15);
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    const int r = 4 * k + (lane >> 4), row = r0 + 32 * (r >> 4) + 16 * wm + (r & 15);
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(own + r * 256 + 16 * ((lane & 15) ^ (r & 15)));
    if (row < r1 && n0 + c0 < p.ncols) *reinterpret_cast<u32x4_t*>(p.c + (int64_t)row * p.ldc + n0 + c0) = v;
  }
}

static int band_rows() {
  static const int b = [] {
    const char* e = getenv("NXD_GRG_BAND");   // 8: +2..7 % over 4 on most Mixtral shapes (r3_grouped_rowgemm_variants)
    const int v = e ? atoi(e) : 8;
    return v > 0 ? v : 8;
  }();
  return b;
}

}  // namespace grg

// Floats of ws and the number of tickets for a product of `rows` rows of E experts, a reduction of `red` and `ncols` columns (0: its tiles are
// never split)
int64_t grouped_rowgemm_workspace(int red, int ncols, int rows, int E, int* tickets) {
  int slots, frags;
  grg::room_for(red, ncols, rows, E, &slots, &frags);
  *tickets = grg::XCDS * slots;
  return (int64_t)*tickets * frags * grg::FRAG_FLOATS;
}

// mode 0 FWD:   a = x [rows, K],  W [E, K, N], c = y  [rows, N]
// mode 1 DGRAD: a = dy [rows, N], W [E, K, N], c = dx [rows, K]
// Requires the reduction length % 32 == 0 and K, N % 8 == 0 (checked; returns -1 otherwise, the
// caller then takes the 128-tile kernel).  Rows past offs[E] are not written.
// ws, tickets: of grouped_rowgemm_workspace()'s sizes (tickets zeroed), or null: unsplit.
int grouped_rowgemm_launch(int mode, const void* a, const void* w, void* c, const int* offs, int E, int rows, int K,
                           int N, hipStream_t stream, float* ws, int* tickets) {
  if (E <= 0 || K <= 0 || N <= 0 || rows < 0 || K % 8 || N % 8) return -1;
  grg::Params p{};
  p.a = static_cast<const uint16_t*>(a);
  p.b = static_cast<const uint16_t*>(w);
  p.c = static_cast<uint16_t*>(c);
  p.offs = offs;
  p.E = E;
  p.rows = rows;
  p.b_es = (int64_t)K * N;
  p.ldb = N;
  if (mode == grg::FWD) {
    p.red = K; p.ncols = N; p.lda = K; p.ldc = N;
  } else if (mode == grg::DGRAD) {
    p.red = N; p.ncols = K; p.lda = N; p.ldc = K;
  } else {
    return -1;
  }
  if (p.red % 32) return -1;
  if (rows == 0) return 0;
  p.rt = ceil_div(rows, grg::BM) + E;
  p.nt = ceil_div(p.ncols, grg::BN);
  p.band = grg::band_rows();
  grg::room_for(p.red, p.ncols, rows, E, &p.slots, &p.frags);
  p.ws = tickets && p.slots ? ws : nullptr;
  p.tickets = tickets;
  const int64_t nwg = (ceil_div64((int64_t)p.rt * p.nt, grg::XCDS) + (p.ws ? grg::XCD_CUS : 0)) * grg::XCDS;
  if (nwg > INT32_MAX) return -2;
  const bool half = p.red % grg::BK != 0;
  auto* f = mode == grg::FWD ? (half ? &grg::rowgemm_kernel<grg::FWD, true> : &grg::rowgemm_kernel<grg::FWD, false>)
                             : (half ? &grg::rowgemm_kernel<grg::DGRAD, true> : &grg::rowgemm_kernel<grg::DGRAD, false>);
  hipLaunchKernelGGL(f, dim3((unsigned)nwg), dim3(grg::NT), 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace nxd
