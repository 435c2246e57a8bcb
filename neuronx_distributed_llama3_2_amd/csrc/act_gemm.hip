// Products of a prompt's rows with the activation as their epilogue: y = silu(x Wg^T) (x Wu^T) for W = [Wg; Wu], and y = max(x W^T, 0)^2, bf16.
//
// A product and an elementwise pass after it write the product to memory and read it back; here a tile's results, rounded to bf16 as the product would
// leave them, take the activation on their way out.  The loop is that of gemm_tile.h (4 waves, 256 x 256 tile, one workgroup a CU, clock- and
// feed-bound); reductions are not split, so the sums are in the order of the reduction.
//
// The tiles are dealt to the XCDs in equal runs of an L2 band raster, in rounds of its 32 CUs.  What is left of a run after whole rounds would keep a few CUs for
// a whole tile's time, so these tiles are cut into 2 or 4 pieces of 128 or 64 rows when all CUs can have one.
// A workgroup has up to four tiles of rounds one after the other.  The ring of steps goes on from one to the next: during the last two steps of a tile the next one's
// first two are loaded, and its first sums need no registers cleared, so that a round costs no launch of workgroups, no first trip to memory and no wait for its stores, which
// are left in flight.  Results go out of the
// registers, 64 contiguous bytes of 16 rows a store; SwiGLU's gates and the columns they go with are in one wave for that.  (No more than four, so that CUs that
// something else holds keep no more than that waiting.)
// One tile a workgroup, results through LDS / now, us, one card in turn: SwiGLU of 8,192 columns, reduction 2,048: 2,304 rows 133 / 123; squared ReLU of 12,288, 2,048, 4,096 rows
// 154 / 143; rounds of 256 tiles of 512 20.4 / 16.9 each, of 2,048 51 / 47.5.
// Against a library product and the activation's own launch: act_pays in ops/gemm.py.
// The products are the library's to the bit there (its unsplit kernels sum in the same order).  Fewer rows: the library, with smaller tiles.
#include "gemm_tile.h"

namespace nxd {
namespace act {

using tile::BK;
using tile::BM;
using tile::BN;
enum Act { SWIGLU = 0, RELU2 = 1 };

struct Params {
  const uint16_t* x;   // [R][K]
  const uint16_t* w;   // [N][K]; SWIGLU: [2 N][K], the gate's rows and then the other's
  uint16_t* y;         // [R][N]
  int R, N, K;
  int rt, ct;          // tiles of rows, of columns
};

constexpr int XCDS = 8, XCD_CUS = 32, BAND = 8;   // row tiles of a band
constexpr int RUN = 4;                            // tiles of a workgroup at most

// An XCD's share of so many tiles, in rounds of its CUs: what is left after whole rounds is cut into 2 or 4 pieces of a tile when all CUs can have
// one (`cut` tiles), else it is a round too
struct Share {
  int tiles, rounds, cut, pieces;
  __host__ __device__ explicit Share(int tiles_) : tiles(tiles_) {
    const int tail = tiles % XCD_CUS;
    pieces = 4 * tail <= XCD_CUS ? 4 : 2 * tail <= XCD_CUS ? 2 : 1;
    cut = pieces > 1 ? tail : 0;
    rounds = (tiles - cut + XCD_CUS - 1) / XCD_CUS;
  }
  __host__ __device__ int runs(bool pipe) const { return pipe ? (rounds + RUN - 1) / RUN : rounds; }
  __host__ __device__ int workgroups(bool pipe) const { return runs(pipe) * XCD_CUS + cut * pieces; }
};

// PIPE (whole steps, two or more): a workgroup has up to RUN tiles, of rounds one after the other, and loads the next one's first steps during the last ones of a
// tile: its results go out of the registers while those are on their way.
template <int ACT, bool HALF, bool PIPE>
__global__ void __launch_bounds__(tile::THREADS, 1) kernel(Params p) {
  __shared__ __attribute__((aligned(16))) char smem[tile::LDS_BYTES];
  constexpr int COLS = ACT == SWIGLU ? BN / 2 : BN;   // results of a row
  const int total = p.rt * p.ct, xcd = blockIdx.x % XCDS, idx = blockIdx.x / XCDS;
  const int base = xcd * (total / XCDS) + min(xcd, total % XCDS);
  const Share share(total / XCDS + (xcd < total % XCDS));
  const int run = idx / XCD_CUS, runs = share.runs(PIPE);
  int items, first, pieces = 1, piece = 0;   // tiles of this workgroup, the XCD_CUS-th one after the other
  if (run < runs) {
    first = run * (PIPE ? RUN : 1) * XCD_CUS + idx % XCD_CUS;
    items = min(PIPE ? RUN : 1, (share.tiles - share.cut - first + XCD_CUS - 1) / XCD_CUS);
  } else {
    const int j = idx - runs * XCD_CUS;
    pieces = share.pieces, piece = j % pieces, first = share.tiles - share.cut + j / pieces;
    items = first < share.tiles ? 1 : 0;
  }
  if (items <= 0) return;
  int r0, r1, n0;
  auto place = [&](int k) __attribute__((always_inline)) {   // of the workgroup's k-th tile
    const int id = base + first + k * XCD_CUS, band = id / (BAND * p.ct), rem = id - band * BAND * p.ct, h = min(BAND, p.rt - band * BAND);
    const int rows = BM / pieces;
    r0 = __builtin_amdgcn_readfirstlane((band * BAND + rem % h) * BM + piece * rows), n0 = __builtin_amdgcn_readfirstlane(rem / h * COLS);
    r1 = min(p.R, r0 + rows);
  };
  place(0);
  if (r0 >= r1) return;   // (a piece past the last row)
  const auto x = [&](int row) { return p.x + (int64_t)row * p.K; };
  const auto w = [&](int row) { return p.w + (int64_t)row * p.K; };
  const auto cols = [&](int col) { return ACT == SWIGLU ? BN : min(BN, p.N - col); };
  tile::Loop<false> loop(smem, x(r0), p.K, r1 - r0, w(n0), p.K, cols(n0));
  const int lane = loop.lane, wid = loop.wid, wm = loop.wm, wn = loop.wn;
  // SwiGLU: a wave's 128 columns are 64 gates and the 64 others that they are multiplied with (of whole tiles: N % 128 == 0), 64 rows of the image each
  auto pairs = [&]() __attribute__((always_inline)) {
    if (ACT == SWIGLU) {
      const uint32_t by = (uint32_t)((wid & 1) * p.N + 64 * (wid >> 1) - 64 * wid) * (uint32_t)p.K * 2;
#pragma unroll
      for (int i = 8; i < 16; ++i) loop.off[i] += by;
    }
  };
  pairs();
  f32x4_t acc[8][8];
  // a tile's results, rounded as the product leaves them, with the activation: 8 columns of a row a lane, 64 contiguous bytes of 16 rows a store
  constexpr int FRAG_STORES = ACT == SWIGLU ? 2 : 4, STORES = 8 * FRAG_STORES;   // of a row fragment, of a tile
  auto out = [&](auto ok) __attribute__((always_inline)) {
    const int c0 = n0 + (ACT == SWIGLU ? 64 : 128) * wn + 8 * (lane >> 4);
    uint16_t* y = p.y + (int64_t)(r0 + 16 * wm + (lane & 15)) * p.N + c0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < 2 * FRAG_STORES; j += 2) {
        auto rounded = [&](int jj, float (&v)[8]) __attribute__((always_inline)) {
          unpack8(u32x4_t{pack2bf(acc[i][jj][0], acc[i][jj][1]), pack2bf(acc[i][jj][2], acc[i][jj][3]), pack2bf(acc[i][jj + 1][0], acc[i][jj + 1][1]),
                          pack2bf(acc[i][jj + 1][2], acc[i][jj + 1][3])}, v);
        };
        float v[8];
        rounded(j, v);
        if (ACT == SWIGLU) {
          float u[8];
          rounded(j + 4, u);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = v[e] * (1.f / (1.f + __expf(-v[e]))) * u[e];
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = v[e] > 0.f ? v[e] * v[e] : 0.f;
        }
        if (ok(r0 + 32 * i + 16 * wm + (lane & 15), c0 + 16 * j)) *reinterpret_cast<u32x4_t*>(y + (int64_t)32 * i * p.N + 16 * j) = pack8(v);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int steps = (p.K + BK - 1) / BK;
  if (PIPE && pieces == 1) {
    tile::Loop<false>::Frags<8> frags;
    loop.template begin<false>(frags, steps, false);
    bool stored = false;
#pragma unroll 1
    for (int k = 0; k < items; ++k) {
      const int R0 = r0, R1 = r1, N0 = n0;
      const bool another = k + 1 < items;
      if (another) place(k + 1);
      const int nr0 = r0, nr1 = r1, nn0 = n0;
      loop.template run_tile<STORES>(acc, frags, steps, stored, another, [&]() __attribute__((always_inline)) {
        loop.set(x(nr0), p.K, nr1 - nr0, w(nn0), p.K, cols(nn0));
        pairs();
      });
      r0 = R0, r1 = R1, n0 = N0;
      const bool whole = r1 - r0 == BM && n0 + COLS <= p.N;
      if (whole) out([](int, int) { return true; });
      else out([&](int row, int col) { return row < r1 && col < p.N; });
      stored = whole;
      r0 = nr0, r1 = nr1, n0 = nn0;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (loads that nothing reads)
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (!PIPE && r1 - r0 > BM / 2) loop.template run<8, HALF>(acc, steps, HALF);
  else if (r1 - r0 > BM / 4) loop.template run<4, HALF>(acc, steps, HALF);
  else loop.template run<2, HALF>(acc, steps, HALF);
  out([&](int row, int col) { return row < r1 && col < p.N; });
}

}  // namespace act

// y [R, N] = act(x [R, K] w^T): act 0 SwiGLU, w [2 N, K], N % 128 == 0; act 1 squared ReLU, w [N, K], N % 8 == 0; K % 32 == 0, contiguous, 16-byte aligned.
// -1: not such sizes
int act_gemm_launch(int act, const void* x, const void* w, void* y, int64_t R, int64_t N, int64_t K, hipStream_t stream) {
  if (act < 0 || act > 1 || R < 0 || R > INT32_MAX / 2 || N <= 0 || K <= 0 || K % 32 || N % (act ? 8 : 128)) return -1;
  // 32-bit offsets in a tile's operands: 256 rows, of SwiGLU's weights from the gate's to the other's
  if ((act ? tile::BN : N + tile::BN) * K * 2 > UINT32_MAX || N > INT32_MAX / 2) return -1;
  if (R == 0) return 0;
  act::Params p{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), (int)R, (int)N, (int)K,
                (int)ceil_div64(R, tile::BM), (int)ceil_div64(N, act ? tile::BN : tile::BN / 2)};
  const int64_t total = (int64_t)p.rt * p.ct;
  if (total > INT32_MAX / 64) return -1;
  const bool half = K % tile::BK != 0, pipe = !half && K >= 2 * tile::BK;
  int most = 0;
  for (int64_t tiles : {total / act::XCDS, ceil_div64(total, act::XCDS)}) {
    const int n = act::Share((int)tiles).workgroups(pipe);
    most = n > most ? n : most;
  }
  auto* f = act ? (half ? &act::kernel<act::RELU2, true, false> : pipe ? &act::kernel<act::RELU2, false, true> : &act::kernel<act::RELU2, false, false>)
                : (half ? &act::kernel<act::SWIGLU, true, false> : pipe ? &act::kernel<act::SWIGLU, false, true> : &act::kernel<act::SWIGLU, false, false>);
  hipLaunchKernelGGL(f, dim3((unsigned)most * act::XCDS), dim3(tile::THREADS), 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace nxd
