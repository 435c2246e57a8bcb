// Products of a prompt's rows with the activation as their epilogue: y = silu(x Wg^T) (x Wu^T) for W = [Wg; Wu], and y = max(x W^T, 0)^2, bf16.
//
// A product and an elementwise pass after it write the product to memory and read it back; here a tile's results, rounded to bf16 as the product would
// leave them, take the activation on their way out.  The loop is that of gemm_tile.h (4 waves, 256 x 256 tile, one workgroup a CU, clock- and
// feed-bound); reductions are not split, so the sums are in the order of the reduction.
//
// The tiles are dealt to the XCDs in equal runs of an L2 band raster.  What is left of a run after whole rounds of its 32 CUs would keep a few CUs for
// a whole tile's time, so these tiles are cut into 2 or 4 pieces of 128 or 64 rows when all CUs can have one.
// Against a library product and the activation's own launch, us, weights from memory: SwiGLU of 8,192 columns, reduction 2,048: 1,024 rows 68 -> 62, 2,304 150 ->
// 152 (147 on another card), 4,096 232 -> 231; squared ReLU of 12,288, 2,048: 1,024 rows 60 -> 60, 4,096 182 -> 170 (1.2 PFLOP/s, the product alone at 1.4 in the library).
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

// of so many tiles of an XCD: those of whole rounds, and the pieces of each one left
__host__ __device__ inline int whole_of(int share) { return share / XCD_CUS * XCD_CUS; }
__host__ __device__ inline int pieces_of(int tail) { return 4 * tail <= XCD_CUS ? 4 : 2 * tail <= XCD_CUS ? 2 : 1; }

template <int ACT, bool HALF>
__global__ void __launch_bounds__(tile::THREADS, 1) kernel(Params p) {
  __shared__ __attribute__((aligned(16))) char smem[tile::LDS_BYTES];
  constexpr int COLS = ACT == SWIGLU ? BN / 2 : BN;   // results of a row
  const int total = p.rt * p.ct, xcd = blockIdx.x % XCDS, idx = blockIdx.x / XCDS;
  const int share = total / XCDS + (xcd < total % XCDS), base = xcd * (total / XCDS) + min(xcd, total % XCDS);
  const int whole = whole_of(share), tail = share - whole;
  int pieces = 1, piece = 0, id = base + idx;
  if (idx >= whole) {
    pieces = pieces_of(tail);
    const int j = idx - whole;
    if (j >= tail * pieces) return;
    piece = j % pieces;
    id = base + whole + j / pieces;
  }
  const int band = id / (BAND * p.ct), rem = id - band * BAND * p.ct, h = min(BAND, p.rt - band * BAND);
  const int rows = BM / pieces, r0 = (band * BAND + rem % h) * BM + piece * rows, n0 = rem / h * COLS;
  const int r1 = min(p.R, r0 + rows);
  if (r0 >= r1) return;   // (a piece past the last row)
  tile::Loop<false> loop(smem, p.x + (int64_t)r0 * p.K, p.K, r1 - r0, p.w + (int64_t)n0 * p.K, p.K, ACT == SWIGLU ? BN : min(BN, p.N - n0));
  if (ACT == SWIGLU && loop.wid >= 2) {   // rows 128 .. of the weights' tile: the other half's (of whole tiles: N % 128 == 0)
#pragma unroll
    for (int i = 8; i < 16; ++i) loop.off[i] += (uint32_t)(p.N - BN / 2) * (uint32_t)p.K * 2;
  }
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int steps = (p.K + BK - 1) / BK;
  if (r1 - r0 > BM / 2) loop.template run<8, HALF>(acc, steps, HALF);
  else if (r1 - r0 > BM / 4) loop.template run<4, HALF>(acc, steps, HALF);
  else loop.template run<2, HALF>(acc, steps, HALF);
  const int lane = loop.lane, wid = loop.wid, wm = loop.wm, wn = loop.wn;

  // ---- results through LDS, a wave's 128 x 128 in 32 KB of its own (16-byte chunks XORed with the row)
  __syncthreads();
  char* own = smem + wid * (tile::LDS_BYTES / 4);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const int r = 16 * i + (lane & 15), c = tile::col<false>(0, j, lane);
      *reinterpret_cast<u32x4_t*>(own + r * 256 + 16 * ((c >> 3) ^ (r & 15))) =
          u32x4_t{pack2bf(acc[i][j][0], acc[i][j][1]), pack2bf(acc[i][j][2], acc[i][j][3]),
                  pack2bf(acc[i][j + 1][0], acc[i][j + 1][1]), pack2bf(acc[i][j + 1][2], acc[i][j + 1][3])};
    }
  if (ACT == SWIGLU) __syncthreads();   // a wave takes half the rows of its gates and of its neighbour's columns (or the other way round)
  else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const char* gate = ACT == SWIGLU ? smem + (wid & ~1) * (tile::LDS_BYTES / 4) : own;
  const int c0 = (ACT == SWIGLU ? 0 : 128 * wn) + 8 * (lane & 15);
#pragma unroll 4
  for (int k = 0; k < (ACT == SWIGLU ? 16 : 32); ++k) {
    const int r = 4 * (ACT == SWIGLU ? 16 * wn + k : k) + (lane >> 4), row = r0 + 32 * (r >> 4) + 16 * wm + (r & 15);
    const char* at = gate + r * 256 + 16 * ((lane & 15) ^ (r & 15));
    float v[8];
    unpack8(*reinterpret_cast<const u32x4_t*>(at), v);
    if (ACT == SWIGLU) {
      float u[8];
      unpack8(*reinterpret_cast<const u32x4_t*>(at + tile::LDS_BYTES / 4), u);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * (1.f / (1.f + __expf(-v[e]))) * u[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] > 0.f ? v[e] * v[e] : 0.f;
    }
    if (row < r1 && n0 + c0 < p.N) *reinterpret_cast<u32x4_t*>(p.y + (int64_t)row * p.N + n0 + c0) = pack8(v);
  }
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
  int most = 0;
  for (int share : {(int)(total / act::XCDS), (int)ceil_div64(total, act::XCDS)}) {
    const int whole = act::whole_of(share), tail = share - whole, n = whole + tail * act::pieces_of(tail);
    most = n > most ? n : most;
  }
  const bool half = K % tile::BK != 0;
  auto* f = act ? (half ? &act::kernel<act::RELU2, true> : &act::kernel<act::RELU2, false>)
                : (half ? &act::kernel<act::SWIGLU, true> : &act::kernel<act::SWIGLU, false>);
  hipLaunchKernelGGL(f, dim3((unsigned)most * act::XCDS), dim3(tile::THREADS), 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace nxd
