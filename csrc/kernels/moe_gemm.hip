// The experts' products for many pairs (moe.h), bf16: one BM x BN tile of one expert per workgroup on the
// tile core of the projection GEMM (gemm_sk_core.h). The up product gathers its rows of h by the sorted
// pair list while they are staged, and its epilogue is silu(gate) * up, or relu squared.
#include "gemm_sk_core.h"
#include "moe.h"

namespace {

// Work item g of the tiles' products: a tile and its columns
template <int BM, int BN, int UP, int NB>
LSA_DEVICE void moe_tile(unsigned char* smem, const MoeTile* __restrict__ tiles, int g, const int* __restrict__ order, int top,
                         const bf16_raw* __restrict__ A, const bf16_raw* __restrict__ W, SkParams& prm, const EpiArgs& ep) {
  using K_ = Kern<BM, BN, UP == MOE_GLU ? EPI_SWIGLU : EPI_STORE, NB, UP != MOE_DOWN>;
  int ti, nt;
  tile_coords(prm, g, ti, nt);
  const MoeTile tile = tiles[ti];
  if (tile.expert < 0) return;
  prm.M = tile.start + tile.count;
  K_ k;
  k.smem = smem;
  k.A = A;
  k.W = W + (size_t)tile.expert * prm.N * prm.K;
  k.p = &prm;
  k.order = order;
  k.per = top;
  k.tid = threadIdx.x;
  k.lane = threadIdx.x & 63;
  k.w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  k.wr = k.w / K_::WN;
  k.wc = k.w % K_::WN;
  k.group = k.w >> 2;
  f32x4_t acc[K_::FM][K_::FN];
#pragma unroll
  for (int i = 0; i < K_::FM; ++i)
#pragma unroll
    for (int j = 0; j < K_::FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  k.run_segment(acc, tile.start, nt, 0, prm.NKT, []() {});
  k.epilogue(ep, acc, tile.start, nt, 0);
}

template <int BM, int BN, int UP, int NB>
__global__ __launch_bounds__(NTHR) void moe_gemm_kernel(const MoeTile* __restrict__ tiles, int n_tiles,
                                                         const int* __restrict__ order, int top,
                                                         const bf16_raw* __restrict__ A, const bf16_raw* __restrict__ W,
                                                         SkParams prm, EpiArgs ep) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[Geo<BM, BN, NB>::SMEM];
  // Workgroups of one XCD get consecutive work; group_m tiles (mostly of one expert) share a column sweep. The table is as
  // long as it could have to be (an eighth longer than its tiles for 25512 pairs and 32 experts): shared out by its length,
  // the XCD that got the missing tiles stood idle while the others had a round more (up 257 -> 221 us, down 146 -> 131).
  const int used = tiles[0].used;
  if (used > 0 && used < prm.MT) prm.MT = used;
  const int G = prm.MT * prm.NT, q = G / 8, r = G % 8, x = blockIdx.x % 8;
  if ((int)blockIdx.x >= G) return;
  moe_tile<BM, BN, UP, NB>(smem, tiles, (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + blockIdx.x / 8, order, top, A, W, prm,
                           ep);
}

// The same with the height that the pairs' counts chose (MoePick): one of four bodies. How many rounds the tiles make is known when
// they are counted and not before: 32 experts of 1024 x 2048 with 900 pairs each are 127 tiles of 256 rows, four rounds in either
// product, and 96 of 320, three (365 -> 330 us); with 700 each 96 and 96. One workgroup a CU takes tile after tile of its
// XCD's (as above): with one for as many as there could be of the lowest, those too many held a CU for 1.5 us each and made 470 us of 64
// experts with 1100 pairs 495. Four lists of experts, 200 to 1500 pairs each, evenly and unevenly drawn (profiles/cost_moe_bf16.csv): 0.94
// times the time of 128 rows up to 320 pairs an expert and 256 above, which the host chose (0.72 to 1.03 times; by the mean it could
// get to 0.98). Tiles of several heights in one table, to fill all but 64 rows of an expert's, were slower on average (0.97).
template <int BM, int UP>
LSA_DEVICE void moe_tiles(unsigned char* smem, const MoeTile* __restrict__ tiles, const int* __restrict__ order, int top,
                          const bf16_raw* __restrict__ A, const bf16_raw* __restrict__ W, SkParams& prm, const EpiArgs& ep) {
  const int G = prm.MT * prm.NT, q = G / 8, r = G % 8, x = blockIdx.x % 8, step = gridDim.x / 8;
  const int first = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q, end = first + (x < r ? q + 1 : q);
  for (int g = first + blockIdx.x / 8; g < end; g += step) {
    moe_tile<BM, 256, UP, 2>(smem, tiles, g, order, top, A, W, prm, ep);
    __syncthreads();
  }
}
template <int UP>
__global__ __launch_bounds__(NTHR) void moe_pick_kernel(const MoeTile* __restrict__ tiles, const int* __restrict__ order, int top,
                                                         const bf16_raw* __restrict__ A, const bf16_raw* __restrict__ W,
                                                         SkParams prm, EpiArgs ep) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[Geo<MOE_ROWS[3], 256, 2>::SMEM];
  const int used = __builtin_amdgcn_readfirstlane(tiles[0].used);
  prm.MT = min(prm.MT, used & ((1 << MOE_HEIGHT) - 1));
  switch (used >> MOE_HEIGHT) {
    case 0: return moe_tiles<MOE_ROWS[0], UP>(smem, tiles, order, top, A, W, prm, ep);
    case 1: return moe_tiles<MOE_ROWS[1], UP>(smem, tiles, order, top, A, W, prm, ep);
    case 2: return moe_tiles<MOE_ROWS[2], UP>(smem, tiles, order, top, A, W, prm, ep);
    default: return moe_tiles<MOE_ROWS[3], UP>(smem, tiles, order, top, A, W, prm, ep);
  }
}

template <int BM, int BN, int UP, int NB>
int launch(const MoeTile* t, int n_tiles, const int* order, int top, const void* A, const void* W, SkParams prm,
           const EpiArgs& ep, hipStream_t s) {
  prm.MT = n_tiles;
  prm.NT = prm.N / BN;
  prm.group_m = 8;
  moe_gemm_kernel<BM, BN, UP, NB><<<n_tiles * prm.NT, NTHR, 0, s>>>(t, n_tiles, order, top, (const bf16_raw*)A,
                                                                     (const bf16_raw*)W, prm, ep);
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

template <int UP>
int launch_pick(const MoeTile* t, int n_tiles, const int* order, int top, const void* A, const void* W, SkParams prm,
                const EpiArgs& ep, hipStream_t s) {
  prm.MT = n_tiles;
  prm.NT = prm.N / 256;
  prm.group_m = 8;
  moe_pick_kernel<UP><<<256, NTHR, 0, s>>>(t, order, top, (const bf16_raw*)A, (const bf16_raw*)W, prm, ep);
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

}  // namespace

// As lsa_moe_gemm (bf16) for tiles of at most tile_rows = 128 / 256 pairs, or 0: of the height in the table (lsa_moe_group with
// heights; N % 256 == 0); a_rows: rows of A
extern "C" int lsa_moe_gemm_big(int up, const void* tiles, int n_tiles, int tile_rows, const int* order, int top,
                                const void* A, int a_rows, int lda, const void* W, int N, int K, void* out, int ldo,
                                hipStream_t s) {
  if (n_tiles < 1 || n_tiles > (1 << 20) || top < 1 || N < 128 || N % 128 || K < BK || K % BK || lda < K || lda % 8 ||
      up < MOE_DOWN || up > MOE_RELU2 || ldo < (up == MOE_GLU ? N / 2 : N) || ldo % 8 || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)out) % 16 || !order || !tiles ||
      (tile_rows != 128 && tile_rows != 256 && (tile_rows || N % 256)) || (size_t)a_rows * lda * 2 >= (1ull << 31))
    return LSA_BAD_SHAPE;
  SkParams prm = {};
  prm.N = N;
  prm.K = K;
  prm.lda = lda;
  prm.NKT = K / BK;
  EpiArgs ep = {};
  ep.out = (bf16_raw*)out;
  ep.ldo = ldo;
  ep.act = up == MOE_RELU2 ? 2 : 0;
  const MoeTile* t = (const MoeTile*)tiles;
#define LSA_B(BM, BN, NB)                                                                             \
  return up == MOE_GLU ? launch<BM, BN, MOE_GLU, NB>(t, n_tiles, order, top, A, W, prm, ep, s)        \
         : up          ? launch<BM, BN, MOE_RELU2, NB>(t, n_tiles, order, top, A, W, prm, ep, s)      \
                       : launch<BM, BN, MOE_DOWN, NB>(t, n_tiles, order, top, A, W, prm, ep, s)
  if (!tile_rows)
    return up == MOE_GLU ? launch_pick<MOE_GLU>(t, n_tiles, order, top, A, W, prm, ep, s)
           : up          ? launch_pick<MOE_RELU2>(t, n_tiles, order, top, A, W, prm, ep, s)
                         : launch_pick<MOE_DOWN>(t, n_tiles, order, top, A, W, prm, ep, s);
  if (tile_rows == 256) {
    if (N % 256 == 0) LSA_B(256, 256, 2);
    LSA_B(256, 128, 2);
  }
  if (N % 256 == 0) LSA_B(128, 256, 2);
  LSA_B(128, 128, 3);
#undef LSA_B
}
