// Projections of the fp32 engine: C[M][N] = A[M][K] . W[N][K]^T with products and sums of fp32 accuracy (f32_core.h). Epilogues:
// store, or the gated unit over interleaved 16-row gate / up blocks (ops/packing.py fuse_gate_up), as EPI_STORE /
// EPI_SWIGLU / EPI_GEGLU of the bf16 GEMMs.
#include "epilogue.h"
#include "f32_core.h"

namespace {

// epi_store1 with fp32 in the place of bf16 (ep.out, ep.gate)
LSA_DEVICE void store_f32(const EpiArgs& ep, int m, int n, float v) {
  v += epi_bias(ep, n);
  if (ep.act && epi_acts(ep, n)) v = epi_activate(ep.act, v);
  if (!ep.out32 || n < ep.col32) {
    ((float*)ep.out)[(size_t)m * ep.ldo + n] = v;
    return;
  }
  float* o = ep.out32 + (size_t)m * ep.ldo32 + (n - ep.col32);
  if (!ep.gate) *o = v;
  else if (n < ep.cols) *o += sigmoid(((const float*)ep.gate)[(size_t)m * ep.ldg + n]) * v;
}

// gate and up value of columns n and n + 16 (n % 32 < 16)
template <int EPI>
LSA_DEVICE void store_glu(const EpiArgs& ep, int m, int n, float g, float u) {
  ep.out32[(size_t)m * ep.ldo + (n >> 5) * 16 + (n & 15)] = epi_glu<EPI>(ep, g + epi_bias(ep, n), u + epi_bias(ep, n + 16));
}

template <int EPI, int MT, int NT, int NW>
__global__ __launch_bounds__(NW * 64) void stream_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                             int M, int N, int K, EpiArgs ep) {
  using S = F32Stream<MT, NT, NW>;
  __shared__ __attribute__((aligned(16))) float s_acc[S::LDS];
  const int lane = threadIdx.x & 63, n0 = blockIdx.x * NT * 16, m0 = blockIdx.y * MT * 16;
  const float *ar[MT], *wr[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)  // rows past M and columns past N are computed and not stored
    ar[m] = A + (size_t)min(m0 + m * 16 + (lane & 15), M - 1) * lda + 4 * (lane >> 4);
#pragma unroll
  for (int n = 0; n < NT; ++n) wr[n] = f32_block(W, min(n0 / 16 + n, N / 16 - 1), K);
  S::run(ar, wr, K, s_acc);
  const int rows = min(MT * 16, M - m0);
  if constexpr (epi_gated(EPI)) {
    for (int t = threadIdx.x; t < rows * NT * 8; t += NW * 64) {
      const int m = t / (NT * 8), c = t % (NT * 8), n = (c >> 4) * 32 + (c & 15);
      if (n0 + n < N) store_glu<EPI>(ep, m0 + m, n0 + n, S::sum(s_acc, m, n), S::sum(s_acc, m, n + 16));
    }
  } else {
    for (int t = threadIdx.x; t < rows * NT * 16; t += NW * 64) {
      const int m = t / (NT * 16), n = t % (NT * 16);
      if (n0 + n < N) store_f32(ep, m0 + m, n0 + n, S::sum(s_acc, m, n));
    }
  }
}

template <int EPI, int MT, int NW, int KG>
__global__ __launch_bounds__(NW * KG * 64) void tile_f32_kernel(
    const float* __restrict__ A, int lda, const float* __restrict__ W, int M, int N, int K, int mt, int nt, int whole, int S,
    float* slab, unsigned* counters, EpiArgs ep) {
  using T = F32Split<MT, NW, KG>;
  __shared__ u32x4_t lds[T::LDS];
  __shared__ int s_last;
  // workgroups of one XCD get consecutive work; 8 row tiles share a sweep over the columns
  const int part = (int)blockIdx.x - whole, q = whole / 8, r = whole % 8, x = blockIdx.x % 8;
  const int g = part >= 0 ? whole + part / S : (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + blockIdx.x / 8;
  const int first = g / (8 * nt) * 8, gm = min(mt - first, 8), in = g - first * nt;
  const int m0 = (first + in % gm) * T::BM, n0 = in / gm * T::BN;
  const int p = part >= 0 ? part % S : 0, u0 = part >= 0 ? K / 32 * p / S : 0, u1 = part >= 0 ? K / 32 * (p + 1) / S : K / 32;
  const float* wr[T::NT];
#pragma unroll
  for (int n = 0; n < T::NT; ++n) wr[n] = f32_block(W, min(n0 / 16 + T::wave() * T::NT + n, N / 16 - 1), K) + u0 * 512;
  T t;  // of a tile past the whole ones one of the S parts of K
  t.run([&](int i) { return A + (size_t)min(m0 + i, M - 1) * lda + u0 * 32; }, wr, (u1 - u0) * 32, lds);
  if (part >= 0 && !t.meet(p, S, slab + (size_t)(part / S) * S * (T::BM * T::BN), counters + part / S, &s_last)) return;
  t.each([&](int m, int n, float v, float u) {
    if (m0 + m >= M || n0 + n >= N) return;
    if constexpr (epi_gated(EPI)) {
      store_glu<EPI>(ep, m0 + m, n0 + n, v, u);
    } else {
      store_f32(ep, m0 + m, n0 + n, v);
      if (n0 + n + 16 < N) store_f32(ep, m0 + m, n0 + n + 16, u);
    }
  });
}

// A product's tiles, and how many parts of K for each of the last `rem` ones, which fill the CUs only in part (S; `whole` before
// them that fill them). Modelled us: a round of tiles its steps of 32 k and 5.2 to begin and end, a part its share of the steps;
// the meeting by the parts of a tile and by their bytes. Fitted to 176 products (11 of 512 to 8192 k by 640 to 16384 columns at 20
// to 2567 rows, all forms and splits): what it takes is 1.005 times the fastest (geometric mean; worst 1.08; timed without the operands' scaling, which adds 2 %
// to the large tiles' products and up to 9 % to the others). The largest tiles
// split least and read least (1.14 us for 128 x 128 of 32 k against 1.52 of the smallest), the smallest leave the fewest CUs idle.
struct Plan {
  int rows, cols, whole, S;
};
Plan plan(int M, int N, int K, long long slab_floats, int counters) {
  struct Form {
    int rows, cols;
    double busy, idle;  // us for 32 k: all CUs at it, few
  };
  constexpr Form forms[] = {{128, 256, 2.08, 1.74}, {128, 128, 1.14, 0.92}, {64, 128, 0.635, 0.525}, {64, 64, 0.38, 0.31}};
  Plan best{};
  double least = 0;
  for (const Form& f : forms) {
    const int tiles = ((M + f.rows - 1) / f.rows) * ((N + f.cols - 1) / f.cols), rem = tiles % 256, rounds = tiles / 256;
    const double kb = f.rows * f.cols / 256.0;
    for (int S : {1, 2, 3, 4, 6, 8, 12, 16}) {
      const long long parts = (long long)rem * S;
      if (S > 1 && (!rem || K / 32 < 2 * S || parts > 1024 || parts * f.rows * f.cols > slab_floats || rem > counters)) continue;
      double us = rounds * (K / 32 * f.busy + 5.2);
      if (rem) {
        const int n = (int)((parts + 255) / 256), per = (K / 32 + S - 1) / S;
        us += n * (per * (rounds || n > 1 ? f.busy : f.idle + (f.busy - f.idle) * parts / 256) + 5.2);
        if (S > 1) us += (0.28 + S * (0.22 + 0.0065 * kb) + 0.00051 * kb * parts) * (rounds ? 1.42 : 1.0);
      }
      if (!best.rows || us < least) best = Plan{f.rows, f.cols, S > 1 ? tiles - rem : tiles, S}, least = us;
    }
  }
  return best;
}

// The stream form: up to 16 rows; up to 32 of a product that is not large (20 rows, K = 2048, N = 4352 16 against 19 us of tiles,
// N = 8448 28 and 25, N = 16384 35 and 31; 4096 x 4096 19 and 25); where one 16 x 16 tile per workgroup does not fill the CUs
// (N = 128 48 rows 7 against 13 us), or a pair of columns of them does not and K is not long (N = 2048 64 rows: K = 2048 12
// against 16, K = 4096 20 and 20, K = 8192 36 and 26; K = 1024, N = 1024, 128 rows 8 and 14).
// Tiles of 16 rows that a workgroup of that form has; 0: not that form.
int stream_tiles(int M, int N, int K, bool gated) {
  const int t = N / 16, mt16 = (M + 15) / 16;
  const bool alone = (long long)(gated ? t / 2 : t) * mt16 <= 256, pairs = (long long)(t + 1) / 2 * mt16 <= 256 && K <= 4096;
  if (M <= 16 || alone || pairs) return 1;
  return K % 32 || (M <= 32 && (long long)N * K <= 1 << 24) ? 2 : 0;
}

template <int EPI>
void launch(const float* a, int lda, const float* w, int M, int N, int K, const EpiArgs& ep, float* slab, long long slab_floats,
            unsigned* counters, int n_counters, hipStream_t s) {
#define LSA_STREAM(MT, NT) \
  stream_f32_kernel<EPI, MT, NT, 8><<<dim3((t + NT - 1) / NT, (M + MT * 16 - 1) / (MT * 16)), 512, 0, s>>>(a, lda, w, M, N, K, ep)
  // A CU takes 3 us for a tile's products, so that the tiles are as many per workgroup as the fullest CU has anyway:
  // N = 4352 (272 tiles) two 12.2, one 14.8; N = 8448 (528) two 26.5, one 21.4; from N = 8192 on one streams better up to 8 rows
  // (N = 16384, 8 rows 24.6 against 28.4, 16 rows 28.5 and 28.7).
  const int t = N / 16;
  if (const int m = stream_tiles(M, N, K, epi_gated(EPI))) {
    const int rows = (M + 16 * m - 1) / (16 * m);
    const int one = (t * rows + 255) / 256, two = ((t + 1) / 2 * rows + 255) / 256 * 2;
    if constexpr (epi_gated(EPI)) {
      if (m == 1) LSA_STREAM(1, 2);
      else LSA_STREAM(2, 2);
    } else {
      const bool pair = two <= one && (t <= 512 || M > 8);
      if (m == 1 && pair) LSA_STREAM(1, 2);
      else if (m == 1) LSA_STREAM(1, 1);
      else if (pair) LSA_STREAM(2, 2);
      else LSA_STREAM(2, 1);
    }
    return;
  }
#undef LSA_STREAM
  const Plan p = plan(M, N, K, slab_floats, n_counters);
  const int mt = (M + p.rows - 1) / p.rows, nt = (N + p.cols - 1) / p.cols, grid = p.whole + (mt * nt - p.whole) * p.S;
#define LSA_TILE(MT, NW, KG)                                                                                               \
  tile_f32_kernel<EPI, MT, NW, KG><<<grid, NW * KG * 64, 0, s>>>(a, lda, w, M, N, K, mt, nt, p.whole, p.S, slab, counters, ep)
  if (p.cols == 256) LSA_TILE(8, 8, 1);
  else if (p.rows == 128) LSA_TILE(8, 4, 2);
  else if (p.cols == 128) LSA_TILE(4, 4, 2);
  else LSA_TILE(4, 2, 4);
#undef LSA_TILE
}

}  // namespace

// slab (16-byte aligned floats) and counters (zeros, left so): scratch of this stream for products in parts; none: whole tiles
extern "C" int lsa_linear_f32(const float* a, int lda, const float* w, int M, int N, int K, int epi, const EpiArgs* ep,
                              float* slab, long long slab_floats, unsigned* counters, int n_counters, hipStream_t stream) {
  if (M < 1 || N < 16 || N % 16 || K < 16 || K % 16 || lda < K || lda % 4 || !ep || !(ep->out32 || ep->out)) return LSA_BAD_SHAPE;
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)slab) % 16 || (!slab && slab_floats) || (!counters && n_counters))
    return LSA_BAD_SHAPE;
  if (epi_gated(epi)) {
    if (N % 32 || ep->ldo < N / 2 || !ep->out32) return LSA_BAD_SHAPE;
    if (epi == EPI_GEGLU) launch<EPI_GEGLU>(a, lda, w, M, N, K, *ep, slab, slab_floats, counters, n_counters, stream);
    else launch<EPI_SWIGLU>(a, lda, w, M, N, K, *ep, slab, slab_floats, counters, n_counters, stream);
  } else if (epi == EPI_STORE) {
    if (bad_store(*ep, N)) return LSA_BAD_SHAPE;
    launch<EPI_STORE>(a, lda, w, M, N, K, *ep, slab, slab_floats, counters, n_counters, stream);
  } else {
    return LSA_UNSUPPORTED;
  }
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

// What a product becomes: form[0..3] = rows and columns of a tile, tiles in one piece, parts of K of each tile past those; rows 16 or
// 32 with no columns: the stream form
extern "C" int lsa_linear_f32_form(int M, int N, int K, int gated, long long slab_floats, int n_counters, int* form) {
  if (M < 1 || N < 16 || N % 16 || K < 16 || K % 16 || (gated && N % 32) || !form) return LSA_BAD_SHAPE;
  const int m = stream_tiles(M, N, K, gated);
  const Plan p = m ? Plan{16 * m, 0, 0, 1} : plan(M, N, K, slab_floats, n_counters);
  form[0] = p.rows;
  form[1] = p.cols;
  form[2] = p.whole;
  form[3] = p.S;
  return LSA_OK;
}
