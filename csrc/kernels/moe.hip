// Mixture of experts (moe.h): routing, grouping and the expert products (bf16 on MFMA, and fp32 for the
// fp32 engine).
#include "f32_core.h"
#include "moe.h"

namespace {

// one wave per row: the ``top`` largest choice scores (ties: the smaller index), each lane ranking its own among all.
// ``s_c`` [E + groups]: this wave's LDS.
constexpr int MAX_E = 1024;
LSA_DEVICE void wave_sync() {  // LDS written by this wave's lanes is visible to all of them
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int NE>  // logits per lane: at most 64 NE experts
LSA_DEVICE void route_row(const RouteArgs& ra, const float* __restrict__ logits, int ldl, int row, int E, int top,
                          int* __restrict__ expert, float* __restrict__ weight, float* s_c) {
  const int lane = threadIdx.x & 63;
  const float* z = logits + (size_t)row * ldl;
  float v[NE], c[NE];  // score, choice score
  wave_sync();         // the row before has been read
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int e = j * 64 + lane;
    v[j] = c[j] = -INFINITY;
    if (e >= E) continue;
    v[j] = ra.sigmoid ? 1.f / (1.f + expf(-z[e])) : z[e];
    c[j] = v[j] + (ra.correction ? ra.correction[e] : 0.f);
    s_c[e] = c[j];
  }
  wave_sync();
  if (ra.groups > 1) {
    const int per = E / ra.groups;
    float* s_g = s_c + E;
    for (int g = lane; g < ra.groups; g += 64) {
      float b1 = -INFINITY, b2 = -INFINITY;
      for (int i = 0; i < per; ++i) {
        const float x = s_c[g * per + i];
        b2 = fmaxf(b2, fminf(b1, x));
        b1 = fmaxf(b1, x);
      }
      s_g[g] = per > 1 ? b1 + b2 : b1;
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < NE; ++j) {
      const int e = j * 64 + lane;
      if (e >= E) continue;
      const int g = e / per;
      const float mine = s_g[g];
      int better = 0;
      for (int o = 0; o < ra.groups; ++o) better += s_g[o] > mine || (s_g[o] == mine && o < g);
      if (better >= ra.keep) s_c[e] = c[j] = -INFINITY;
    }
    wave_sync();
  }
  int rank[NE];
#pragma unroll
  for (int j = 0; j < NE; ++j) rank[j] = 0;
  for (int o = 0; o < E; ++o) {
    const float x = s_c[o];
#pragma unroll
    for (int j = 0; j < NE; ++j) rank[j] += x > c[j] || (x == c[j] && o < j * 64 + lane);
  }
  float first = 0.f, sum = 0.f;
  if (!ra.sigmoid) {
    first = v[0];
#pragma unroll
    for (int j = 1; j < NE; ++j) first = fmaxf(first, v[j]);
    first = wave_max(first);
  }
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    if (j * 64 + lane >= E || rank[j] >= top) continue;
    if (!ra.sigmoid) v[j] = expf(v[j] - first);
    sum += v[j];
  }
  sum = wave_sum(sum);
  const float inv = ra.sigmoid ? ra.scale / (sum + 1e-20f) : 1.f / sum;
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    if (j * 64 + lane >= E || rank[j] >= top) continue;
    expert[(size_t)row * top + rank[j]] = j * 64 + lane;
    weight[(size_t)row * top + rank[j]] = v[j] * inv;
  }
}

template <int NE>
__global__ __launch_bounds__(256) void route_kernel(RouteArgs ra, const float* __restrict__ logits, int ldl, int rows,
                                                    int E, int top, int* __restrict__ expert, float* __restrict__ weight) {
  extern __shared__ float s_route[];
  const int w = threadIdx.x >> 6, row = blockIdx.x * 4 + w;
  if (row < rows) route_row<NE>(ra, logits, ldl, row, E, top, expert, weight, s_route + w * (E + ra.groups));
}

// Exclusive sums over the experts, one thread each: where expert tid's pairs and tiles start, with its count c and its tiles nt;
// and the number of all tiles. 1024 threads.
struct MoeSpan {
  int pairs, tiles, used;
};
LSA_DEVICE MoeSpan expert_spans(int c, int nt, int (*s_w)[16], int* s_n) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int a = c, b = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(a, o, 64), y = __shfl_up(b, o, 64);
    if (lane >= o) {
      a += x;
      b += y;
    }
  }
  if (lane == 63) {
    s_w[0][w] = a;
    s_w[1][w] = b;
  }
  __syncthreads();
  int ba = 0, bb = 0;
  for (int x = 0; x < w; ++x) {
    ba += s_w[0][x];
    bb += s_w[1][x];
  }
  if (tid == 1023) *s_n = bb + b;
  __syncthreads();
  return MoeSpan{ba + a - c, bb + b - nt, *s_n};
}
// the tile table: expert tid's tiles, and the rest of the table
LSA_DEVICE void write_tiles(MoeTile* __restrict__ tiles, const MoeSpan& sp, int E, int c, int nt, int tile_rows, int h, int max_tiles) {
  const int tid = threadIdx.x, used = sp.used | h << MOE_HEIGHT;
  if (tid < E)
    for (int t = 0; t < nt; ++t)
      if (sp.tiles + t < max_tiles)
        tiles[sp.tiles + t] = MoeTile{tid, sp.pairs + t * tile_rows, min(tile_rows, c - t * tile_rows), used};
  for (int t = sp.used + tid; t < max_tiles; t += 1024) tiles[t] = MoeTile{-1, 0, 0, used};
}
// The height of the tiles (MoePick), thread tid with expert tid's pairs c; tile_rows becomes it. CUs without a tile in the last
// round leave the others more of the clock (ops/hip.py gemm_sk_cost).
LSA_DEVICE int pick_height(const MoePick& pick, int c, int& tile_rows, int (*s_w)[16]) {
  if (!pick.nt[0]) return 0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int n[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) n[i] = wave_sum((c + MOE_ROWS[i] - 1) / MOE_ROWS[i]);
  if (lane < 4) s_w[lane][w] = lane & 2 ? (lane & 1 ? n[3] : n[2]) : (lane & 1 ? n[1] : n[0]);
  __syncthreads();
  int h = 0;
  float best = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int all = 0;
#pragma unroll
    for (int x = 0; x < 16; ++x) all += s_w[i][x];
    float us = 0.f;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int tiles = all * pick.nt[p], rem = tiles & 255;
      us += (float)(tiles >> 8) * (pick.step[i][p] + pick.own[i]);
      us += rem ? pick.step[i][p] * (1.f - 0.47f * (1.f - (float)rem / 256.f)) + pick.own[i] : 0.f;
    }
    if (i == 0 || us < best) {
      best = us;
      h = i;
    }
  }
  tile_rows = h & 2 ? (h & 1 ? MOE_ROWS[3] : MOE_ROWS[2]) : (h & 1 ? MOE_ROWS[1] : MOE_ROWS[0]);
  __syncthreads();  // s_w is read
  return h;
}

// One workgroup: counting sort of the pairs by expert, and the tile table. NE > 0: few rows, whose routing
// comes first.
template <int NE>
__global__ __launch_bounds__(1024) void group_kernel(RouteArgs ra, const float* __restrict__ logits, int ldl, int top,
                                                     float* __restrict__ weight, int* expert, int pairs, int E,
                                                     int tile_rows, MoePick pick, int max_tiles, int* __restrict__ order,
                                                     int* __restrict__ place, MoeTile* __restrict__ tiles) {
  __shared__ int s_cnt[MAX_E], s_off[MAX_E], s_n[1], s_w[4][16];
  const int tid = threadIdx.x;
  s_cnt[tid] = 0;
  if constexpr (NE > 0) {
    extern __shared__ float s_route[];
    const int w = tid >> 6;
    for (int row = w; row < pairs / top; row += 16)
      route_row<NE>(ra, logits, ldl, row, E, top, expert, weight, s_route + w * (E + ra.groups));
    __threadfence_block();
  }
  __syncthreads();
  constexpr int U = 8;  // loads in flight per thread
  for (int i0 = tid; i0 < pairs; i0 += 1024 * U) {
    int e[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = i0 + u * 1024 < pairs ? expert[i0 + u * 1024] : 0;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + u * 1024 < pairs) place[i0 + u * 1024] = atomicAdd(&s_cnt[e[u]], 1);  // rank within its expert
  }
  __syncthreads();
  const int c = tid < E ? s_cnt[tid] : 0, hi = pick_height(pick, c, tile_rows, s_w), nt = (c + tile_rows - 1) / tile_rows;
  const MoeSpan sp = expert_spans(c, nt, s_w, s_n);
  s_off[tid] = sp.pairs;
  __syncthreads();
  write_tiles(tiles, sp, E, c, nt, tile_rows, hi, max_tiles);
  for (int i0 = tid; i0 < pairs; i0 += 1024 * U) {
    int e[U], rank[U];  // this thread's own ranks
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = min(i0 + u * 1024, pairs - 1);
      e[u] = expert[i];
      rank[u] = place[i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * 1024;
      if (i >= pairs) break;
      const int at = s_off[e[u]] + rank[u];
      place[i] = at;
      order[at] = i;
    }
  }
}

// The same of many pairs in two launches of a workgroup for every GROUP_PAIRS: counts [workgroups][E] and ranks within a
// workgroup's pairs, then the sums over the workgroups (each makes them for itself) and the places. One workgroup is bound by its
// pairs' turns at the counters and at memory; here a thread has two of them. us, 32 experts: 4096 pairs 5.3 and 5.8, 6000 6.2 and
// 5.9, 12000 9.6 and 6.4, 25512 17.2 and 6.7, 65536 38 and 8; 8 experts 25512 19 and 8.7; 256 experts 22 and 7.5 (graphs; in a
// prompt's stream 5868 pairs 7.6 and 10.2, 25512 25 and 9.5).
constexpr int GROUP_PAIRS = 2048, GROUP_MANY = 10240;
__global__ __launch_bounds__(1024) void count_kernel(const int* __restrict__ expert, int pairs, int E, int* __restrict__ place,
                                                     int* __restrict__ counts) {
  __shared__ int s_cnt[MAX_E];
  const int tid = threadIdx.x, i0 = blockIdx.x * GROUP_PAIRS + tid, i1 = i0 + 1024;
  const int e0 = i0 < pairs ? expert[i0] : 0, e1 = i1 < pairs ? expert[i1] : 0;
  s_cnt[tid] = 0;
  __syncthreads();
  if (i0 < pairs) place[i0] = atomicAdd(&s_cnt[e0], 1);
  if (i1 < pairs) place[i1] = atomicAdd(&s_cnt[e1], 1);
  __syncthreads();
  if (tid < E) counts[(size_t)blockIdx.x * E + tid] = s_cnt[tid];
}
__global__ __launch_bounds__(1024) void place_kernel(const int* __restrict__ expert, int pairs, int E, int tile_rows, MoePick pick,
                                                     int max_tiles, int* __restrict__ order, int* __restrict__ place,
                                                     const int* __restrict__ counts, MoeTile* __restrict__ tiles) {
  __shared__ int s_all[MAX_E], s_before[MAX_E], s_n[1], s_w[4][16];
  const int tid = threadIdx.x, i0 = blockIdx.x * GROUP_PAIRS + tid, i1 = i0 + 1024;
  const int j0 = min(i0, pairs - 1), j1 = min(i1, pairs - 1);
  const int e0 = expert[j0], e1 = expert[j1], r0 = place[j0], r1 = place[j1];
  s_all[tid] = s_before[tid] = 0;
  __syncthreads();
  const int n = gridDim.x * E, mine = blockIdx.x * E;
  for (int i = tid; i < n; i += 1024) {
    const int c = counts[i], e = i % E;
    atomicAdd(&s_all[e], c);
    if (i < mine) atomicAdd(&s_before[e], c);
  }
  __syncthreads();
  const int c = tid < E ? s_all[tid] : 0, hi = blockIdx.x == 0 ? pick_height(pick, c, tile_rows, s_w) : 0;  // (it writes the tiles)
  const int nt = (c + tile_rows - 1) / tile_rows;
  const MoeSpan sp = expert_spans(c, nt, s_w, s_n);
  s_before[tid] += sp.pairs;
  __syncthreads();
  if (blockIdx.x == 0) write_tiles(tiles, sp, E, c, nt, tile_rows, hi, max_tiles);
  if (i0 < pairs) {
    const int at = s_before[e0] + r0;
    place[i0] = at;
    order[at] = i0;
  }
  if (i1 < pairs) {
    const int at = s_before[e1] + r1;
    place[i1] = at;
    order[at] = i1;
  }
}

// One tile of MT x 16 pairs x 64 columns of one expert's product; four waves share K and meet in LDS.
// MOE_GLU: the columns are gate / up 16-tiles in turn and the output is silu(gate) * up (32 columns). The rows
// of A are the pairs' rows of h (up), or the sorted pairs themselves (down).
template <int MT, int UP>
__global__ __launch_bounds__(256) void moe_small_kernel(const MoeTile* __restrict__ tiles, const int* __restrict__ order,
                                                        int top, const bf16_raw* __restrict__ A, int lda,
                                                        const bf16_raw* __restrict__ W, int N, int K,
                                                        bf16_raw* __restrict__ out, int ldo) {
  constexpr int NT = 4;
  constexpr bool GLU = UP == MOE_GLU;
  __shared__ __attribute__((aligned(16))) float s_acc[4][MT * 16][NT * 16 + 4];
  const MoeTile tile = tiles[blockIdx.y];
  if (tile.expert < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nt0 = blockIdx.x * NT, KT = K / 32, ntn = min(NT, N / 16 - nt0);
  const bf16_raw* ar[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int i = tile.start + min(m * 16 + l16, tile.count - 1);  // rows past the count are not stored
    ar[m] = A + (size_t)(UP ? order[i] / top : i) * lda + q4 * 8;
  }
  const bf16_raw* wp = W + (size_t)tile.expert * N * K + ((size_t)nt0 * KT * 64 + lane) * 8;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int k1 = KT * (w + 1) / 4;
  // the next step's operands are requested before this one's products
  auto load = [&](int kt, u32x4_t (&b)[NT], u32x4_t (&x)[MT]) {
#pragma unroll
    for (int n = 0; n < NT; ++n) b[n] = ld16(wp + ((size_t)min(n, ntn - 1) * KT + kt) * 512);
#pragma unroll
    for (int m = 0; m < MT; ++m) x[m] = ld16(ar[m] + kt * 32);
  };
  auto mul = [&](const u32x4_t (&b)[NT], const u32x4_t (&x)[MT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = mfma16(x[m], b[n], acc[m][n]);
  };
  u32x4_t b0[NT], x0[MT], b1[NT], x1[MT];
  int kt = KT * w / 4;
  if (kt < k1) load(kt, b0, x0);
  for (; kt + 2 < k1; kt += 2) {
    load(kt + 1, b1, x1);
    mul(b0, x0);
    load(kt + 2, b0, x0);
    mul(b1, x1);
  }
  if (kt + 1 < k1) load(kt + 1, b1, x1);
  if (kt < k1) mul(b0, x0);
  if (kt + 1 < k1) mul(b1, x1);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) s_acc[w][m * 16 + q4 * 4 + r][n * 16 + l16] = acc[m][n][r];
  __syncthreads();
  const int cols = GLU ? ntn * 8 : ntn * 16;  // output columns of this workgroup
  for (int t = tid; t < tile.count * (cols / 4); t += 256) {
    const int m = t / (cols / 4), c = (t % (cols / 4)) * 4;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
    const int cc = GLU ? (c / 16) * 32 + c % 16 : c;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      v += *reinterpret_cast<const f32x4_t*>(&s_acc[x][m][cc]);
      if (GLU) u += *reinterpret_cast<const f32x4_t*>(&s_acc[x][m][cc + 16]);
    }
    if (GLU)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = v[j] / (1.f + __expf(-v[j])) * u[j];
    if (UP == MOE_RELU2)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = fmaxf(v[j], 0.f) * fmaxf(v[j], 0.f);
    st4(out + (size_t)(tile.start + m) * ldo + (GLU ? nt0 * 8 : nt0 * 16) + c, v);
  }
}

// fp32 (f32_core.h): gate / up 16-tiles in turn, or the output's own columns
template <int UP>
LSA_DEVICE float up_f32(float g, float u) {
  if constexpr (UP == MOE_GLU) return g / (1.f + expf(-g)) * u;
  if constexpr (UP == MOE_RELU2) return fmaxf(g, 0.f) * fmaxf(g, 0.f);
  return g;
}

// few pairs per expert: MT x 16 pairs x NT x 16 columns
template <int UP, int MT, int NT, int NW>
__global__ __launch_bounds__(NW * 64) void moe_stream_f32_kernel(const MoeTile* __restrict__ tiles, const int* __restrict__ order,
                                                                 int top, const float* __restrict__ A, int lda,
                                                                 const float* __restrict__ W, int N, int K,
                                                                 float* __restrict__ out, int ldo) {
  using S = F32Stream<MT, NT, NW>;
  constexpr bool GLU = UP == MOE_GLU;
  constexpr int OC = GLU ? NT * 8 : NT * 16;  // output columns
  __shared__ __attribute__((aligned(16))) float s_acc[S::LDS];
  const MoeTile tile = tiles[blockIdx.y];
  if (tile.expert < 0) return;
  const int lane = threadIdx.x & 63, n0 = blockIdx.x * NT * 16;
  const float *ar[MT], *wr[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int i = tile.start + min(m * 16 + (lane & 15), tile.count - 1);  // rows past the count are not stored
    ar[m] = A + (size_t)(UP ? order[i] / top : i) * lda + 4 * (lane >> 4);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
    wr[n] = f32_block(W, (size_t)tile.expert * (N / 16) + min(n0 / 16 + n, N / 16 - 1), K);
  S::run(ar, wr, K, s_acc);
  for (int t = threadIdx.x; t < tile.count * OC; t += NW * 64) {
    const int m = t / OC, c = t % OC, n = GLU ? (c >> 4) * 32 + (c & 15) : c;
    if (n0 + n >= N) continue;
    const float v = S::sum(s_acc, m, n);
    out[(size_t)(tile.start + m) * ldo + (GLU ? n0 / 2 : n0) + c] = up_f32<UP>(v, GLU ? S::sum(s_acc, m, n + 16) : 0.f);
  }
}

// many: MT x 16 pairs x NW x 32 columns. 20536 pairs, 32 experts of 2048 x 1024: up 776 -> 477, down 769 -> 465 us (64 x 64 tiles
// on the fp32 matrix instructions before); about 90 pairs an expert, gated, of 1024 columns 509 -> 346 in 64 x 128 tiles; 8 experts
// of 1024 x 2048, 40 pairs each 35 -> 29 in 64 x 64 (64 x 128 44, 128 x 256 117: which of them, ops/moe.py).
template <int UP, int MT, int NW, int KG>
__global__ __launch_bounds__(NW * KG * 64) void moe_tile_f32_kernel(const MoeTile* __restrict__ tiles, const int* __restrict__ order,
                                                                    int top, const float* __restrict__ A, int lda,
                                                                    const float* __restrict__ W, int N, int K,
                                                                    float* __restrict__ out, int ldo) {
  using T = F32Split<MT, NW, KG>;
  __shared__ u32x4_t lds[T::LDS];
  // Workgroups of one XCD get consecutive work, 8 tiles (mostly of one expert) share a sweep over the columns.
  const int nx = gridDim.x, b = blockIdx.y * nx + blockIdx.x, told = tiles[0].used;
  const int used = told > 0 ? min(told, (int)gridDim.y) : gridDim.y;
  const int G = used * nx, q = G / 8, r = G % 8, x = b % 8;
  if (b >= G) return;
  const int g = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + b / 8;
  const int first = g / (8 * nx) * 8, gm = min(used - first, 8), in = g - first * nx;
  const MoeTile tile = tiles[first + in % gm];
  if (tile.expert < 0) return;
  const int n0 = in / gm * T::BN;
  const float* wr[T::NT];
#pragma unroll
  for (int n = 0; n < T::NT; ++n)
    wr[n] = f32_block(W + (size_t)tile.expert * N * K, min(n0 / 16 + T::wave() * T::NT + n, N / 16 - 1), K);
  T t;
  t.run([&](int i) {
    const int at = tile.start + min(i, tile.count - 1);  // rows past the count are not stored
    return A + (size_t)(UP ? order[at] / top : at) * lda;
  }, wr, K, lds);
  t.each([&](int m, int n, float v, float u) {
    if (m >= tile.count || n0 + n >= N) return;
    float* o = out + (size_t)(tile.start + m) * ldo;
    if (UP == MOE_GLU) {
      o[((n0 + n) >> 5) * 16 + (n & 15)] = up_f32<UP>(v, u);
    } else {
      o[n0 + n] = up_f32<UP>(v, 0.f);
      o[n0 + n + 16] = up_f32<UP>(u, 0.f);  // N % 32 == 0
    }
  });
}

template <int UP>
int launch_f32(const MoeTile* t, int max_tiles, int tile_rows, bool narrow, const int* order, int top, const float* A, int lda,
               const float* W, int N, int K, float* out, int ldo, hipStream_t s) {
  constexpr int NT = UP == MOE_GLU ? 2 : 1;
  const dim3 grid((N + NT * 16 - 1) / (NT * 16), max_tiles);
  if (tile_rows <= 16) moe_stream_f32_kernel<UP, 1, NT, 8><<<grid, 512, 0, s>>>(t, order, top, A, lda, W, N, K, out, ldo);
  else if (tile_rows <= 32) moe_stream_f32_kernel<UP, 2, NT, 8><<<grid, 512, 0, s>>>(t, order, top, A, lda, W, N, K, out, ldo);
  else if (tile_rows <= 64 && narrow)
    moe_tile_f32_kernel<UP, 4, 2, 4><<<dim3((N + 63) / 64, max_tiles), 512, 0, s>>>(t, order, top, A, lda, W, N, K, out, ldo);
  else if (tile_rows <= 64)
    moe_tile_f32_kernel<UP, 4, 4, 2><<<dim3((N + 127) / 128, max_tiles), 512, 0, s>>>(t, order, top, A, lda, W, N, K, out, ldo);
  else if (tile_rows <= 128)
    moe_tile_f32_kernel<UP, 8, 8, 1><<<dim3((N + 255) / 256, max_tiles), 512, 0, s>>>(t, order, top, A, lda, W, N, K, out, ldo);
  else return LSA_UNSUPPORTED;
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

}  // namespace

static bool bad_route(const RouteArgs* ra, int E) {
  return !ra || ra->groups < 1 || ra->keep < 1 || ra->keep > ra->groups || E % ra->groups;
}

extern "C" int lsa_moe_route(const RouteArgs* ra, const float* logits, int ldl, int rows, int E, int top, int* expert,
                             float* weight, hipStream_t s) {
  if (rows < 1 || E < 1 || E > MAX_E || top < 1 || top > E || ldl < E || bad_route(ra, E)) return LSA_BAD_SHAPE;
  const size_t lds = (size_t)4 * (E + ra->groups) * 4;
#define LSA_RT(NE) route_kernel<NE><<<(rows + 3) / 4, 256, lds, s>>>(*ra, logits, ldl, rows, E, top, expert, weight)
  if (E <= 64) LSA_RT(1);
  else if (E <= 256) LSA_RT(4);
  else LSA_RT(MAX_E / 64);
#undef LSA_RT
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

// max_tiles >= min(E, pairs) + pairs / tile_rows; counts: n_counts ints of scratch, or none; heights: tiles of the height that the
// pairs make best (tile_rows: the lowest, 128), or null
extern "C" int lsa_moe_group(const int* expert, int pairs, int E, int tile_rows, int max_tiles, int* order, int* place,
                             void* tiles, int* counts, int n_counts, const MoePick* heights, hipStream_t s) {
  if (pairs < 1 || E < 1 || E > MAX_E || tile_rows < 1 || max_tiles < (E < pairs ? E : pairs) + pairs / tile_rows ||
      (!counts && n_counts))
    return LSA_BAD_SHAPE;
  const MoePick pick = heights ? *heights : MoePick{};
  if (heights && (tile_rows != MOE_ROWS[0] || max_tiles >= 1 << MOE_HEIGHT || pick.nt[0] < 1 || pick.nt[1] < 1 ||
                  pick.nt[0] > 4096 || pick.nt[1] > 4096 || (long long)max_tiles * 4096 >= 1ll << 31))
    return LSA_BAD_SHAPE;
  const int wg = (pairs + GROUP_PAIRS - 1) / GROUP_PAIRS;
  if (pairs >= GROUP_MANY && (long long)wg * E <= n_counts) {
    count_kernel<<<wg, 1024, 0, s>>>(expert, pairs, E, place, counts);
    place_kernel<<<wg, 1024, 0, s>>>(expert, pairs, E, tile_rows, pick, max_tiles, order, place, counts, (MoeTile*)tiles);
    LSA_CHECK_LAUNCH();
    return LSA_OK;
  }
  group_kernel<0><<<1, 1024, 0, s>>>(RouteArgs{}, nullptr, 0, 1, nullptr, const_cast<int*>(expert), pairs, E, tile_rows,
                                     pick, max_tiles, order, place, (MoeTile*)tiles);
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

// lsa_moe_route and lsa_moe_group of few rows in one launch
extern "C" int lsa_moe_route_group(const RouteArgs* ra, const float* logits, int ldl, int rows, int E, int top, int* expert,
                                   float* weight, int tile_rows, int max_tiles, int* order, int* place, void* tiles,
                                   hipStream_t s) {
  const int pairs = rows * top;
  if (rows < 1 || rows > 64 || E < 1 || E > 256 || top < 1 || top > E || ldl < E || tile_rows < 1 || bad_route(ra, E) ||
      max_tiles < (E < pairs ? E : pairs) + pairs / tile_rows)
    return LSA_BAD_SHAPE;
  const size_t lds = (size_t)16 * (E + ra->groups) * 4;
#define LSA_RG(NE)                                                                                                  \
  group_kernel<NE><<<1, 1024, lds, s>>>(*ra, logits, ldl, top, weight, expert, pairs, E, tile_rows, MoePick{}, max_tiles, order, \
                                        place, (MoeTile*)tiles)
  if (E <= 64) LSA_RG(1);
  else LSA_RG(4);
#undef LSA_RG
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}

// up (MoeUp): A = h rows, out [pairs][ldo >= N / 2 (glu) or N]; down: A = act [pairs], out [pairs][ldo >= N]
// narrow (fp32, tiles of 64 rows): 64 columns a workgroup instead of 128
extern "C" int lsa_moe_gemm(int f32, int up, const void* tiles, int max_tiles, int tile_rows, int narrow, const int* order, int top,
                            const void* A, int lda, const void* W, int N, int K, void* out, int ldo, hipStream_t s) {
  if (max_tiles < 1 || max_tiles > 65535 || top < 1 || N < 32 || N % 32 || K < 32 || K % 32 || lda < K || lda % 8 ||
      up < MOE_DOWN || up > MOE_RELU2 || ldo < (up == MOE_GLU ? N / 2 : N) || ldo % 4 ||
      ((uintptr_t)A | (uintptr_t)W | (uintptr_t)out) % 16)
    return LSA_BAD_SHAPE;
  const dim3 grid((N + 63) / 64, max_tiles);
  const MoeTile* t = (const MoeTile*)tiles;
  if (f32) {
    auto* f = up == MOE_GLU ? launch_f32<MOE_GLU> : up ? launch_f32<MOE_RELU2> : launch_f32<MOE_DOWN>;
    return f(t, max_tiles, tile_rows, narrow, order, top, (const float*)A, lda, (const float*)W, N, K, (float*)out, ldo, s);
  }
#define LSA_M(MT)                                                                                                     \
  if (tile_rows == MT * 16) {                                                                                         \
    auto* f = up == MOE_GLU ? moe_small_kernel<MT, MOE_GLU> : up ? moe_small_kernel<MT, MOE_RELU2> : moe_small_kernel<MT, MOE_DOWN>; \
    f<<<grid, 256, 0, s>>>(t, order, top, (const bf16_raw*)A, lda, (const bf16_raw*)W, N, K, (bf16_raw*)out, ldo);    \
    LSA_CHECK_LAUNCH();                                                                                               \
    return LSA_OK;                                                                                                    \
  }
  LSA_M(1) LSA_M(2) LSA_M(4)
#undef LSA_M
  return LSA_UNSUPPORTED;
}
