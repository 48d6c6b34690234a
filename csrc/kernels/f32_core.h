// Products C[m][n] = sum_k A[m][k] W[n][k] of fp32 operands on the matrix unit, for the fp32 engine's projections
// (linear_f32.hip) and experts (moe.hip). A is row-major with K consecutive. W is packed (ops/packing.py pack_f32): blocks of 16
// columns x 16 k of 1 KiB, in which lane l has column l & 15 and k 4 (l >> 4) .., so that a wave's load is 1 KiB in one piece.
// From row-major weights (16 pieces of 64 bytes) 16 rows took N = K = 2048 10.5 instead of 8.3 us, N = 8704 27.7 instead of 20.3,
// N = 32000 72 instead of 50. The sum over k runs in the order of that layout, the same for A and W.
//
// Two forms, chosen by the caller:
//   F32Stream  few rows, on the fp32 matrix instructions (v_mfma_f32_*_f32: true fp32 products and sums): a lane loads four
//              consecutive k and gives them to four instructions in turn; the weights go once from memory to operand registers;
//              the waves of a workgroup share K and meet in LDS. Bound by launch and one round trip, then by reading the weights:
//              8 rows, N = K = 2048 7 us (2.4 TB/s), N = 16384 25 us (5.5 TB/s).
//   F32Split   many rows, on the bf16 matrix instructions, which are 16 times as fast: each operand is taken apart into three
//              bf16 (8 + 8 + 8 bits of its 24), and of their nine products the six of more than 2^-24 of the whole are made.
//              Bound by the matrix unit and by the splitting, which take turns: at 2567 rows, N = 16384, K = 2048 the one is busy
//              for 66 % of the time, at the 1.75 GHz that its six products leave it (1835 of 2500 TFLOP/s, 306 of fp32 product), and 1.9
//              other vector instructions for each of its take 31 %. That product 1343 -> 806 us (214 TFLOP/s; the fp32 instructions
//              reach 157 at best), 963 rows, N = 16384 512 -> 302, N = 2048 78 -> 54, K = 8192 257 -> 171.
//              Errors against 64 bits are lower than those of fp32 instructions, since a sum is rounded once for 32 k instead
//              of once for 2 (the five smaller products have sums of their own): K = 2048 3.3e-7 to 5.7e-7 -> 1.1e-7 to 2.7e-7 of the
//              result's norm, K = 8192 6.6e-7 to 1.15e-6 -> 2.2e-7 to 5.7e-7. With all six in one sum it was 7e-7.
#pragma once
#include "elem.h"
#include "mfma_pair.h"

// this lane's part of block (columns 16 t .., k 0 ..) of packed weights; the next block of k lies 256 floats behind it
LSA_DEVICE const float* f32_block(const float* W, size_t t, int K) { return W + t * 16 * K + (threadIdx.x & 63) * 4; }

// MT x 16 rows by NT x 16 columns; NW waves, each with a part of K (in units of 16).
template <int MT, int NT, int NW>
struct F32Stream {
  static constexpr int UN = MT + NT <= 2 ? 4 : 2;  // units requested together (another UN are in flight meanwhile)
  static constexpr int LD = NT * 16 + 4, LDS = NW * MT * 16 * LD;
  struct Unit {
    f32x4_t a[UN][MT], w[UN][NT];
  };

  // ar: this lane's rows (lane & 15 of each tile) from k = 4 * (lane >> 4) on; wr: this lane's part of the first blocks
  // (f32_block); s_acc: LDS floats
  LSA_DEVICE static void run(const float* const (&ar)[MT], const float* const (&wr)[NT], int K, float* s_acc) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int u0 = (K / 16) * w / NW, u1 = (K / 16) * (w + 1) / NW;
    f32x4_t acc[2][MT][NT];  // of every other instruction: half as long sums round less, 2.1e-7 of the result at K = 2048 for 2.9e-7
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[0][m][n] = acc[1][m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int u, Unit& x) {
#pragma unroll
      for (int i = 0; i < UN; ++i) {
        const int k = 16 * min(u + i, u1 - 1);  // past the end: the last unit again, not used
#pragma unroll
        for (int n = 0; n < NT; ++n) x.w[i][n] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(wr[n] + k * 16));
#pragma unroll
        for (int m = 0; m < MT; ++m) x.a[i][m] = *reinterpret_cast<const f32x4_t*>(ar[m] + k);
      }
    };
    auto mul = [&](int u, const Unit& x) {
#pragma unroll
      for (int i = 0; i < UN; ++i) {
        if (u + i >= u1) break;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
              acc[j & 1][m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.a[i][m][j], x.w[i][n][j], acc[j & 1][m][n], 0, 0, 0);
      }
    };
    Unit x0, x1;
    if (u0 < u1) load(u0, x0);
    for (int u = u0; u < u1; u += 2 * UN) {
      if (u + UN < u1) load(u + UN, x1);
      mul(u, x0);
      if (u + UN >= u1) break;
      if (u + 2 * UN < u1) load(u + 2 * UN, x0);
      mul(u + UN, x1);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s_acc[(w * MT * 16 + m * 16 + (lane >> 4) * 4 + r) * LD + n * 16 + (lane & 15)] = acc[0][m][n][r] + acc[1][m][n][r];
    __syncthreads();
  }
  LSA_DEVICE static float sum(const float* s_acc, int m, int n) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += s_acc[(w * MT * 16 + m) * LD + n];
    return v;
  }
};

// MT x 16 rows by NW x 32 columns of C; KG groups of NW waves, each with its part of K, every wave 32 columns of all rows. A
// wave splits its columns for itself, from memory to operand registers, and an NW-th of the rows for all, through LDS: were the
// columns shared too, twice as much would go through LDS. The pieces are rounded to nearest, so that they hold 24 bits and the
// dropped products have either sign. Operands are split 2^16 times as large: the last bit of an fp32 number, 2^-149 for
// the smallest, is then one that a bf16 holds (2^-133), and every finite value is the sum of its pieces. The sums are 2^32 times as
// large in turn: values from 2^112 and results from 2^96 on give infinities in them and are made again from the values
// (whole). Unscaled, values under 2^-109 had fewer bits (1e-6 off at 2^-115, nothing left at 2^-134); the two products with 2^16 of
// a pair of values take 2 % of a product's time (2567 rows, N = 16384, K = 2048 797 -> 812 us, 963 rows 300 -> 307). Tile sizes
// (linear_f32.hip plan) by how many there are of them.
template <int MT, int NW, int KG>
struct F32Split {
  static_assert(MT % NW == 0 && MT % KG == 0);
  static constexpr int NT = 2, BM = MT * 16, BN = NW * NT * 16, THREADS = NW * KG * 64;
  static constexpr int SF = MT / NW;       // 16-row fragments that a wave splits for all
  static constexpr int BUF = MT * 3 * 64;  // 32 k of the rows: fragments of three pieces, 16 bytes a lane
  static constexpr int LDS = KG * 2 * BUF;
  static constexpr int MO = MT / KG;       // fragments that a wave holds in the end: from MO * group on
  static constexpr float UP = 0x1p16f, DOWN = 0x1p-32f;
  f32x4_t acc[MT][NT];

  LSA_DEVICE static int group() { return KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / NW; }
  LSA_DEVICE static int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % NW; }

  // row(r): where row r of the tile starts; wr: this lane's part of this wave's blocks of columns (f32_block); K % 32 == 0
  template <typename R>
  LSA_DEVICE void run(R row, const float* const (&wr)[NT], int K, u32x4_t* lds) {
    const int grp = group(), steps = (K / 32 + KG - 1) / KG;  // of the groups with the most
    const int u = K / 32 * grp / KG, mine = K / 32 * (grp + 1) / KG - u, from = mine ? u * 32 : 0;
    const int last = max(mine - 1, 0) * 32;
    const float* w2[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) w2[n] = wr[n] + from * 16;
    sums([&](int r) { return row(r) + from; }, w2, steps, mine, last, lds + grp * 2 * BUF);
    whole([&](int r) { return row(r) + from; }, w2, mine * 32);
    if constexpr (KG > 1) {  // every group gets the others' sums of its rows
      static_assert(KG * (KG - 1) * MO * NT * NW * 64 <= LDS);
      const int at = wave() * 64 + (threadIdx.x & 63);
      auto part = [&](int to, int from, int m, int n) -> u32x4_t& {  // from: groups behind `to`
        return lds[(((to * (KG - 1) + from - 1) * MO + m) * NT + n) * NW * 64 + at];
      };
      f32x4_t own[MO][NT];
      __syncthreads();  // the fragments are read
#pragma unroll
      for (int to = 0; to < KG; ++to)
#pragma unroll
        for (int m = 0; m < MO; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            if (to == grp) own[m][n] = acc[to * MO + m][n];
            else part(to, (grp + KG - to) % KG, m, n) = __builtin_bit_cast(u32x4_t, acc[to * MO + m][n]);
          }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          acc[m][n] = own[m][n];
#pragma unroll
          for (int y = 1; y < KG; ++y) acc[m][n] += __builtin_bit_cast(f32x4_t, part(grp, y, m, n));
        }
    }
  }

  template <typename R>
  LSA_DEVICE void sums(R row, const float* const (&wr)[NT], int steps, int mine, int last, u32x4_t* lds) {
    const int lane = threadIdx.x & 63, w = wave();
    f32x4_t low[MT][NT];  // the products with second and third pieces: 2^-8 of the others and less, as are their roundings
    const float* ar[SF];
#pragma unroll
    for (int i = 0; i < SF; ++i) ar[i] = row((w + NW * i) * 16 + (lane & 15)) + 4 * (lane >> 4);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = low[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t g[SF + NT][2];  // 8 k of a row or column: from 4 (lane / 16) on and from 16 behind that
    auto load = [&](int i, int k0) {
      k0 = min(k0, last);  // past the end: the last ones again, not used
      const float* p = i < SF ? ar[i < SF ? i : 0] + k0 : wr[i < SF ? 0 : i - SF] + k0 * 16;
      g[i][0] = *reinterpret_cast<const f32x4_t*>(p);
      g[i][1] = *reinterpret_cast<const f32x4_t*>(p + (i < SF ? 16 : 256));
    };
    u32x4_t sa[3], b[2][NT][3], a[2][3];
    float u, v;
    // A third of the split of two values; after the last two of a fragment it goes to LDS (rows) and the next is requested.
    constexpr int THIRDS = 12 * (SF + NT);
    auto third = [&](int s, int k0, u32x4_t* nxt, u32x4_t (&bn)[NT][3]) {
      const int i = s / 12, j = s / 3 % 4, x = s % 3;
      u32x4_t(&to)[3] = i < SF ? sa : bn[i < SF ? 0 : i - SF];
      if (x == 0) u = g[i][j >> 1][2 * j & 3] * UP, v = g[i][j >> 1][(2 * j & 3) + 1] * UP;
      const unsigned h = pack2(u, v);
      to[x][j] = h;
      if (x < 2) u -= __uint_as_float(h << 16), v -= __uint_as_float(h & 0xffff0000u);
      if (s % 12 < 11) return;
      if (i < SF)
#pragma unroll
        for (int p = 0; p < 3; ++p) nxt[((w + NW * i) * 3 + p) * 64 + lane] = sa[p];
      load(i, k0);
    };
    // 32 k that are split already. Between their products the next 32 are split, what their registers get next is requested,
    // and each fragment of the rows comes from LDS while the one before is used. The barrier stands before the last one, whose
    // way from LDS is over: after it this buffer is written again, and the next one's first fragment is read.
    constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};  // the pieces of each product
    auto step = [&](int k0, const u32x4_t* cur, u32x4_t* nxt, const u32x4_t (&b)[NT][3], u32x4_t (&bn)[NT][3]) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if (m == MT - 1) __syncthreads();
#pragma unroll
        for (int q = 0; q < 6; ++q) {
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            f32x4_t& c = q < 5 ? low[m][n] : acc[m][n];
            c = mfma16(a[m & 1][pa[q]], b[n][pb[q]], c);
          }
          if (q < 3) a[(m + 1) & 1][2 - q] = m + 1 < MT ? cur[((m + 1) * 3 + 2 - q) * 64 + lane] : nxt[(2 - q) * 64 + lane];
          const int z = m * 6 + q;
#pragma unroll
          for (int s = z * THIRDS / (6 * MT); s < (z + 1) * THIRDS / (6 * MT); ++s) third(s, k0 + 64, nxt, bn);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
#pragma unroll
    for (int i = 0; i < SF + NT; ++i) load(i, 0);
#pragma unroll
    for (int s = 0; s < THIRDS; ++s) third(s, 32, lds, b[0]);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 3; ++p) a[0][p] = lds[p * 64 + lane];
    for (int s = 0; s < steps; s += 2) {
      if (s < mine) step(s * 32, lds, lds + BUF, b[0], b[1]);
      else __syncthreads();
      if (s + 1 >= steps) break;
      if (s + 1 < mine) step(s * 32 + 32, lds + BUF, lds, b[1], b[0]);
      else __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = (acc[m][n] + low[m][n]) * DOWN;
  }

  // Sums that are no finite numbers again from the values as they are: the pieces of an infinity, and of a value that rounds
  // to one, are infinities and NaN, and an infinity times a piece that is zero is NaN where the whole product is none.
  template <typename R>
  LSA_DEVICE void whole(R row, const float* const (&wr)[NT], int K) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      bool bad = false;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) bad |= !(fabsf(acc[m][n][r]) < INFINITY);
      if (!__any(bad)) continue;
      const float* a = row(m * 16 + (lane & 15)) + 4 * (lane >> 4);
      f32x4_t c[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) c[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      for (int k = 0; k < K; k += 16) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + k);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const f32x4_t y = *reinterpret_cast<const f32x4_t*>(wr[n] + k * 16);
#pragma unroll
          for (int j = 0; j < 4; ++j) c[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], y[j], c[n], 0, 0, 0);
        }
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!(fabsf(acc[m][n][r]) < INFINITY)) acc[m][n][r] = c[n][r];
    }
  }

  // This workgroup's sums are part q of S of a tile: whoever is the last to bring its part gets all of them, added in the
  // order of the parts, and true. slab: S * BM * BN floats of this tile; counter: 0, and 0 again when the last has come.
  // Parts are written and read past the L2 (sc1), each is drained before its ticket is drawn, and nobody waits. A part's offset
  // is in the vector register: behind a 16-byte store with a scalar one the compiler leaves no wait states before it writes
  // the store's data registers again, and what was stored here was then an address instead of a sum (csrc/isa_audit.py R5).
  LSA_DEVICE bool meet(int q, int S, float* slab, unsigned* counter, int* s_last) {
    const int tid = threadIdx.x;
    constexpr int PART = BM * BN * 4;  // bytes
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)slab, (short)0, S * PART, 0x00020000);
#pragma unroll
    for (int c = 0; c < MO * NT; ++c)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[c / NT][c % NT]), r,
                                             q * PART + (c * THREADS + tid) * 16, 0, 16);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0)
      *s_last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
    __syncthreads();
    if (!*s_last) return false;
#pragma unroll
    for (int c = 0; c < MO * NT; ++c) acc[c / NT][c % NT] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int p0 = 0; p0 < S; p0 += 2) {
      const int p1 = min(p0 + 1, S - 1);
      f32x4_t v[2][MO * NT];
#pragma unroll
      for (int c = 0; c < MO * NT; ++c) {
        v[0][c] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (c * THREADS + tid) * 16, p0 * PART, 16));
        v[1][c] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (c * THREADS + tid) * 16, p1 * PART, 16));
      }
#pragma unroll
      for (int c = 0; c < MO * NT; ++c) acc[c / NT][c % NT] += v[0][c];
      if (p0 + 1 < S)
#pragma unroll
        for (int c = 0; c < MO * NT; ++c) acc[c / NT][c % NT] += v[1][c];
    }
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  // f(row of the tile, column of the tile, value, value 16 columns further)
  template <typename F>
  LSA_DEVICE void each(F f) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        f((group() * MO + m) * 16 + (lane >> 4) * 4 + r, wave() * 32 + (lane & 15), acc[m][0][r], acc[m][1][r]);
  }
};
