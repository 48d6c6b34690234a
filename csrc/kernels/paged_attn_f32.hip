// Paged grouped-query attention of the fp32 engine (paged_attn.h) on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32:
// true fp32 products and sums); paged_attn.hip's plain kernel takes the sizes this does not.
//
// A workgroup takes up to 16 (row, head) pairs of one kv head as the columns of its tiles: the heads of one row, or of
// as many rows of one sequence as fit. Scores are keys (rows of a tile) by pairs, values channels by pairs, so that a
// lane's four weights are operands of the value product as they are (step r: key 4 g + r of lane = 16 g + c), and a pair's
// numbers stay in its lanes. Keys lie token by token, values channel by channel with four tokens of a lane side by side
// (att_vidx): both go to registers in 16-byte pieces. Each wave takes 32 keys at a time with sums of its own, and
// they meet in LDS at the end; no barrier in the loop. Where every workgroup has a CU to itself there are eight waves.
// Bound by the latency of its reads; at 2560 rows of up to 200 keys, 16 heads of 128 over 4 kv heads, it takes 84 us (softmax)
// and 97 us (sigmoids), at 16 rows in a decoding step 15.2 and 18 (19.5 and 23.9 with four waves and pages looked up one by one). The plain kernel, a
// workgroup per row and head, takes 2300 at 2560 rows.
#include <type_traits>
#include "paged_attn.h"

namespace {

LSA_DEVICE f32x4_t mfma(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
LSA_DEVICE f32x4_t ldf4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }

// DV: dvp / 64. U: scores' operands are requested for 16 U channels together: 4 for as few workgroups as have a CU's registers
// to themselves (16 rows, 16 heads of 128 over 4: 15.0 us, with 2 15.8), else 2 and a wave more per SIMD (256 rows 35 us, with
// 4 45).
template <int DV, bool SIG, int U, int NW>
__global__ __launch_bounds__(NW * 64, U == 4 || DV == 1 ? 2 : DV == 2 ? 4 : 3) void attend_f32_kernel(
    AttnArgs a, int n, int per, const float* __restrict__ q, int ldq, const float* __restrict__ gate, int ldg,
    float* __restrict__ out, int ldo) {
  constexpr int DVP = 64 * DV, LO = DVP + 4, NT = NW * 64, NO = NW / 2;
  extern __shared__ __attribute__((aligned(16))) float s_q[];  // [16][dkp + 4]
  __shared__ __attribute__((aligned(16))) float s_o[NO][16 * LO], s_ml[2][NW][16];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.heads / a.kv_heads, kvh = blockIdx.y, lq = a.dkp + 4;
  const int e0 = blockIdx.x * per, ne = min(per, n - e0);
  for (int s0 = 0, s1; s0 < ne; s0 = s1) {
    const int row0 = a.index ? a.index[e0 + s0] : e0 + s0, slot = __builtin_amdgcn_readfirstlane(a.slot[row0]);
    const int pos0 = __builtin_amdgcn_readfirstlane(a.pos[row0]);
    auto queries = [&](int cols) {
      for (int t = tid; t < cols * a.dkp; t += NT) {
        const int x = t / a.dkp, d = t % a.dkp, e = e0 + s0 + x / G;
        s_q[x * lq + d] = q[(size_t)(a.index ? a.index[e] : e) * ldq + (size_t)(kvh * G + x % G) * a.dkp + d];
      }
    };
    // Reads that wait for one another are most of a few rows' time: the first 64 pages of the sequence come in one, beside a
    // single row's queries.
    const bool live = pos0 >= 0 && pos0 < a.max_pages * ATT_PAGE;
    const int first_pages = live ? a.table[(size_t)slot * a.max_pages + min(lane, a.max_pages - 1)] : -1;
    if (per == 1) queries(G);
    auto table = [&](int b) {
      return b < 64 ? __builtin_amdgcn_readlane(first_pages, b) : a.table[(size_t)slot * a.max_pages + b];
    };
    int p0 = -1;
    if (live) {
      const int pg = table(pos0 / ATT_PAGE);
      if (pg >= 0 && pg < a.n_pages) p0 = pos0;
    }
    s1 = s0 + 1;
    if (p0 < 0) {  // an idle row
      for (int d = tid; d < G * a.dvp; d += NT) out[(size_t)row0 * ldo + (size_t)kvh * G * a.dvp + d] = 0.f;
      continue;
    }
    int lo = p0, hi = p0;
    for (; s1 < ne; ++s1) {  // rows of the same sequence
      const int r = a.index ? a.index[e0 + s1] : e0 + s1, p = att_pos(a, r);
      if (p < 0 || a.slot[r] != slot) break;
      lo = min(lo, p);
      hi = max(hi, p);
    }
    const int cols = (s1 - s0) * G;
    const int mine = s0 + min(c, cols - 1) / G;  // columns past the last are computed and not stored
    const int row = a.index ? a.index[e0 + mine] : e0 + mine, h = kvh * G + min(c, cols - 1) % G, p = a.pos[row];
    const float hs = att_scale(a, h, p);
    float r1 = 0.f, r2 = 0.f, b2 = 0.f;
    if constexpr (SIG) {
      r1 = a.sig[h];
      r2 = a.sig[a.heads + h];
      b2 = a.sig[2 * a.heads + h];
    }
    if (per != 1) queries(cols);
    __syncthreads();
    const float* sq = s_q + min(c, cols - 1) * lq + 4 * g4;
    const AttBlocks blocks(a, lo, hi);
    const int pooled = att_pooled(a, hi), mine_pooled = att_pooled(a, p);
    f32x4_t o[4 * DV];
    float m, l;
    // A value that a pair does not see, or whose weight is 0, has no part in its sums, whatever it is: a tile's product is 0
    // times it, which an infinity or a NaN would make a NaN of. A wave whose sums are not all finite takes its keys once more,
    // each pair without what it gives no weight to, by the maximum of all waves' keys (m0; a sum that is an infinity is not
    // scaled down to 0). (The check is 1 to 3 % of 16 to 67 us: one row of 64 to 256 sequences.)
    auto sums = [&](auto apart, float m0) {
#pragma unroll
      for (int t = 0; t < 4 * DV; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      m = m0, l = 0.f;
      for (int i = w; i < 2 * blocks.n; i += NW) {
        const bool pool = blocks.is_pooled(i >> 1);
        const int half = 32 * (i & 1), key0 = blocks.at(i >> 1) * ATT_PAGE + half;
        const int last = pool ? pooled - 1 : hi;  // behind it nothing was written
        if (key0 > last) continue;
        AttKv kv;
        if (pool) {
          kv = att_kv(a, blocks, slot, i >> 1);
        } else {
          const int pg = table(__builtin_amdgcn_readfirstlane(blocks.at(i >> 1)));
          kv = AttKv{a.k, a.v, pg < 0 || pg >= a.n_pages ? 0 : pg};
        }
        const size_t page = (size_t)kv.page * a.kv_heads + kvh;
        const float* kb = (const float*)kv.k + page * ATT_PAGE * a.dkp + 4 * g4;
        const float* k0 = kb + (size_t)(half + min(c, last - key0)) * a.dkp;
        const float* k1 = kb + (size_t)(half + min(c + 16, last - key0)) * a.dkp;
        // A score is added up from sums of every fourth of 16 U values, pair by pair: in one sum of all its rounding is twice
        // the plain kernel's, so it is nine tenths of it.
        f32x4_t sc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
        for (int d = 0; d < a.dkp; d += 16 * U) {  // dkp % 64 == 0
          f32x4_t x[U], y[U], z[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            x[u] = ldf4(k0 + d + 16 * u);
            y[u] = ldf4(k1 + d + 16 * u);
            z[u] = ldf4(sq + d + 16 * u);
          }
          __builtin_amdgcn_sched_barrier(0);  // all requested before the first is waited for
          f32x4_t sum[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            f32x4_t p[2][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              p[0][j] = p[1][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int u = 0; u < U; ++u) {
                p[0][j] = mfma(x[u][2 * h + j], z[u][2 * h + j], p[0][j]);
                p[1][j] = mfma(y[u][2 * h + j], z[u][2 * h + j], p[1][j]);
              }
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) sum[k] = h ? sum[k] + (p[k][0] + p[k][1]) : p[k][0] + p[k][1];
            if constexpr (U == 2) __builtin_amdgcn_sched_barrier(0);  // (else all eight are kept)
          }
          sc[0] += sum[0];
          sc[1] += sum[1];
        }
        float wt[2][4], mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = key0 + 16 * u + 4 * g4 + r;
            const bool sees = pool ? key < mine_pooled : att_sees(a, p, key);
            float s = sc[u][r] * hs;
            if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
            if constexpr (SIG) {
              s += b2 - r1 * log1pf(r2 * (float)(p - key));
              wt[u][r] = sees ? 1.f / (1.f + expf(-s)) : 0.f;
            } else {
              wt[u][r] = sees ? s : -INFINITY;
              mx = fmaxf(mx, wt[u][r]);
            }
          }
        float alpha = 1.f;
        if constexpr (!SIG) {
          mx = fmaxf(mx, lane_xor<16>(mx));
          mx = fmaxf(mx, lane_xor<32>(mx));
          const float mn = fmaxf(m, mx), at = mn == -INFINITY ? 0.f : mn;  // (no key of these 32 or before is this pair's)
          alpha = expf(m - at);
          float sum = 0.f;
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              wt[u][r] = expf(wt[u][r] - at);
              sum += wt[u][r];
            }
          l = l * alpha + sum;
          m = mn;
        }
        // tokens half + 16 u + 4 g4 + r of a channel lie at half + 8 g4 + 4 u + r
        const float* vb = (const float*)kv.v + page * a.dvp * ATT_PAGE + (size_t)c * ATT_PAGE + half + 8 * g4;
        const bool cut = key0 + 31 > last;
#pragma unroll
        for (int t = 0; t < 4 * DV; ++t) {
          f32x4_t v[2] = {ldf4(vb + (size_t)t * 16 * ATT_PAGE), ldf4(vb + (size_t)t * 16 * ATT_PAGE + 4)};
          if (cut) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (key0 + 16 * u + 4 * g4 + r > last) v[u][r] = 0.f;
          }
          if constexpr (!SIG) o[t] *= alpha;
          if constexpr (decltype(apart)::value) {
            f32x4_t own = o[t];
            for (int x = 0; x < cols; ++x) {
              f32x4_t y = o[t];
#pragma unroll
              for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  y = mfma(__shfl(wt[u][r], (lane & 48) | x, 64) != 0.f ? v[u][r] : 0.f, wt[u][r], y);
              if (c == x) own = y;
            }
            o[t] = own;
          } else {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[t] = mfma(v[u][r], wt[u][r], o[t]);
          }
        }
      }
    };
    sums(std::false_type{}, -INFINITY);
    bool finite = true;
#pragma unroll
    for (int t = 0; t < 4 * DV; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) finite = finite && fabsf(o[t][r]) < INFINITY;
    const bool again = !__all(finite);
    float f = 1.f, F = a.oscale, M = -INFINITY;
    if constexpr (!SIG) {
      l += lane_xor<16>(l);
      l += lane_xor<32>(l);
      if (g4 == 0) {
        s_ml[0][w][c] = m;
        s_ml[1][w][c] = l;
      }
      __syncthreads();
      float L = 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) M = fmaxf(M, s_ml[0][x][c]);
#pragma unroll
      for (int x = 0; x < NW; ++x)
        if (s_ml[0][x][c] != -INFINITY) L += s_ml[1][x][c] * expf(s_ml[0][x][c] - M);
      f = again ? 1.f : m == -INFINITY ? 0.f : expf(m - M);
      const float t = a.sink ? fmaxf(M, 0.f) : M, e = expf(M - t);
      F *= e / (L * e + (a.sink ? expf(-t) : 0.f));
    }
    if (again) sums(std::true_type{}, M);
    f *= F;
    // the first half of the waves write, the others add: channels 16 t + 4 g4 + r of pair c
    float* so = s_o[w % NO] + c * LO + 4 * g4;
#pragma unroll
    for (int turn = 0; turn < 2; ++turn) {
      if (w / NO == turn) {
#pragma unroll
        for (int t = 0; t < 4 * DV; ++t) {
          f32x4_t v = o[t] * f;
          f32x4_t* to = reinterpret_cast<f32x4_t*>(so + 16 * t);
          if (turn) v += *to;
          *to = v;
        }
      }
      __syncthreads();
    }
    for (int t = tid; t < cols * a.dvp; t += NT) {
      const int x = t / a.dvp, d = t % a.dvp, e = e0 + s0 + x / G, r = a.index ? a.index[e] : e, hh = kvh * G + x % G;
      float y = s_o[0][x * LO + d];
#pragma unroll
      for (int k = 1; k < NO; ++k) y += s_o[k][x * LO + d];
      out[(size_t)r * ldo + (size_t)hh * a.dvp + d] = y * att_gate(a, gate, r, ldg, hh, d);
    }
    __syncthreads();  // s_q, s_o and s_ml serve the next sequence
  }
}

}  // namespace

bool attn_f32(const AttnArgs& a, int n, bool singles, const float* q, int ldq, const float* gate, int ldg, float* out, int ldo,
              hipStream_t s) {
  const int G = a.heads / a.kv_heads;
  if (G > 16 || a.dkp > 256 || (a.dvp != 64 && a.dvp != 128 && a.dvp != 256) ||
      ((uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.pk | (uintptr_t)a.pv) % 16)
    return false;
  // Rows of one sequence share its keys' reads once there are 1024 workgroups of a row each, as many as leave one for every CU:
  // 128 rows of a sequence, 8 heads over 8 kv heads 12.1 us, with a row each 24.8, with 16 each 18.1; 256 rows, 16 heads over 4
  // 14.8 and with a row each 26.5. Rows of as many sequences would run one after another in a workgroup: up to 200 keys, 128 rows
  // of 8 over 8 219 us with 16 each, 46 with one; 256 of 16 over 4 57 and 35 (the plain kernel 122 and 303).
  const long all = (long)n * a.kv_heads;
  const int per = singles || all < 1024 ? 1 : (int)min(16L / G, all / 256);
  const dim3 grid((n + per - 1) / per, a.kv_heads);
  const size_t lds = (size_t)16 * (a.dkp + 4) * 4;
  const bool few = all <= 512, alone = all <= 256;
#define LSA_K(DV, SIG, U, NW) attend_f32_kernel<DV, SIG, U, NW><<<grid, NW * 64, lds, s>>>(a, n, per, q, ldq, gate, ldg, out, ldo)
#define LSA_S(DV, SIG)                 \
  if (alone) LSA_K(DV, SIG, 4, 8);     \
  else if (few) LSA_K(DV, SIG, 4, 4);  \
  else LSA_K(DV, SIG, 2, 4)
#define LSA_A(DV)                              \
  if (a.sig) {                                 \
    LSA_S(DV, true);                           \
  } else {                                     \
    LSA_S(DV, false);                          \
  }
  if (a.dvp == 64) {
    LSA_A(1)
  } else if (a.dvp == 128) {
    LSA_A(2)
  } else {
    LSA_A(4)
  }
#undef LSA_A
#undef LSA_S
#undef LSA_K
  return true;
}
