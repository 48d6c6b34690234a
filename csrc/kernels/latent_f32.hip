// Latent attention of the fp32 engine in the absorbed form on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32: true fp32
// products and sums); latent.hip's plain kernels take the sizes these do not. All operands go straight to registers in
// 16-byte pieces; which four values of a sum an instruction takes is chosen so that no operand is moved between lanes.
//
// With lane = 16 g + c and step j of four, an operand value belongs to row (or column) c and to summand 4 g + j; a
// result's register r to row 4 g + r and column c. Where the summed index is the slow one in memory, a lane's 16 bytes
// are four rows' (tile t has rows 4 c + t of 64), and its four steps are four loads.
#include "latent.h"

namespace {

LSA_DEVICE f32x4_t mfma(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
LSA_DEVICE f32x4_t ldf4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
constexpr f32x4_t ZERO4 = {0.f, 0.f, 0.f, 0.f};

// qt = W_uk^T q of 16 RT entries and one head: four waves take 64 columns each in turn. One read of the head's matrix per
// workgroup (from L2) bounds it, with few entries the waits for its parts, each requested during the products of the one
// before (4 entries, 16 heads, krp 256: 14.5 -> 6.0 us).
template <int RT>
__global__ __launch_bounds__(256) void absorb_f32_kernel(LatentArgs a, int n, const float* __restrict__ q, int ldq,
                                                         const float* __restrict__ wk, float* __restrict__ qt) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.y, e0 = blockIdx.x * 16 * RT, cw = a.krp + a.rp;
  const float* qr[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int e = min(e0 + 16 * i + c, n - 1), row = a.index ? a.index[e] : e;
    qr[i] = q + (size_t)row * ldq + (size_t)h * (a.dkp + a.rp) + 4 * g;
  }
  const float* wh = wk + (size_t)h * a.dkp * a.krp + (size_t)4 * g * a.krp + 4 * c;
  for (int b = w; b < a.krp / 64; b += 4) {
    f32x4_t acc[RT][4];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[i][t] = ZERO4;
    struct Part {
      f32x4_t x[2][RT], y[2][4];
    };
    auto load = [&](int d, Part& p) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int j = 0; j < 4; ++j) p.y[u][j] = ldf4(wh + (size_t)(d + 16 * u + j) * a.krp + 64 * b);
#pragma unroll
        for (int i = 0; i < RT; ++i) p.x[u][i] = ldf4(qr[i] + d + 16 * u);
      }
    };
    auto mul = [&](const Part& p) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[i][t] = mfma(p.x[u][i][j], p.y[u][j][t], acc[i][t]);
    };
    Part p0;  // dkp % 64 == 0
    if constexpr (RT == 1) {
      Part p1;
      load(0, p0);
#pragma unroll 1
      for (int d = 0; d < a.dkp; d += 64) {
        load(d + 32, p1);
        __builtin_amdgcn_sched_barrier(0);  // requested here, not where it is used
        mul(p0);
        if (d + 64 < a.dkp) load(d + 64, p0);
        __builtin_amdgcn_sched_barrier(0);
        mul(p1);
      }
    } else {
      for (int d = 0; d < a.dkp; d += 32) {
        load(d, p0);
        mul(p0);
      }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = e0 + 16 * i + 4 * g + r;
        if (e < n)
          *reinterpret_cast<f32x4_t*>(qt + ((size_t)e * a.heads + h) * cw + 64 * b + 4 * c) =
              f32x4_t{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
      }
  }
  for (int t = threadIdx.x; t < 16 * RT * a.rp; t += 256) {
    const int e = e0 + t / a.rp, j = t % a.rp;
    if (e >= n) break;
    const int row = a.index ? a.index[e] : e;
    const float* qh = q + (size_t)row * ldq + (size_t)h * (a.dkp + a.rp) + a.dkp;
    qt[((size_t)e * a.heads + h) * cw + a.krp + j] =
        j < a.rot_dim && lat_keys(a, row) > 0 ? lat_rot(a, qh, j, a.pos[row]) : 0.f;
  }
}

// Split softmax attention of one entry and 16 heads: each of four waves takes 16 keys at a time with a maximum, a sum and
// [16 heads][krp] sums of its own, and they meet in LDS at the end; no barrier in the loop. Scores are keys (rows) by heads
// (columns), so that a lane's weights are operands of the value product as they are, and the value product is
// latent dimensions by heads: a head's numbers stay in its lanes. A key's latent is read twice, from L2 the second time.
// Bound by those reads: 963 rows of up to 500 keys, 16 heads, krp 256: the plain kernel, a workgroup per row and head
// with one key per thread, took 1216 us, this 81 (three times the time of its products; 102 with the first rows first, whose
// last ones ran alone; with two neighbouring rows to a workgroup and one read for both 103).
template <int KR>  // krp / 64; rp == 64
__global__ __launch_bounds__(256, KR <= 4 ? 2 : 1) void attend_f32_kernel(LatentArgs a, const float* __restrict__ qt, int ns,
                                                         float* __restrict__ po, float* __restrict__ pm) {
  constexpr int KRP = 64 * KR, CW = KRP + 64, LQ = CW + 4, LO = KRP + 4;
  __shared__ __attribute__((aligned(16))) float s_q[16 * LQ], s_o[2][16 * LO], s_ml[2][4][16];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e = gridDim.x - 1 - blockIdx.x;  // a prompt's last rows see most keys: they begin
  const int h0 = blockIdx.y * 16, s = blockIdx.z, row = a.index ? a.index[e] : e;
  const int len = lat_keys(a, row), first = lat_first(a, len), slot = a.slot[row];
  const int fb = first / LAT_PAGE, nb = (len + LAT_PAGE - 1) / LAT_PAGE - fb;
  const int k0 = max(first, (fb + nb * s / ns) * LAT_PAGE), k1 = min(len, (fb + nb * (s + 1) / ns) * LAT_PAGE);
  const float sl2 = a.scale * 1.4426950408889634f;
  for (int t = tid; t < 16 * (CW / 4); t += 256) {
    const int h = t / (CW / 4), d = t % (CW / 4) * 4;
    const f32x4_t v = ldf4(qt + ((size_t)e * a.heads + min(h0 + h, a.heads - 1)) * CW + d);
    *reinterpret_cast<f32x4_t*>(s_q + h * LQ + d) = v * sl2;
  }
  __syncthreads();
  f32x4_t o[KR][4];
#pragma unroll
  for (int b = 0; b < KR; ++b)
#pragma unroll
    for (int t = 0; t < 4; ++t) o[b][t] = ZERO4;
  float m = -INFINITY, l = 0.f;
  const float* cache = static_cast<const float*>(a.cache);
  const float* sq = s_q + c * LQ + 4 * g;
  for (int kb = (k0 & ~15) + 16 * w; kb < k1; kb += 64) {
    const float* page = cache + (size_t)lat_page(a, slot, kb / LAT_PAGE) * LAT_PAGE * CW;
    // keys outside [k0, k1) weigh nothing; their places are taken by keys of this row's that do
    const int at = min(max(kb + c, k0), k1 - 1) % LAT_PAGE;
    const float* kr = page + (size_t)at * CW + 4 * g;
    f32x4_t sc = ZERO4, sc2 = ZERO4;
#pragma unroll
    for (int d = 0; d < CW; d += 32) {
      const f32x4_t x = ldf4(kr + d), y = ldf4(kr + d + 16), p = ldf4(sq + d), q = ldf4(sq + d + 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sc = mfma(x[j], p[j], sc);
        sc2 = mfma(y[j], q[j], sc2);
      }
    }
    sc += sc2;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = kb + 4 * g + r;
      if (key < k0 || key >= k1) sc[r] = -INFINITY;
      mx = fmaxf(mx, sc[r]);
    }
    mx = fmaxf(mx, lane_xor<16>(mx));
    mx = fmaxf(mx, lane_xor<32>(mx));
    const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
    float p[4], sum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = __builtin_amdgcn_exp2f(sc[r] - mn);
      sum += p[r];
    }
    l = l * alpha + sum;  // this lane's keys
    m = mn;
    const float* vr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) vr[r] = page + (size_t)(min(max(kb + 4 * g + r, k0), k1 - 1) % LAT_PAGE) * CW + 4 * c;
#pragma unroll
    for (int b = 0; b < KR; ++b) {
      f32x4_t v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = ldf4(vr[r] + 64 * b);
#pragma unroll
      for (int t = 0; t < 4; ++t) o[b][t] *= alpha;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t) o[b][t] = mfma(v[r][t], p[r], o[b][t]);
    }
  }
  l += lane_xor<16>(l);
  l += lane_xor<32>(l);
  if (g == 0) {
    s_ml[0][w][c] = m;
    s_ml[1][w][c] = l;
  }
  __syncthreads();
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) M = fmaxf(M, s_ml[0][x][c]);
#pragma unroll
  for (int x = 0; x < 4; ++x)
    if (s_ml[0][x][c] != -INFINITY) L += s_ml[1][x][c] * __builtin_amdgcn_exp2f(s_ml[0][x][c] - M);
  const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
  // waves 0 and 1 write, 2 and 3 add
  float* so = s_o[w & 1] + c * LO + 16 * g;  // dimensions 64 b + 16 g + 4 r + t of head c
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (w >> 1 == half) {
#pragma unroll
      for (int b = 0; b < KR; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4_t v = f32x4_t{o[b][0][r], o[b][1][r], o[b][2][r], o[b][3][r]} * f;
          f32x4_t* to = reinterpret_cast<f32x4_t*>(so + 64 * b + 4 * r);
          if (half) v += *to;
          *to = v;
        }
    }
    __syncthreads();
  }
  for (int t = tid; t < 16 * (KRP / 4); t += 256) {
    const int h = t / (KRP / 4), d = t % (KRP / 4) * 4;
    if (h0 + h >= a.heads) break;
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(s_o[0] + h * LO + d) + *reinterpret_cast<const f32x4_t*>(s_o[1] + h * LO + d);
    *reinterpret_cast<f32x4_t*>(po + (((size_t)e * a.heads + h0 + h) * ns + s) * KRP + d) = v;
  }
  if (tid < 16 && h0 + tid < a.heads) {  // (c == tid)
    const size_t at = ((size_t)e * a.heads + h0 + tid) * ns + s;
    pm[at * 2] = M;
    pm[at * 2 + 1] = L;
  }
}

// Merge of the splits, W_uv and gate of 16 entries and one head: four waves share K and meet in LDS, 64 columns at a time, whose
// weights are requested before the merge and before the last columns meet (4 entries, 16 heads, krp 256: 15.5 -> 10.6 us).
template <int KR>
__global__ __launch_bounds__(256) void value_f32_kernel(LatentArgs a, int n, const float* __restrict__ po,
                                                        const float* __restrict__ pm, int ns, const float* __restrict__ wv,
                                                        const float* __restrict__ gate, int ldg, float* __restrict__ out,
                                                        int ldo) {
  constexpr int KRP = 64 * KR;
  __shared__ __attribute__((aligned(16))) float s_acc[4][16][68], s_f[16][65];  // factor of every split
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.y, e0 = blockIdx.x * 16;
  // this wave's part of K: 16 KR of the latent's dimensions
  const float* wh = wv + (size_t)h * KRP * a.dvp + (size_t)(16 * KR * w + 4 * g) * a.dvp + 4 * c;
  f32x4_t y[KR][4];
  auto load_w = [&](int b) {
#pragma unroll
    for (int u = 0; u < KR; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) y[u][j] = ldf4(wh + (size_t)(16 * u + j) * a.dvp + 64 * b);
  };
  const int step = gridDim.z;  // columns 64 b ..: all of them, or each 64 a workgroup's
  load_w(blockIdx.z);
  __builtin_amdgcn_sched_barrier(0);  // requested here, not where it is used
  if (tid < 16) {
    const float* pe = pm + ((size_t)min(e0 + tid, n - 1) * a.heads + h) * ns * 2;
    float M = -INFINITY, L = 0.f;
    for (int s = 0; s < ns; ++s) M = fmaxf(M, pe[2 * s]);
    if (M == -INFINITY) M = 0.f;
    for (int s = 0; s < ns; ++s) L += pe[2 * s + 1] * __builtin_amdgcn_exp2f(pe[2 * s] - M);
    L += lat_sink(a, h, M);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    for (int s = 0; s < ns; ++s) s_f[tid][s] = __builtin_amdgcn_exp2f(pe[2 * s] - M) * inv;
  }
  __syncthreads();
  f32x4_t x[KR];
#pragma unroll
  for (int u = 0; u < KR; ++u) x[u] = ZERO4;
  const float* pr = po + ((size_t)min(e0 + c, n - 1) * a.heads + h) * ns * KRP + 16 * KR * w + 4 * g;
  for (int s = 0; s < ns; ++s) {
    const float f = s_f[c][s];
#pragma unroll
    for (int u = 0; u < KR; ++u) x[u] += ldf4(pr + (size_t)s * KRP + 16 * u) * f;
  }
  for (int b = blockIdx.z; b < a.dvp / 64; b += step) {
    f32x4_t acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = ZERO4;
#pragma unroll
    for (int u = 0; u < KR; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = mfma(x[u][j], y[u][j][t], acc[t]);
    if (b + step < a.dvp / 64) load_w(b + step);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<f32x4_t*>(&s_acc[w][4 * g + r][4 * c]) = f32x4_t{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
    __syncthreads();
    const int i = tid >> 4, e = e0 + i, j = (tid & 15) * 4;
    if (e < n) {
      f32x4_t v = ZERO4;
#pragma unroll
      for (int k = 0; k < 4; ++k) v += *reinterpret_cast<const f32x4_t*>(&s_acc[k][i][j]);
      const int row = a.index ? a.index[e] : e;
      const size_t at = (size_t)h * a.dvp + 64 * b + j;
      if (gate) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] *= sigmoid(gate[(size_t)row * ldg + at + k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) out[(size_t)row * ldo + at + k] = v[k];
    }
    __syncthreads();
  }
}

bool aligned(const void* p, int ld) { return (uintptr_t)p % 16 == 0 && ld % 4 == 0; }
bool latent_size(const LatentArgs& a) {
  return a.rp == 64 && (a.krp == 64 || a.krp == 128 || a.krp == 256 || a.krp == 512);
}

}  // namespace

bool latent_absorb_f32(const LatentArgs& a, int n, const float* q, int ldq, const float* wk, float* qt, hipStream_t s) {
  if (!aligned(q, ldq) || !aligned(wk, 0) || !aligned(qt, 0)) return false;
  // 32 entries per workgroup (half the reads of the matrix) where that still makes two workgroups per CU
  if ((long)(n + 31) / 32 * a.heads >= 512) absorb_f32_kernel<2><<<dim3((n + 31) / 32, a.heads), 256, 0, s>>>(a, n, q, ldq, wk, qt);
  else absorb_f32_kernel<1><<<dim3((n + 15) / 16, a.heads), 256, 0, s>>>(a, n, q, ldq, wk, qt);
  return true;
}

bool latent_attend_f32(const LatentArgs& a, int n, const float* qt, int ns, float* po, float* pm, hipStream_t s) {
  if (!latent_size(a) || !aligned(a.cache, 0) || !aligned(qt, 0) || !aligned(po, 0)) return false;
  const dim3 grid(n, (a.heads + 15) / 16, ns);
  auto* f = a.krp == 64 ? attend_f32_kernel<1> : a.krp == 128 ? attend_f32_kernel<2> : a.krp == 256 ? attend_f32_kernel<4>
                                                                                                 : attend_f32_kernel<8>;
  f<<<grid, 256, 0, s>>>(a, qt, ns, po, pm);
  return true;
}

bool latent_value_f32(const LatentArgs& a, int n, const float* po, const float* pm, int ns, const float* wv, const float* gate,
                      int ldg, float* out, int ldo, hipStream_t s) {
  if (!latent_size(a) || !aligned(po, 0) || !aligned(wv, 0)) return false;
  auto* f = a.krp == 64 ? value_f32_kernel<1> : a.krp == 128 ? value_f32_kernel<2> : a.krp == 256 ? value_f32_kernel<4>
                                                                                               : value_f32_kernel<8>;
  const int wg = (n + 15) / 16 * a.heads, blocks = a.dvp / 64;
  f<<<dim3((n + 15) / 16, a.heads, wg * blocks <= 256 ? blocks : 1), 256, 0, s>>>(a, n, po, pm, ns, wv, gate, ldg, out, ldo);
  return true;
}
