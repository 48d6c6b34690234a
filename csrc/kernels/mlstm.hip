// Matrix memory step by step (mlstm.h): one workgroup per (run, head) keeps the head's state in registers and walks
// the run's rows; everything between the projections and the output projection in one launch. The fp32 engine runs whole
// portions this way.
#include "mlstm.h"

namespace {

template <typename T>
LSA_DEVICE void ml_row(const MlArgs& a, int row, int h, int DK, int DV, float* sq, float* sk, float* sv) {
  const T* in = (const T*)a.in + (size_t)row * a.ldi;
  for (int c = threadIdx.x; c < 2 * DK + DV; c += 256) {
    if (c < DK) sq[c] = ld1(in + a.oq + h * DK + c) * a.q_scale;
    else if (c < 2 * DK) sk[c - DK] = ld1(in + a.ok + h * DK + c - DK);
    else sv[c - 2 * DK] = ld1(in + a.ov + h * DV + c - 2 * DK);
  }
}

template <typename T>
LSA_DEVICE void ml_store(const MlArgs& a, int row, int h, int d, float o, float rs, float g) {
  st1((T*)a.out + (size_t)row * a.ldo + h * a.dv + d, o * rs * a.norm[h * a.dv + d] * sigmoid(g));
}
template <typename T>
LSA_DEVICE float ml_out_gate(const MlArgs& a, int row, int h, int d) {
  return ld1((const T*)a.in + (size_t)row * a.ldi + a.og + h * a.dv + d);
}

template <typename T>
LSA_DEVICE bool ml_idle(const MlArgs& a, const MlRun& r, int h) {
  if (r.n) return false;
  if (!a.runs)
    for (int d = threadIdx.x; d < a.dv; d += blockDim.x) st1((T*)a.out + (size_t)r.row0 * a.ldo + h * a.dv + d, 0.f);
  return true;
}

LSA_DEVICE float lane_at(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// Row by row: all threads share the key channels, one wave norms the read-out, the next row's operands are requested while
// this one is computed. ONE: a launch of single rows (decoding) has a kernel without the loop, whose operands took a 128 x 128
// state's workgroups from four to two waves per SIMD: 4 sequences, 16 heads 5.1 us, with the loop 5.8; 64 sequences 21.8 and 24.3.
// With it, such a state is bounded to three: 128 runs of 4 rows 68 -> 59 us, of 8 106 -> 86.
template <typename T, int DK, int DV, bool ONE>
__global__ __launch_bounds__(256, !ONE && DK * DV == 128 * 128 ? 3 : 1) void ml_rows_kernel(MlArgs a) {
  // a thread holds RPT rows x 4 value channels of S and the same rows of n
  constexpr int NG = 1024 / DV, RPT = DK / NG, NX = (2 * DK + DV + 255) / 256;
  constexpr int NO = (DV + 63) / 64;  // channels per lane of the wave that stores
  static_assert(RPT >= 1 && NG * RPT == DK, "geometry");
  __shared__ __attribute__((aligned(16))) float s_in[2 * DK + DV], s_b[NG][DV], s_n[NG];
  const MlRun r = ml_run(a, blockIdx.x);
  const int h = blockIdx.y, tid = threadIdx.x, v = (tid % (DV / 4)) * 4, grp = tid / (DV / 4), d0 = grp * RPT;
  if (ml_idle<T>(a, r, h)) return;
  const size_t head = (size_t)r.slot * a.heads + h;
  float* st = a.S + head * DK * DV + (size_t)d0 * DV + v;
  float* sn = a.n + head * a.copies * DK;
  struct Row {
    float x[NX], gate[NO], i, f;
  };
  auto load = [&](int row, Row& y) {
    const T* in = (const T*)a.in + (size_t)row * a.ldi;
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int c = tid + 256 * u;
      y.x[u] = ld1(in + (c < DK ? a.oq + h * DK + c : c < 2 * DK ? a.ok + h * DK + c - DK : a.ov + h * DV + min(c - 2 * DK, DV - 1)));
    }
#pragma unroll
    for (int u = 0; u < NO; ++u) y.gate[u] = ml_out_gate<T>(a, row, h, ((tid & 63) + 64 * u) % DV);
    y.i = ml_input_gate(a, row, h);
    y.f = ml_forget_gate(a, row, h);
  };
  Row y;
  load(r.row0, y);
  const bool fresh = r.pos0 == 0;
  float m = fresh ? 0.f : a.m[head * a.copies];
  f32x4_t S[RPT];
  float n[RPT];
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    S[j] = fresh ? f32x4_t{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4_t*>(st + (size_t)j * DV);
    n[j] = fresh ? 0.f : sn[d0 + j];
  }
  for (int t = 0; t < (ONE ? 1 : r.n); ++t) {
    const bool last = ONE || t + 1 == r.n;
    const float i = y.i, fm = y.f + m;
    m = fmaxf(fm, i);
    const float keep = expf(fm - m), add = expf(i - m);
    float gate[NO];
#pragma unroll
    for (int u = 0; u < NO; ++u) gate[u] = y.gate[u];
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int c = tid + 256 * u;
      if (c < 2 * DK + DV) s_in[c] = c < DK ? y.x[u] * a.q_scale : y.x[u];
    }
    __syncthreads();
    if (!last) load(r.row0 + t + 1, y);
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where it is first used
    const f32x4_t u4 = *reinterpret_cast<const f32x4_t*>(&s_in[2 * DK + v]) * add;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    float nq = 0.f;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const float q = s_in[d0 + j], k = s_in[DK + d0 + j];
      S[j] = S[j] * keep + u4 * k;
      o += S[j] * q;
      n[j] = n[j] * keep + add * k;
      nq += n[j] * q;
      if (last) *reinterpret_cast<f32x4_t*>(st + (size_t)j * DV) = S[j];
    }
    *reinterpret_cast<f32x4_t*>(&s_b[grp][v]) = o;
    if (v == 0) s_n[grp] = nq;
    __syncthreads();
    if (tid >= 64) continue;  // s_in is written again by now, s_b and s_n behind the next row's first barrier
    float z = 0.f, x[NO], ss = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g) z += s_n[g];
    const float den = ml_denominator(z, m);
#pragma unroll
    for (int u = 0; u < NO; ++u) {
      const int d = tid + 64 * u;
      x[u] = 0.f;
      if (d < DV) {
#pragma unroll
        for (int g = 0; g < NG; ++g) x[u] += s_b[g][d];
        x[u] /= den;
      }
      ss += x[u] * x[u];
    }
    const float rs = 1.f / sqrtf(wave_sum(ss) / (float)a.vdim + a.eps);
#pragma unroll
    for (int u = 0; u < NO; ++u)
      if (tid + 64 * u < DV) ml_store<T>(a, r.row0 + t, h, tid + 64 * u, x[u], rs, gate[u]);
  }
  for (int c = 0; c < a.copies; ++c) {
    if (v == 0) {
#pragma unroll
      for (int j = 0; j < RPT; ++j) sn[(size_t)c * DK + d0 + j] = n[j];
    }
    if (tid == 0) a.m[head * a.copies + c] = m;
  }
}

// over the lanes with the same lane % 4
LSA_DEVICE float over_quads(float x) {
  x += dpp_mov<0x124>(x);
  x += dpp_mov<0x128>(x);
  x += lane_xor<16>(x);
  return x + lane_xor<32>(x);
}

// Rows in batches of BR: their operands and gates come together, the next batch's are requested while this one is computed,
// and the read-outs are normed and stored together, so that a batch has two barriers. A wave has 16 value channels and all
// key channels of the state, and no step waits for another wave. Bound by the vector unit: three operations per element of
// the state and row, what a wave does for n and the sums over its lanes make 0.7 us a row at 128 x 128. 4 portions of 300
// rows, 16 heads, fp32: 267 us; with two barriers a row 500, without the operands requested ahead 805.
template <typename T, int DK, int DV>
__global__ __launch_bounds__(DV * 4) void ml_steps_kernel(MlArgs a) {
  constexpr int NT = DV * 4, BR = 16, W = 2 * DK + DV, NX = (BR * W + NT - 1) / NT;
  constexpr int KPL = DK / 16, KV = KPL < 4 ? KPL : 4;  // key channels of a lane, together in groups of KV
  constexpr int L = DV / 4;                             // threads per row of the read-out, 4 channels each
  static_assert(KPL % KV == 0 && NT / L == BR, "geometry");
  __shared__ __attribute__((aligned(16))) float s_in[BR][W], so[BR][DV];  // q, k, v
  __shared__ float s_nq[BR], s_m[BR];
  const MlRun r = ml_run(a, blockIdx.x);
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 2, v = w * 16 + (lane & 3) * 4;
  if (ml_idle<T>(a, r, h)) return;
  const size_t head = (size_t)r.slot * a.heads + h;
  float* const st = a.S + head * DK * DV + v;
  float* const sn = a.n + head * a.copies * DK;
  const auto key = [&](int j) { return (j / KV * 16 + kg) * KV + j % KV; };
  f32x4_t S[KPL];
  float n[KPL], m = r.pos0 == 0 ? 0.f : a.m[head * a.copies];
#pragma unroll
  for (int j = 0; j < KPL; ++j) {
    S[j] = r.pos0 == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4_t*>(st + (size_t)key(j) * DV);
    n[j] = r.pos0 == 0 ? 0.f : sn[key(j)];
  }
  float x[NX], zi, zf;
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + NT * u, t = e / W, c = e % W;
      const int at = c < DK ? a.oq + h * DK + c : c < 2 * DK ? a.ok + h * DK + c - DK : a.ov + h * DV + c - 2 * DK;
      x[u] = t < BR && t0 + t < r.n ? ld1((const T*)a.in + (size_t)(r.row0 + t0 + t) * a.ldi + at) : 0.f;
    }
    const float* z = a.in32 + (size_t)(r.row0 + min(t0 + (lane & (BR - 1)), r.n - 1)) * a.ldi32 + h;
    zi = z[a.oi];
    zf = z[a.of];
  };
  load(0);
  const int rt = tid / L, rl = tid % L;  // this thread's row and channels rl + L j of the read-out
  for (int t0 = 0; t0 < r.n; t0 += BR) {
    const int nb = min(BR, r.n - t0);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + NT * u, c = e % W;
      if (e < BR * W) (&s_in[0][0])[e] = c < DK ? x[u] * a.q_scale : x[u];
    }
    // a lane's gates, the running maximum of its row, and from these what its step keeps and adds
    const float i = ml_in(a, zi), f = ml_forget(a, zf);
    float fm = 0.f, mx = 0.f;
    for (int t = 0; t < nb; ++t) {
      const float y = lane_at(f, t) + m;
      m = fmaxf(y, lane_at(i, t));
      if ((lane & (BR - 1)) == t) fm = y, mx = m;
    }
    const float keep = expf(fm - mx), add = expf(i - mx);
    __syncthreads();
    if (tid < BR) s_m[tid] = mx;
    const int row = r.row0 + t0 + min(rt, nb - 1);
    float gate[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) gate[j] = ml_out_gate<T>(a, row, h, rl + L * j);
    if (t0 + BR < r.n) load(t0 + BR);
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where they are first used
    typedef float kvec __attribute__((ext_vector_type(KV)));
    struct Row {
      kvec q[KPL / KV], k[KPL / KV];
      f32x4_t v;
    };
    auto fetch = [&](int t, Row& y) {
#pragma unroll
      for (int g = 0; g < KPL / KV; ++g) {
        y.q[g] = *reinterpret_cast<const kvec*>(&s_in[t][key(g * KV)]);
        y.k[g] = *reinterpret_cast<const kvec*>(&s_in[t][DK + key(g * KV)]);
      }
      y.v = *reinterpret_cast<const f32x4_t*>(&s_in[t][2 * DK + v]);
    };
    auto step = [&](int t, const Row& y) {
      const float kp = lane_at(keep, t), ad = lane_at(add, t);
      const f32x4_t u = y.v * ad;
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
      float nq = 0.f;
#pragma unroll
      for (int j = 0; j < KPL; ++j) {
        const float q = y.q[j / KV][j % KV], k = y.k[j / KV][j % KV];
        S[j] = S[j] * kp + u * k;
        o += S[j] * q;
        n[j] = n[j] * kp + ad * k;
        nq += n[j] * q;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = over_quads(o[e]);
      nq = over_quads(nq);
      if (kg == 0) *reinterpret_cast<f32x4_t*>(&so[t][v]) = o;
      if (tid == 0) s_nq[t] = nq;
    };
    Row y0, y1;
    fetch(0, y0);
    for (int t = 0; t < nb; t += 2) {  // (a row past the batch is read and not used)
      fetch(t + 1, y1);
      step(t, y0);
      if (t + 1 >= nb) break;
      fetch(min(t + 2, BR - 1), y0);
      step(t + 1, y1);
    }
    __syncthreads();
    if (rt >= nb) continue;  // whole rows; s_in and so are written again behind this barrier and the next
    const float den = ml_denominator(s_nq[rt], s_m[rt]);
    float y[4], ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      y[j] = so[rt][rl + L * j] / den;
      ss += y[j] * y[j];
    }
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float rs = 1.f / sqrtf(ss / (float)a.vdim + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) ml_store<T>(a, row, h, rl + L * j, y[j], rs, gate[j]);
  }
#pragma unroll
  for (int j = 0; j < KPL; ++j) *reinterpret_cast<f32x4_t*>(st + (size_t)key(j) * DV) = S[j];
  for (int c = 0; c < a.copies; ++c) {
    if (w == 0 && (lane & 3) == 0) {
#pragma unroll
      for (int j = 0; j < KPL; ++j) sn[(size_t)c * DK + key(j)] = n[j];
    }
    if (tid == 0) a.m[head * a.copies + c] = m;
  }
}

// As above for runs that leave CUs idle: 32 value channels a workgroup, a wave 8 of them, so that a head has DV / 32 workgroups
// of one wave per SIMD, and a lane 16 elements of the state instead of 32. The four sums over 32 lanes are halved with their
// lanes. Read-outs go out as they are; n and m, which every workgroup reads and only the first writes, go to nm
// [run][head][DK + 1]; ml_finish_kernel norms the ones and puts the others in their place.
// Bound by the vector unit, some 100 instructions a row and 700 a batch for its gates and operands: 0.35 us a row. 4 portions
// of 300 rows, 16 heads of 128 x 128: 267 -> 117 us (ml_steps_kernel, these two kernels).
template <int DK, int DV>
__global__ __launch_bounds__(256) void ml_split_kernel(MlArgs a, float* __restrict__ nm) {
  constexpr int BR = 16, V = 32, W = 2 * DK + V, Q = W / 4, NX = (BR * Q + 255) / 256, KPL = DK / 32;
  __shared__ __attribute__((aligned(16))) float s_in[BR][W], so[BR][V];  // q, k, v
  __shared__ float s_nq[BR], s_m[BR];
  const MlRun r = ml_run(a, blockIdx.x);
  const int h = blockIdx.y, v0 = blockIdx.z * V, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 1;
  if (!r.n) return;
  const size_t head = (size_t)r.slot * a.heads + h;
  const int v = w * 8 + (lane & 1) * 4;
  float* const st = a.S + head * DK * DV + v0 + v;
  const float* const sn = a.n + head * a.copies * DK;
  const bool fresh = r.pos0 == 0;
  f32x4_t S[KPL];
  float n[KPL], m = fresh ? 0.f : a.m[head * a.copies];
#pragma unroll
  for (int j = 0; j < KPL; ++j) {
    S[j] = fresh ? f32x4_t{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4_t*>(st + (size_t)(kg * KPL + j) * DV);
    n[j] = fresh ? 0.f : sn[kg * KPL + j];
  }
  const float* const in = (const float*)a.in + (size_t)r.row0 * a.ldi;
  f32x4_t x[NX];
  float zi, zf;
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u, t = min(t0 + e / Q, r.n - 1), c = e % Q * 4;
      const int at = c < DK ? a.oq + h * DK + c : c < 2 * DK ? a.ok + h * DK + c - DK : a.ov + h * DV + v0 + c - 2 * DK;
      x[u] = *reinterpret_cast<const f32x4_t*>(in + (size_t)t * a.ldi + at);
    }
    const float* z = a.in32 + (size_t)(r.row0 + min(t0 + (lane & (BR - 1)), r.n - 1)) * a.ldi32 + h;
    zi = z[a.oi];
    zf = z[a.of];
  };
  load(0);
  for (int t0 = 0; t0 < r.n; t0 += BR) {
    const int nb = min(BR, r.n - t0);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u, c = e % Q * 4;
      if (e >= BR * Q) continue;
      f32x4_t y = c < DK ? x[u] * a.q_scale : x[u];
      if (e / Q >= nb) y = f32x4_t{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4_t*>(&s_in[0][0] + 4 * e) = y;
    }
    // a lane's gates, the running maximum of its row, and from these what its step keeps and adds
    const float i = ml_in(a, zi), f = ml_forget(a, zf);
    float fm = 0.f, mx = 0.f;
    for (int t = 0; t < nb; ++t) {
      const float y = lane_at(f, t) + m;
      m = fmaxf(y, lane_at(i, t));
      if ((lane & (BR - 1)) == t) fm = y, mx = m;
    }
    const float keep = expf(fm - mx), add = (lane & (BR - 1)) < nb ? expf(i - mx) : 0.f;  // rows past the batch change nothing
    __syncthreads();
    if (tid < BR) s_m[tid] = mx;
    if (t0 + BR < r.n) load(t0 + BR);
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where they are first used
    typedef float kvec __attribute__((ext_vector_type(KPL)));
    struct Row {
      kvec q, k;
      f32x4_t v;
    };
    auto fetch = [&](int t, Row& y) {
      y.q = *reinterpret_cast<const kvec*>(&s_in[t][kg * KPL]);
      y.k = *reinterpret_cast<const kvec*>(&s_in[t][DK + kg * KPL]);
      y.v = *reinterpret_cast<const f32x4_t*>(&s_in[t][2 * DK + v]);
    };
    auto step = [&](int t, const Row& y) {
      const float kp = lane_at(keep, t), ad = lane_at(add, t);
      const f32x4_t u = y.v * ad;
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
      float nq = 0.f;
#pragma unroll
      for (int j = 0; j < KPL; ++j) {
        const float q = y.q[j], k = y.k[j];
        S[j] = S[j] * kp + u * k;
        o += S[j] * q;
        n[j] = n[j] * kp + ad * k;
        nq += n[j] * q;
      }
      float z = quarters(halves(o[0], o[1]), halves(o[2], o[3]));
      z += dpp_mov<0x4E>(z);
      z += dpp_mov<0x124>(z);
      z += dpp_mov<0x128>(z);
      nq += dpp_mov<0x4E>(nq);
      nq += dpp_mov<0x124>(nq);
      nq += dpp_mov<0x128>(nq);
      nq += lane_xor<16>(nq);
      nq += lane_xor<32>(nq);
      so[t][v + (lane >> 3 & 2) + (lane >> 5)] = z;  // lanes with the same sum store it all: no branch
      s_nq[t] = nq;
    };
    Row y[2][2];  // two rows in one block of code: the sums of one are made beside the products of the other
    fetch(0, y[0][0]);
    fetch(1, y[0][1]);
    for (int t = 0; t < nb; t += 4) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int u = t + 2 * p;
        fetch((u + 2) % BR, y[1 - p][0]);
        fetch((u + 3) % BR, y[1 - p][1]);
        step(u, y[p][0]);
        step(u + 1, y[p][1]);
      }
    }
    __syncthreads();
    const int rt = tid / 16, c = tid % 16 * 2;
    if (rt >= nb) continue;  // s_in and so are written again behind this barrier and the next
    const float den = ml_denominator(s_nq[rt], s_m[rt]);
    *reinterpret_cast<float2*>((float*)a.out + (size_t)(r.row0 + t0 + rt) * a.ldo + h * DV + v0 + c) =
        make_float2(so[rt][c] / den, so[rt][c + 1] / den);
  }
#pragma unroll
  for (int j = 0; j < KPL; ++j) *reinterpret_cast<f32x4_t*>(st + (size_t)(kg * KPL + j) * DV) = S[j];
  if (blockIdx.z) return;
  float* to = nm + ((size_t)blockIdx.x * a.heads + h) * (DK + 1);
  if (w == 0 && (lane & 1) == 0) {
#pragma unroll
    for (int j = 0; j < KPL; ++j) to[kg * KPL + j] = n[j];
  }
  if (tid == 0) to[DK] = m;
}

// What ml_split_kernel left: rows of a run by blockIdx.y, dv / 4 lanes per head, in place; n and m into all their copies.
__global__ __launch_bounds__(256) void ml_finish_kernel(MlArgs a, const float* __restrict__ nm) {
  const MlRun r = ml_run(a, blockIdx.x);
  const int g4 = a.dv / 4, n = a.heads * g4;
  for (int t = blockIdx.y; t < r.n; t += gridDim.y) {
    const size_t row = r.row0 + t;
    for (int c = threadIdx.x; c < n; c += 256) {  // whole heads leave together
      float* const o = (float*)a.out + row * a.ldo + 4 * c;
      const f32x4_t y = *reinterpret_cast<const f32x4_t*>(o), nw = *reinterpret_cast<const f32x4_t*>(a.norm + 4 * c);
      const f32x4_t g = *reinterpret_cast<const f32x4_t*>((const float*)a.in + row * a.ldi + a.og + 4 * c);
      float ss = y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3];
      for (int s = g4 / 2; s > 0; s >>= 1) ss += __shfl_xor(ss, s, 64);
      const float rs = 1.f / sqrtf(ss / (float)a.vdim + a.eps);
      f32x4_t z;
#pragma unroll
      for (int j = 0; j < 4; ++j) z[j] = y[j] * rs * nw[j] * sigmoid(g[j]);
      *reinterpret_cast<f32x4_t*>(o) = z;
    }
  }
  if (blockIdx.y || !r.n) return;
  for (int e = threadIdx.x; e < a.heads * (a.dk + 1); e += 256) {
    const int h = e / (a.dk + 1), d = e % (a.dk + 1);
    const size_t head = (size_t)r.slot * a.heads + h;
    const float x = nm[((size_t)blockIdx.x * a.heads + h) * (a.dk + 1) + d];
    for (int c = 0; c < a.copies; ++c) {
      if (d < a.dk) a.n[(head * a.copies + c) * a.dk + d] = x;
      else a.m[head * a.copies + c] = x;
    }
  }
}

// any size (one copy): the state stays in memory; thread <-> value channels, and key channels of n
template <typename T>
__global__ __launch_bounds__(256) void ml_plain_kernel(MlArgs a) {
  extern __shared__ float smem[];
  const int DK = a.dk, DV = a.dv, tid = threadIdx.x, h = blockIdx.y;
  float *sq = smem, *sk = sq + DK, *sv = sk + DK, *so = sv + DV;
  __shared__ float s_ss[4], s_n[4];
  const MlRun r = ml_run(a, blockIdx.x);
  if (ml_idle<T>(a, r, h)) return;
  const size_t head = (size_t)r.slot * a.heads + h;
  float *st = a.S + head * DK * DV, *sn = a.n + head * DK;
  float m = r.pos0 == 0 ? 0.f : a.m[head];
  for (int t = 0; t < r.n; ++t) {
    const bool fresh = t == 0 && r.pos0 == 0;
    const int row = r.row0 + t;
    __syncthreads();
    ml_row<T>(a, row, h, DK, DV, sq, sk, sv);
    const float i = ml_input_gate(a, row, h), fm = ml_forget_gate(a, row, h) + m;
    m = fmaxf(fm, i);
    const float keep = expf(fm - m), add = expf(i - m);
    __syncthreads();
    float nq = 0.f;
    for (int d = tid; d < DK; d += 256) {
      const float z = (fresh ? 0.f : sn[d] * keep) + add * sk[d];
      sn[d] = z;
      nq = fmaf(z, sq[d], nq);
    }
    nq = wave_sum(nq);
    if ((tid & 63) == 0) s_n[tid >> 6] = nq;
    __syncthreads();
    const float den = ml_denominator(s_n[0] + s_n[1] + s_n[2] + s_n[3], m);
    float ss = 0.f;
    for (int v = tid; v < DV; v += 256) {
      float o = 0.f;
      const float u = sv[v] * add;
      for (int d = 0; d < DK; ++d) {
        const float x = fmaf(sk[d], u, fresh ? 0.f : st[(size_t)d * DV + v] * keep);
        st[(size_t)d * DV + v] = x;
        o = fmaf(x, sq[d], o);
      }
      o /= den;
      so[v] = o;
      ss = fmaf(o, o, ss);
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_ss[tid >> 6] = ss;
    __syncthreads();
    const float rs = 1.f / sqrtf((s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)a.vdim + a.eps);
    for (int d = tid; d < DV; d += 256) ml_store<T>(a, row, h, d, so[d], rs, ml_out_gate<T>(a, row, h, d));
  }
  if (tid == 0) a.m[head] = m;  // read before the first barrier
}

// Up to how many rows of the longest run go row by row. A batch costs its filling however few rows it has, and of many
// workgroups one's rows fill another's waits. us row by row and in batches: 16 heads, 4 runs: 128 x 128, 2 rows 7.7 and 8.1, 3
// 9.7 and 8.9; 128 x 64 (twice the operands a thread), 3 rows 7.9 and 8, 4 9.6 and 8.5; 128 x 32 (three times), 4 rows 9.4 and
// 11.2, 6 13 and 12.2. 128 x 128, 32 runs of 8 rows 29.6 and 28.9 (fp32), 27.4 and 30.5 (bf16), of 12 39.5 and 36.3, 38.1 and
// 38.9; 64 of 12 68.9 and 68.2 (fp32), of 24 118 and 128 (bf16); 128 of 24 204 and 214 (fp32), of 32 287 and 269, 253 and 305.
// Fewer keys: 8 heads of 64 x 64, 64 runs of 2 rows 7 and 7.8, 3 8.7 and 8.2, 128 of 4 14.2 and 14.2, 6 19.1 and 16.5; 4 heads of
// 32 x 128, 128 runs of 3 rows 9.1 and 9.9, 4 11 and 10.7.
int few_rows(int f32, const MlArgs& a, int n) {
  const int wg = n * a.heads, fill = 4 * (2 * a.dk + a.dv) / a.dv;  // operands a thread stages for a batch
  if (wg < 512) return fill >= 36 ? 4 : fill >= 20 ? 3 : 2;
  if (a.dk < 128) return wg >= 1024 ? 4 : a.dv > a.dk ? 3 : 2;
  if (f32) return wg < 2048 ? 8 : 24;
  return wg < 1024 ? 12 : wg < 2048 ? 24 : 32;
}

// Runs for the split form: its second launch takes 6 us, and a CU that two of its workgroups share gains nothing. us in batches
// and split, 16 heads of 128 x 128: 4 runs of 12 rows 17 and 15.5, of 8 13.9 and 14.5, of 60 59 and 33; 8 runs of 12 rows 17.6 and
// 17.1, of 300 268 and 160; 16 of 60 63 and 67, of 300 270 and 270; 64 of 60 227 and 208. 8 heads of 64 x 64, 4 of 100 57 and 33.
bool split_form(const MlArgs& a, int n, int longest) { return longest >= 12 && (long long)n * a.heads * (a.dv / 32) <= 512; }

}  // namespace

// n runs (a->runs), or n single rows (a->slot / a->pos); longest: none has more rows (0: not known); nm: scratch, nm_floats
// n heads (dk + 1) or no form that needs it
extern "C" int lsa_ml_steps(int f32, const MlArgs* a, int n, int longest, float* nm, long long nm_floats, hipStream_t s) {
  if (bad_ml(a) || n < 1 || longest < 0 || (!nm && nm_floats)) return LSA_BAD_SHAPE;
  const dim3 grid(n, a->heads);
  const bool few = longest > 0 && longest <= few_rows(f32, *a, n);
  const bool split = f32 && a->runs && !few && split_form(*a, n, longest) &&
                     nm_floats >= (long long)n * a->heads * (a->dk + 1) && !((a->ldi | a->ldo | a->oq | a->ok | a->ov | a->og) % 4) &&
                     !(((uintptr_t)a->in | (uintptr_t)a->out | (uintptr_t)a->norm | (uintptr_t)a->S) % 16);
#define LSA_D(K, V)                                                                      \
  if (a->dk == K && a->dv == V) {                                                        \
    if (!a->runs && f32) ml_rows_kernel<float, K, V, true><<<grid, 256, 0, s>>>(*a);     \
    else if (!a->runs) ml_rows_kernel<bf16_raw, K, V, true><<<grid, 256, 0, s>>>(*a);    \
    else if (few && f32) ml_rows_kernel<float, K, V, false><<<grid, 256, 0, s>>>(*a);    \
    else if (few) ml_rows_kernel<bf16_raw, K, V, false><<<grid, 256, 0, s>>>(*a);        \
    else if (split) {                                                                    \
      ml_split_kernel<K, V><<<dim3(n, a->heads, V / 32), 256, 0, s>>>(*a, nm);           \
      ml_finish_kernel<<<dim3(n, longest < 512 ? longest : 512), 256, 0, s>>>(*a, nm);   \
    } else if (f32) ml_steps_kernel<float, K, V><<<grid, V * 4, 0, s>>>(*a);               \
    else ml_steps_kernel<bf16_raw, K, V><<<grid, V * 4, 0, s>>>(*a);                     \
    LSA_CHECK_LAUNCH();                                                                  \
    return LSA_OK;                                                                       \
  }
  LSA_D(32, 32) LSA_D(32, 64) LSA_D(32, 128) LSA_D(64, 32) LSA_D(64, 64) LSA_D(64, 128) LSA_D(128, 32) LSA_D(128, 64)
  LSA_D(128, 128)
#undef LSA_D
  if (a->copies != 1) return LSA_BAD_SHAPE;
  const size_t lds = (size_t)(2 * a->dk + 2 * a->dv) * 4;
  if (lds > 60000) return LSA_UNSUPPORTED;
  if (f32) ml_plain_kernel<float><<<grid, 256, lds, s>>>(*a);
  else ml_plain_kernel<bf16_raw><<<grid, 256, lds, s>>>(*a);
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}
