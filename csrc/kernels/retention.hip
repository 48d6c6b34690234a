// Retention step by step (retention.h): one workgroup per (run, head) keeps the head's state in registers and
// walks the run's rows; everything between the projections and the output projection in one launch. Decoded
// tokens are runs of one row; the fp32 engine runs whole portions this way.
#include "retention.h"

namespace {

template <typename T>
LSA_DEVICE void ret_row(const RetArgs& a, const RetRun& r, int t, int h, int DK, int DV, float* sq, float* sk, float* sv) {
  const T* in = (const T*)a.in + (size_t)(r.row0 + t) * a.ldi;
  const int p = r.pos0 + t;
  for (int c = threadIdx.x; c < 2 * DK + DV; c += 256) {
    if (c < 2 * DK) {
      const bool q = c < DK;
      const int d = q ? c : c - DK;
      const float x = ret_turn(a, in + (q ? a.oq : a.ok) + h * DK, d, p);
      (q ? sq : sk)[d] = q ? x : x * a.k_scale;
    } else {
      const int d = c - 2 * DK;
      sv[d] = ld1(in + a.ov + h * DV + d);
    }
  }
}

template <typename T>
LSA_DEVICE float ret_gate(const RetArgs& a, int row, int h, int d) {
  return ld1((const T*)a.in + (size_t)row * a.ldi + a.og + h * a.dv + d);
}
template <typename T>
LSA_DEVICE void ret_store(const RetArgs& a, int row, int h, int d, float o, float rs, float g) {
  st1((T*)a.out + (size_t)row * a.ldo + h * a.dv + d, o * rs * (g / (1.f + expf(-g))) * a.oscale);
}

template <typename T>
LSA_DEVICE bool ret_idle(const RetArgs& a, const RetRun& r, int h) {
  if (r.n) return false;
  if (!a.runs)
    for (int d = threadIdx.x; d < a.dv; d += 256) st1((T*)a.out + (size_t)r.row0 * a.ldo + h * a.dv + d, 0.f);
  return true;
}

// What one row brings, requested a row ahead: a step is a chain of three barriers, and waiting in it for its own operands
// and its output gate took half of its time. Portions of 200 rows, fp32: 1.8 us a row before, now 1.1.
template <typename T, int DK, int DV>
struct RetNext {
  static constexpr int NX = (2 * DK + DV + 255) / 256;
  float x[NX], y[NX], c[NX], s[NX], g;  // a value, the other of its pair, and its angle's cosine and sine
  LSA_DEVICE void load(const RetArgs& a, int row, int p, int h) {
    const T* in = (const T*)a.in + (size_t)row * a.ldi;
    const int half = a.rot_dims / 2;
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = threadIdx.x + 256 * u, d = e < DK ? e : e - DK;
      const T* head = in + (e < 2 * DK ? (e < DK ? a.oq : a.ok) + h * DK : a.ov + h * DV);
      x[u] = ld1(head + (e < 2 * DK ? d : min(e - 2 * DK, DV - 1)));
      y[u] = c[u] = s[u] = 0.f;
      if (e < 2 * DK && a.cos && d < a.rot_dims) {
        const int f = d < half ? d : d - half;
        y[u] = ld1(head + (d < half ? d + half : f));
        c[u] = a.cos[(size_t)p * half + f];
        s[u] = a.sin[(size_t)p * half + f];
      }
    }
    g = ret_gate<T>(a, row, h, min((int)threadIdx.x, DV - 1));
  }
  LSA_DEVICE void store(const RetArgs& a, float* sq, float* sk, float* sv) const {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = threadIdx.x + 256 * u, d = e < DK ? e : e - DK;
      if (e < 2 * DK) {
        float t = x[u];
        if (a.cos && d < a.rot_dims) t = d < a.rot_dims / 2 ? x[u] * c[u] - y[u] * s[u] : x[u] * c[u] + y[u] * s[u];
        if (e < DK) sq[d] = t;
        else sk[d] = t * a.k_scale;
      } else if (e < 2 * DK + DV) {
        sv[e - 2 * DK] = x[u];
      }
    }
  }
};

template <typename T, int DK, int DV>
__global__ __launch_bounds__(256) void ret_steps_kernel(RetArgs a) {
  // a thread holds RPT rows x 4 value channels of the state
  constexpr int NG = 1024 / DV, RPT = DK / NG;
  static_assert(RPT >= 1 && NG * RPT == DK, "geometry");
  __shared__ __attribute__((aligned(16))) float sq[DK], sk[DK], sv[DV], s_b[NG][DV];
  __shared__ float s_ss[4];
  const RetRun r = ret_run(a, blockIdx.x);
  const int h = blockIdx.y, tid = threadIdx.x, v = (tid % (DV / 4)) * 4, grp = tid / (DV / 4), d0 = grp * RPT;
  if (ret_idle<T>(a, r, h)) return;
  float* st = a.state + ((size_t)r.slot * a.heads + h) * DK * DV + (size_t)d0 * DV + v;
  f32x4_t S[RPT];
#pragma unroll
  for (int j = 0; j < RPT; ++j) S[j] = *reinterpret_cast<const f32x4_t*>(st + (size_t)j * DV);
  if (r.pos0 == 0) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) S[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  const float decay = a.decay[h];
  RetNext<T, DK, DV> x1;
  x1.load(a, r.row0, r.pos0, h);
  for (int t = 0; t < r.n; ++t) {
    x1.store(a, sq, sk, sv);
    const float gate = x1.g;
    __syncthreads();
    if (t + 1 < r.n) x1.load(a, r.row0 + t + 1, r.pos0 + t + 1, h);
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where it is first used
    const f32x4_t u = *reinterpret_cast<const f32x4_t*>(&sv[v]);
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      S[j] = S[j] * decay + u * sk[d0 + j];
      o += S[j] * sq[d0 + j];
    }
    *reinterpret_cast<f32x4_t*>(&s_b[grp][v]) = o;
    __syncthreads();
    float x = 0.f;
    if (tid < DV) {
#pragma unroll
      for (int g = 0; g < NG; ++g) x += s_b[g][tid];
    }
    const float ss = wave_sum(x * x);
    if ((tid & 63) == 0) s_ss[tid >> 6] = ss;
    __syncthreads();
    if (tid < DV)
      ret_store<T>(a, r.row0 + t, h, tid, x, 1.f / sqrtf((s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)a.vdim + a.eps), gate);
  }
#pragma unroll
  for (int j = 0; j < RPT; ++j) *reinterpret_cast<f32x4_t*>(st + (size_t)j * DV) = S[j];
}

// fp32 portions that leave CUs idle: 32 value channels a workgroup, a wave 8 of them, so that a head has DV / 32 workgroups, and rows
// in batches of 16 whose operands come together, turned on their way to LDS: no step waits for another wave. A lane has DK / 32 key
// channels by 4 value channels of the state; the four sums over 32 lanes are halved with their lanes. Read-outs go out as they are,
// ret_finish_kernel norms them. Reductions and LDS
// latency, no longer three barriers a row: 8 heads of 128 x 128, one run of 200 rows 260 -> 49 us, 16 of them 262 -> 77.
template <int DK, int DV>
__global__ __launch_bounds__(256) void ret_split_kernel(RetArgs a) {
  constexpr int BR = 16, V = 32, W = 2 * DK + V, Q = W / 4, NX = (BR * Q + 255) / 256, KPL = DK / 32;
  __shared__ __attribute__((aligned(16))) float s_in[BR][W], so[BR][V];  // q, k, v
  const RetRun r = ret_run(a, blockIdx.x);
  const int h = blockIdx.y, v0 = blockIdx.z * V, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 1;
  if (!r.n) return;
  const int v = w * 8 + (lane & 1) * 4, half = a.rot_dims / 2;
  float* const st = a.state + ((size_t)r.slot * a.heads + h) * DK * DV + v0 + v;
  f32x4_t S[KPL];
#pragma unroll
  for (int j = 0; j < KPL; ++j)
    S[j] = r.pos0 == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4_t*>(st + (size_t)(kg * KPL + j) * DV);
  const float* const in = (const float*)a.in + (size_t)r.row0 * a.ldi;
  f32x4_t x[NX], y[NX], co[NX], si[NX];  // values, the others of their pairs, and the angles' cosines and sines
  const auto turns = [&](int c) { return a.cos && c < 2 * DK && c % DK < a.rot_dims; };
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u, t = min(t0 + e / Q, r.n - 1), c = e % Q * 4, d = c % DK;
      const float* row = in + (size_t)t * a.ldi;
      const float* head = row + (c < DK ? a.oq + h * DK : c < 2 * DK ? a.ok + h * DK : a.ov + h * DV + v0);
      x[u] = *reinterpret_cast<const f32x4_t*>(head + (c < 2 * DK ? d : c - 2 * DK));
      if (!turns(c)) continue;
      const int f = d < half ? d : d - half;
      const size_t at = (size_t)(r.pos0 + t) * half + f;
      y[u] = *reinterpret_cast<const f32x4_t*>(head + (d < half ? d + half : f));
      co[u] = *reinterpret_cast<const f32x4_t*>(a.cos + at);
      si[u] = *reinterpret_cast<const f32x4_t*>(a.sin + at);
    }
  };
  const float decay = a.decay[h];
  load(0);
  for (int t0 = 0; t0 < r.n; t0 += BR) {
    const int nb = min(BR, r.n - t0);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u, c = e % Q * 4, d = c % DK;
      if (e >= BR * Q) continue;
      f32x4_t z = x[u];
      if (turns(c)) {
        const f32x4_t w = y[u] * si[u];
        z = __builtin_elementwise_fma(x[u], co[u], d < half ? -w : w);
      }
      if (c >= DK && c < 2 * DK) z *= a.k_scale;
      if (e / Q >= nb) z = f32x4_t{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4_t*>(&s_in[0][0] + 4 * e) = z;
    }
    __syncthreads();
    if (t0 + BR < r.n) load(t0 + BR);
    __builtin_amdgcn_sched_barrier(0);  // requested here, not where they are first used
    typedef float kvec __attribute__((ext_vector_type(KPL)));
    struct Row {
      kvec q, k;
      f32x4_t v;
    };
    auto fetch = [&](int t, Row& z) {
      z.q = *reinterpret_cast<const kvec*>(&s_in[t][kg * KPL]);
      z.k = *reinterpret_cast<const kvec*>(&s_in[t][DK + kg * KPL]);
      z.v = *reinterpret_cast<const f32x4_t*>(&s_in[t][2 * DK + v]);
    };
    auto step = [&](int t, const Row& z) {
      const float keep = t < nb ? decay : 1.f;  // rows past the batch change nothing
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KPL; ++j) {
        // Written out: of two products and their sum the compiler rounded the state's here, the far larger one, and its errors
        // grew by a third (four heads of 128 x 128, 190 rows: 3.0e-7 of its norm, now 2.3e-7 as in ret_steps_kernel).
        S[j] = __builtin_elementwise_fma(S[j], f32x4_t{keep, keep, keep, keep}, z.v * z.k[j]);
        o += S[j] * z.q[j];
      }
      float s = quarters(halves(o[0], o[1]), halves(o[2], o[3]));
      s += dpp_mov<0x4E>(s);
      s += dpp_mov<0x124>(s);
      s += dpp_mov<0x128>(s);
      so[t][v + (lane >> 3 & 2) + (lane >> 5)] = s;  // lanes with the same sum store it all: no branch
    };
    Row z[2][2];  // two rows in one block of code: the sums of one are made beside the products of the other
    fetch(0, z[0][0]);
    fetch(1, z[0][1]);
    for (int t = 0; t < nb; t += 4) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int u = t + 2 * p;
        fetch((u + 2) % BR, z[1 - p][0]);
        fetch((u + 3) % BR, z[1 - p][1]);
        step(u, z[p][0]);
        step(u + 1, z[p][1]);
      }
    }
    __syncthreads();
    const int rt = tid / 16, c = tid % 16 * 2;
    if (rt >= nb) continue;  // s_in and so are written again behind this barrier and the next
    *reinterpret_cast<float2*>((float*)a.out + (size_t)(r.row0 + t0 + rt) * a.ldo + h * DV + v0 + c) =
        make_float2(so[rt][c], so[rt][c + 1]);
  }
#pragma unroll
  for (int j = 0; j < KPL; ++j) *reinterpret_cast<f32x4_t*>(st + (size_t)(kg * KPL + j) * DV) = S[j];
}

// What ret_split_kernel left, in place: rows of a run by blockIdx.y, dv / 4 lanes per head.
__global__ __launch_bounds__(256) void ret_finish_kernel(RetArgs a) {
  const RetRun r = ret_run(a, blockIdx.x);
  const int g4 = a.dv / 4, n = a.heads * g4;
  for (int t = blockIdx.y; t < r.n; t += gridDim.y) {
    const size_t row = r.row0 + t;
    for (int c = threadIdx.x; c < n; c += 256) {  // whole heads leave together
      float* const o = (float*)a.out + row * a.ldo + 4 * c;
      const f32x4_t y = *reinterpret_cast<const f32x4_t*>(o);
      const f32x4_t g = *reinterpret_cast<const f32x4_t*>((const float*)a.in + row * a.ldi + a.og + 4 * c);
      float ss = y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3];
      for (int s = g4 / 2; s > 0; s >>= 1) ss += __shfl_xor(ss, s, 64);
      const float rs = 1.f / sqrtf(ss / (float)a.vdim + a.eps);
      f32x4_t z;
#pragma unroll
      for (int j = 0; j < 4; ++j) z[j] = y[j] * rs * (g[j] / (1.f + expf(-g[j]))) * a.oscale;
      *reinterpret_cast<f32x4_t*>(o) = z;
    }
  }
}

// Runs for the split form, whose second launch takes 6 us. With up to 1024 workgroups it is faster from 12 rows on (heads of 128 x 128,
// 32 runs x 8 heads x 4: 12 rows 22 -> 18 us, 200 rows 264 -> 139; one run of 12 rows 19 -> 10); with 2048 short runs lose (12 rows
// 29 -> 31 us, 17 rows 37 -> 41) and long ones gain little (200 rows 299 -> 256).
bool split_form(const RetArgs& a, int n, int longest) {
  return a.runs && longest >= 12 && (long long)n * a.heads * (a.dv / 32) <= 1024 && a.rot_dims % 8 == 0 &&
         !((a.ldi | a.ldo | a.oq | a.ok | a.ov | a.og) % 4) &&
         !(((uintptr_t)a.in | (uintptr_t)a.out | (uintptr_t)a.state | (uintptr_t)a.cos | (uintptr_t)a.sin) % 16);
}

// any size: the state stays in memory; thread <-> value channels
template <typename T>
__global__ __launch_bounds__(256) void ret_plain_kernel(RetArgs a) {
  extern __shared__ float smem[];
  const int DK = a.dk, DV = a.dv, tid = threadIdx.x, h = blockIdx.y;
  float *sq = smem, *sk = sq + DK, *sv = sk + DK, *so = sv + DV;
  __shared__ float s_ss[4];
  const RetRun r = ret_run(a, blockIdx.x);
  if (ret_idle<T>(a, r, h)) return;
  float* st = a.state + ((size_t)r.slot * a.heads + h) * DK * DV;
  const float decay = a.decay[h];
  for (int t = 0; t < r.n; ++t) {
    const bool fresh = t == 0 && r.pos0 == 0;
    __syncthreads();
    ret_row<T>(a, r, t, h, DK, DV, sq, sk, sv);
    __syncthreads();
    float ss = 0.f;
    for (int v = tid; v < DV; v += 256) {
      float o = 0.f;
      for (int d = 0; d < DK; ++d) {
        const float x = fmaf(sk[d], sv[v], fresh ? 0.f : st[(size_t)d * DV + v] * decay);
        st[(size_t)d * DV + v] = x;
        o = fmaf(x, sq[d], o);
      }
      so[v] = o;
      ss = fmaf(o, o, ss);
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_ss[tid >> 6] = ss;
    __syncthreads();
    const float rs = 1.f / sqrtf((s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)a.vdim + a.eps);
    for (int d = tid; d < DV; d += 256) ret_store<T>(a, r.row0 + t, h, d, so[d], rs, ret_gate<T>(a, r.row0 + t, h, d));
  }
}

}  // namespace

// n runs (a->runs), or n single rows (a->slot / a->pos); longest: none has more rows (0: not known)
extern "C" int lsa_ret_steps(int f32, const RetArgs* a, int n, int longest, hipStream_t s) {
  if (bad_ret(a) || n < 1 || longest < 0) return LSA_BAD_SHAPE;
  const dim3 grid(n, a->heads);
  const bool split = f32 && split_form(*a, n, longest);
#define LSA_D(K, V)                                                                    \
  if (a->dk == K && a->dv == V) {                                                      \
    if (split) {                                                                       \
      ret_split_kernel<K, V><<<dim3(n, a->heads, V / 32), 256, 0, s>>>(*a);            \
      ret_finish_kernel<<<dim3(n, longest < 512 ? longest : 512), 256, 0, s>>>(*a);    \
    } else if (f32) ret_steps_kernel<float, K, V><<<grid, 256, 0, s>>>(*a);            \
    else ret_steps_kernel<bf16_raw, K, V><<<grid, 256, 0, s>>>(*a);                    \
    LSA_CHECK_LAUNCH();                                                                \
    return LSA_OK;                                                                     \
  }
  LSA_D(32, 32) LSA_D(32, 64) LSA_D(32, 128) LSA_D(64, 32) LSA_D(64, 64) LSA_D(64, 128) LSA_D(128, 32) LSA_D(128, 64)
  LSA_D(128, 128)
#undef LSA_D
  const size_t lds = (size_t)(2 * a->dk + 2 * a->dv) * 4;
  if (lds > 60000) return LSA_UNSUPPORTED;
  if (f32) ret_plain_kernel<float><<<grid, 256, lds, s>>>(*a);
  else ret_plain_kernel<bf16_raw><<<grid, 256, lds, s>>>(*a);
  LSA_CHECK_LAUNCH();
  return LSA_OK;
}
