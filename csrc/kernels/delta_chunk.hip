// The gated delta rule over prompt portions in chunks of 32 rows (delta.h), bf16 engine.
//
// With G_i the sum of the log decays of rows 0..i of a chunk (per key channel) and S the state before it,
//
//   u = U - W S             U = T (beta v), W = T (beta k e^G), T = (1 + A)^-1
//   o = (q e^G) S + P u     A_ij = beta_i sum_d k_i k_j e^(G_i - G_j) (j < i),  P_ij the same of q_i, k_j (j <= i)
//   S <- e^G_31 S + (k e^(G_31 - G))^T u
//
// delta_chunk_kernel makes W, U, q e^G, k e^(G_31 - G), P and e^G_31 of every (chunk, head) at once;
// delta_scan_kernel then walks a run's chunks, one workgroup per (run, head). No exponent is ever
// positive: the 16 x 16 blocks on the diagonal of A and P take e^(G_i - G_j) pair by pair, the block
// below them splits it at row 15.
//
// Everything is fp32 or, where it is an operand of a matrix product, a pair of bf16 (the value's
// rounding and the rounding of what that leaves): each product is the sum of three, hi hi + hi lo + lo hi.
// The pairs lie in memory in operand order, the K index in the order in which the accumulators hold it,
// so the state never leaves the scan's registers.
#include "delta.h"

namespace {

constexpr int C = 32;

struct DeltaChunk {  // rows row0 .. row0 + n of one run at positions pos0 ..; before: rows of that run ahead of row0
  int row0, n, slot, pos0, before, pad0, pad1, pad2;
};
struct DeltaSpan {  // chunks [chunk0, chunk0 + chunks) of one run, its rows and first position
  int chunk0, chunks, slot, pos0, row0, n, pad0, pad1;
};

template <int DK>
struct Pieces {  // 1-KiB pieces of a (chunk, head) in the workspace; hi ones first
  static constexpr int KF = DK / 32, W = 0, Q = 4 * KF, K = 8 * KF, P = 12 * KF, E = P + 4, U = E + 1;
};

// 8 values -> operand pieces
LSA_DEVICE void put_pair(unsigned char* hi, unsigned char* lo, int at, const float* f) {
  const u32x4_t h = pack8(f);
  float b[8], r[8];
  unpack8(h, b);
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = f[j] - b[j];
  st16(hi + at * 16, h);
  st16(lo + at * 16, pack8(r));
}
LSA_DEVICE void split_pair(const float* f, u32x4_t& h, u32x4_t& l) {
  h = pack8(f);
  float b[8], r[8];
  unpack8(h, b);
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = f[j] - b[j];
  l = pack8(r);
}
LSA_DEVICE f32x4_t mfma_pair(u32x4_t ah, u32x4_t al, u32x4_t bh, u32x4_t bl, f32x4_t c) {
  return mfma16(al, bh, mfma16(ah, bl, mfma16(ah, bh, c)));
}

// log(1 + e^x) in fp32 on the hardware's exponential and logarithm
LSA_DEVICE float softplus_fast(float x) {
  const float e = __expf(-fabsf(x));
  return fmaxf(x, 0.f) + (e < 0x1p-9f ? e * (1.f - e * (0.5f - e * 0.33333333f)) : __logf(1.f + e));
}
LSA_DEVICE float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// Convolution and silu of one channel over the chunk's rows. load() requests its inputs (up to four taps), so
// that a thread can ask for everything it needs before it waits for any of it; run(f) calls f(row, value),
// zero past the last row.
struct ConvRows {
  bf16_raw raw[C];
  float x1, x2, x3;
  int ch, col;

  // the input j rows before row t
  LSA_DEVICE float past(const DeltaArgs& a, const DeltaChunk& ck, int channels, int t, int j) const {
    if (j - t <= ck.before) return bf2f(((const bf16_raw*)a.in)[(size_t)(ck.row0 + t - j) * a.ldi + col]);
    const int p = ck.pos0 + t - j;
    return p < 0 ? 0.f : a.ring[((size_t)ck.slot * a.taps + p % a.taps) * channels + ch];
  }
  LSA_DEVICE void load(const DeltaArgs& a, const DeltaChunk& ck, int channels, int ch_, int col_) {
    ch = ch_;
    col = col_;
    if (a.taps > 4) return;
    const bf16_raw* in = (const bf16_raw*)a.in + (size_t)ck.row0 * a.ldi + col;
#pragma unroll
    for (int t = 0; t < C; ++t) raw[t] = in[(size_t)min(t, ck.n - 1) * a.ldi];
    x1 = a.taps > 1 ? past(a, ck, channels, 0, 1) : 0.f;
    x2 = a.taps > 2 ? past(a, ck, channels, 0, 2) : 0.f;
    x3 = a.taps > 3 ? past(a, ck, channels, 0, 3) : 0.f;
  }
  template <typename F>
  LSA_DEVICE void run(const DeltaArgs& a, const DeltaChunk& ck, int channels, F f) {
    const float* w = a.conv + (size_t)ch * a.taps + a.taps - 1;
    if (a.taps <= 4) {
      const float w0 = w[0], w1 = a.taps > 1 ? w[-1] : 0.f, w2 = a.taps > 2 ? w[-2] : 0.f, w3 = a.taps > 3 ? w[-3] : 0.f;
#pragma unroll
      for (int t = 0; t < C; ++t) {
        const float x = bf2f(raw[t]);
        const float y = silu_fast(fmaf(x3, w3, fmaf(x2, w2, fmaf(x1, w1, x * w0))));
        f(t, t < ck.n ? y : 0.f);
        x3 = x2;
        x2 = x1;
        x1 = x;
      }
    } else {
#pragma unroll
      for (int t = 0; t < C; ++t) {
        float y = 0.f;
        if (t < ck.n) {
          for (int j = 0; j < a.taps; ++j) y = fmaf(past(a, ck, channels, t, j), w[-j], y);
          y = silu_fast(y);
        }
        f(t, y);
      }
    }
  }
};

// Bound by its vector and LDS instructions (a wave's 4100 and 620, three workgroups a CU). Rows scaled, summed and squared four channels
// at a time, and the second block's diagonal by all threads instead of one a row: 102 chunks, 16 heads of 128 x 128, 92 -> 80 us.
template <int DK, int DV>
__global__ __launch_bounds__(256) void delta_chunk_kernel(DeltaArgs a, const DeltaChunk* __restrict__ chunks,
                                                          unsigned char* __restrict__ ws) {
  using PC = Pieces<DK>;
  constexpr int KF = DK / 32;
  constexpr size_t STRIDE = (size_t)(PC::U + DV / 8) * 1024;
  // Rows without padding, their 16-byte pieces exchanged by the row (at); A below the diagonal of one square, P's columns as
  // its rows on and above it: 53632 bytes, so that three workgroups share a CU.
  __shared__ __attribute__((aligned(16))) float sq[C][DK], sk[C][DK], sg[C][DK], sAP[C][C];
  __shared__ float su[2 * C], sb[C];
  const auto at = [](int t, int d) { return d ^ ((t & (DK / 4 < 16 ? DK / 4 - 1 : 15)) << 2); };
  const auto four = [&](float (*x)[DK], int t, int d) { return *reinterpret_cast<const f32x4_t*>(&x[t][at(t, d)]); };
  const DeltaChunk ck = chunks[blockIdx.x];
  const int h = blockIdx.y, kb = h / (a.heads / a.kv_heads), kc = a.kv_heads * a.dim;
  const int channels = 2 * kc + a.heads * a.vdim;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* out = ws + ((size_t)blockIdx.x * a.heads + h) * STRIDE;

  static_assert(2 * DK <= 256 && DK + DV <= 256, "one channel per thread");
  const int cd = tid % DK, isk = tid / DK;  // thread < 2 DK: channel cd of q / k, and 16 rows of its decay
  ConvRows qk, vc;
  float zz[16];
  if (tid < 2 * DK) {
    const int d = min(cd, a.dim - 1);
    qk.load(a, ck, channels, isk * kc + kb * a.dim + d, (isk ? a.ok : a.oq) + kb * a.dim + d);
    const float* z = a.z + (size_t)ck.row0 * a.ldz + h * a.dim + d;
#pragma unroll
    for (int t = 0; t < 16; ++t) zz[t] = z[(size_t)min(isk * 16 + t, ck.n - 1) * a.ldz];
  }
  if (tid < DV) {
    const int d = min(tid, a.vdim - 1);
    vc.load(a, ck, channels, 2 * kc + h * a.vdim + d, a.ov + h * a.vdim + d);
  }
  if (tid < 2 * DK) {
    auto& dst = isk ? sk : sq;
    qk.run(a, ck, channels, [&](int t, float y) { dst[t][at(t, cd)] = cd < a.dim ? y : 0.f; });
    const float A = cd < a.dim ? -a.decay[h] * 1.4426950408889634f : 0.f, bias = cd < a.dim ? a.dt_bias[h * a.dim + cd] : 0.f;
    float g = 0.f;  // sums of log2 decays, 16 rows at a time
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      g = isk * 16 + t < ck.n ? fmaf(A, softplus_fast(zz[t] + bias), g) : g;
      sg[isk * 16 + t][at(t, cd)] = g;
    }
  }
  if (tid < C) sb[tid] = tid < ck.n ? 1.f / (1.f + __expf(-a.in32[(size_t)(ck.row0 + tid) * a.ld32 + a.ob + h])) : 0.f;
  __syncthreads();
  {  // unit vectors: four threads per vector
    const int v = tid >> 2, t = v & (C - 1);
    const float(*x)[DK] = v < C ? sq : sk;
    float ss = 0.f;
#pragma unroll
    for (int d0 = 0; d0 < DK; d0 += 16) {  // (whole rows: the order of their pieces does not matter, here and below)
      const f32x4_t y = *reinterpret_cast<const f32x4_t*>(&x[t][d0 + (tid & 3) * 4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = fmaf(y[e], y[e], ss);
    }
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    if ((tid & 3) == 0) su[v] = (v < C ? a.q_scale : 1.f) / sqrtf(ss + a.unit_eps);
  }
  for (int e = tid * 4; e < 16 * DK; e += 1024) {
    const int t = 16 + e / DK, d = e % DK;
    *reinterpret_cast<f32x4_t*>(&sg[t][at(t, d)]) = four(sg, t, d) + four(sg, 15, d);
  }
  __syncthreads();
  for (int e = tid * 4; e < C * DK; e += 1024) {
    const int t = e / DK, d = e % DK;
    *reinterpret_cast<f32x4_t*>(&sq[t][d]) *= su[t];
    *reinterpret_cast<f32x4_t*>(&sk[t][d]) *= su[C + t];
  }
  __syncthreads();

  {  // A and P: the two blocks on the diagonal, one pair of rows per thread
    const int r0 = tid >> 4, r1 = tid & 15;
    const int i = r0 >= r1 ? r0 : 16 + r1, j = r0 >= r1 ? r1 : 16 + r0;
    float x = 0.f, y = 0.f;
#pragma unroll 4
    for (int d = 0; d < DK; d += 4) {
      const f32x4_t gi = four(sg, i, d), gj = four(sg, j, d), ki = four(sk, i, d), kj = four(sk, j, d), qi = four(sq, i, d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = kj[e] * __builtin_amdgcn_exp2f(gi[e] - gj[e]);
        x = fmaf(ki[e], z, x);
        y = fmaf(qi[e], z, y);
      }
    }
    if (i != j) sAP[i][j] = sb[i] * x;
    sAP[j][i] = y;
    float p = 0.f;  // the second block's diagonal: 16 threads a row
#pragma unroll
    for (int d0 = 0; d0 < DK; d0 += 64) {
      const int d = d0 + r1 * 4;
      if (DK % 64 && d >= DK) break;
      const f32x4_t qd = *reinterpret_cast<const f32x4_t*>(&sq[16 + r0][d]), kd = *reinterpret_cast<const f32x4_t*>(&sk[16 + r0][d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) p = fmaf(qd[e], kd[e], p);
    }
    p = group_sum<16>(p);
    if (r1 == 0) sAP[16 + r0][16 + r0] = p;
  }
  if (w < 2) {  // the block below, through row 15: wave 0 A, wave 1 P
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    float(*sx)[DK] = w ? sq : sk;
#pragma unroll
    for (int kf = 0; kf < KF; ++kf) {
      float x[8], y[8];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int d = kf * 32 + q4 * 8 + 4 * p;
        const f32x4_t g = four(sg, 15, d), gi = four(sg, 16 + l16, d), gj = four(sg, l16, d), xi = four(sx, 16 + l16, d),
                      kj = four(sk, l16, d);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[4 * p + e] = xi[e] * __builtin_amdgcn_exp2f(gi[e] - g[e]);
          y[4 * p + e] = kj[e] * __builtin_amdgcn_exp2f(g[e] - gj[e]);
        }
      }
      u32x4_t xh, xl, yh, yl;
      split_pair(x, xh, xl);
      split_pair(y, yh, yl);
      acc = mfma_pair(xh, xl, yh, yl, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 + q4 * 4 + r;
      if (w) sAP[l16][i] = acc[r];
      else sAP[i][l16] = sb[i] * acc[r];
    }
  }
  // q e^G (rows x key channels) and k e^(G_31 - G) (key channels x rows)
  for (int e = tid; e < 2 * KF * 64; e += 256) {
    const int ln = e & 63, kf = (e >> 6) % KF, t = (e >> 6) / KF * 16 + (ln & 15), d0 = kf * 32 + (ln >> 4) * 4;
    float f[8];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const f32x4_t y = four(sq, t, d0 + 16 * p), g = four(sg, t, d0 + 16 * p);
#pragma unroll
      for (int j = 0; j < 4; ++j) f[4 * p + j] = y[j] * __builtin_amdgcn_exp2f(g[j]);
    }
    put_pair(out + PC::Q * 1024, out + (PC::Q + 2 * KF) * 1024, e, f);
  }
  for (int e = tid; e < 2 * KF * 64; e += 256) {
    const int ln = e & 63, d = (e >> 6) * 16 + (ln & 15), t0 = (ln >> 4) * 4;
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int t = t0 + (j & 4) * 4 + (j & 3);
      f[j] = sk[t][at(t, d)] * __builtin_amdgcn_exp2f(sg[C - 1][at(C - 1, d)] - sg[t][at(t, d)]);
    }
    put_pair(out + PC::K * 1024, out + (PC::K + 2 * KF) * 1024, e, f);
  }
  for (int d = tid; d < DK; d += 256) reinterpret_cast<float*>(out + PC::E * 1024)[d] = __builtin_amdgcn_exp2f(sg[C - 1][at(C - 1, d)]);
  __syncthreads();
  if (tid < 128) {  // P (rows x rows)
    const int t = (tid >> 6) * 16 + l16;
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = q4 * 4 + (j & 4) * 4 + (j & 3);
      f[j] = i <= t ? sAP[i][t] : 0.f;
    }
    put_pair(out + PC::P * 1024, out + (PC::P + 2) * 1024, tid, f);
  }
  // (1 + A) x = b, one column per thread: beta v -> U, beta k e^G -> W
  if (tid < DV + DK) {
    const int c = tid;
    float x[C];
    if (c < DV) {
      vc.run(a, ck, channels, [&](int t, float y) { x[t] = c < a.vdim ? y * sb[t] : 0.f; });
    } else {
#pragma unroll
      for (int t = 0; t < C; ++t) x[t] = sb[t] * sk[t][at(t, c - DV)] * __builtin_amdgcn_exp2f(sg[t][at(t, c - DV)]);
    }
#pragma unroll
    for (int i = 1; i < C; ++i) {
      float s = x[i];
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const f32x4_t r = *reinterpret_cast<const f32x4_t*>(&sAP[i][j]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j + e < i) s = fmaf(-r[e], x[j + e], s);
      }
      x[i] = s;
    }
    if (c < DV) {
      f32x4_t* u = reinterpret_cast<f32x4_t*>(out + (PC::U + (c / 16) * 2) * 1024);
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e * 16 + (c & 15)] = f32x4_t{x[4 * e], x[4 * e + 1], x[4 * e + 2], x[4 * e + 3]};
    } else {
#pragma unroll
      for (int t = 0; t < C; ++t) sq[t][at(t, c - DV)] = x[t];  // q is in memory already
    }
  }
  __syncthreads();
  for (int e = tid; e < 2 * KF * 64; e += 256) {
    const int ln = e & 63, kf = (e >> 6) % KF, t = (e >> 6) / KF * 16 + (ln & 15), d0 = kf * 32 + (ln >> 4) * 4;
    float f[8];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const f32x4_t y = four(sq, t, d0 + 16 * p);
#pragma unroll
      for (int j = 0; j < 4; ++j) f[4 * p + j] = y[j];
    }
    put_pair(out, out + 2 * KF * 1024, e, f);
  }
}

LSA_DEVICE __amdgpu_buffer_rsrc_t bytes_of(const void* p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, n, 0x00020000);
}
LSA_DEVICE void glds16(__amdgpu_buffer_rsrc_t src, int off, unsigned char* lds_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)lds_base, 16, off, 0, 0, 0);
}

// One workgroup per (run, head, NW 16 value channels): the state in registers (a wave has 16 channels of it), a
// chunk's operands by LDS-DMA two chunks ahead. Leaves the read-outs in fp32 for delta_norm_kernel.
//
// A chunk is one serial chain (operands from LDS, W S, u, the state's own products) on a CU that one workgroup fills.
// Where a head has 64 keys or more they are halved between two waves for each 16 channels, which exchange their W S
// and half of their read-outs through LDS; and the channels lie with as many workgroups as there are CUs (lsa_delta_chunked),
// so that a CU reads the operands out of LDS for fewer waves. Three runs of 34 chunks, 16 heads of 128 x 128: 93 us with
// all keys in a wave, 84 halved (96 workgroups), 65 with half of the channels each (192); 50 of them stay without the DMA.
template <int DK, int DV, int NW>
__global__ __launch_bounds__(NW * (DK > 32 ? 128 : 64)) void delta_scan_kernel(DeltaArgs a,
                                                                                const DeltaSpan* __restrict__ spans,
                                                                                const unsigned char* __restrict__ ws,
                                                                                float* __restrict__ o32) {
  using PC = Pieces<DK>;
  constexpr int KS = DK > 32 ? 2 : 1, NWV = NW * KS;  // key parts, waves
  constexpr int KF = DK / 32, MT = DK / 16, NP = PC::U;
  constexpr int KFW = KF / KS, MTW = MT / KS;  // of one wave
  constexpr int NDMA = (NP + NWV - 1) / NWV, NST = 8 / KS;  // DMA instructions and stores of a wave per chunk
  constexpr size_t STRIDE = (size_t)(PC::U + DV / 8) * 1024;
  // the exchange: 3 KiB a wave, in place of the chunk's W and q e^G (read by then) where LDS is full
  constexpr int EX = KS > 1 ? NWV * 3072 : 0;
  constexpr bool EX_OWN = 3 * NP * 1024 + EX <= 160 * 1024;
  static_assert(EX_OWN || EX <= PC::K * 1024, "room for the exchange");
  __shared__ __attribute__((aligned(16))) unsigned char smem[3 * NP * 1024 + (EX_OWN ? EX : 0)];
  const DeltaSpan sp = spans[blockIdx.x];
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), kh = w / NW;  // kh: this wave's keys
  const int vt = blockIdx.z * NW + w % NW;                              // its channels: 16 vt ..
  const unsigned char* src = ws + ((size_t)sp.chunk0 * a.heads + h) * STRIDE;
  const size_t step = (size_t)a.heads * STRIDE;

  f32x4_t S[MTW], U0[2], U1[2];
  float* st = a.state + (((size_t)sp.slot * a.heads + h) * DK + kh * (DK / KS)) * DV + vt * 16 + l16;
#pragma unroll
  for (int m = 0; m < MTW; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[m][r] = st[(size_t)(m * 16 + q4 * 4 + r) * DV];
  if (sp.pos0 == 0) {
#pragma unroll
    for (int m = 0; m < MTW; ++m) S[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // Chunk c, nothing where there is none: every wave has the same instructions in flight at the same place of each
  // chunk, so that waits can be counted (what is left over of the pieces is requested twice).
  int off[NDMA];
#pragma unroll
  for (int i = 0; i < NDMA; ++i) off[i] = min(i * NWV + w, NP - 1) * 1024 + lane * 16;
  auto stage = [&](int c, int buf, f32x4_t (&U)[2]) {
    const __amdgpu_buffer_rsrc_t r = bytes_of(src + c * step, c < sp.chunks ? (int)STRIDE : 0);
#pragma unroll
    for (int i = 0; i < NDMA; ++i)
      glds16(r, off[i], smem + (buf * NP + min(i * NWV + w, NP - 1)) * 1024);
#pragma unroll
    for (int m = 0; m < 2; ++m)
      U[m] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (PC::U + vt * 2 + m) * 1024 + lane * 16, 0, 0));
    asm volatile("" ::: "memory");
  };
  const int v = vt * 16 + l16, ldo = a.heads * a.vdim;
  const int row_at = v < a.vdim ? ((kh * 16 + q4 * 4) * ldo + v) * 4 : 0x40000000;
  // a chunk's read-outs: rows past the run's last and channels past the head's lie behind the descriptor's end
  auto put = [&](int c, const f32x4_t (&O)[2]) {
    const int left = min(C, sp.n - c * C);
    const __amdgpu_buffer_rsrc_t r =
        bytes_of(o32 + ((size_t)sp.row0 + c * C) * ldo + h * a.vdim, c >= 0 ? ((left - 1) * ldo + a.vdim) * 4 : 0);
#pragma unroll
    for (int m = 0; m < 2 / KS; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(O[m][e]), r, row_at + (m * 16 + e) * ldo * 4, 0, 0);
    asm volatile("" ::: "memory");
  };

  // Chunk c + 2 is requested while chunk c runs: operands into the buffer chunk c - 1 used, U into the registers
  // chunk c's has left. The counted wait leaves what came after chunk c's in flight: the stores of two chunks and the
  // requests for the next one.
  int buf = 0, buf2 = 2;
  auto chunk = [&](int c, f32x4_t (&U)[2]) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(NDMA + 2 + 2 * NST) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    unsigned char* const at = smem + buf * NP * 1024;
    const unsigned char* p = at + lane * 16;
    // operands are read a whole group ahead of their products; pin() is where the wait for a group goes
    auto fetch = [&](u32x4_t* r, int n, int first) {
#pragma unroll
      for (int i = 0; i < n; ++i) r[i] = *reinterpret_cast<const u32x4_t*>(p + (first + i) * 1024);
    };
    auto pin = [](auto& r) {
#pragma unroll
      for (int i = 0; i < (int)(sizeof(r) / sizeof(r[0])); ++i) asm volatile("" : "+v"(r[i]));
    };
    u32x4_t wf[4 * KFW], qf[4 * KFW], kf_[2 * MTW], pf[4];  // [rows or hi / lo][this wave's keys]
    f32x4_t ef[MTW];
#pragma unroll
    for (int m = 0; m < 4; ++m) fetch(wf + m * KFW, KFW, PC::W + m * KF + kh * KFW);
#pragma unroll
    for (int m = 0; m < 4; ++m) fetch(qf + m * KFW, KFW, PC::Q + m * KF + kh * KFW);
    float u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = U[j >> 2][j & 3];
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(u[j]));
    stage(c + 2, buf2, U);
    u32x4_t sh[KFW], sl[KFW];
#pragma unroll
    for (int kf = 0; kf < KFW; ++kf) {
      float f[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[j] = S[2 * kf][j];
        f[4 + j] = S[2 * kf + 1][j];
      }
      split_pair(f, sh[kf], sl[kf]);
    }
    f32x4_t V[2], O[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) V[m] = O[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    pin(wf);
#pragma unroll
    for (int kf = 0; kf < KFW; ++kf)
#pragma unroll
      for (int m = 0; m < 2; ++m) V[m] = mfma_pair(wf[m * KFW + kf], wf[(2 + m) * KFW + kf], sh[kf], sl[kf], V[m]);
#pragma unroll
    for (int m = 0; m < 2; ++m) fetch(kf_ + m * MTW, MTW, PC::K + m * MT + kh * MTW);
    if (KS == 1) {
      fetch(pf, 4, PC::P);
    } else {  // read-outs of rows 16 kh ..: one row tile of P
      fetch(pf, 1, PC::P + kh);
      fetch(pf + 2, 1, PC::P + 2 + kh);
    }
#pragma unroll
    for (int m = 0; m < MTW; ++m)
      ef[m] = *reinterpret_cast<const f32x4_t*>(at + PC::E * 1024 + ((kh * MTW + m) * 16 + q4 * 4) * 4);
    pin(qf);
    unsigned char* const ex = (EX_OWN ? smem + 3 * NP * 1024 : at) + lane * 16;
    if (KS > 1) {
      if (!EX_OWN) {  // every wave has its W and q e^G
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int m = 0; m < 2; ++m) *reinterpret_cast<f32x4_t*>(ex + (w * 3 + m) * 1024) = V[m];
    }
#pragma unroll
    for (int kf = 0; kf < KFW; ++kf)
#pragma unroll
      for (int m = 0; m < 2; ++m) O[m] = mfma_pair(qf[m * KFW + kf], qf[(2 + m) * KFW + kf], sh[kf], sl[kf], O[m]);
    if (KS > 1) {
      *reinterpret_cast<f32x4_t*>(ex + (w * 3 + 2) * 1024) = kh ? O[0] : O[1];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const unsigned char* other = ex + ((w + (kh ? -NW : NW)) * 3) * 1024;
#pragma unroll
      for (int m = 0; m < 2; ++m) V[m] += *reinterpret_cast<const f32x4_t*>(other + m * 1024);
      O[0] = (kh ? O[1] : O[0]) + *reinterpret_cast<const f32x4_t*>(other + 2048);
    }
    u32x4_t vh, vl;
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] -= V[j >> 2][j & 3];
    split_pair(u, vh, vl);
    pin(kf_);
    pin(ef);
#pragma unroll
    for (int m = 0; m < MTW; ++m) S[m] = mfma_pair(kf_[m], kf_[MTW + m], vh, vl, S[m] * ef[m]);
#pragma unroll
    for (int m = 0; m < 2 / KS; ++m) O[m] = mfma_pair(pf[m], pf[2 + m], vh, vl, O[m]);
    put(c, O);
    buf = buf == 2 ? 0 : buf + 1;
    buf2 = buf2 == 2 ? 0 : buf2 + 1;
  };
  // (what a chunk's products read and write has no fixed place in flight before the loop: stores of nothing stand in)
  const f32x4_t none[2] = {};
  stage(0, 0, U0);
  put(-1, none);
  stage(1, 1, U1);
  put(-1, none);
  int c = 0;
  for (; c + 1 < sp.chunks; c += 2) {
    chunk(c, U0);
    chunk(c + 1, U1);
  }
  if (c < sp.chunks) chunk(c, U0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int m = 0; m < MTW; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) st[(size_t)(m * 16 + q4 * 4 + r) * DV] = S[m][r];
}

// Read-outs -> RMS norm over the head's value channels, weight, output gate. One workgroup per (chunk, head), 16
// lanes per row.
__global__ __launch_bounds__(256) void delta_norm_kernel(DeltaArgs a, const DeltaChunk* __restrict__ chunks,
                                                         const float* __restrict__ o32) {
  const DeltaChunk ck = chunks[blockIdx.x];
  const int h = blockIdx.y, l16 = threadIdx.x & 15;
  for (int t = threadIdx.x >> 4; t < ck.n; t += 16) {
    const size_t row = ck.row0 + t;
    const float* o = o32 + (row * a.heads + h) * a.vdim;
    const bf16_raw* g = (const bf16_raw*)a.gate + row * a.ldg + h * a.vdim;
    bf16_raw* out = (bf16_raw*)a.out + row * a.ldo + h * a.vdim;
    float x[8], ss = 0.f;  // vdim <= 128
    if (a.vdim == 128 && !((a.ldg | a.ldo) & 7) && !(((uintptr_t)a.gate | (uintptr_t)a.out) & 15)) {
      *reinterpret_cast<f32x4_t*>(x) = *reinterpret_cast<const f32x4_t*>(o + l16 * 8);
      *reinterpret_cast<f32x4_t*>(x + 4) = *reinterpret_cast<const f32x4_t*>(o + l16 * 8 + 4);
      float z[8];
      unpack8(ld16(g + l16 * 8), z);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = fmaf(x[j], x[j], ss);
      const float rs = 1.f / sqrtf(group_sum<16>(ss) / 128.f + a.eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= rs * a.norm[l16 * 8 + j] * sigmoid(z[j]);
      st16(out + l16 * 8, pack8(x));
      continue;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = j * 16 + l16;
      x[j] = d < a.vdim ? o[d] : 0.f;
      ss = fmaf(x[j], x[j], ss);
    }
    const float rs = 1.f / sqrtf(group_sum<16>(ss) / (float)a.vdim + a.eps);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = j * 16 + l16;
      if (d < a.vdim) out[d] = f2bf(x[j] * rs * a.norm[d] * sigmoid(bf2f(g[d])));
    }
  }
}

}  // namespace

// bytes of one (chunk, head) in the workspace, 0: size not built
extern "C" int lsa_delta_chunk_bytes(int dk, int dv) {
  if ((dk != 32 && dk != 64 && dk != 128) || (dv != 32 && dv != 64 && dv != 128)) return 0;
  return (12 * (dk / 32) + 5 + dv / 8) * 1024;
}

// chunks: n_chunks DeltaChunk; spans: n_spans DeltaSpan over them; ws: n_chunks * heads * lsa_delta_chunk_bytes;
// o32: [rows][heads * vdim]. The scan's workgroups have 32 value channels where those are no more than the 256 CUs (one fits on each) and
// 64 otherwise: a second round of the narrow ones, 65 us each, costs more than one of the wide ones, 84.
extern "C" int lsa_delta_chunked(const DeltaArgs* a, const void* chunks, int n_chunks, const void* spans, int n_spans,
                                 void* ws, float* o32, hipStream_t s) {
  if (!a || bad_delta(a) || !a->gate || n_chunks < 1 || n_spans < 1 || !chunks || !spans || !ws || !o32 || (uintptr_t)ws % 16)
    return LSA_BAD_SHAPE;
#define LSA_S(K, V, NW)                                                                                                  \
  delta_scan_kernel<K, V, NW><<<dim3(n_spans, a->heads, V / (NW * 16)), NW * (K > 32 ? 128 : 64), 0, s>>>(                \
      *a, (const DeltaSpan*)spans, (const unsigned char*)ws, o32)
#define LSA_C(K, V)                                                                                                       \
  if (a->dk == K && a->dv == V) {                                                                                         \
    delta_chunk_kernel<K, V><<<dim3(n_chunks, a->heads), 256, 0, s>>>(*a, (const DeltaChunk*)chunks, (unsigned char*)ws); \
    LSA_CHECK_LAUNCH();                                                                                                   \
    if (K > 32 && V > 32 && n_spans * a->heads * (V / 32) <= 256) LSA_S(K, V, 2);                                         \
    else LSA_S(K, V, (V == 32 ? 2 : 4));                                                                                  \
    LSA_CHECK_LAUNCH();                                                                                                   \
    delta_norm_kernel<<<dim3(n_chunks, a->heads), 256, 0, s>>>(*a, (const DeltaChunk*)chunks, o32);                       \
    LSA_CHECK_LAUNCH();                                                                                                   \
    return LSA_OK;                                                                                                        \
  }
  LSA_C(32, 32) LSA_C(32, 64) LSA_C(32, 128) LSA_C(64, 32) LSA_C(64, 64) LSA_C(64, 128) LSA_C(128, 32) LSA_C(128, 64)
  LSA_C(128, 128)
#undef LSA_C
#undef LSA_S
  return LSA_UNSUPPORTED;
}
