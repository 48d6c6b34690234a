// Grouped-query attention over a paged cache: per-head scale, soft-capped scores, a sliding window that
// keeps the first tokens or sees what lies behind it as means of blocks, a softmax (with or without a sink) or
// a sigmoid per key (less a logarithm of the distance), and an output gate per head or per value.
//
// A page holds 64 tokens of one layer. Keys lie token by token, values channel by channel:
//   k [n_pages][kv_heads][64][dkp]      v [n_pages][kv_heads][dvp][64]
// so that both are read as MFMA operands in 16-byte pieces. The 64 tokens of a value row are stored in
// the order in which the scores' accumulators hold them (att_vidx), which lets the weights go from
// the score tile straight into the value product.
//
// Pooled blocks: block b holds the means of the keys and values at positions b pool .. b pool + pool - 1. They
// lie in pages of 64 blocks of the same layout, which have a table of their own; a row at position i sees
// those whose last position is at most i - window.
#pragma once
#include "elem.h"

constexpr int ATT_PAGE = 64;

// Mirrored by llm_sharding_amd/ops/paged_attn.py::AttnArgs (ctypes) - keep the field order in sync.
struct AttnArgs {
  void* k;
  void* v;
  const int* table;     // [slots][max_pages] page of each 64-token stretch, -1: none
  const int* slot;      // [rows]
  const int* pos;       // [rows]
  const int* index;     // optional: entry i of the launch is row index[i]
  const float* hscale;  // [heads] score scale times the head's own number
  int max_pages;
  int n_pages;
  int heads, kv_heads;
  int dim, vdim, dkp, dvp;  // dkp, dvp: padded head parts (zeros behind)
  int window;               // a row sees keys less than this far back (INT_MAX: all) ..
  int keep;                 // .. and keys before this position
  float softcap;            // 0: none
  void* pk;                 // pooled blocks
  void* pv;
  const int* ptable;        // [slots][pmax_pages] page of each 64 blocks
  int pool, pmax_pages, pn_pages;  // pool 0: no blocks
  const float* sig;         // null: softmax; else [3][heads] r1, r2 and the number added to a score: weights are
                            // sigmoid(score - r1 ln(1 + r2 distance) + number)
  int sink;                 // softmax over one more score of 0
  int elem_gate;            // the gate has a value per output value, not per head
  int temp_every;           // queries times 1 + temp_coef ln(floor((p + 1) / temp_every) + 1)
  float temp_coef;
  float oscale;             // factor of the output
};

// place of token r (0..63) in a value row
LSA_DEVICE int att_vidx(int r) { return (r & 32) | ((r & 12) << 1) | ((r & 16) >> 2) | (r & 3); }

LSA_DEVICE bool att_sees(const AttnArgs& a, int p, int key) {
  return key <= p && (p - key < a.window || key < a.keep);
}

// position of a live row, -1 for one whose slot holds no page there (an idle row of a decode graph)
LSA_DEVICE int att_pos(const AttnArgs& a, int row) {
  const int p = a.pos[row];
  if (p < 0 || p >= a.max_pages * ATT_PAGE) return -1;
  const int pg = a.table[(size_t)a.slot[row] * a.max_pages + p / ATT_PAGE];
  return pg < 0 || pg >= a.n_pages ? -1 : p;
}

LSA_DEVICE int att_page(const AttnArgs& a, int slot, int b) {
  const int pg = a.table[(size_t)slot * a.max_pages + b];
  return pg < 0 || pg >= a.n_pages ? 0 : pg;
}

// pooled blocks that a row at position p sees: the first ones
LSA_DEVICE int att_pooled(const AttnArgs& a, int p) {
  const int n = p - a.window + 1;
  return a.pool > 0 && n > 0 ? n / a.pool : 0;
}

LSA_DEVICE int att_ppage(const AttnArgs& a, int slot, int b) {
  const int pg = b < a.pmax_pages ? a.ptable[(size_t)slot * a.pmax_pages + b] : 0;
  return pg < 0 || pg >= a.pn_pages ? 0 : pg;
}

// The key blocks (of one page each) that rows at positions p0..p1 see some key of: pages of pooled blocks, then
// the kept pages, then those from the window's first on.
struct AttBlocks {
  int pooled, kept, first, n;
  LSA_DEVICE AttBlocks(const AttnArgs& a, int p0, int p1) {
    const int last = p1 / ATT_PAGE;
    pooled = (att_pooled(a, p1) + ATT_PAGE - 1) / ATT_PAGE;
    kept = a.keep > 0 ? (min(a.keep, p1 + 1) - 1) / ATT_PAGE + 1 : 0;
    const int w = p0 - a.window + 1;  // oldest key in the first row's window
    first = max(kept, w > 0 ? w / ATT_PAGE : 0);
    n = pooled + kept + max(0, last - first + 1);
  }
  LSA_DEVICE bool is_pooled(int i) const { return i < pooled; }
  LSA_DEVICE int at(int i) const {  // number of the page among its kind
    if (i < pooled) return i;
    i -= pooled;
    return i < kept ? i : first + i - kept;
  }
};

// page of listed block i and where its kind of pages begins
struct AttKv {
  const void* k;
  const void* v;
  int page;
};
LSA_DEVICE AttKv att_kv(const AttnArgs& a, const AttBlocks& bl, int slot, int i) {
  if (bl.is_pooled(i)) return AttKv{a.pk, a.pv, att_ppage(a, slot, i)};
  return AttKv{a.k, a.v, att_page(a, slot, bl.at(i))};
}

// head h's factor of a row's scores at position p
LSA_DEVICE float att_scale(const AttnArgs& a, int h, int p) {
  const float s = a.hscale[h];
  return a.temp_coef == 0.f ? s : s * (1.f + a.temp_coef * logf((float)((p + 1) / a.temp_every + 1)));
}

// sum l of exp2(score - m): factor that turns the sum of values into the output (0: no key)
LSA_DEVICE float att_norm(const AttnArgs& a, float m, float l) {
  if (!a.sink) return l > 0.f ? 1.f / l : 0.f;
  const float t = fmaxf(m, 0.f), e = __builtin_amdgcn_exp2f(m - t);
  return e / (l * e + __builtin_amdgcn_exp2f(-t));
}

// output gate of value d of head h
template <typename T>
LSA_DEVICE float att_gate(const AttnArgs& a, const T* gate, size_t row, int ldg, int h, int d) {
  return gate ? 1.f / (1.f + __expf(-ld1(gate + row * ldg + (a.elem_gate ? h * a.dvp + d : h)))) : 1.f;
}
LSA_DEVICE f32x4_t att_gate4(const AttnArgs& a, const bf16_raw* gate, size_t row, int ldg, int h, int d) {
  if (gate && a.elem_gate) {
    const u32x2_t v = *reinterpret_cast<const u32x2_t*>(gate + row * ldg + h * a.dvp + d);
    return f32x4_t{sigmoid(__uint_as_float(v[0] << 16)), sigmoid(__uint_as_float(v[0] & 0xffff0000u)),
                   sigmoid(__uint_as_float(v[1] << 16)), sigmoid(__uint_as_float(v[1] & 0xffff0000u))};
  }
  const float g = gate ? sigmoid(bf2f(gate[row * ldg + h])) : 1.f;
  return f32x4_t{g, g, g, g};
}

// A sigmoid weight from a score s2 in exponents of two (times log2 e): 1 / (1 + exp2(-s2 + r1 log2(1 + r2 d) - b2))
struct AttSig {
  float r1, r2, b2;
  AttSig() = default;
  LSA_DEVICE AttSig(const AttnArgs& a, int h) {
    r1 = a.sig[h];
    r2 = a.sig[a.heads + h];
    b2 = a.sig[2 * a.heads + h] * 1.4426950408889634f;
  }
  LSA_DEVICE float offset(float d) const { return r1 * __builtin_amdgcn_logf(fmaf(r2, d, 1.f)) - b2; }
  static LSA_DEVICE float weight(float s2, float off) {
    return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(off - s2));
  }
};

// score (q . k) times the head's factor -> soft-capped
LSA_DEVICE float att_cap(float s, float cap, float icap) {
  // cap tanh(s / cap) = cap (1 - 2 / (exp(2 s / cap) + 1))
  return cap - 2.f * cap * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(s * icap) + 1.f);  // icap = 2 log2(e) / cap
}

// lsa_attn_plain's work in fp32 (paged_attn_f32.hip); false: not a size or alignment for it, nothing launched.
bool attn_f32(const AttnArgs& a, int n, bool singles, const float* q, int ldq, const float* gate, int ldg, float* out, int ldo,
              hipStream_t s);
