// How workgroups that each have a part of a tile's sum finish the tile together.
//
// Each writes its part through to memory (sc1 stores, drained before it arrives), and then finishes one of ``ns`` shares of the tile: it
// waits until all parts have arrived and reads its share of the others. Against the last to arrive reading all parts, which is one CU
// at some 50 GB/s (256 x 128 in four parts: 512 KB there, 96 KB here), gemm_sk takes for 512 rows by 4096 x 11008 in four parts 59.3 -> 49.5
// us, by 4096 x 4096 in four 36.1 -> 28.0 and in two 29.1 -> 26.9, 1256 by 3072 x 8192 in two 65.2 -> 61.2, and 1984 products in parts
// within one round of tiles 0.89 of their time (geometric mean); whole steps of 512 sequences (Llama-2-7B) 6993 -> 6884.
// Nobody waits for a workgroup that may have no place to run: after ``looks`` looks at the counter a workgroup leaves its share to the
// last to arrive, who finds that in the counter it arrives at. Two streams' launches that wait for each other's places end this way. A pair of
// products beside each other, with 64 looks and with none (and through the last to arrive alone): 512 rows by 4096 x 11008 in four parts 105 and 117
// us (118), by 4096 x 4096 in two 53.4 and 55.2 (54.8), 384 by 4096 x 11008 in five 98.4 and 100 (103), 128 by 3072 x 3072 in four 22.8 and 24.0
// (24.6); in six parts of 256 x 128, 256 by 4096 x 11008, the wait costs 2 of 73.
// The sums are the same whoever makes them: parts are added in their order.
#pragma once
#include "common.h"

// A tile's counter, zero before the launch and behind it: parts that arrived, shares that were left (bits), workgroups that are through.
constexpr unsigned HO_PARTS = 4095u, HO_LEFT = 12, HO_DONE = 20;
// From one tile's counter to the next, in words: lines and channels of their own. With 64 counters in two lines the looks of all tiles'
// workgroups held up each other's arrivals: 3072 x 3072 of 128 rows in four parts 16.8 us instead of 13.0 from first start to last end.
constexpr int HO_STRIDE = 64;
constexpr int HO_SHARES = HO_DONE - HO_LEFT;  // at most
constexpr int HO_LAST = -1;                   // instead of looks: the last to arrive finishes all, for launches with more workgroups than CUs

// One thread, what other shares need of its workgroup's part written through: arrives at ``c`` with part ``s`` of ``S``. The shares that
// are this workgroup's to finish, as bits; ``last``: all other parts had arrived. HO_TIRED: it has looked often enough. Then all of its part
// is to be written, and ho_leave says whether the share is still its own.
constexpr unsigned HO_TIRED = 1u << 31;
LSA_DEVICE unsigned ho_arrive(unsigned* c, int s, int S, int ns, int looks, bool& last) {
  unsigned v = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
  last = (v & HO_PARTS) == (unsigned)S;
  if (looks < 0) return last ? (1u << ns) - 1u : 0u;
  const unsigned mine = s < ns ? 1u << s : 0u;
  if (last) return mine | ((v >> HO_LEFT) & ((1u << HO_SHARES) - 1u));
  if (!mine) return 0u;
  for (int i = 0; i < looks; ++i) {
    __builtin_amdgcn_s_sleep(1);
    v = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((v & HO_PARTS) == (unsigned)S) return mine;
  }
  return HO_TIRED;
}

LSA_DEVICE unsigned ho_leave(unsigned* c, int s, int S) {
  unsigned v = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while ((v & HO_PARTS) < (unsigned)S)  // (where the exchange fails, v is what has arrived meanwhile)
    if (__hip_atomic_compare_exchange_strong(c, &v, v | (1u << (HO_LEFT + s)), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return 0u;
  return 1u << s;
}

// One thread: the last one through leaves the counter as it was. Other waves of its workgroup may still be reading parts: neither they nor
// the counter are used for anything else before the launch has ended.
LSA_DEVICE void ho_through(unsigned* c, int s, int ns, int looks, unsigned mine, bool last) {
  if (looks < 0) {
    if (last) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  // every share finished by its own part's workgroup counts for one, and the last to arrive, who has what others left, for one more
  const unsigned own = (s < ns ? (mine >> s) & 1u : 0u) + (last ? 1u : 0u);
  if (!own) return;
  const unsigned v = __hip_atomic_fetch_add(c, own << HO_DONE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((v >> HO_DONE) + own + __builtin_popcount((v >> HO_LEFT) & ((1u << HO_SHARES) - 1u)) == (unsigned)ns + 1u)
    __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// compute units of the current device
inline int device_cus() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int v = 0;
    cached[dev] = hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0 ? v : 256;
  }
  return cached[dev];
}
