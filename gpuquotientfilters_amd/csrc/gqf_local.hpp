// gqf_local.hpp -- localized updates: the parts that the SQF's and the RSQF's
// in-place inserts and deletes of small sorted batches share.
//
// A table is cut into windows of LW_SLOTS slots, one wave64 each.  A batch
// key changes only the slots from its quotient to the end of the cluster
// there (insert: up to the empty slot it takes; delete: up to the next slot
// that holds nothing or an entry at its own quotient).  Keys whose ranges
// meet form a region; a region is updated by one lane, key after key, and
// regions never share a slot, so they run in parallel.  Three steps:
//   1. k_*_plan   per window, from the table as it was: what the keys of the
//                 window need (below), and the window's scan state;
//   2. lw_scan    the states' exclusive scan over the windows;
//   3. k_*_apply  per window with keys: the window's slots in LDS, a lane per
//                 region that starts in the window, the changed 64-slot
//                 blocks written back.
// Which keys start a region ("heads"):
//   insert  with E_k the empty slots before key k's quotient, key k takes the
//           empty slot of rank J_k = max(E_k, J_{k-1} + 1) at the latest (a
//           key that is already stored takes none); it starts a region iff
//           J_{k-1} < E_k.  Over a window with n keys and e empty slots, the
//           keys that overflow into the next window are x -> max(0, x + n - e,
//           max_k(E_k - k) + n - e) of those that overflow into it: the
//           state (a, b) of x -> max(x + a, b).
//   delete  key k starts a region iff a boundary (a slot that is empty or
//           whose entry is at its own quotient) lies after key k-1's quotient
//           and at or before its own; the state is the last boundary.
// A region that passes its window's end is held with it, up to some blocks of
// the next window; the next window's wave leaves those slots, and the keys
// there, alone.  The 64-slot block where a window's first region starts may hold the
// end of an earlier window's region: it too is updated in the table, slot by
// slot, and never written back as a whole.
//   Work is per key and per keyed window; a window without keys is read only
// when its predecessor has some (it must absorb what overflows).  Batches
// that do not fit this form raise ctr[CTR_MISC] before anything is written
// and the call takes its general path: more than LW_KEYS keys in a window, a
// whole aligned group of 64 keys without a head, fewer than LW_SPILL empty
// slots in a window (clusters longer than a window), an overflow above
// LW_SPILL, a region that reaches past the blocks held of the next window, a
// region that would take longer than the general path (lw_budget), too few
// regions (lw_scan).  After such a batch the next 4, 8, ... 256 of its kind on
// the stream go straight to the general path.
#pragma once

#include "gqf_rebuild.hpp"

namespace gqf {

constexpr uint32_t LW_SLOTS = 4096;  // slots per window: 64 lanes x one 64-slot block
constexpr uint32_t LW_KEYS = 512;    // keys per window
constexpr int32_t LW_SPILL = 64;     // keys that may overflow into a window
constexpr uint32_t LW_MAX_WINDOWS = RBS_PER * 64;  // one state per window: the scan's limit

// Automatic choice: batches of up to 1/32 of the slots, 1/80 where the
// windows do not fill the chip twice over and the time is that of the
// longest regions.  SQF inserts, ms per call, localized / rebuild:
//   q=26 r=5  fill 0.45  2^20 keys 0.134 / 0.286   2^21 0.212 / 0.342   2^22 0.315 / 0.376
//             fill 0.75  2^20 keys 0.152 / 0.347   2^21 0.267 / 0.401   2^22 0.476 / 0.438
//             fill 0.8   2^10 keys 0.057 / 0.317   2^21 0.312 / 0.414   2^22 0.612 / 0.457
//   q=22 r=5  fill 0.75  2^13 keys 0.061 / 0.098   2^16 0.087 / 0.097   2^18 0.179 / 0.103
//   q=19 r=13 fill 0.8   2^10 keys 0.049 / 0.073   2^13 0.089 / 0.086   2^16 0.118 / 0.091
// Deletes:
//   q=26 r=5  fill 0.75  2^10 keys 0.056 / 0.314   2^20 0.182 / 0.370   2^21 0.316 / 0.423
//             fill 0.8   2^20 keys 0.204 / 0.390   2^21 0.385 / 0.441
//   q=22 r=5  fill 0.75  2^10 keys 0.050 / 0.079   2^13 0.075 / 0.092
// RSQF inserts, localized / by windows:
//   q=26 r=8  fill 0.5   2^10 keys 0.072 / 0.195   2^18 0.144 / 0.382   2^21 0.262 / 0.440
//             fill 0.8   2^10 keys 0.072 / 0.293   2^18 0.158 / 0.392   2^20 0.232 / 0.400
//   q=24 r=5  fill 0.7   2^10 keys 0.058 / 0.145   2^16 0.088 / 0.197
//   q=22 r=8  fill 0.8   2^10 keys 0.055 / 0.073   2^13 0.070 / 0.084
// RSQF deletes, localized / rebuild:
//   q=26 r=8  fill 0.5   2^10 keys 0.077 / 0.375   2^18 0.155 / 0.419   2^21 0.288 / 0.497
//             fill 0.8   2^10 keys 0.083 / 0.472   2^18 0.216 / 0.549   2^20 0.333 / 0.574
//   q=24 r=5  fill 0.7   2^10 keys 0.062 / 0.182   2^16 0.110 / 0.191
static inline bool lw_auto(uint64_t n, uint64_t slots) { return n * (slots >= (8192ull * LW_SLOTS) ? 32 : 80) <= slots; }

static inline uint32_t lw_windows(uint64_t slots) { return (uint32_t)((slots + LW_SLOTS - 1) / LW_SLOTS); }

// Bits of a word that regions share: only a region's own change.
__host__ __device__ __forceinline__ void lw_xor(unsigned long long* p, uint64_t d) {
#ifdef __HIP_DEVICE_COMPILE__
  if (d) atomicXor(p, (unsigned long long)d);
#else
  *p ^= d;
#endif
}

// Scan state of a window: the map x -> max(x + a, b), lb, and the keys that
// start a region.
//   insert  the overflow map; lb = 1 + the largest overflow into the window
//           whose region ends in the blocks held of it (lw_room).
//   delete  a = -2, b = 1 where the last key's region reaches the window's end
//           (else 0): of the windows before, the map at 0 is the last one's b;
//           lb = 1 + the last boundary slot (0: none), with LW_FAR where the
//           first one lies past the blocks held.
struct LW {
  int32_t a, b;
  uint32_t lb, heads;
};
constexpr uint32_t LW_FAR = 0x80000000u;
__host__ __device__ __forceinline__ LW lw_combine(LW x, LW y) {
  const int32_t b = x.b + y.a;
  const uint32_t xl = x.lb & ~LW_FAR, yl = y.lb & ~LW_FAR;
  return LW{x.a + y.a, b > y.b ? b : y.b, xl > yl ? xl : yl, x.heads + y.heads};
}
// The region of an overflow x takes an empty slot for each of the x keys and
// for each of the window's keys before the first with v = E_k - k >= x, which
// starts the next region: the largest x for which these fit `held` slots is
// the maximum of lw_fit over the window's keys and of held - nk (all of them).
__host__ __device__ __forceinline__ int32_t lw_fit(int32_t v, int32_t held, int32_t k) { return v < held - k ? v : held - k; }
__host__ __device__ __forceinline__ uint32_t lw_room(int32_t fit) {
  return 1u + (uint32_t)(fit < 0 ? 0 : fit < LW_SPILL ? fit : LW_SPILL);
}
// b of a window that the localized form does not take: an overflow that no
// window absorbs.
constexpr int32_t LW_BAD = 1 << 28;
__device__ __forceinline__ LW lw_none() { return LW{0, 0, 0u, 0u}; }
__device__ __forceinline__ uint4 lw_pack(LW x) { return make_uint4((uint32_t)x.a, (uint32_t)x.b, x.lb, x.heads); }
__device__ __forceinline__ LW lw_unpack(uint4 w) { return LW{(int32_t)w.x, (int32_t)w.y, w.z, w.w}; }
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ LW lw_dpp(LW x) {
  return LW{(int32_t)dpp_u32<CTRL, ROW_MASK>(0u, (uint32_t)x.a), (int32_t)dpp_u32<CTRL, ROW_MASK>(0u, (uint32_t)x.b),
            dpp_u32<CTRL, ROW_MASK>(0u, x.lb), dpp_u32<CTRL, ROW_MASK>(0u, x.heads)};
}
__device__ __forceinline__ LW lw_wave_excl(LW x, LW* total) {
  LW inc = x;
  inc = lw_combine(lw_dpp<DPP_ROW_SHR | 1>(inc), inc);
  inc = lw_combine(lw_dpp<DPP_ROW_SHR | 2>(inc), inc);
  inc = lw_combine(lw_dpp<DPP_ROW_SHR | 4>(inc), inc);
  inc = lw_combine(lw_dpp<DPP_ROW_SHR | 8>(inc), inc);
  inc = lw_combine(lw_dpp<DPP_ROW_BCAST15, 0xA>(inc), inc);
  inc = lw_combine(lw_dpp<DPP_ROW_BCAST31, 0xC>(inc), inc);
  *total = LW{(int32_t)wave_read((uint32_t)inc.a, 63), (int32_t)wave_read((uint32_t)inc.b, 63), wave_read(inc.lb, 63),
              wave_read(inc.heads, 63)};
  return lw_dpp<DPP_WAVE_SHR1>(inc);
}
// Exclusive scan of the window states: pre[w] = {insert: keys that overflow
// into window w; 1 + the last boundary before it}.  More of the former than
// there is room for, or any past the last window, a region that reaches a
// boundary past the blocks held, and LW_BAD raise the flag, in the counters and
// in host memory (report); so do fewer regions than min_heads (lw_min_heads).  Resets the counters before.  One workgroup and one launch
// for up to LW_ONE windows a thread (5.2 us for 4097; a loop over more of them
// took 34 us for 16385), two launches as rb_scan for more (7 us).
constexpr uint32_t LW_ONE = 8;
__device__ __forceinline__ void lw_raise(uint32_t* ctr, uint32_t* report) {
  ctr[CTR_MISC] = 1u;
  __hip_atomic_store(report, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Stores window w's prefix; whether it or (the last window) the end is bad.
template <bool INS>
__host__ __device__ __forceinline__ bool lw_put(LW p, LW x, uint32_t w, uint32_t W, uint2* __restrict__ pre,
                                                uint32_t min_heads) {
  const int32_t o = p.a > p.b ? p.a : p.b;  // the map of the windows before, at 0
  pre[w] = make_uint2(o > 0 ? (uint32_t)o : 0u, p.lb);
  // (windows that are not read have no overflow)
  const bool bad = INS ? o > LW_SPILL || (o > 0 && (uint32_t)o >= x.lb) : o > 1 || (o > 0 && (x.lb & LW_FAR));
  if (w + 1 < W) return bad;
  const LW all = lw_combine(p, x);
  return bad || (all.a > all.b ? all.a : all.b) > (INS ? 0 : 1) || all.heads < min_heads;
}
template <bool INS>
__global__ __launch_bounds__(1024) void k_lw_one(const uint4* __restrict__ st, uint32_t W, uint2* __restrict__ pre,
                                                 uint32_t min_heads, uint32_t* __restrict__ ctr,
                                                 uint32_t* __restrict__ report) {
  __shared__ uint4 s_wave[16];
  __shared__ uint4 s_st[1024 * (LW_ONE + 1)];  // a thread's windows, one word of 16 bytes apart (banks)
  const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (tid >= CTR_OP && tid < CTR_TOTAL) ctr[tid] = 0u;
  const uint32_t w0 = tid * LW_ONE;
  uint4 x[LW_ONE];
#pragma unroll
  for (uint32_t j = 0; j < LW_ONE; ++j) x[j] = j * 1024 + tid < W ? st[j * 1024 + tid] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
  for (uint32_t j = 0; j < LW_ONE; ++j) {
    const uint32_t i = j * 1024 + tid;
    s_st[i + i / LW_ONE] = x[j];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < LW_ONE; ++j) x[j] = s_st[w0 + tid + j];
  LW own = lw_unpack(x[0]);
#pragma unroll
  for (uint32_t j = 1; j < LW_ONE; ++j) own = lw_combine(own, lw_unpack(x[j]));
  LW wt;
  const LW ex = lw_wave_excl(own, &wt);
  if (lane == 0) s_wave[wid] = lw_pack(wt);
  __syncthreads();  // (orders the counters' reset as well)
  if (wid == 0) {
    LW tot;
    const LW xe = lw_wave_excl(lane < 16 ? lw_unpack(s_wave[lane]) : lw_none(), &tot);
    if (lane < 16) s_wave[lane] = lw_pack(xe);
  }
  __syncthreads();
  LW p = lw_combine(lw_unpack(s_wave[wid]), ex);
  bool bad = false;
#pragma unroll
  for (uint32_t j = 0; j < LW_ONE; ++j) {
    if (w0 + j < W) bad |= lw_put<INS>(p, lw_unpack(x[j]), w0 + j, W, pre, min_heads);
    p = lw_combine(p, lw_unpack(x[j]));
  }
  if (bad) lw_raise(ctr, report);
}
[[maybe_unused]] static __global__ __launch_bounds__(1024) void k_lw_reduce(const uint4* __restrict__ st, uint32_t W,
                                                                            uint4* __restrict__ part,
                                                                            uint32_t* __restrict__ ctr) {
  __shared__ uint4 s_wave[16];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, i = blockIdx.x * RBS_PER + tid;
  if (blockIdx.x == 0 && tid >= CTR_OP && tid < CTR_TOTAL) ctr[tid] = 0u;
  LW t;
  (void)lw_wave_excl(i < W ? lw_unpack(st[i]) : lw_none(), &t);
  if (lane == 0) s_wave[wid] = lw_pack(t);
  __syncthreads();
  if (wid == 0) {
    LW tot;
    (void)lw_wave_excl(lane < 16 ? lw_unpack(s_wave[lane]) : lw_none(), &tot);
    if (lane == 0) part[blockIdx.x] = lw_pack(tot);
  }
}

template <bool INS>
__global__ __launch_bounds__(1024) void k_lw_scan(const uint4* __restrict__ st, uint32_t W, const uint4* __restrict__ part,
                                                  uint2* __restrict__ pre, uint32_t min_heads, uint32_t* __restrict__ ctr,
                                                  uint32_t* __restrict__ report) {
  __shared__ uint4 s_wave[17];  // wave aggregates, then their prefixes; [16] = carry
  const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, i = blockIdx.x * RBS_PER + tid;
  const LW x = i < W ? lw_unpack(st[i]) : lw_none();
  if (wid == 0) {
    LW carry;
    (void)lw_wave_excl(lane < blockIdx.x ? lw_unpack(part[lane]) : lw_none(), &carry);
    if (lane == 0) s_wave[16] = lw_pack(carry);
  }
  LW wt;
  const LW ex = lw_wave_excl(x, &wt);
  if (lane == 0) s_wave[wid] = lw_pack(wt);
  __syncthreads();
  if (wid == 0) {
    const LW carry = lw_unpack(s_wave[16]);
    LW tot;
    const LW xe = lw_wave_excl(lane < 16 ? lw_unpack(s_wave[lane]) : lw_none(), &tot);
    if (lane < 16) s_wave[lane] = lw_pack(lw_combine(carry, xe));
  }
  __syncthreads();
  if (i >= W) return;
  if (lw_put<INS>(lw_combine(lw_unpack(s_wave[wid]), ex), x, i, W, pre, min_heads)) lw_raise(ctr, report);
}

// The regions a batch must have, 24 (insert) or 25 (delete) per 32 keys
// where there is a key per window: long clusters with several keys in each
// make a wave wait for a few lanes.  RSQF q=26 r=8 without that rule, ms per
// call, localized / general path, and the keys per region:
//   insert  fill 0.8   2^20 keys 0.235 / 0.399 (1.20)   2^21 0.429 / 0.453 (1.39)
//           fill 0.9   2^18 keys 0.307 / 0.401 (1.17)   2^20 0.950 / 0.412 (1.67)
//   delete  fill 0.85  2^20 keys 0.515 / 0.597 (1.27)
//           fill 0.9   2^18 keys 0.458 / 0.601 (1.18)   2^19 0.688 / 0.611 (1.29)
static inline uint32_t lw_min_heads(bool insert, uint32_t n, uint32_t W) {
  return n < W ? 0u : (uint32_t)((uint64_t)n * (insert ? 24 : 25) / 32);
}

// The longest region a batch may have, in quarters of a microsecond of its
// lane: a region is updated key after key, and every key moves the entries from
// its place to the cluster's end.  A key's time on MI355X, with the 64-slot
// blocks from its quotient to that end (single regions of 1 .. 60 keys in
// clusters of 1 .. 32 blocks): a + b per block, lw_key.  Past the budget the
// general path is the faster one: it takes about 75 us (RSQF inserts 65) and
// 4.5 or more per 2^20 slots, the call without its longest region about 40.
// Without this rule, us a call, localized / general path:
//   SQF   q=22 r=5 fill 0.9   30011 keys deleted 326 / 111
//   RSQF  q=20 r=8 fill 0.9   64 copies of a key inserted 477 / 68, deleted 971 / 175
//         q=24 r=8 fill 0.9   100003 keys inserted 264 / 161, deleted 498 / 204
//         q=26 r=8 fill 0.95  1000 keys, 16 different ones, deleted 5197 / 645
static inline uint32_t lw_budget(bool rsqf_insert, uint64_t slots) {
  return (uint32_t)((rsqf_insert ? 96 : 128) + 18 * slots / (1u << 20));
}
struct LwKey {
  uint32_t a, b;
};
// SQF slots of bpe bytes; RSQF remainders of r bits.
template <bool INS>
__host__ __device__ __forceinline__ LwKey lw_key_sqf(uint32_t bpe) {
  return INS ? (bpe == 1 ? LwKey{5, 3} : LwKey{4, 5}) : (bpe == 1 ? LwKey{7, 5} : LwKey{8, 7});
}
template <bool INS>
__host__ __device__ __forceinline__ LwKey lw_key_rsqf(uint32_t r) {
  return INS ? LwKey{5, 1 + r * 5 / 16} : LwKey{10, 3 + r / 2};
}
// The longest region among a window's keys, 64 at a time -- in a loop of its
// own, which few windows need (may): a key's cluster spans no more blocks than
// lie without empty slots (boundaries) together, and the two beside them.
template <bool INS>
struct LwChain {
  LwKey key;
  uint64_t nz;      // blocks with empty slots (insert) or boundaries (delete)
  uint32_t spread;  // insert: sixteenths of a block to the next empty slot
  uint32_t carry = 0, keys = 0, longest = 0;
  __device__ __forceinline__ LwChain(LwKey k, uint64_t nz_, uint32_t empties)
      : key(k), nz(nz_), spread(INS ? 1024u / (empties ? empties : 1u) : 0u) {}
  // Whether the longest region of nk keys with so many heads may be past the
  // budget.
  __device__ __forceinline__ bool may(uint32_t nk, uint32_t heads, uint32_t budget) const {
    const uint32_t most = nk - heads + 1u;
    uint32_t gap = 2;
    for (uint64_t z = ~nz; z; z &= z << 1) ++gap;
    return most * (key.a + key.b * (gap + (most * spread >> 4))) > budget;
  }
  // A key of block blk and its slot s there, whose word of the plane is mask;
  // the heads of the 64 keys: heads.
  __device__ __forceinline__ void add(bool on, uint64_t mask, uint32_t s, uint32_t blk, bool head, uint64_t heads) {
    const uint32_t lane = threadIdx.x & 63;
    uint32_t n = 1;  // blocks to the cluster's end
    if (!(mask & (INS ? ~0ull << s : ~((2ull << s) - 1ull)))) {
      const uint64_t later = nz & ~((2ull << blk) - 1ull);
      n += (later ? (uint32_t)__builtin_ctzll(later) : 64u) - blk;
    }
    if (INS) {  // the empty slots that the region's keys before it have taken
      const uint64_t h = heads & ((2ull << lane) - 1ull);
      const uint32_t before = h ? lane - 63u + (uint32_t)__clzll(h) : lane + keys;
      n += before * spread >> 4;
      keys = heads ? (uint32_t)__clzll(heads) + 1u : keys + 64u;
    }
    const uint32_t cost = on ? key.a + key.b * n : 0u, sum = wave_incl_add(cost);
    const uint32_t from = wave_incl_max(head ? sum - cost + 1 : 0u);  // 1 + the costs before the last head
    const uint32_t since = from ? sum + 1 - from : sum + carry;
    carry = wave_read(since, 63);
    longest = since > longest ? since : longest;
  }
};

static inline size_t lw_scan_bytes(uint32_t W) { return aligned_bytes((size_t)((W + RBS_PER - 1) / RBS_PER) * 16); }
template <bool INS>
static gqf_status lw_scan(hipStream_t s, DeviceState& ds, Arena& ar, const uint4* st, uint32_t W, uint2* pre,
                          uint32_t min_heads) {
  const uint32_t P = (W + RBS_PER - 1) / RBS_PER;
  uint4* part = ar.take<uint4>(P ? P : 1);
  if (ar.used > ar.cap) {
    set_error("internal: window scan workspace overflow");
    return GQF_ERR_INVALID;
  }
  *reinterpret_cast<volatile uint32_t*>(ds.h_local) = 0u;
  if (W <= LW_ONE * 1024) {
    GQF_LAUNCH(k_lw_one<INS>, dim3(1), dim3(1024), 0, s, st, W, pre, min_heads, ds.counters, ds.d_local);
    return GQF_OK;
  }
  GQF_LAUNCH(k_lw_reduce, dim3(P), dim3(RBS_PER), 0, s, st, W, part, ds.counters);
  GQF_LAUNCH(k_lw_scan<INS>, dim3(P), dim3(RBS_PER), 0, s, st, W, part, pre, min_heads, ds.counters, ds.d_local);
  return GQF_OK;
}
// After the call's work: whether the localized form took the batch.
static inline bool lw_done(DeviceState& ds) { return *reinterpret_cast<volatile uint32_t*>(ds.h_local) == 0u; }

// Entries of the sorted batch with quotients below the windows w - 1, w and
// w + 1 (the calling wave's three searches, 8 lanes each).
template <typename K>
__device__ __forceinline__ void lw_bounds(const K* __restrict__ B, uint32_t n, uint32_t r, uint32_t w, uint32_t* prev,
                                          uint32_t* b0, uint32_t* b1) {
  const uint32_t g = (threadIdx.x & 63) / 8, x = w + g - 1;  // (w = 0: no window before)
  const bool on = g < 3 && (w || g);
  const uint64_t key = ((uint64_t)x * LW_SLOTS) << r;
  const uint32_t b = group8_search(0u, on ? n : 0u, [&](uint32_t m) { return (uint64_t)B[m] < key; });
  *prev = wave_read(b, 0);
  *b0 = wave_read(b, 8);
  *b1 = wave_read(b, 16);
}

// Each window's range of the sorted batch: bstart[x] = first fingerprint with
// quotient >= LW_SLOTS x (x = 0 .. W), 8 lanes per window (group8_search).
// Also resets the counters.
constexpr uint32_t WB_LANES = 8;
template <typename K>
__global__ __launch_bounds__(256) void k_wm_bounds(const K* __restrict__ B, uint32_t n, uint32_t r, uint32_t W,
                                                   uint32_t* __restrict__ bstart, uint32_t* __restrict__ ctr) {
  if (blockIdx.x == 0 && threadIdx.x >= CTR_OP && threadIdx.x < CTR_TOTAL) ctr[threadIdx.x] = 0u;
  const uint32_t gt = blockIdx.x * 256 + threadIdx.x;
  const uint32_t x = gt / WB_LANES;
  // every lane stays for the ballots; groups past W search an empty range
  const uint64_t key = ((uint64_t)x * LW_SLOTS) << r;
  const uint32_t b = group8_search(0u, x <= W ? n : 0u, [&](uint32_t m) { return (uint64_t)B[m] < key; });
  if (gt % WB_LANES == 0 && x <= W) bstart[x] = b;
}

// The largest value of the lanes of a wave.
__device__ __forceinline__ int32_t lw_wave_max(int32_t x) {
  return (int32_t)(wave_read(wave_incl_max((uint32_t)x ^ 0x80000000u), 63) ^ 0x80000000u);
}
// Heads among the 64 keys [k0, k0 + 64) of a window, one per lane, from
// v = E_k - k (valid lanes only) and the running maximum M of the keys before
// (initially the overflow into the window): bit of the calling lane.
__device__ __forceinline__ bool lw_insert_head(int32_t v, bool valid, int32_t& M) {
  // maxima over values shifted to unsigned, 0 the identity
  const uint32_t u = valid ? (uint32_t)v ^ 0x80000000u : 0u;
  const uint32_t inc = wave_incl_max(u);
  const uint32_t ex = dpp_u32<DPP_WAVE_SHR1>(0u, inc);
  const uint32_t m0 = (uint32_t)M ^ 0x80000000u;
  const uint32_t before = ex > m0 ? ex : m0;
  const uint32_t all = wave_read(inc, 63);
  M = (int32_t)((all > m0 ? all : m0) ^ 0x80000000u);
  return valid && u >= before;
}

}  // namespace gqf
