// gqf_plookup.hpp -- large batches of lookups by quotient range instead of
// one random table access per key:
//
//   k_ps_scatter<.., true>  the keys by group (gqf_dbuild.hpp), and what brings
//                 the answers back: every key's place in its tile, and per tile
//                 and group the place of the tile's first key and its region;
//   k_pl_sqf / k_pl_rsqf   a group's part of the table in LDS, the walks there,
//                 every answer in its key's place;
//   k_pl_gather   a tile's answers, run by run, to LDS and in the order of the
//                 keys to the output.
// The direct walk costs a cache line from beyond the L2 per key and is bound
// by their number: 38 G/s (SQF) and 30 G/s (RSQF) on tables of 2^26 slots.
// Here every pass streams: about 32 bytes per key and the table once.  2^24
// keys, 2^26 slots: SQF 437 -> 235 us (partition 68, walks 106, answers 55),
// RSQF (r = 8) 552 -> 223 us (77, 89, 50).  The walks are bound by their
// instructions, the other two by the number of their runs (16 keys each).
//   A walk that leaves the group's part (clusters that reach far past it) and
// a key that its group's region has no room for (hot keys) answer PL_PENDING;
// k_pl_gather walks the table for them.
#pragma once

#include "gqf_dbuild.hpp"
#include "gqf_sqf_dev.hpp"

namespace gqf {

constexpr uint32_t PL_PENDING = 0xFFFFFFFEu;  // no slot (tables have fewer than 2^31)
constexpr int PL_THREADS = 512;
// Where the direct walk ends (us, direct : by groups).  SQF, q = 26: 71 : 87 at
// 2^21 keys, 116 : 103 at 2^22, 381 : 226 at 2^24; q = 20, whose table stays in
// the L2: 68 : 75, 111 : 104, 373 : 279 (the direct walk's instructions).
// RSQF, q = 26: 78 : 92, 136 : 107, 480 : 223; q = 24: 93 : 72, 156 : 89; its
// cheaper walk stays ahead where the table does in the L2s: q = 22, 2^24 keys
// 216 : 225.
constexpr uint64_t PL_MIN = 7u << 19;
constexpr uint32_t PL_QMIN_SQF = 20, PL_QMIN_RSQF = 24;
// SQF walks through long clusters: the group's walk takes as many steps as the
// direct one, with a workgroup per group (256 up to q = 23) and the way there
// and back on top.  64ths of a step of 32 slots per key (0.3 steps at fill
// 0.85, 0.85 at 0.9, 3.7 at 0.95, 8 at 0.97, 71 when full) up to which the
// groups stay ahead.  us, direct : by groups, for 2^22 and 2^24 keys: q = 20 at
// 0.85 158 : 147, 553 : 458, at 0.9 240 : 317, 863 : 1032; q = 23 at 0.85
// 154 : 145, 544 : 406, at 0.9 242 : 264, 862 : 816; q = 24 at 0.95
// 554 : 503, 2026 : 1801, at 0.98 1590 : 1672, 5833 : 5694, full 7685 : 13122,
// 28264 : 45663; q = 26 at 0.98 889 : 698, 3274 : 2081.
// Counted in PL_SAMPLE of the groups (by all of them, one counter for the waves
// takes 125 us at q = 26; a sum in the gather, 5 to 8).
constexpr uint32_t PL_SAMPLE = 64, PL_SAMPLE_WAVES = PL_SAMPLE * (PL_THREADS / 64);
inline uint32_t pl_steps_max(uint32_t q) { return q <= 23 ? 40 : q == 24 ? 400 : 1280; }

struct PlPlan {
  PsPlan p;
  uint32_t tiles, lanes;  // tiles; log2 of the lanes that move a run
};
// The plan of n lookups in a table of 2^q quotients; false where the direct
// walk is the faster one.
inline bool pl_plan(uint64_t n, uint32_t q, uint32_t r, uint32_t qmin, PlPlan* o) {
  if (n < PL_MIN || q < qmin || q > DB_QB + PS_GB_MAX || r > 8 || n >= (1ull << 30)) return false;
  PsPlan& p = o->p;
  o->tiles = ps_tiles(n, q, r, &p);
  const uint64_t mean = n >> p.gb;
  p.cap = (uint32_t)((mean + mean / 4 + 1024 + 63) & ~63ull);
  o->lanes = 3;
  while (o->lanes < 6 && (1u << o->lanes) < 3 * (p.tile >> p.gb) / 2) ++o->lanes;
  return true;
}
static inline size_t pl_bytes(const PlPlan& o, uint64_t n) {
  const size_t nd = o.p.ngroups;
  return aligned_bytes(nd * o.p.cap * 4) + aligned_bytes((nd + 2) * 4) + aligned_bytes(n * 2) +
         aligned_bytes(o.tiles * nd * 4) + aligned_bytes(o.tiles * nd * 2) + 4096;
}

// ---------------------------------------------------------------- SQF walks
// A group's slots in LDS: PL_BACK before its first quotient and PL_FWD past
// its last one (clusters that cross), the table bytes and the three flag
// planes.
constexpr uint32_t PL_BACK = 256, PL_FWD = 512, PL_SLOTS = DB_NQ + PL_BACK + PL_FWD, PL_WORDS = PL_SLOTS / 32 + 1;

// 32 bits of a plane from bit `at` on (the word after them is read).
__device__ __forceinline__ uint32_t pl_bits(const uint32_t* s_plane, uint32_t at) {
  return __builtin_amdgcn_alignbit(s_plane[(at >> 5) + 1], s_plane[at >> 5], at & 31u);
}
// Position of the k-th set bit of x (1 <= k <= their number).
__device__ __forceinline__ uint32_t pl_select(uint32_t x, uint32_t k) {
  uint32_t pos = 0;
#pragma unroll
  for (uint32_t h = 16; h; h >>= 1) {
    const uint32_t c = (uint32_t)__popc((x >> pos) & ((1u << h) - 1u));
    const bool up = k > c;
    k -= up ? c : 0u;
    pos += up ? h : 0u;
  }
  return pos;
}

// sqf_lookup_win's walk for the quotient at `at` in the loaded slots (end of
// them, at least 32 before `at`): the slot, SQF_NOT_FOUND or PL_PENDING.  In
// 32-bit steps from where the walk stands (counted), not words of the table: 64-bit
// shifts and counts of whole words took 142 us at 2^24 keys.
__device__ __forceinline__ uint32_t pl_sqf_walk(const uint32_t* s_raw, const uint32_t* s_occ, const uint32_t* s_cont,
                                                const uint32_t* s_shf, uint32_t end, uint32_t at, uint32_t fr,
                                                uint32_t& steps) {
  uint32_t s = at - 31, occ = pl_bits(s_occ, s);  // (bit 31: the quotient's)
  if (!(occ >> 31)) return SQF_NOT_FOUND;
  // the cluster's start, and the run starts to skip after it
  uint32_t ns = ~pl_bits(s_shf, s), k = 0;
  while (ns == 0) {
    k += (uint32_t)__popc(occ);
    if (s < 32) return PL_PENDING;
    ++steps;
    s -= 32;
    ns = ~pl_bits(s_shf, s);
    occ = pl_bits(s_occ, s);
  }
  const uint32_t d = (uint32_t)__builtin_clz(ns);
  k += (uint32_t)__popc((occ >> 1) >> (31u - d));
  s += 31u - d;
  if (k) {  // the k-th slot after it without a continuation bit
    ++s;
    uint32_t rs = ~pl_bits(s_cont, s), c;
    while ((c = (uint32_t)__popc(rs)) < k) {
      k -= c;
      s += 32;
      ++steps;
      if (s + 32 > end) return PL_PENDING;
      rs = ~pl_bits(s_cont, s);
    }
    s += pl_select(rs, k);
  }
  // its run, four slots at a time: the first remainder >= fr
  const uint32_t frs = fr * 0x01010101u;
  uint32_t head = 0x00000080u;  // (the first slot belongs to the run)
  for (;;) {
    if (s + 8 > end) return PL_PENDING;
    const uint32_t x = __builtin_amdgcn_alignbyte(s_raw[(s >> 2) + 1], s_raw[s >> 2], s & 3u);
    const uint32_t stop = ~(x << 6) & 0x80808080u & ~head;
    uint32_t ge = ((((x >> 3) & 0x1F1F1F1Fu) | 0x80808080u) - frs) & 0x80808080u;
    ge &= stop ? (stop & (0u - stop)) - 1u : ~0u;
    if (ge) {
      const uint32_t p = (uint32_t)__builtin_ctz(ge) >> 3;
      return ((x >> (8 * p + 3)) & 0x1Fu) == fr ? s + p : SQF_NOT_FOUND;
    }
    if (stop) return SQF_NOT_FOUND;
    head = 0;
    s += 4;
  }
}

// p[0 .. m) = walk(p[i]), four at a time and the next four on their way (up to
// three words past m, of the same region, change).
template <typename F>
__device__ __forceinline__ void pl_each(uint32_t* p, uint32_t m, F walk) {
  uint4* p4 = reinterpret_cast<uint4*>(p);
  const uint32_t n4 = (m + 3) / 4;
  uint32_t i = threadIdx.x;
  uint4 next = i < n4 ? p4[i] : make_uint4(0u, 0u, 0u, 0u);
  for (; i < n4; i += PL_THREADS) {
    const uint4 k = next;
    if (i + PL_THREADS < n4) next = p4[i + PL_THREADS];
    uint4 a;
    a.x = walk(k.x);
    a.y = walk(k.y);
    a.z = walk(k.z);
    a.w = walk(k.w);
    p4[i] = a;
  }
}

// The sampled waves' steps and how many of the waves are done, in one word; the
// last wave compares.  *crowded: raised for more than 64 steps_max steps.
__device__ __forceinline__ void pl_count(unsigned long long* steps, uint32_t took, uint32_t steps_max,
                                         uint32_t* crowded) {
  for (int x = 32; x; x >>= 1) took += (uint32_t)__shfl_xor((int)took, x);
  if (threadIdx.x & 63u) return;
  const uint32_t sum = took >> 6;
  const unsigned long long old = atomicAdd(steps, ((unsigned long long)sum << 16) + 1ull);
  if ((uint32_t)(old & 0xFFFFu) == PL_SAMPLE_WAVES - 1 && (old >> 16) + sum > steps_max) *crowded = 1u;
}

// Group blockIdx.x of a table of 1-byte slots (16-byte aligned, S slots).
[[maybe_unused]] static __global__ __launch_bounds__(PL_THREADS) void k_pl_sqf(
    const uint8_t* __restrict__ t, uint32_t S, uint32_t qb, uint32_t r, const uint32_t* __restrict__ gsize, uint32_t cap,
    uint32_t* __restrict__ io, unsigned long long* __restrict__ steps, uint32_t steps_max, uint32_t* __restrict__ crowded) {
  __shared__ __align__(16) uint32_t s_raw[PL_SLOTS / 4];
  __shared__ uint32_t s_occ[PL_WORDS], s_cont[PL_WORDS], s_shf[PL_WORDS];
  const uint32_t g = blockIdx.x, q0 = g << qb, m = gsize[g] < cap ? gsize[g] : cap;
  const bool sampled = g % (gridDim.x / PL_SAMPLE) == 0;
  if (m == 0) {
    if (sampled) pl_count(steps, 0u, steps_max, crowded);
    return;
  }
  // (group 0: PL_BACK slots that read as empty stand before slot 0, a cluster
  // start to the walk as slot 0 itself is)
  const uint32_t lo = q0 - PL_BACK, end = (1u << qb) + PL_BACK + PL_FWD;
  for (uint32_t c = threadIdx.x; c < end / 16; c += PL_THREADS) {
    const uint32_t s0 = lo + 16 * c;  // (wraps before slot 0: past the table's end, too)
    uint4 x = make_uint4(0u, 0u, 0u, 0u);  // slots outside the table read as empty
    if (s0 < S && s0 + 16 <= S) {
      x = *reinterpret_cast<const uint4*>(t + s0);
    } else if (s0 < S) {
      uint32_t b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (uint32_t i = 0; i < 16; ++i)
        if (s0 + i < S) b[i >> 2] |= (uint32_t)t[s0 + i] << (8 * (i & 3));
      x = make_uint4(b[0], b[1], b[2], b[3]);
    }
    reinterpret_cast<uint4*>(s_raw)[c] = x;
    auto plane = [&](uint32_t bit) {
      return byte_bits8((x.x >> bit) & 0x01010101u, (x.y >> bit) & 0x01010101u) |
             byte_bits8((x.z >> bit) & 0x01010101u, (x.w >> bit) & 0x01010101u) << 8;
    };
    reinterpret_cast<uint16_t*>(s_occ)[c] = (uint16_t)plane(2);
    reinterpret_cast<uint16_t*>(s_cont)[c] = (uint16_t)plane(1);
    // (slot 0 starts a cluster whatever its bit says)
    reinterpret_cast<uint16_t*>(s_shf)[c] = (uint16_t)(s0 == 0 ? plane(0) & ~1u : plane(0));
  }
  __syncthreads();
  uint32_t* p = io + (uint64_t)g * cap;
  const uint32_t qmask = (1u << qb) - 1u, rmask = (1u << r) - 1u;
  uint32_t took = 0;
  pl_each(p, m, [&](uint32_t key) {
    const uint32_t a = pl_sqf_walk(s_raw, s_occ, s_cont, s_shf, end, ((key >> r) & qmask) + PL_BACK, key & rmask, took);
    return a >= PL_PENDING ? a : a + lo;
  });
  if (sampled) pl_count(steps, took, steps_max, crowded);
}

// The direct walk, for k_pl_gather.
struct SqfWalk {
  const uint8_t* t;
  uint32_t S, q, r, hflag;
  __device__ __forceinline__ uint32_t operator()(uint32_t key) const {
    const uint32_t fp = fingerprint32(key, q + r + hflag);
    return sqf_lookup_win<1>(t, S, (fp >> r) & (uint32_t)mask64(q), fp & ((1u << r) - 1u));
  }
};

// ---------------------------------------------------------------- answers
// Tile blockIdx.x: the answers of its keys from the groups' regions, in the
// order of the keys; direct(key): the walk in the table.  *crowded is raised
// for keys without a place in their region.
template <typename Walk>
__global__ __launch_bounds__(PS_THREADS) void k_pl_gather(Walk direct, const uint32_t* __restrict__ keys, uint32_t n,
                                                          uint32_t nd, uint32_t tile, uint32_t cap, uint32_t lanes,
                                                          const uint32_t* __restrict__ tbase,
                                                          const uint16_t* __restrict__ tfirst,
                                                          const uint16_t* __restrict__ place,
                                                          const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                          uint32_t* __restrict__ crowded) {
  __shared__ uint32_t s_ans[PS_TILE];
  __shared__ uint32_t s_base[PS_ND];
  __shared__ uint16_t s_first[PS_ND + 2];
  const uint32_t t = threadIdx.x;
  const uint64_t t0 = (uint64_t)blockIdx.x * tile;
  const uint32_t tn = (uint32_t)(n - t0 < tile ? n - t0 : tile);
  for (uint32_t d = t; d < nd; d += PS_THREADS) {
    s_base[d] = tbase[(uint64_t)blockIdx.x * nd + d];
    s_first[d] = tfirst[(uint64_t)blockIdx.x * nd + d];
  }
  if (t == 0) s_first[nd] = (uint16_t)tn;  // (32768 at most)
  uint2 pl[PS_ITEMS / 4];
#pragma unroll
  for (uint32_t c = 0; c < PS_ITEMS / 4; ++c) {
    const uint32_t at = ps_at(4 * c);
    if (at < tn) pl[c] = *reinterpret_cast<const uint2*>(place + t0 + at);  // (has room for whole fours)
  }
  __syncthreads();
  // 1 << lanes lanes per run; the first so many keys of eight runs at once (a
  // loop per run waits for every load in turn: 87 us at 2^24 keys)
  const uint32_t sub = t & ((1u << lanes) - 1u), step = PS_THREADS >> lanes;
  for (uint32_t d0 = t >> lanes; d0 < nd; d0 += 8 * step) {
    uint32_t p[8], v[8];
    bool longer = false;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t d = d0 + i * step < nd ? d0 + i * step : nd - 1;
      const uint32_t e = d0 + i * step < nd ? s_first[d + 1] : 0u, at = s_base[d] + s_first[d] + sub;
      p[i] = s_first[d] + sub;
      longer |= p[i] + (1u << lanes) < e;
      if (p[i] >= e) p[i] = PS_TILE;
      v[i] = in[d * cap + (p[i] < PS_TILE && at < cap ? at : 0u)];
      if (at >= cap) v[i] = PL_PENDING;
      if (at == cap && p[i] < PS_TILE) *crowded = 1u;  // (one tile has the group's first key too many)
    }
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i)
      if (p[i] < PS_TILE) s_ans[p[i]] = v[i];
    if (__ballot(longer)) {
#pragma unroll 1
      for (uint32_t i = 0; i < 8; ++i) {
        const uint32_t d = d0 + i * step;
        if (d >= nd) break;
        const uint32_t e = s_first[d + 1], b = s_base[d];
        for (uint32_t z = s_first[d] + sub + (1u << lanes); z < e; z += 1u << lanes) {
          const uint32_t at = b + z;
          s_ans[z] = at < cap ? in[d * cap + at] : PL_PENDING;
          if (at == cap) *crowded = 1u;
        }
      }
    }
  }
  __syncthreads();
  bool pending = false;
#pragma unroll
  for (uint32_t c = 0; c < PS_ITEMS / 4; ++c) {
    const uint32_t at = ps_at(4 * c);
    if (at >= tn) continue;
    uint32_t a[4] = {s_ans[pl[c].x & 0x7FFFu], s_ans[(pl[c].x >> 16) & 0x7FFFu], s_ans[pl[c].y & 0x7FFFu],
                     s_ans[(pl[c].y >> 16) & 0x7FFFu]};
    const bool open = a[0] == PL_PENDING || a[1] == PL_PENDING || a[2] == PL_PENDING || a[3] == PL_PENDING;
    if (at + 4 <= tn && !open) {
      st16_dw(out + t0 + at, make_uint4(a[0], a[1], a[2], a[3]));
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k)
        if (at + k < tn && a[k] != PL_PENDING) out[t0 + at + k] = a[k];
    }
    pending |= open;
  }
  if (!pending) return;
  // (out may be keys: those left to walk for are still there)
#pragma unroll 1
  for (uint32_t i = 0; i < PS_ITEMS; ++i) {
    const uint32_t at = ps_at(i);
    if (at < tn && s_ans[place[t0 + at]] == PL_PENDING) out[t0 + at] = direct(keys[t0 + at]);
  }
}

// ---------------------------------------------------------------- host
// After the call: a stream whose keys crowd into few groups, or whose walks
// are long, takes the direct walk for its next calls.
static inline void pl_report(DeviceState& ds, LocalKind k) {
  lw_report(ds, k, *static_cast<volatile uint32_t*>(ds.h_local) == 0);
}
// walks(gsize, cap, io, steps) launches the walks of all groups; steps: a
// cleared word of 64 bits.  No host wait.
template <bool WIDE, typename Walk, typename F>
static gqf_status pl_lookup(hipStream_t s, DeviceState& ds, const PlPlan& o, const uint32_t* keys, uint32_t fp_bits,
                            uint32_t n, uint32_t* out, const Walk& direct, F walks) {
  const PsPlan& p = o.p;
  const uint32_t nd = p.ngroups, bits = p.shift + p.gb, hbits = bits > 32 ? bits - 32 : 0u;
  Arena ar(ds.ws, ds.ws_cap);
  uint32_t* mid = ar.take<uint32_t>((size_t)nd * p.cap);
  uint32_t* gsize = ar.take<uint32_t>(nd + 2);
  uint16_t* place = ar.take<uint16_t>((size_t)n + 4);
  uint32_t* tbase = ar.take<uint32_t>((size_t)o.tiles * nd);
  uint16_t* tfirst = ar.take<uint16_t>((size_t)o.tiles * nd);
  if (ar.used > ar.cap) {
    set_error("internal: lookup workspace overflow");
    return GQF_ERR_INVALID;
  }
  *ds.h_local = 0;
  GQF_LAUNCH(k_ps_reset, dim3(1), dim3(PS_THREADS), 0, s, gsize, nd + 2, ds.counters);
  GQF_LAUNCH_B((double)n * 10.0, (k_ps_scatter<WIDE, true>), dim3(p.wgs), dim3(PS_THREADS), 0, s, keys, n, fp_bits,
               p.shift, nd, hbits, p.tile, p.cap, gsize, mid, ds.counters, PsBack{place, tbase, tfirst});
  walks(gsize, p.cap, mid, reinterpret_cast<unsigned long long*>(gsize + nd));
  GQF_LAUNCH_B((double)n * 10.0, (k_pl_gather<Walk>), dim3(o.tiles), dim3(PS_THREADS), 0, s, direct, keys, n, nd, p.tile,
               p.cap, o.lanes, tbase, tfirst, place, mid, out, ds.d_local);
  return GQF_OK;
}

}  // namespace gqf
