// gqf_rsqf_local.hpp -- localized inserts and deletes of the RSQF: the plan
// and apply kernels over 4096-slot windows (see gqf_local.hpp), and the
// update of one region by one lane.
//
// With D(s) the runs of quotients below s that end at or after slot s (the
// occupied bits before s less the run ends before s), slot s is empty iff
// D(s) = 0 and its quotient is not occupied, and a boundary (no entry of a
// smaller quotient at or after it) iff D(s) = 0.  The plan derives D from
// counts over the whole table, so it does not rely on the 8-bit offsets; per
// batch key it leaves D at the key's quotient, from which its region is
// decoded, and per window the empty slots.
//   One wave per window: 2^18 keys into q=26 r=8 at fill 0.8 take 77 us
// (every window has keys: 100 MB of table read, the changed blocks written),
// plan and counts 35; rewriting every window takes 264 and 68 us.  Bound by
// the dependent LDS reads of the longest region of each wave.
#pragma once

#include "gqf_local.hpp"

namespace gqf {

// Blocks of the next window that a region may reach.  45: 10,204 bytes of LDS
// per deleting wave, 16 of them per CU (48: 15; steps of 2^18 keys 339 us, now
// 330).
constexpr uint32_t RL_HALO = 45;
constexpr uint32_t RL_BLOCKS = 64 + RL_HALO;
constexpr uint32_t RL_E_BITS = 13;  // a key's word: E_k or the head bit, D above

// ---------------------------------------------------------------- one key
// A window and the blocks after it that its last region reaches: occupied
// and run-end bits and the remainder bit string (slot s at bits [s r, s r +
// r)).  Regions may share words: a lane changes bits of its own region only,
// by xor.  Slots are relative to the window.  R: r at compile time, or 0.
template <int R>
struct RlPlanes {
  using U = unsigned long long;
  U *occ, *ends, *rem;
  const U* empty;  // insert: the slots that were empty before the batch
  int32_t* off;    // changes of the blocks' offsets
  uint32_t end, r;
  uint64_t dirty[2];

  __host__ __device__ __forceinline__ uint32_t rb() const { return R ? (uint32_t)R : r; }
  __host__ __device__ __forceinline__ static uint64_t upto(uint32_t i) { return (2ull << i) - 1ull; }
  __host__ __device__ __forceinline__ static uint64_t from(uint32_t i) { return ~0ull << i; }
  __host__ __device__ __forceinline__ void mark(uint32_t b0, uint32_t b1) {
    if (b0 < 64) dirty[0] |= from(b0) & (b1 < 63 ? upto(b1) : ~0ull);
    if (b1 >= 64) dirty[1] |= upto(b1 - 64) & (b0 > 64 ? from(b0 - 64) : ~0ull);
  }
  __host__ __device__ __forceinline__ uint32_t get_rem(uint32_t s) const {
    const uint32_t bit = s * rb(), w = bit >> 6, o = bit & 63;
    uint64_t v = rem[w] >> o;
    if (o + rb() > 64) v |= (uint64_t)rem[w + 1] << (64 - o);
    return (uint32_t)v & ((1u << rb()) - 1u);
  }
  // The first set bit of m at or after slot s; end if none is held.
  __host__ __device__ __forceinline__ uint32_t next(const U* m, uint32_t s) const {
    if (s >= end) return end;
    uint32_t w = s >> 6;
    uint64_t x = m[w] & from(s & 63);
    while (!x) {
      if (++w >= end / 64) return end;
      x = m[w];
    }
    return 64 * w + (uint32_t)__builtin_ctzll(x);
  }
  // The k-th run end (k >= 1) at or after slot a, and the one before it
  // (*prev; a - 1 when k = 1); end if it is not held.
  __host__ __device__ __forceinline__ uint32_t run_end(uint32_t a, uint32_t k, uint32_t* prev) const {
    uint32_t w = a >> 6, last = a - 1;
    uint64_t x = ends[w] & from(a & 63);
    for (;;) {
      const uint32_t c = (uint32_t)__builtin_popcountll(x);
      if (c >= k) break;
      k -= c;
      if (x) last = 64 * w + 63 - (uint32_t)__builtin_clzll(x);
      if (++w >= end / 64) return end;
      x = ends[w];
    }
    const uint32_t b = select_bit64(x, k);
    const uint64_t low = x & ((1ull << b) - 1ull);
    *prev = low ? 64 * w + 63 - (uint32_t)__builtin_clzll(low) : last;
    return 64 * w + b;
  }
  // Occupied quotients of [a, b).
  __host__ __device__ __forceinline__ uint32_t occupied(uint32_t a, uint32_t b) const {
    uint32_t c = 0;
    for (uint32_t w = a >> 6; w <= b >> 6 && w < end / 64; ++w) {
      uint64_t x = occ[w];
      if (w == a >> 6) x &= from(a & 63);
      if (w == b >> 6) x &= ~from(b & 63);
      c += (uint32_t)__builtin_popcountll(x);
    }
    return c;
  }

  // Inserts (fq, fr), which takes the empty slot e.  a, D: the region's first
  // quotient and the runs open there.
  __host__ __device__ __forceinline__ void insert(uint32_t fq, uint32_t fr, uint32_t a, uint32_t D, uint32_t e) {
    const uint32_t fw = fq >> 6, ew = e >> 6;
    const bool stored = (occ[fw] >> (fq & 63)) & 1ull;
    const uint32_t t = D + occupied(a, fq) + (stored ? 1u : 0u);
    uint32_t p = fq, y = fq;  // the slot, and where its run-end bit comes in
    if (t) {
      uint32_t prev;
      const uint32_t x = run_end(a, t, &prev);
      if (x >= e && x >= end) return;  // not reached: the region is held
      if (stored) {
        const uint32_t start = (int32_t)prev >= (int32_t)fq ? prev + 1 : fq;
        for (p = x + 1; p > start && get_rem(p - 1) > fr;) --p;
        y = x;
      } else {
        if (x + 1 > p) p = x + 1;
        y = p;
      }
    }
    if (p > e || y > e || e >= end) return;  // not reached: the region is held
    if (!stored) lw_xor(&occ[fw], 1ull << (fq & 63));
    // run ends of [y, e]: those of [y, e) move up by one; slot y ends a run
    // iff the quotient is new
    uint64_t top = 0;
    for (uint32_t w = y >> 6; w <= ew; ++w) {
      uint64_t reg = ~0ull;
      const uint64_t old = ends[w];
      uint64_t v = (old << 1) | top;
      top = old >> 63;
      if (w == y >> 6) {
        reg = from(y & 63);
        v = (v & ~(1ull << (y & 63))) | ((stored ? 0ull : 1ull) << (y & 63));
      }
      if (w == ew) reg &= upto(e & 63);
      lw_xor(&ends[w], (old ^ v) & reg);
    }
    // remainders of [p, e]
    const uint32_t b0 = p * rb(), b1 = (e + 1) * rb() - 1, i0 = b0 >> 6, i1 = b1 >> 6, o = b0 & 63;
    uint64_t in = 0;
    for (uint32_t i = i0; i <= i1; ++i) {
      const uint64_t old = rem[i];
      uint64_t v, mask = ~0ull;
      if (i == i0) {
        mask = from(o);
        v = ((old & mask) << rb()) | ((uint64_t)fr << o);
        in = ((old & mask) >> (64 - rb())) | (o + rb() > 64 ? (uint64_t)fr >> (64 - o) : 0ull);
      } else {
        v = (old << rb()) | in;
        in = old >> (64 - rb());
      }
      if (i == i1) mask &= upto(b1 & 63);
      if (mask == ~0ull) rem[i] = v;
      else lw_xor(&rem[i], (old ^ v) & mask);
    }
    // entries of quotients below their first slots: one more in these blocks
    for (uint32_t j = fw + 1; j <= ew; ++j) off[j] += 1;
    mark(fw, ew);
  }

  // Removes one copy of (fq, fr) if it is stored.
  __host__ __device__ __forceinline__ void erase(uint32_t fq, uint32_t fr, uint32_t a, uint32_t D) {
    const uint32_t fw = fq >> 6;
    if (!((occ[fw] >> (fq & 63)) & 1ull)) return;
    uint32_t prev;
    const uint32_t x = run_end(a, D + occupied(a, fq) + 1, &prev);
    if (x >= end) return;  // not reached
    const uint32_t start = (int32_t)prev >= (int32_t)fq ? prev + 1 : fq;
    uint32_t p = x;
    while (p > start && get_rem(p) > fr) --p;
    if (get_rem(p) != fr) return;
    // l: the last slot of the entries that move back, the first from x on
    // where no run is open: the occupied quotients of (fq, l] are as many as
    // the run ends of (x, l].  Their difference falls only at run ends on
    // unoccupied slots, so 16 slots with fewer of those are passed at once.
    uint32_t l = x;
    int32_t open = (int32_t)occupied(fq + 1, x + 1);
    if (open) {
      l = end - 1;
      uint32_t s = x + 1;
      for (bool found = false; !found && s < end; s = (s | 15u) + 1) {
        const uint32_t sh = s & 48, m = 0xFFFFu & (0xFFFFu << (s & 15));
        const uint32_t oc = (uint32_t)(occ[s >> 6] >> sh) & m, en = (uint32_t)(ends[s >> 6] >> sh) & m;
        if (open <= (int32_t)__builtin_popcount(en & ~oc)) {
          for (uint32_t c = en; c; c &= c - 1u) {
            const uint32_t up = c ^ (c - 1u);
            if (open + (int32_t)__builtin_popcount(oc & up) == (int32_t)__builtin_popcount(en & up)) {
              l = (s & ~15u) + (uint32_t)__builtin_ctz(c);
              found = true;
              break;
            }
          }
        }
        open += (int32_t)__builtin_popcount(oc) - (int32_t)__builtin_popcount(en);
      }
    }
    const uint32_t lw = l >> 6;
    // run ends of [start, l]: one entry fewer in the run, or no run
    for (uint32_t w = start >> 6; w <= lw; ++w) {
      uint64_t reg = ~0ull;
      const uint64_t old = ends[w];
      uint64_t v = old >> 1;
      if (w == start >> 6) reg = from(start & 63);
      if (w < lw) {
        v |= (uint64_t)ends[w + 1] << 63;
      } else {
        v &= ~(1ull << (l & 63));
        reg &= upto(l & 63);
      }
      lw_xor(&ends[w], (old ^ v) & reg);
    }
    if (start == x) lw_xor(&occ[fw], 1ull << (fq & 63));
    // remainders of [p, l]; slot l's becomes 0
    const uint32_t b0 = p * rb(), bl = l * rb(), b1 = bl + rb() - 1, i0 = b0 >> 6, i1 = b1 >> 6;
    for (uint32_t i = i0; i <= i1; ++i) {
      const uint64_t old = rem[i];
      uint64_t v = old >> rb(), mask = i == i0 ? from(b0 & 63) : ~0ull;
      if (i < i1) v |= (uint64_t)rem[i + 1] << (64 - rb());
      if (i == i1) mask &= upto(b1 & 63);
      if (64 * i + 63 >= bl) v = 64 * i >= bl ? 0ull : v & ~from(bl & 63);
      if (mask == ~0ull) rem[i] = v;
      else lw_xor(&rem[i], (old ^ v) & mask);
    }
    for (uint32_t j = fw + 1; j <= lw; ++j) off[j] -= 1;
    mark(fw, lw);
  }
};

// ---------------------------------------------------------------- plan
// Window w's occupied quotients less its run ends (dw) and their sums over
// groups of 64 windows (gs), 64 windows per workgroup; the windows' ranges of
// the sorted batch (bstart).
template <typename K>
__global__ __launch_bounds__(1024) void k_rl_pop(const uint64_t* __restrict__ meta, uint32_t nb, uint32_t W,
                                                 const K* __restrict__ B, uint32_t n, uint32_t r,
                                                 uint32_t* __restrict__ bstart, uint32_t* __restrict__ dw,
                                                 uint32_t* __restrict__ gs) {
  __shared__ uint32_t s_sum[16];
  const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6, w0 = blockIdx.x * 64 + 4 * wid;
  uint4 x[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t b = (w0 + i) * 64 + lane;
    x[i] = b < nb ? reinterpret_cast<const uint4*>(meta)[2 * (size_t)b] : make_uint4(0u, 0u, 0u, 0u);
  }
  {
    const uint32_t w = w0 + lane / 8;
    const bool on = lane < 32 && w < W;
    const uint64_t key = ((uint64_t)w * LW_SLOTS) << r;
    const uint32_t b = group8_search(0u, on ? n : 0u, [&](uint32_t m) { return (uint64_t)B[m] < key; });
    if (on && (lane & 7) == 0) bstart[w] = b;
    if (blockIdx.x == 0 && threadIdx.x == 0) bstart[W] = n;
  }
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t d = wave_read(wave_incl_add((uint32_t)__popc(x[i].x) + (uint32_t)__popc(x[i].y) -
                                               (uint32_t)__popc(x[i].z) - (uint32_t)__popc(x[i].w)), 63);
    if (lane == 0 && w0 + i < W) dw[w0 + i] = d;
    sum += d;
  }
  if (lane == 0) s_sum[wid] = sum;
  __syncthreads();
  if (wid == 0) {
    const uint32_t a = wave_read(wave_incl_add(lane < 16 ? s_sum[lane] : 0u), 63);
    if (lane == 0) gs[blockIdx.x] = a;
  }
}

// One wave per window, a lane per block.  dw, gs: from k_rl_pop.  key[i]:
// insert E_k within the window, delete 1 iff a boundary of the window lies
// after the key before it and at or before it; D above (RL_E_BITS).  Insert: empty[block] of the windows
// read; delete: fb[w] = the window's first boundary (LW_SLOTS: none).
template <typename K, bool INS>
__global__ __launch_bounds__(64) void k_rl_plan(const uint64_t* __restrict__ meta, uint32_t nb, uint32_t r,
                                                const uint32_t* __restrict__ dw, const uint32_t* __restrict__ gs,
                                                const K* __restrict__ B, const uint32_t* __restrict__ bstart, uint32_t W,
                                                uint32_t* __restrict__ key, uint64_t* __restrict__ empty,
                                                uint16_t* __restrict__ fb, uint4* __restrict__ st, uint32_t budget) {
  __shared__ uint64_t s_mask[64], s_occ[64], s_end[64];
  __shared__ uint32_t s_pre[64];
  __shared__ int32_t s_D[64];
  const uint32_t w = blockIdx.x, lane = threadIdx.x;
  const uint32_t b0 = bstart[w], nk = bstart[w + 1] - b0;
  const uint32_t base = w * LW_SLOTS;
  const bool after = w > 0 && bstart[w - 1] != b0;  // the window before has keys
  if (nk == 0 && !after) {
    // not read: what overflows into it is absorbed by the window before, and
    // a boundary of that window separates keys on both sides
    if (lane == 0) {
      st[w] = lw_pack(LW{-LW_SPILL, 0, base + 1, 0u});
      if (!INS) fb[w] = 0;
    }
    return;
  }
  const uint32_t blk = w * 64 + lane;
  uint64_t occ = 0, end = 0;
  if (blk < nb) {
    const uint4 x = reinterpret_cast<const uint4*>(meta)[2 * (size_t)blk];
    occ = ((uint64_t)x.y << 32) | x.x;
    end = ((uint64_t)x.w << 32) | x.z;
  }
  const uint32_t step = (uint32_t)__popcll(occ) - (uint32_t)__popcll(end);
  // runs that begin before the window's quotients' and end in or past it: the
  // sums of the 64-window groups before, and of the windows of its own
  uint32_t d = (w & ~63u) + lane < w ? dw[(w & ~63u) + lane] : 0u;
  for (uint32_t i = lane; i < w / 64; i += 64) d += gs[i];
  d = wave_read(wave_incl_add(d), 63);
  int32_t D = (int32_t)(d + wave_incl_add(step) - step);
  s_occ[lane] = occ;
  s_end[lane] = end;
  s_D[lane] = D;
  // insert: the empty slots; delete: the boundaries
  uint64_t mask = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t o = (uint32_t)(occ >> (32 * h)), e = (uint32_t)(end >> (32 * h));
    uint32_t m = 0;
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      if (!INS) m |= (D <= 0 ? 1u : 0u) << s;
      D += (int32_t)((o >> s) & 1u);
      if (INS) m |= (D <= 0 ? 1u : 0u) << s;
      D -= (int32_t)((e >> s) & 1u);
    }
    mask |= (uint64_t)m << (32 * h);
  }
  if (blk >= nb) mask = 0;
  s_mask[lane] = mask;
  const uint64_t nz = __ballot(mask != 0);
  uint32_t e = 0, first = LW_SLOTS, last = 0;
  int32_t held = 1 << 20;  // insert: empty slots of the blocks that the window before may hold (a short last window: all)
  bool bad = nk > LW_KEYS;
  if (INS) {
    if (blk < nb) empty[blk] = mask;
    const uint32_t c = (uint32_t)__popcll(mask), inc = wave_incl_add(c);
    s_pre[lane] = inc - c;
    e = wave_read(inc, 63);
    if (w + 1 < W) bad = bad || e < (uint32_t)LW_SPILL;
    if (nb > w * 64 + RL_HALO) held = (int32_t)wave_read(inc, RL_HALO - 1);
  } else {
    const uint32_t own = mask ? 64 * lane + 64 - (uint32_t)__clzll(mask) : 0u;
    const uint32_t inc = wave_incl_max(own);
    s_pre[lane] = dpp_u32<DPP_WAVE_SHR1>(0u, inc);
    last = wave_read(inc, 63);
    if (nz) {
      const uint32_t fl = (uint32_t)__builtin_ctzll(nz);
      const uint32_t lo = wave_read((uint32_t)mask, (int)fl), hi = wave_read((uint32_t)(mask >> 32), (int)fl);
      first = 64 * fl + (uint32_t)__builtin_ctzll(((uint64_t)hi << 32) | lo);
    }
    bad = bad || first == LW_SLOTS;
  }
  __syncthreads();
  int32_t M = 0, fit = held - (int32_t)nk;
  uint32_t heads = 0, last_key = 0;  // delete: 1 + the window's last key (0: none)
  LwChain<INS> chain(lw_key_rsqf<INS>(r), nz, e);
  if (nk <= LW_KEYS) {
    uint32_t prev = 0;  // delete: 1 + the key before the group (0: none)
    const K kbase = (K)base << r;
    for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
      const uint32_t k = k0 + lane;
      const bool on = k < nk;
      const uint32_t rel = on ? (uint32_t)((B[b0 + k] - kbase) >> r) & (LW_SLOTS - 1) : 0u;
      const uint32_t bk = rel >> 6;
      const uint64_t below = (1ull << (rel & 63u)) - 1ull, m = s_mask[bk];
      const int32_t Dk = s_D[bk] + (int32_t)__popcll(s_occ[bk] & below) - (int32_t)__popcll(s_end[bk] & below);
      if (on && (Dk < 0 || Dk >= (1 << (32 - RL_E_BITS)))) bad = true;  // not a valid table, or a very long run
      bool head;
      uint32_t info;
      if (INS) {
        info = s_pre[bk] + (uint32_t)__popcll(m & below);
        const int32_t v = (int32_t)info - (int32_t)k, f = lw_fit(v, held, (int32_t)k);
        if (on && f > fit) fit = f;
        head = lw_insert_head(v, on, M);
      } else {
        const uint64_t at = m & (below | (1ull << (rel & 63u)));
        const uint32_t lb = at ? 64 * bk + 64 - (uint32_t)__clzll(at) : s_pre[bk];
        uint32_t p = dpp_u32<DPP_WAVE_SHR1>(0u, rel + 1);
        if (lane == 0) p = prev;
        prev = wave_read(rel + 1, 63);
        last_key = wave_read(rel + 1, (int)((nk - 1 - k0) & 63u));
        head = on && lb > p;
        info = head ? 1u : 0u;
      }
      if (on) key[b0 + k] = info | ((uint32_t)Dk << RL_E_BITS);
      const uint64_t hm = __ballot(head);
      heads += (uint32_t)__popcll(hm);
      if (k0 + 64 <= nk && hm == 0) bad = true;
    }
    if (nk && chain.may(nk, heads, budget)) {
      int32_t M2 = 0;
      for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
        const uint32_t k = k0 + lane;
        const bool on = k < nk;
        const uint32_t rel = on ? (uint32_t)((B[b0 + k] - kbase) >> r) & (LW_SLOTS - 1) : 0u;
        const uint32_t x = on ? key[b0 + k] & ((1u << RL_E_BITS) - 1u) : 0u;
        const bool head = INS ? lw_insert_head((int32_t)x - (int32_t)k, on, M2) : on && x != 0;
        chain.add(on, s_mask[rel >> 6], rel & 63u, rel >> 6, head, __ballot(head));
      }
    }
  }
  bad = __any(bad || chain.longest > budget);
  if (INS) fit = lw_wave_max(fit);
  if (lane == 0) {
    const int32_t a = INS ? (int32_t)nk - (int32_t)e : -2;
    int32_t b = INS ? (nk ? M + a : 0) : last <= last_key;
    if (b < 0) b = 0;
    if (bad) b = LW_BAD;
    const uint32_t lb = INS ? lw_room(fit) : (last ? base + last : 0u) | (first > 64 * RL_HALO ? LW_FAR : 0u);
    st[w] = lw_pack(LW{a, b, lb, heads});
    if (!INS) fb[w] = (uint16_t)first;
  }
}

// ---------------------------------------------------------------- apply
template <typename K, int R, bool INS>
__global__ __launch_bounds__(64) void k_rl_apply(uint64_t* __restrict__ meta, uint64_t* __restrict__ remg, uint32_t nb,
                                                 uint32_t r, const K* __restrict__ B, uint32_t n,
                                                 const uint32_t* __restrict__ bstart, uint32_t W,
                                                 const uint2* __restrict__ pre, const uint32_t* __restrict__ key,
                                                 const uint64_t* __restrict__ empty, const uint16_t* __restrict__ fb,
                                                 const uint32_t* __restrict__ ctr) {
  using U = unsigned long long;
  constexpr uint32_t RW = R ? R : 16;  // remainder words per block, at most
  __shared__ U s_rem[RL_BLOCKS * RW + 1];
  __shared__ U s_occ[RL_BLOCKS], s_end[RL_BLOCKS], s_empty[INS ? RL_BLOCKS : 1];
  __shared__ int32_t s_off[RL_BLOCKS];
  __shared__ uint16_t s_head[LW_KEYS];
  __shared__ uint32_t s_dirty[4];
  const uint32_t w = blockIdx.x, lane = threadIdx.x, rr = R ? (uint32_t)R : r;
  const uint32_t b0 = bstart[w], b1 = bstart[w + 1], nk = b1 - b0;
  if (nk == 0 || nk > LW_KEYS || ctr[CTR_MISC]) return;
  const uint32_t base = w * LW_SLOTS, bw = w * 64;
  const K kbase = (K)base << rr;
  // block i of the window: metadata (a lane each)
  auto load = [&](uint32_t i) {
    uint64_t o = 0, e = 0, m = 0;
    if (bw + i < nb) {
      const uint4 x = reinterpret_cast<const uint4*>(meta)[2 * (size_t)(bw + i)];
      o = ((uint64_t)x.y << 32) | x.x;
      e = ((uint64_t)x.w << 32) | x.z;
      if (INS) m = empty[bw + i];
    }
    s_occ[i] = o;
    s_end[i] = e;
    if (INS) s_empty[i] = m;
    s_off[i] = 0;
  };
  load(lane);
#pragma unroll 8
  for (uint32_t k = 0; k < rr; ++k) {
    const uint32_t i = k * 64 + lane;  // word of the window
    const uint64_t at = (uint64_t)bw * rr + i;
    s_rem[i] = at < (uint64_t)nb * rr ? remg[at] : 0ull;
  }
  if (lane < 4) s_dirty[lane] = 0u;
  // heads
  const uint2 pw = pre[w];
  const uint32_t fbw = INS ? 0u : fb[w];
  uint32_t nh = 0;
  int32_t M = (int32_t)pw.x;
  for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
    const uint32_t k = k0 + lane;
    const bool on = k < nk;
    const uint32_t x = on ? key[b0 + k] & ((1u << RL_E_BITS) - 1u) : 0u;
    bool head;
    if (INS) {
      head = lw_insert_head((int32_t)x - (int32_t)k, on, M);
    } else {
      head = on && x != 0;
      // the window's first key, before its first boundary: dependent on the
      // key before it iff no boundary lies between the two
      if (k == 0 && !head) head = b0 == 0 || pw.y > (uint32_t)(B[b0 - 1] >> rr) + 1;
    }
    const uint64_t hm = __ballot(head);
    if (head) s_head[nh + (uint32_t)__popcll(hm & ((1ull << lane) - 1ull))] = (uint16_t)k;
    nh += (uint32_t)__popcll(hm);
  }
  if (nh == 0) return;  // every key belongs to an earlier window's region
  // keys of later windows that the last region takes, and hi: the last slot
  // it may change (relative; inside the window unless it leaves it)
  uint32_t k1 = b1, hi = LW_SLOTS - 1;
  if (INS) {
    uint32_t need = w + 1 < W ? pre[w + 1].x : 0u;
    if (need) {
      uint32_t c = bw + 64;  // block
      uint64_t em = c < nb ? empty[c] : 0ull;
      while ((uint32_t)__popcll(em) < need && c + 1 < nb && c + 1 < bw + RL_BLOCKS) {
        need -= (uint32_t)__popcll(em);
        em = empty[++c];
      }
      for (; need > 1; --need) em &= em - 1ull;
      for (;;) {  // the empty slot that the region's last key takes
        while (em == 0 && c + 1 < nb && c + 1 < bw + RL_BLOCKS) em = empty[++c];
        if (em == 0) break;  // not reached: the scan found room (lw_room)
        hi = 64 * (c - bw) + (uint32_t)__builtin_ctzll(em);
        em &= em - 1ull;
        if (k1 >= n || (uint32_t)(B[k1] >> rr) > base + hi) break;
        ++k1;
      }
    }
  } else {
    uint32_t hp = (uint32_t)(B[b1 - 1] >> rr);
    if (w + 1 < W && fb[w + 1] && pre[w + 1].y <= hp + 1) hi = LW_SLOTS + fb[w + 1] - 1;  // no boundary after the last key
    while (k1 < n) {
      const uint32_t h = (uint32_t)(B[k1] >> rr), w2 = h / LW_SLOTS;
      if (h - w2 * LW_SLOTS >= fb[w2] || pre[w2].y > hp + 1) break;
      hp = h;
      ++k1;
    }
  }
  uint32_t held = hi / 64 + 1;  // blocks held
  if (held > RL_BLOCKS) held = RL_BLOCKS;  // not reached: the scan's bounds
  if (lane < held - 64) load(64 + lane);
  for (uint32_t i = 64 * rr + lane; i < held * rr; i += 64) {
    const uint64_t at = (uint64_t)bw * rr + i;
    s_rem[i] = at < (uint64_t)nb * rr ? remg[at] : 0ull;
  }
  __syncthreads();
  const uint32_t h0 = (uint32_t)((B[b0 + s_head[0]] - kbase) >> rr);
  RlPlanes<R> m;
  m.occ = s_occ;
  m.ends = s_end;
  m.rem = s_rem;
  m.empty = s_empty;
  m.off = s_off;
  m.end = 64 * held;
  m.r = rr;
  m.dirty[0] = m.dirty[1] = 0;
  // the regions
  const uint32_t rmask = (1u << rr) - 1u;
  for (uint32_t ri = lane; ri < nh; ri += 64) {
    const uint32_t ka = b0 + s_head[ri], kb = ri + 1 < nh ? b0 + s_head[ri + 1] : k1;
    const uint32_t a = (uint32_t)((B[ka] - kbase) >> rr), D = key[ka] >> RL_E_BITS;
    uint32_t e = a - 1;
    for (uint32_t k = ka; k < kb; ++k) {
      const uint32_t x = (uint32_t)(B[k] - kbase);
      const uint32_t fq = (uint32_t)((B[k] - kbase) >> rr);
      if (fq >= m.end) break;  // not reached: hi covers the region's keys
      if (INS) {
        e = m.next(s_empty, e + 1);
        m.insert(fq, x & rmask, a, D, e);
      } else {
        m.erase(fq, x & rmask, a, D);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t d = (uint32_t)(m.dirty[k >> 1] >> (32 * (k & 1)));
    if (d) atomicOr(&s_dirty[k], d);
  }
  __syncthreads();
  // the changed blocks: whole, but for the one in which an earlier window's
  // region may end (before the first region) and the one in which the last
  // region ends, whose own slots [lo, hi] change by xor
  const uint32_t lo = (INS ? pw.x > 0 : fbw > 0) ? h0 : 0u;
  auto dirty = [&](uint32_t i) { return (s_dirty[i >> 5] >> (i & 31)) & 1u; };
  auto own = [&](uint32_t i) {  // the block's slots in [lo, hi]
    uint64_t x = ~0ull;
    if (i == lo >> 6) x &= m.from(lo & 63);
    if (i == hi >> 6) x &= m.upto(hi & 63);
    return x;
  };
  for (uint32_t i = lane; i < held; i += 64) {
    if (!dirty(i) || bw + i >= nb) continue;
    uint64_t* rec = meta + 4 * (size_t)(bw + i);
    const uint64_t x = own(i);
    if (x == ~0ull) {
      *reinterpret_cast<uint4*>(rec) = make_uint4((uint32_t)s_occ[i], (uint32_t)(s_occ[i] >> 32), (uint32_t)s_end[i],
                                                  (uint32_t)(s_end[i] >> 32));
    } else {
      lw_xor(reinterpret_cast<U*>(rec), (rec[0] ^ s_occ[i]) & x);
      lw_xor(reinterpret_cast<U*>(rec) + 1, (rec[1] ^ s_end[i]) & x);
    }
    if (s_off[i]) rec[2] = (rec[2] + (uint64_t)(int64_t)s_off[i]) & 0xFFull;
  }
  for (uint32_t i = lane; i < held * rr; i += 64) {
    const uint32_t bk = i / rr;
    if (!dirty(bk) || bw + bk >= nb) continue;
    uint64_t* g = remg + (uint64_t)bw * rr + i;
    uint64_t x = ~0ull;  // the word's bits of the block's own slots
    if (bk == lo >> 6) {
      const uint32_t bit = lo * rr;
      x &= 64 * i + 63 < bit ? 0ull : (64 * i >= bit ? ~0ull : m.from(bit & 63));
    }
    if (bk == hi >> 6) {
      const uint32_t bit = (hi + 1) * rr;  // the first bit past them
      x &= 64 * i >= bit ? 0ull : (64 * i + 64 <= bit ? ~0ull : ~m.from(bit & 63));
    }
    if (x == ~0ull) *g = s_rem[i];
    else if (x) lw_xor(reinterpret_cast<U*>(g), (*g ^ s_rem[i]) & x);
  }
}

}  // namespace gqf
