// gqf_sqf_local.hpp -- localized inserts and deletes of the SQF: the plan and
// apply kernels over 4096-slot windows (see gqf_local.hpp), and the update of
// one region by one lane.
#pragma once

#include "gqf_local.hpp"
#include "gqf_sqf_dev.hpp"

namespace gqf {

// ---------------------------------------------------------------- one key
// An update on single elements: what SlPlanes does on bits, step by step, for
// the checks of the region rules on the CPU.  Both work on any accessor a with
// a.get(slot) (elements at or past the last slot S read as 0) and a.put(slot,
// element), on a canonical table.  Slots before b, the last slot at or before
// fq that is empty or holds an entry at its own quotient, belong to earlier
// quotients' runs and play no part.

// The start of fq's run, or where it would start, given a non-empty slot fq.
template <class A>
__host__ __device__ __forceinline__ uint32_t sl_run_start(A& a, uint32_t S, uint32_t fq) {
  uint32_t b = fq;
  while (b > 0 && (a.get(b) & 1u)) --b;
  uint32_t s = b;
  for (; b < fq; ++b)
    if (a.get(b) & 4u) {
      do {
        ++s;
      } while (s < S && (a.get(s) & 2u));
    }
  return s;
}

// Inserts (fq, fr) unless it is stored.  An empty slot must follow.
template <class A>
__host__ __device__ __forceinline__ void sl_insert(A& a, uint32_t S, uint32_t fq, uint32_t fr) {
  const uint32_t e0 = a.get(fq);
  if ((e0 & 7u) == 0) {
    a.put(fq, (fr << 3) | 4u);
    return;
  }
  uint32_t p = sl_run_start(a, S, fq);
  const bool occ = (e0 & 4u) != 0;
  bool first = true;
  if (occ) {
    uint32_t e = a.get(p);
    for (;;) {
      if ((e >> 3) == fr) return;
      if ((e >> 3) > fr) break;
      ++p;
      first = false;
      e = a.get(p);
      if (!(e & 2u)) break;
    }
  } else {
    a.put(fq, e0 | 4u);  // p > fq: another quotient's entry holds slot fq
  }
  uint32_t carry = (fr << 3) | (first ? 0u : 2u) | (p != fq ? 1u : 0u);
  uint32_t cont = occ && first ? 2u : 0u;  // the run's old first entry continues it
  for (; p < S; ++p) {
    const uint32_t old = a.get(p);
    a.put(p, (old & 4u) | carry);
    if ((old & 7u) == 0) return;
    carry = (old & ~4u) | 1u | cont;
    cont = 0u;
  }
}

// Removes one copy of (fq, fr) if it is stored.
template <class A>
__host__ __device__ __forceinline__ void sl_erase(A& a, uint32_t S, uint32_t fq, uint32_t fr) {
  if (!(a.get(fq) & 4u)) return;
  uint32_t p = sl_run_start(a, S, fq);
  uint32_t e = a.get(p);
  bool first = true;
  while ((e >> 3) != fr) {
    if ((e >> 3) > fr || p + 1 >= S) return;
    ++p;
    first = false;
    e = a.get(p);
    if (!(e & 2u)) return;
  }
  uint32_t nx = a.get(p + 1);
  const bool single = first && !(nx & 2u);
  bool heir = first && !single;  // the next entry becomes the run's first
  uint32_t qcur = fq;
  while (nx & 1u) {  // an entry away from its quotient moves back one slot
    uint32_t el = nx & ~4u;
    if (heir) {
      el &= ~2u;
      if (p == fq) el &= ~1u;
      heir = false;
    } else if (!(nx & 2u)) {
      // a run start: the next occupied quotient's
      do {
        ++qcur;
      } while (qcur < S && !(a.get(qcur) & 4u));
      if (qcur == p) el &= ~1u;
    }
    a.put(p, (a.get(p) & 4u) | el);
    ++p;
    nx = a.get(p + 1);
  }
  a.put(p, a.get(p) & 4u);
  if (single) a.put(fq, a.get(fq) & ~4u);
}

// Blocks of the next window that a region may reach: 7.6 KB of LDS, 21 waves
// per CU (16: 8.1 KB; 2^20-key steps 309 us, 11: 300).
constexpr uint32_t SL_HALO = 11;
constexpr uint32_t SL_BLOCKS = 64 + SL_HALO;

// ---------------------------------------------------------------- plan
// One wave per window.  Insert: el[i] = E_k within the window of batch key i,
// the state (a, b).  Delete: el[i] = 1 iff a boundary of the window lies
// after the key before it in the window (or after the window's start) and at
// or before it, fb[w] = the window's first boundary (LW_SLOTS: none), the
// state's last boundary.
template <int BPE, bool INS>
__global__ __launch_bounds__(64) void k_sl_plan(const uint8_t* __restrict__ t, uint32_t S, uint32_t r,
                                                const uint32_t* __restrict__ B, uint32_t n,
                                                uint32_t* __restrict__ bstart, uint32_t W, uint16_t* __restrict__ el,
                                                uint16_t* __restrict__ fb, uint4* __restrict__ st, uint32_t budget) {
  __shared__ uint64_t s_mask[64];
  __shared__ uint16_t s_pre[64];
  const uint32_t w = blockIdx.x, lane = threadIdx.x;
  uint32_t bp, b0, nk;
  lw_bounds(B, n, r, w, &bp, &b0, &nk);
  nk -= b0;
  if (lane == 0) {
    bstart[w] = b0;
    if (w + 1 == W) bstart[W] = b0 + nk;
  }
  const uint32_t base = w * LW_SLOTS;
  if (nk == 0 && (w == 0 || bp == b0)) {
    // not read: what overflows into it is absorbed by the window before, and
    // a boundary of that window separates keys on both sides
    if (lane == 0) {
      st[w] = lw_pack(LW{-LW_SPILL, 0, base + 1, 0u});
      if (!INS) fb[w] = 0;
    }
    return;
  }
  SqfWin<BPE> x;
  sqf_win_load<BPE>(t, S, w * 64 + lane, x);
  const uint32_t s0 = base + 64 * lane;
  const uint64_t valid = s0 + 64 <= S ? ~0ull : (s0 < S ? (1ull << (S - s0)) - 1ull : 0ull);
  const uint64_t mask = (INS ? ~(x.occ | x.cont | x.shf) : ~x.shf) & valid;
  s_mask[lane] = mask;
  const uint64_t nz = __ballot(mask != 0);
  uint32_t e = 0, first = LW_SLOTS, last = 0;
  int32_t held = 1 << 20;  // empty slots of the blocks that the window before may hold (a short last window: all)
  if (INS) {
    const uint32_t c = (uint32_t)__popcll(mask), inc = wave_incl_add(c);
    s_pre[lane] = (uint16_t)(inc - c);
    e = wave_read(inc, 63);
    if (base + 64 * SL_HALO < S) held = (int32_t)wave_read(inc, SL_HALO - 1);
  } else {
    // 1 + the last boundary before each 64-slot block
    const uint32_t own = mask ? 64 * lane + 64 - (uint32_t)__clzll(mask) : 0u;
    const uint32_t inc = wave_incl_max(own);
    s_pre[lane] = (uint16_t)dpp_u32<DPP_WAVE_SHR1>(0u, inc);
    last = wave_read(inc, 63);
    if (nz) {
      const uint32_t fl = (uint32_t)__builtin_ctzll(nz);
      const uint32_t lo = wave_read((uint32_t)mask, (int)fl), hi = wave_read((uint32_t)(mask >> 32), (int)fl);
      first = 64 * fl + (uint32_t)__builtin_ctzll(((uint64_t)hi << 32) | lo);
    }
  }
  __syncthreads();
  bool bad = nk > LW_KEYS || (INS ? e < (uint32_t)LW_SPILL && w + 1 < W : first == LW_SLOTS);
  int32_t M = 0, fit = held - (int32_t)nk;
  uint32_t heads = 0, end = 0;  // delete: 1 + the window's last key (0: none)
  LwChain<INS> chain(lw_key_sqf<INS>(BPE), nz, e);
  if (!bad) {
    uint32_t prev = 0;  // delete: 1 + the key before the group (0: none)
    for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
      const uint32_t k = k0 + lane;
      const bool on = k < nk;
      const uint32_t rel = on ? (B[b0 + k] >> r) - base : 0u;
      const uint32_t blk = (rel >> 6) & 63u;
      const uint64_t m = s_mask[blk];
      bool head;
      if (INS) {
        const uint32_t E = s_pre[blk] + (uint32_t)__popcll(m & ((1ull << (rel & 63u)) - 1ull));
        if (on) el[b0 + k] = (uint16_t)E;
        const int32_t v = (int32_t)E - (int32_t)k, f = lw_fit(v, held, (int32_t)k);
        if (on && f > fit) fit = f;
        head = lw_insert_head(v, on, M);
      } else {
        const uint64_t at = m & ((2ull << (rel & 63u)) - 1ull);
        const uint32_t lb = at ? 64 * blk + 64 - (uint32_t)__clzll(at) : s_pre[blk];
        uint32_t p = dpp_u32<DPP_WAVE_SHR1>(0u, rel + 1);
        if (lane == 0) p = prev;
        prev = wave_read(rel + 1, 63);
        end = wave_read(rel + 1, (int)((nk - 1 - k0) & 63u));
        head = on && lb > p;  // boundary lb - 1 after the key p - 1
        if (on) el[b0 + k] = head ? 1 : 0;
      }
      const uint64_t hm = __ballot(head);
      heads += (uint32_t)__popcll(hm);
      if (k0 + 64 <= nk && hm == 0) bad = true;
    }
    if (nk && chain.may(nk, heads, budget)) {
      int32_t M2 = 0;
      for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
        const uint32_t k = k0 + lane;
        const bool on = k < nk;
        const uint32_t rel = on ? (B[b0 + k] >> r) - base : 0u, x = on ? el[b0 + k] : 0u;
        const bool head = INS ? lw_insert_head((int32_t)x - (int32_t)k, on, M2) : on && x != 0;
        chain.add(on, s_mask[(rel >> 6) & 63u], rel & 63u, (rel >> 6) & 63u, head, __ballot(head));
      }
      if (__any(chain.longest > budget)) bad = true;
    }
  }
  if (INS) fit = lw_wave_max(fit);
  if (lane == 0) {
    const int32_t a = INS ? (int32_t)nk - (int32_t)e : -2;
    int32_t b = INS ? (nk ? M + a : 0) : last <= end;
    if (b < 0) b = 0;
    if (bad) b = LW_BAD;
    const uint32_t lb = INS ? lw_room(fit) : (last ? base + last : 0u) | (first > 64 * SL_HALO ? LW_FAR : 0u);
    st[w] = lw_pack(LW{a, b, lb, heads});
    if (!INS) fb[w] = (uint16_t)first;
  }
}

// ---------------------------------------------------------------- apply
// A window and the slots after it that its last region reaches (up to
// SL_HALO 64-slot blocks), held as bit planes and remainders: a run is found
// with popcounts and selects, and an update moves 64 flags or 64 / (8 BPE)
// remainders per step.  Regions may share a word of a plane or of the
// remainders: a lane changes bits of its own region only, by xor.  Slots are
// relative to the window.
//   One wave per window: a batch of 1/64 of the slots has a region for most
// lanes, and 8 KB of LDS leave room for 21 waves per CU.  The time is the
// wave's longest region (dependent LDS reads) times the waves per CU: 2^20
// keys into q=26 r=5 at fill 0.75 take 77 us, 559 us when the lanes walked
// element bytes one by one (1.9 and 0.26 TB/s of table bytes read and
// written); the rebuild's decode, state and write passes take 250 us.  As
// many deletes take 104 us, 160 when every run start that moves was paired
// with its quotient one by one; decode, mark and rebuild take 290 us.

template <int BPE>
struct SlPlanes {
  using E = typename std::conditional<BPE == 1, uint8_t, uint16_t>::type;
  using U = unsigned long long;
  static constexpr uint32_t RB = 8 * BPE;  // bits per remainder
  static constexpr uint32_t PW = 64 / RB;  // remainders per word
  U *occ, *cont, *shf, *rem;
  uint32_t end;       // slots held
  uint32_t pend;      // runs of quotients before the window that start in it
  uint64_t dirty[2];  // blocks changed

  __host__ __device__ __forceinline__ static uint64_t upto(uint32_t i) { return (2ull << i) - 1ull; }  // bits 0..i
  __host__ __device__ __forceinline__ static uint64_t from(uint32_t i) { return ~0ull << i; }
  __host__ __device__ __forceinline__ void mark(uint32_t b0, uint32_t b1) {  // blocks b0..b1
    if (b0 < 64) dirty[0] |= from(b0) & (b1 < 63 ? upto(b1) : ~0ull);
    if (b1 >= 64) dirty[1] |= upto(b1 - 64) & (b0 > 64 ? from(b0 - 64) : ~0ull);
  }
  // (memcpy: the same words are read and written whole)
  __host__ __device__ __forceinline__ uint32_t get_rem(uint32_t s) const {
    E v;
    __builtin_memcpy(&v, reinterpret_cast<const char*>(rem) + s * BPE, BPE);
    return v;
  }
  __host__ __device__ __forceinline__ void put_rem(uint32_t s, uint32_t x) {
    const E v = (E)x;
    __builtin_memcpy(reinterpret_cast<char*>(rem) + s * BPE, &v, BPE);
  }
  __host__ __device__ __forceinline__ bool bit(const U* m, uint32_t s) const { return (m[s >> 6] >> (s & 63)) & 1ull; }

  // The first slot >= s whose bit is set in f(word); end if none is held.
  template <class F>
  __host__ __device__ __forceinline__ uint32_t next(uint32_t s, F f) const {
    if (s >= end) return end;
    uint32_t w = s >> 6;
    uint64_t m = f(w) & from(s & 63);
    while (!m) {
      if (++w >= end / 64) return end;
      m = f(w);
    }
    return 64 * w + (uint32_t)__builtin_ctzll(m);
  }
  // The start of fq's run when it is stored, else the slot after the runs of
  // smaller quotients; slot fq is not empty.  end: not held.
  __host__ __device__ __forceinline__ uint32_t run_start(uint32_t fq, bool stored) const {
    uint32_t w = fq >> 6, k = stored ? 0u : 1u;
    uint64_t sel = upto(fq & 63), fr = ~0ull;
    for (;;) {
      const uint64_t m = ~(uint64_t)shf[w] & sel;
      if (m) {  // an entry at its own quotient begins the runs that count
        fr = from(63 - (uint32_t)__builtin_clzll(m));
        k += (uint32_t)__builtin_popcountll(occ[w] & sel & fr);
        break;
      }
      k += (uint32_t)__builtin_popcountll(occ[w] & sel);
      if (w == 0) {
        k += pend;
        break;
      }
      --w;
      sel = ~0ull;
    }
    for (;;) {  // the k-th slot from there on that continues no run
      const uint64_t starts = ~(uint64_t)cont[w] & fr;
      const uint32_t c = (uint32_t)__builtin_popcountll(starts);
      if (c >= k) return 64 * w + select_bit64(starts, k);
      k -= c;
      fr = ~0ull;
      if (++w >= end / 64) return end;
    }
  }
  // fr's slot in the run that starts at s, or the slot it would take.
  __host__ __device__ __forceinline__ bool find(uint32_t s, uint32_t fr, uint32_t* p) const {
    uint32_t x = get_rem(s);
    while (x < fr) {
      if (++s >= end || !bit(cont, s)) {
        *p = s;
        return false;
      }
      x = get_rem(s);
    }
    *p = s;
    return x == fr;
  }

  // Inserts (fq, fr) unless it is stored.
  __host__ __device__ __forceinline__ void insert(uint32_t fq, uint32_t fr) {
    const uint32_t fw = fq >> 6;
    const uint64_t fbit = 1ull << (fq & 63);
    const bool stored = (occ[fw] & fbit) != 0;
    if (((occ[fw] | cont[fw] | shf[fw]) & fbit) == 0) {
      lw_xor(&occ[fw], fbit);
      put_rem(fq, fr);
      mark(fw, fw);
      return;
    }
    const uint32_t s = run_start(fq, stored);
    uint32_t p = s;
    if (s >= end || (stored && find(s, fr, &p))) return;
    const uint32_t e = next(p, [&](uint32_t w) { return ~(uint64_t)(occ[w] | cont[w] | shf[w]); });
    if (e >= end) return;  // not reached: the region is held
    if (!stored) lw_xor(&occ[fw], fbit);
    // flags of [p, e]: the entries after p moved up by one, away from their
    // quotients; a run's old first entry continues it
    const bool first = p == s;
    const uint32_t pw = p >> 6, ew = e >> 6;
    uint64_t top = 0;
    for (uint32_t w = pw; w <= ew; ++w) {
      const uint64_t reg = (w == pw ? from(p & 63) : ~0ull) & (w == ew ? upto(e & 63) : ~0ull);
      const uint64_t old = cont[w];
      uint64_t c = (old << 1) | top, z = ~0ull;
      top = old >> 63;
      if (w == pw) {
        const uint64_t pb = 1ull << (p & 63);
        c = first ? c & ~pb : c | pb;
        if (p == fq) z = ~pb;
      }
      if (stored && first && (p + 1) >> 6 == w) c |= 1ull << ((p + 1) & 63);
      lw_xor(&cont[w], (old ^ c) & reg);
      lw_xor(&shf[w], ((uint64_t)shf[w] ^ z) & reg);
    }
    uint64_t in = fr;
    const uint32_t i0 = p / PW, i1 = e / PW;
    for (uint32_t i = i0; i <= i1; ++i) {
      const uint64_t old = rem[i];
      const uint32_t at = i == i0 ? RB * (p % PW) : 0u;
      const uint64_t up = from(at);
      const uint64_t v = ((old & up) << RB) | (in << at);
      const uint64_t mask = i == i1 ? up & (~0ull >> (64 - RB * (e % PW + 1))) : up;
      in = old >> (64 - RB);
      if (mask == ~0ull) rem[i] = v;
      else lw_xor(&rem[i], (old ^ v) & mask);
    }
    mark(fw, ew);
  }

  // Removes one copy of (fq, fr) if it is stored.
  __host__ __device__ __forceinline__ void erase(uint32_t fq, uint32_t fr) {
    const uint32_t fw = fq >> 6;
    if (!bit(occ, fq)) return;
    const uint32_t s = run_start(fq, true);
    uint32_t p;
    if (s >= end || !find(s, fr, &p)) return;
    // the entries of (p, l] move back by one; after l comes a slot that is
    // empty or holds an entry at its own quotient
    const uint32_t l = next(p + 1, [&](uint32_t w) { return ~(uint64_t)shf[w]; }) - 1;
    const bool first = p == s, more = l > p && bit(cont, p + 1);
    const uint32_t pw = p >> 6, lw = l >> 6;
    // the j-th run start among them belongs to the j-th occupied quotient
    // after fq: it comes to its own quotient z (and is no longer shifted) iff
    // z is occupied and R, the occupied quotients of (fq, z] less the run
    // starts up to z, is 0 there.  R falls only at run starts on unoccupied
    // slots, so 16 slots with fewer of those than R are passed at once.
    int32_t R = 0;
    for (uint32_t w = fw; w <= pw; ++w) {
      const uint64_t sel = (w == fw ? ~upto(fq & 63) : ~0ull) & (w == pw ? ~from(p & 63) : ~0ull);
      R += __builtin_popcountll(occ[w] & sel);
    }
    for (uint32_t w = pw; w <= lw; ++w) {
      const uint64_t reg = (w == pw ? from(p & 63) : ~0ull) & (w == lw ? upto(l & 63) : ~0ull);
      const uint64_t gap = w == lw ? 1ull << (l & 63) : 0ull;  // becomes empty
      const uint64_t old = cont[w];
      uint64_t c = ((old >> 1) | (w < lw ? (uint64_t)cont[w + 1] << 63 : 0ull)) & ~gap, z = ~gap;
      const uint64_t heads = ~c & ~gap & reg;
      const uint64_t own = occ[w] & reg & (w == fw ? ~upto(fq & 63) : ~0ull);
      for (uint32_t k = 0; k < 64; k += 16) {
        const uint32_t h = (uint32_t)(heads >> k) & 0xFFFFu, o = (uint32_t)(own >> k) & 0xFFFFu;
        if (R <= (int32_t)__builtin_popcount(h & ~o)) {
          for (uint32_t m = h & o; m; m &= m - 1u) {
            const uint32_t up = m ^ (m - 1u);  // up to the candidate's bit
            if (R + (int32_t)__builtin_popcount(o & up) == (int32_t)__builtin_popcount(h & up))
              z &= ~((uint64_t)(m & (0u - m)) << k);
          }
        }
        R += (int32_t)__builtin_popcount(o) - (int32_t)__builtin_popcount(h);
      }
      if (w == pw && first && more) {  // the run's next entry becomes its first
        const uint64_t pb = 1ull << (p & 63);
        c &= ~pb;
        if (p == fq) z &= ~pb;
      }
      lw_xor(&cont[w], (old ^ c) & reg);
      lw_xor(&shf[w], ((uint64_t)shf[w] ^ z) & reg);
    }
    if (first && !more) lw_xor(&occ[fw], 1ull << (fq & 63));
    const uint32_t i0 = p / PW, i1 = l / PW;
    for (uint32_t i = i0; i <= i1; ++i) {
      const uint64_t old = rem[i];
      uint64_t v = old >> RB, mask = i == i0 ? from(RB * (p % PW)) : ~0ull;
      if (i < i1) {
        v |= (uint64_t)rem[i + 1] << (64 - RB);
      } else {
        const uint32_t at = RB * (l % PW);
        v &= ~from(at);  // slot l holds nothing
        mask &= ~0ull >> (64 - RB - at);
      }
      if (mask == ~0ull) rem[i] = v;
      else lw_xor(&rem[i], (old ^ v) & mask);
    }
    mark(fw, lw);
  }
};

// Bit i of n (4 bits) to bit 0 of byte i: the product's terms do not overlap.
__device__ __forceinline__ uint32_t nib_bytes(uint32_t n) { return __umul24(n, 0x204081u) & 0x01010101u; }

// Table words (4 / BPE slots each) of the 16 slots [s, s + 16) of the planes.
template <int BPE>
__device__ __forceinline__ void sl_pack16(const SlPlanes<BPE>& m, uint32_t s, uint32_t (&x)[4 * BPE]) {
  const uint32_t sh = s & 48;
  const uint32_t o = (uint32_t)(m.occ[s >> 6] >> sh) & 0xFFFFu, c = (uint32_t)(m.cont[s >> 6] >> sh) & 0xFFFFu,
                 f = (uint32_t)(m.shf[s >> 6] >> sh) & 0xFFFFu;
  const uint4* r4 = reinterpret_cast<const uint4*>(reinterpret_cast<const typename SlPlanes<BPE>::E*>(m.rem) + s);
#pragma unroll
  for (int k = 0; k < BPE; ++k) {
    const uint4 v = r4[k];
    const uint32_t rw[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int q = 4 * k + j;
      if (BPE == 1) {
        x[q] = (rw[j] << 3) | (nib_bytes((o >> (4 * q)) & 15u) << 2) | (nib_bytes((c >> (4 * q)) & 15u) << 1) |
               nib_bytes((f >> (4 * q)) & 15u);
      } else {
        auto two = [&](uint32_t b) { return ((b >> (2 * q)) & 1u) | (((b >> (2 * q)) & 2u) << 15); };
        const uint32_t e = (rw[j] << 3) | (two(o) << 2) | (two(c) << 1) | two(f);
        x[q] = ((e & 0x00FF00FFu) << 8) | ((e >> 8) & 0x00FF00FFu);
      }
    }
  }
}

template <int BPE, bool INS>
__global__ __launch_bounds__(64) void k_sl_apply(uint8_t* __restrict__ t, uint32_t S, uint32_t r,
                                                 const uint32_t* __restrict__ B, uint32_t n,
                                                 const uint32_t* __restrict__ bstart, uint32_t W,
                                                 const uint2* __restrict__ pre, const uint16_t* __restrict__ el,
                                                 const uint16_t* __restrict__ fb, const uint32_t* __restrict__ ctr) {
  using U = unsigned long long;
  __shared__ __align__(16) U s_rem[SL_BLOCKS * 8 * BPE];
  __shared__ U s_occ[SL_BLOCKS], s_cont[SL_BLOCKS], s_shf[SL_BLOCKS];
  __shared__ uint16_t s_head[LW_KEYS];
  __shared__ uint32_t s_dirty[4];
  const uint32_t w = blockIdx.x, lane = threadIdx.x;
  const uint32_t b0 = bstart[w], b1 = bstart[w + 1], nk = b1 - b0;
  if (nk == 0 || nk > LW_KEYS || ctr[CTR_MISC]) return;
  const uint32_t base = w * LW_SLOTS;
  // block `blk` of the window (64 slots) to the planes
  auto load = [&](uint32_t blk) {
    SqfWin<BPE> x;
    sqf_win_load<BPE>(t, S, w * 64 + blk, x);
    s_occ[blk] = x.occ;
    s_cont[blk] = x.cont;
    s_shf[blk] = x.shf;
    uint4* d = reinterpret_cast<uint4*>(s_rem + blk * 8 * BPE);
#pragma unroll
    for (int k = 0; k < 4 * BPE; ++k) {
      uint32_t v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a = x.raw[4 * k + j];
        if (BPE == 1) v[j] = (a >> 3) & 0x1F1F1F1Fu;
        else v[j] = ((((a & 0x00FF00FFu) << 8) | ((a >> 8) & 0x00FF00FFu)) >> 3) & 0x1FFF1FFFu;
      }
      d[k] = make_uint4(v[0], v[1], v[2], v[3]);
    }
  };
  load(lane);
  if (lane < 4) s_dirty[lane] = 0u;
  // heads
  const uint2 pw = pre[w];
  const uint32_t fbw = INS ? 0u : fb[w];
  uint32_t nh = 0;
  int32_t M = (int32_t)pw.x;
  for (uint32_t k0 = 0; k0 < nk; k0 += 64) {
    const uint32_t k = k0 + lane;
    const bool on = k < nk;
    const uint32_t x = on ? el[b0 + k] : 0u;
    bool head;
    if (INS) {
      head = lw_insert_head((int32_t)x - (int32_t)k, on, M);
    } else {
      head = on && x != 0;
      // the window's first key, before its first boundary: dependent on the
      // key before it iff no boundary lies between the two
      if (k == 0 && !head) head = b0 == 0 || pw.y > (B[b0 - 1] >> r) + 1;
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
      uint32_t cs = base + LW_SLOTS;
      const uint32_t stop = base + 64 * SL_BLOCKS < S ? base + 64 * SL_BLOCKS : S;  // (the scan found room before it)
      auto empties = [&]() { return __ballot(cs + lane < stop && (sqf_get<BPE>(t, S, cs + lane) & 7u) == 0); };
      uint64_t em = empties();
      while ((uint32_t)__popcll(em) < need && cs + 64 < stop) {
        need -= (uint32_t)__popcll(em);
        cs += 64;
        em = empties();
      }
      for (; need > 1; --need) em &= em - 1ull;
      for (;;) {  // the empty slot that the region's last key takes at the latest
        while (em == 0 && cs + 64 < stop) {
          cs += 64;
          em = empties();
        }
        if (em == 0) break;  // not reached
        hi = cs + (uint32_t)__builtin_ctzll(em) - base;
        em &= em - 1ull;
        if (k1 >= n || (B[k1] >> r) > base + hi) break;
        ++k1;
      }
    }
  } else {
    uint32_t hp = B[b1 - 1] >> r;
    if (w + 1 < W && fb[w + 1] && pre[w + 1].y <= hp + 1) hi = LW_SLOTS + fb[w + 1] - 1;  // no boundary after the last key
    while (k1 < n) {
      const uint32_t h = B[k1] >> r, w2 = h / LW_SLOTS;
      if (h - w2 * LW_SLOTS >= fb[w2] || pre[w2].y > hp + 1) break;
      hp = h;
      ++k1;
    }
  }
  if (hi >= 64 * SL_BLOCKS) hi = 64 * SL_BLOCKS - 1;  // not reached: the scan's bounds
  const uint32_t nb = hi / 64 + 1;  // blocks held
  if (lane < nb - 64) load(64 + lane);
  __syncthreads();
  const uint32_t h0 = (B[b0 + s_head[0]] >> r) - base;
  SlPlanes<BPE> m;
  m.occ = s_occ;
  m.cont = s_cont;
  m.shf = s_shf;
  m.rem = s_rem;
  m.end = 64 * nb;
  m.pend = 0;
  m.dirty[0] = m.dirty[1] = 0;
  {
    // a first region whose cluster began before the window: the runs of the
    // quotients back to its last entry in place that start in the window
    const uint32_t hb = h0 >> 6;
    const uint64_t z = ~(uint64_t)s_shf[lane] & (lane < hb ? ~0ull : lane == hb ? m.upto(h0 & 63) : 0ull);
    if (__ballot(z != 0) == 0) {
      for (uint32_t c = base; c >= 64;) {
        c -= 64;
        const uint32_t e = sqf_get<BPE>(t, S, c + lane);
        const uint64_t o = __ballot((e & 4u) != 0), st = __ballot((e & 2u) == 0), in_place = __ballot((e & 1u) == 0);
        const uint64_t fr = in_place ? m.from(63 - (uint32_t)__builtin_clzll(in_place)) : ~0ull;
        m.pend += (uint32_t)__popcll(o & fr) - (uint32_t)__popcll(st & fr);
        if (in_place) break;
      }
    }
  }
  // the regions
  const uint32_t rmask = (1u << r) - 1u;
  for (uint32_t ri = lane; ri < nh; ri += 64) {
    const uint32_t ka = b0 + s_head[ri], kb = ri + 1 < nh ? b0 + s_head[ri + 1] : k1;
    for (uint32_t k = ka; k < kb; ++k) {
      const uint32_t fp = B[k];
      if (INS) m.insert((fp >> r) - base, fp & rmask);
      else m.erase((fp >> r) - base, fp & rmask);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t d = (uint32_t)(m.dirty[k >> 1] >> (32 * (k & 1)));
    if (d) atomicOr(&s_dirty[k], d);
  }
  __syncthreads();
  // the changed blocks, 16 slots per lane and step: whole, but for the block
  // in which an earlier window's region may end (before the first region) and
  // the one in which the last region ends
  const uint32_t lo = (INS ? pw.x > 0 : fbw > 0) ? h0 : 0u;
  const uint32_t last = base + hi < S ? hi : S - base - 1;
  for (uint32_t s = 16 * lane; s < 64 * nb; s += 1024) {
    const uint32_t blk = s >> 6;
    if (!((s_dirty[blk >> 5] >> (blk & 31)) & 1u)) continue;
    uint32_t x[4 * BPE];
    sl_pack16<BPE>(m, s, x);
    uint8_t* d = t + ((size_t)base + s) * BPE;
    if (s >= lo && s + 15 <= last) {
#pragma unroll
      for (int k = 0; k < BPE; ++k)
        st16_dw(reinterpret_cast<uint32_t*>(d) + 4 * k, make_uint4(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]));
    } else {
#pragma unroll
      for (uint32_t j = 0; j < 16 * BPE; ++j) {
        const uint32_t sl = s + j / BPE;
        if (sl >= lo && sl <= last) d[j] = (uint8_t)(x[j >> 2] >> (8 * (j & 3)));
      }
    }
  }
}

}  // namespace gqf
