// gqf_dbuild.hpp -- bulk builds without a sort: one partition by quotient
// range, then the runs of every range in LDS, then the layout.
//
//   k_ps_scatter  every key to its group: hashed, ranked by one LDS atomic
//                 and written as runs of equal digits (the fingerprint's top
//                 bits, so a digit is a range of quotients, up to 2^15) to
//                 places that one global atomic per tile and digit reserves;
//   k_db_runs     a group's runs: a byte counter per quotient ranks every key
//                 in its run, the counters are scanned, every remainder goes
//                 to its run's bytes, and runs of several entries are sorted
//                 (and thinned out, NoDup).  Leaves a count per quotient, the
//                 remainders in order and the group's scan state;
//   rb_scan       the locations before every group;
//   k_db_spill    the entries that reach past each group's end;
//   k_db_sqf / k_db_rsqf   the table from counts and remainders.
// A sort moves whole fingerprints through several LDS passes per key; here a
// key costs one LDS atomic, two reads and one byte store after the partition,
// and what remains is a byte per quotient and one per key.  Fingerprints of
// 33 and 34 bits are partitioned as their low words.  53.7 M keys into 2^26
// quotients: SQF (r = 5, NoDup) 790 -> 474 us, RSQF (r = 8) 1380 -> 470 us.
//   Groups of more keys than they have room for, runs past 255 entries (hot
// keys), more than 255 keys in 32 neighbouring quotients and spills past 512
// slots raise ctr[CTR_MISC] before the table is written, and the call takes
// the sort (and the stream's next ones, for a while: lw_report).
#pragma once

#include "gqf_rebuild.hpp"

namespace gqf {

constexpr int PS_THREADS = 1024;
constexpr uint32_t PS_ITEMS = 32;                         // keys per thread of a tile or group
constexpr uint32_t PS_TILE = PS_THREADS * PS_ITEMS;       // keys per tile
constexpr uint32_t PS_GB_MIN = 8, PS_GB_MAX = 11;
constexpr uint32_t PS_ND = 1u << PS_GB_MAX;
constexpr uint32_t PS_SPARSE_SQF = 6, PS_SPARSE_RSQF = 32;
constexpr uint32_t DB_QB = 15;                            // log2 of a group's quotients, at most
constexpr uint32_t DB_NQ = 1u << DB_QB;
constexpr uint32_t DB_Q = DB_NQ / PS_THREADS;             // quotients per thread
static_assert(DB_Q == 32, "a thread's occupied bits are one word");

struct PsPlan {
  uint32_t gb, shift, ngroups, qb;  // digit bits, bits below them, 1 << gb, log2 of a group's quotients
  uint32_t tile, wgs, cap;          // keys per tile, workgroups of the partition, keys a group has room for
};
// The partition of n keys of a table of 2^q quotients: digits and tiles.  A
// workgroup takes a CU's LDS: 256 of them, the same number of tiles each.
// Returns the tiles.
inline uint32_t ps_tiles(uint64_t n, uint32_t q, uint32_t r, PsPlan* p) {
  p->gb = q > DB_QB + PS_GB_MIN ? q - DB_QB : PS_GB_MIN;
  p->qb = q - p->gb;
  p->shift = p->qb + r;
  p->ngroups = 1u << p->gb;
  const uint64_t rounds = (n + 256ull * PS_TILE - 1) / (256ull * PS_TILE);
  p->tile = (uint32_t)(((n + 256 * rounds - 1) / (256 * rounds) + 3) & ~3ull);
  const uint32_t tiles = (uint32_t)((n + p->tile - 1) / p->tile);
  p->wgs = tiles < 256 ? tiles : 256;
  return tiles;
}
// The plan of n keys into a table of 2^q quotients; false where the sort
// applies: few keys (their launches count, not their moves), tables of more
// than 2^26 quotients (more digits than runs of stores allow), remainders
// past a byte, more than `sparse` quotients per key (the passes over the
// counts outweigh the sort: an SQF of q = 26 breaks even near 6, 288 : 256 us
// at 8 M keys, 327 : 346 at 16 M; an RSQF near 32, 208 : 200 us at 2 M), and
// batches that uniform keys would hand over as well: groups with no room for
// three standard deviations past their mean, or more than 208 keys per 32
// quotients (their bytes count to 255).
constexpr uint32_t PS_MEAN_MAX = PS_TILE - 640, DB_LOAD_MAX = 208;
inline bool ps_plan(uint64_t n, uint32_t q, uint32_t r, uint32_t sparse, PsPlan* p) {
  if (n <= 256ull * 7600 || n * sparse < (1ull << q) || q < 20 || q > DB_QB + PS_GB_MAX || r > 8 || n >= (1ull << 30)) return false;
  (void)ps_tiles(n, q, r, p);
  const uint64_t mean = n >> p->gb, cap = (2 * mean + 2048 + 63) & ~63ull;
  if (mean > PS_MEAN_MAX || 32 * n > ((uint64_t)DB_LOAD_MAX << q)) return false;
  p->cap = (uint32_t)(cap < PS_TILE ? cap : PS_TILE);
  return true;
}

// A key's fingerprint: digit and low 32 bits.
template <bool WIDE>
__device__ __forceinline__ uint32_t ps_split(uint32_t key, uint32_t fp_bits, uint32_t shift, uint32_t* low) {
  if (WIDE) {
    const uint64_t f = fingerprint(key, fp_bits);
    *low = (uint32_t)f;
    return (uint32_t)(f >> shift);
  }
  const uint32_t f = fingerprint32(key, fp_bits);
  *low = f;
  return f >> shift;
}

// The keys of [t0, t0 + tn) in a thread's order: item i is key
// (i / 4) * 4096 + 4 t + i % 4 (16-byte loads).
__device__ __forceinline__ uint32_t ps_at(uint32_t i) { return (i >> 2) * (4 * PS_THREADS) + 4 * threadIdx.x + (i & 3); }
__device__ __forceinline__ void ps_load(const uint32_t* __restrict__ p, uint32_t tn, uint32_t (&w)[PS_ITEMS]) {
#pragma unroll
  for (uint32_t c = 0; c < PS_ITEMS / 4; ++c) {
    const uint32_t at = ps_at(4 * c);
    if (at + 4 <= tn) {
      const uint4 x = ld16_dw(p + at);
      w[4 * c] = x.x, w[4 * c + 1] = x.y, w[4 * c + 2] = x.z, w[4 * c + 3] = x.w;
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) w[4 * c + k] = at + k < tn ? p[at + k] : 0u;
    }
  }
}

// f(i) for the items of a thread that hold one of tn keys.  Items come in
// blocks of 4 * PS_THREADS keys, tested as a whole except for the last one: a
// test per item would put every item's LDS access into a basic block of its
// own, which waits for it.
template <typename F>
__device__ __forceinline__ void ps_each(uint32_t tn, F f) {
#pragma unroll
  for (uint32_t c = 0; c < PS_ITEMS / 4; ++c) {
    if (4 * PS_THREADS * (c + 1) <= tn) {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) f(4 * c + k);
    } else if (4 * PS_THREADS * c < tn) {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k)
        if (ps_at(4 * c + k) < tn) f(4 * c + k);
    }
  }
}

// Group sizes and the build's counters to zero.
[[maybe_unused]] static __global__ __launch_bounds__(PS_THREADS) void k_ps_reset(uint32_t* __restrict__ gsize, uint32_t nd,
                                                                                 uint32_t* __restrict__ ctr) {
  for (uint32_t d = threadIdx.x; d < nd; d += PS_THREADS) gsize[d] = 0u;
  if (threadIdx.x >= CTR_OP && threadIdx.x < CTR_TOTAL) ctr[threadIdx.x] = 0u;
}

// Where a tile's keys went: key p of the tile in order of digits (d: its own)
// lies at place base[tile][d] + p of d's region, the digit's first key of the
// tile is p = first[tile][d], and key i of all is its tile's place[i].
struct PsBack {
  uint16_t* place;
  uint32_t* base;
  uint16_t* first;
};

// Tiles blockIdx.x, + gridDim.x, ... to their groups, each a region of `cap`
// keys in `out`: every key takes its rank in its digit from an LDS counter,
// one global atomic per digit reserves the tile's places (in flight while
// the counts are scanned and the tile is laid out by digit in LDS), and the
// tile is written in runs of equal digits (16 keys on average at 2^11).
// Order within a group is of no account: its runs are sorted later.  So no
// pass counts the keys first and hashes them twice (that took 70 us more at
// 53.7 M keys).  175 us at that size (r = 8, 64-bit hash: 230), bound by the
// number of its runs and the hash: the same stores in order take 153 us, half
// the tile (two workgroups per CU, runs of 8 keys) 355 us.  The next tile is
// loaded before this one is written; interleaving its hashes with the stores
// gained nothing.
//   BACK leaves the way back to the keys' order (gqf_plookup.hpp).
template <bool WIDE, bool BACK>
__global__ __launch_bounds__(PS_THREADS) void k_ps_scatter(const uint32_t* __restrict__ keys, uint32_t n,
                                                           uint32_t fp_bits, uint32_t shift, uint32_t nd,
                                                           uint32_t hbits, uint32_t tile, uint32_t cap,
                                                           uint32_t* __restrict__ gsize, uint32_t* __restrict__ out,
                                                           uint32_t* __restrict__ ctr, PsBack back) {
  __shared__ uint32_t s_key[PS_TILE];
  __shared__ uint32_t s_cnt[PS_ND], s_base[PS_ND];
  __shared__ uint32_t s_tmp[PS_THREADS / 64];
  __shared__ uint32_t s_hi[4];
  const uint32_t t = threadIdx.x, d0 = 2 * t;  // (a thread's two digits)
  uint64_t t0 = (uint64_t)blockIdx.x * tile;
  uint32_t w[PS_ITEMS];
  uint32_t tn = (uint32_t)(n - t0 < tile ? n - t0 : tile);
  ps_load(keys + t0, tn, w);
  while (t0 < n) {
    if (d0 < nd) *reinterpret_cast<uint2*>(s_cnt + d0) = make_uint2(0u, 0u);
    __syncthreads();
    // digit and rank of every key (rank below 2^15, digit above it)
    uint32_t dr[PS_ITEMS];
#pragma unroll
    for (uint32_t i = 0; i < PS_ITEMS; ++i) {
      uint32_t low;
      const uint32_t d = ps_split<WIDE>(w[i], fp_bits, shift, &low);
      w[i] = low;
      dr[i] = ps_at(i) < tn ? (d << 16) | atomicAdd(&s_cnt[d], 1u) : 0xFFFFFFFFu;
    }
    __syncthreads();
    const uint2 c = d0 < nd ? *reinterpret_cast<const uint2*>(s_cnt + d0) : make_uint2(0u, 0u);
    uint32_t b0 = 0, b1 = 0;
    if (c.x) b0 = atomicAdd(&gsize[d0], c.x);
    if (c.y) b1 = atomicAdd(&gsize[d0 + 1], c.y);
    const uint32_t e = block_excl_scan<PS_THREADS>(c.x + c.y, s_tmp);
    if (d0 < nd) {
      *reinterpret_cast<uint2*>(s_cnt + d0) = make_uint2(e, e + c.x);
      if (WIDE && (d0 & ((nd >> hbits) - 1u)) == 0) s_hi[d0 / (nd >> hbits)] = e;  // first of a high word
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < PS_ITEMS; ++i)
      if (dr[i] != 0xFFFFFFFFu) {
        const uint32_t p = s_cnt[dr[i] >> 16] + (dr[i] & 0xFFFFu);
        s_key[p] = w[i];
        if (BACK) dr[i] = p;
      }
    if (BACK) {
#pragma unroll
      for (uint32_t i = 0; i < PS_ITEMS; i += 4)
        if (ps_at(i) < tn)  // (the last four may be part of one: place has room)
          *reinterpret_cast<uint2*>(back.place + t0 + ps_at(i)) =
              make_uint2((dr[i] & 0xFFFFu) | dr[i + 1] << 16, (dr[i + 2] & 0xFFFFu) | dr[i + 3] << 16);
      if (d0 < nd) {
        const uint64_t row = (t0 / tile) * nd + d0;
        *reinterpret_cast<uint2*>(back.base + row) = make_uint2(b0 - e, b1 - (e + c.x));
        *reinterpret_cast<uint32_t*>(back.first + row) = e | (e + c.x) << 16;
      }
    }
    if (d0 < nd) {
      *reinterpret_cast<uint2*>(s_base + d0) = make_uint2(b0 - e, b1 - (e + c.x));
      if (b0 + c.x > cap || b1 + c.y > cap) {  // a group is full: its further keys are not written
        ctr[CTR_MISC] = 1u;
        if (!BACK) gsize[nd] = 1u;
      }
    }
    __syncthreads();
    const uint32_t tw = tn;
    t0 += (uint64_t)gridDim.x * tile;
    if (t0 < n) {
      tn = (uint32_t)(n - t0 < tile ? n - t0 : tile);
      ps_load(keys + t0, tn, w);
    }
    const uint32_t h1 = WIDE ? s_hi[1] : 0u, h2 = WIDE && hbits > 1 ? s_hi[2] : ~0u, h3 = WIDE && hbits > 1 ? s_hi[3] : ~0u;
#pragma unroll 8
    for (uint32_t j = 0; j < PS_ITEMS; ++j) {
      const uint32_t p = t + j * PS_THREADS;
      if (p < tw) {
        const uint32_t x = s_key[p];
        uint32_t d = shift < 32 ? x >> shift : 0u;
        if (WIDE) d |= ((uint32_t)(p >= h1) + (uint32_t)(p >= h2) + (uint32_t)(p >= h3)) << (32 - shift);
        const uint32_t at = s_base[d] + p;
        if (at < cap) out[(uint64_t)d * cap + at] = x;
      }
    }
    // (s_base and s_key are written again after barriers that follow these reads)
  }
}

// ---------------------------------------------------------------- runs
// Group g: gsize[g] keys from g cap on, as many remainder bytes at most from
// byte g cap on (cap: a multiple of 64).

// LDS writes of the wave's lanes before, reads after.
__device__ __forceinline__ void db_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Sorts the n (2 at least) bytes of a run from p on (rem8 may be read three
// bytes further); UNIQUE: clears the kept bits of repeats and returns their
// number.
template <bool UNIQUE>
__device__ __forceinline__ uint32_t db_sort_run(uint8_t* rem8, uint32_t p, uint32_t n, uint32_t* s_keep) {
  auto order = [](uint32_t& a, uint32_t& b) {
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
  };
  uint32_t repeats = 0;
  auto repeat = [&](uint32_t z) {
    atomicAnd(&s_keep[z >> 5], ~(1u << (z & 31)));
    ++repeats;
  };
  if (n <= 4) {
    // a missing value is larger than any byte
    uint32_t x0 = rem8[p], x1 = rem8[p + 1], x2 = rem8[p + 2], x3 = rem8[p + 3];
    x2 = n > 2 ? x2 : 0x100u;
    x3 = n > 3 ? x3 : 0x200u;
    order(x0, x1), order(x2, x3), order(x0, x2), order(x1, x3), order(x1, x2);
    rem8[p] = (uint8_t)x0;
    rem8[p + 1] = (uint8_t)x1;
    if (n > 2) rem8[p + 2] = (uint8_t)x2;
    if (n > 3) rem8[p + 3] = (uint8_t)x3;
    if (UNIQUE)
      for (uint32_t d = (x0 == x1 ? 1u : 0u) | (x1 == x2 ? 2u : 0u) | (x2 == x3 ? 4u : 0u); d; d &= d - 1u)
        repeat(p + 1 + (uint32_t)__builtin_ctz(d));
  } else if (n <= 8) {
    // Batcher's network on 8 values
    uint32_t x[8];
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) x[i] = i < n ? (uint32_t)rem8[p + i] : 0x100u + i;
    order(x[0], x[1]), order(x[2], x[3]), order(x[0], x[2]), order(x[1], x[3]), order(x[1], x[2]);
    order(x[4], x[5]), order(x[6], x[7]), order(x[4], x[6]), order(x[5], x[7]), order(x[5], x[6]);
    order(x[0], x[4]), order(x[1], x[5]), order(x[2], x[6]), order(x[3], x[7]);
    order(x[2], x[4]), order(x[3], x[5]);
    order(x[1], x[2]), order(x[3], x[4]), order(x[5], x[6]);
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i)
      if (i < n) rem8[p + i] = (uint8_t)x[i];
    if (UNIQUE)
#pragma unroll
      for (uint32_t i = 1; i < 8; ++i)
        if (x[i] == x[i - 1]) repeat(p + i);
  } else {
    for (uint32_t a = p + 1; a < p + n; ++a) {
      const uint8_t x = rem8[a];
      uint32_t b = a;
      for (; b > p; --b) {
        const uint8_t y = rem8[b - 1];
        if (y <= x) break;
        rem8[b] = y;
      }
      rem8[b] = x;
    }
    if (UNIQUE)
      for (uint32_t a = p + 1; a < p + n; ++a)
        if (rem8[a] == rem8[a - 1]) repeat(a);
  }
  return repeats;
}

// The same by a wave, for a run of 2 .. 255 bytes: every byte's rank among
// them, a few per lane.  A lane sorting 64 bytes of two values in place takes
// 1000 dependent moves, and its wave waits; this takes 64 steps.
constexpr uint32_t DB_LONG = 24;  // longer runs are sorted so
template <bool UNIQUE>
__device__ __forceinline__ void db_sort_long(uint8_t* rem8, uint32_t p, uint32_t n, uint8_t* tmp, uint32_t* s_keep) {
  const uint32_t lane = threadIdx.x & 63;
#pragma unroll 1
  for (uint32_t i = lane; i - lane < n; i += 64) {
    const uint32_t x = i < n ? (uint32_t)rem8[p + i] : 0x100u;
    uint32_t rank = 0;
#pragma unroll 4
    for (uint32_t j = 0; j < n; ++j) {
      const uint32_t y = rem8[p + j];
      rank += y < x + (j < i ? 1u : 0u) ? 1u : 0u;
    }
    if (i < n) tmp[rank] = (uint8_t)x;
  }
  db_wave_sync();
#pragma unroll 1
  for (uint32_t i = lane; i < n; i += 64) {
    const uint32_t x = tmp[i];
    rem8[p + i] = (uint8_t)x;
    if (UNIQUE && i && tmp[i - 1] == x) atomicAnd(&s_keep[(p + i) >> 5], ~(1u << ((p + i) & 31)));
  }
  db_wave_sync();
}

// A thread's 32 quotients on the way from k_db_runs to the table: the kept
// entries before them in the group, and 1 + the last location before them
// when nothing precedes the group (0: none).
struct DbThread {
  uint32_t kept, lp;
};
constexpr uint32_t DB_LIST = 128;  // listed runs per wave
constexpr uint32_t DB_MANY = 8;    // repeats that one lane meets: many

// Group blockIdx.x: counts[quotient] (kept entries), their remainders in
// order (db_stream), th[1024 g + t], agg[g].
//   LDS atomics give every key its rank in its run; a key's byte then goes to
// run start + rank, in the order of arrival.  Every wave lists the runs of
// several entries among its quotients and sorts 64 of them at a time, a lane
// per run (up to 8 entries in registers, up to 24 in a loop, longer runs by
// the wave).  Repeats
// (UNIQUE) are dropped from the bytes at the end.
//   A thread sorting its own 32 quotients' runs in place costs its wave the
// longest run at every quotient: 342 us for 53.7 M keys; this: 201 us, 151 us
// with repeats kept.  Bound by instructions and LDS accesses in about equal
// parts (rank, placing and sorting 15, 15 and 25% of the time).
//   A thread takes Q quotients, a group's by its 1024 threads (32 for 2^15; with
// 32 for 2^12 as well, two of sixteen waves had work).  Fewer than 2^15
// quotients: 256 groups, one to a CU, with all its registers.
//   MANY, for keys with many copies: runs past 24 entries are sorted by their
// wave, and where a lane has met 8 repeats the offsets are recounted from the
// kept bits instead of lowered past each.  Builds (NoDup) of 2^25 keys, q = 26,
// so many copies of each on average: 1: 366 us (368 with MANY), 4: 715 -> 575,
// 32: 1520 -> 706; the sort takes 573, 620 and 983.  q = 22, 2^21 keys: 32
// copies 302 -> 118 (the sort 153); q = 20, 2^21 keys, 4 copies: 278 -> 119 (124).
template <bool UNIQUE, uint32_t Q, bool MANY>
__global__ __launch_bounds__(PS_THREADS, Q == DB_Q ? 8 : 4) void k_db_runs(const uint32_t* __restrict__ in,
                                                           const uint32_t* __restrict__ gsize, uint32_t nd, uint32_t cap,
                                                           uint32_t qb, uint32_t r, uint8_t* __restrict__ counts,
                                                           uint8_t* __restrict__ rems,
                                                           DbThread* __restrict__ th, uint4* __restrict__ agg,
                                                           uint32_t* __restrict__ ctr) {
  __shared__ __align__(16) uint32_t s_cnt[DB_NQ / 4];    // counts, then offsets within a thread's range
  __shared__ __align__(16) uint32_t s_rem[PS_TILE / 4 + 4];  // remainder bytes
  __shared__ __align__(16) uint32_t s_keep[UNIQUE ? PS_TILE / 32 + 4 : 4];
  constexpr uint32_t NW = Q / 4;  // a thread's counter words
  __shared__ uint16_t s_base[PS_THREADS + 1];
  __shared__ __align__(16) uint16_t s_list[PS_THREADS / 64][MANY ? DB_LIST + 64 : DB_LIST];  // (MANY: room for 255 bytes past 64)
  __shared__ uint32_t s_tmp[PS_THREADS / 64];
  __shared__ uint4 s_wave[PS_THREADS / 64 + 1];
  __shared__ uint32_t s_many, s_handed;  // MANY: repeats enough to recount; handed over
  const uint32_t t = threadIdx.x, lane = t & 63;
  const uint32_t shift = qb + r, lmask = (1u << shift) - 1u, rmask = (1u << r) - 1u;
  const uint32_t g = blockIdx.x, m = gsize[g];
  if (gsize[nd]) return;  // (uniform) some group is too full: handed over
  uint4* c4 = reinterpret_cast<uint4*>(s_cnt);
  uint32_t k[PS_ITEMS];
  ps_load(in + (uint64_t)g * cap, m, k);
  c4[t] = make_uint4(0u, 0u, 0u, 0u);
  c4[PS_THREADS + t] = make_uint4(0u, 0u, 0u, 0u);
  if (UNIQUE) {
    if (MANY && t == 0) s_many = 0u;
    s_keep[t] = ~0u;
    if (t < 4) s_keep[PS_TILE / 32 + t] = ~0u;
  }
  __syncthreads();
  bool bad = false;
  // every key's rank in its run, above its bits (at most 23)
  ps_each(m, [&](uint32_t i) {
    k[i] &= lmask;
    const uint32_t fq = k[i] >> r, sh = 8 * (fq & 3u);
    const uint32_t x = (atomicAdd(&s_cnt[fq >> 2], 1u << sh) >> sh) & 0xFFu;
    bad |= x == 255u;
    k[i] |= x << 24;
  });
  __syncthreads();
  // this thread's quotients: counts, first key, offsets
  uint32_t* own = s_cnt + NW * t;
  auto words = [&](uint32_t (&o)[NW]) {
    if constexpr (NW == 8) {
      const uint4 x = c4[2 * t], y = c4[2 * t + 1];
      o[0] = x.x, o[1] = x.y, o[2] = x.z, o[3] = x.w, o[4] = y.x, o[5] = y.y, o[6] = y.z, o[7] = y.w;
    } else if constexpr (NW == 4) {
      const uint4 x = c4[t];
      o[0] = x.x, o[1] = x.y, o[2] = x.z, o[3] = x.w;
    } else {
#pragma unroll
      for (uint32_t j = 0; j < NW; ++j) o[j] = own[j];
    }
  };
  auto put_words = [&](void* at, const uint32_t (&o)[NW]) {
    if constexpr (NW >= 4) {
#pragma unroll
      for (uint32_t j = 0; j < NW; j += 4) reinterpret_cast<uint4*>(at)[j / 4] = make_uint4(o[j], o[j + 1], o[j + 2], o[j + 3]);
    } else {
#pragma unroll
      for (uint32_t j = 0; j < NW; ++j) reinterpret_cast<uint32_t*>(at)[j] = o[j];
    }
  };
  uint32_t first, sum = 0;
  {
    uint32_t c[NW], o[NW];
    words(c);
#pragma unroll
    for (uint32_t j = 0; j < NW; ++j) {
      const uint32_t h = (c[j] & 0x00FF00FFu) + ((c[j] >> 8) & 0x00FF00FFu);
      o[j] = (c[j] * 0x01010100u) + (sum & 0xFFu) * 0x01010101u;  // bytes: sums of those below (if all are at most 255)
      sum += (h & 0xFFFFu) + (h >> 16);
    }
    uint32_t near = sum;  // of 32 neighbouring quotients
#pragma unroll
    for (uint32_t x = 1; x < DB_Q / Q; x *= 2) near += (uint32_t)__shfl_xor((int)near, (int)x);
    bad |= near > 255u;
    put_words(own, o);
    first = block_excl_scan<PS_THREADS>(sum, s_tmp);
    s_base[t] = (uint16_t)first;
    if (t == PS_THREADS - 1) s_base[PS_THREADS] = (uint16_t)(first + sum);
  }
  if (__syncthreads_or(bad)) {
    if (t == 0) ctr[CTR_MISC] = 1u;
    return;
  }
  uint8_t* rem8 = reinterpret_cast<uint8_t*>(s_rem);
  const uint8_t* off8 = reinterpret_cast<const uint8_t*>(s_cnt);
  ps_each(m, [&](uint32_t i) {
    const uint32_t fq = (k[i] & lmask) >> r;
    rem8[s_base[fq / Q] + off8[fq] + (k[i] >> 24)] = (uint8_t)(k[i] & rmask);
  });
  // counts of the thread's quotients 4 w .. 4 w + 3, from the offsets
  auto cnt4 = [&](uint32_t w) {
    const uint32_t o = own[w], nx = w + 1 < NW ? own[w + 1] : sum;
    return ((o >> 8) | (nx << 24)) - o;  // no byte borrows: offsets do not decrease
  };
  // handed over by another group meanwhile (where all groups run at once)
  if (Q < DB_Q && t == 0) s_handed = __hip_atomic_load(&ctr[CTR_MISC], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (Q < DB_Q && s_handed) return;  // (uniform)
  // runs of several entries
  {
    uint16_t* list = s_list[t >> 6];
    uint32_t listed = 0, x = 0, repeats = 0;  // (listed: the same in all lanes)
#pragma unroll 1
    for (uint32_t j = 0;;) {
      if (j < Q) {
        if ((j & 3) == 0) x = cnt4(j >> 2);
        const bool several = (x & 0xFFu) > 1;
        const uint64_t who = __ballot(several);
        if (several) list[listed + __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u))] = (uint16_t)(Q * t + j);
        listed += (uint32_t)__popcll(who);
        x >>= 8;
        ++j;
      }
      if (j < Q && listed < 64) continue;
      if (listed == 0) break;
      db_wave_sync();
      const uint32_t nl = listed < 64 ? listed : 64u;
      listed -= nl;
      uint32_t longer = 0;  // a run's place and length (MANY)
      if (lane < nl) {
        const uint32_t q = list[listed + lane], b0 = s_base[q / Q], o = off8[q], p = b0 + o;
        const uint32_t n = (q % Q == Q - 1 ? s_base[q / Q + 1] - b0 : off8[q + 1]) - o;
        if (MANY && n > DB_LONG) longer = p << 8 | n;
        else repeats += db_sort_run<UNIQUE>(rem8, p, n, s_keep);
      }
      if (MANY) {
        for (uint64_t who = __ballot(longer != 0); who; who &= who - 1ull) {
          const uint32_t x = wave_read(longer, __builtin_ctzll(who));
          db_sort_long<UNIQUE>(rem8, x >> 8, x & 0xFFu, reinterpret_cast<uint8_t*>(list + 64), s_keep);
          repeats = DB_MANY;
        }
      }
      db_wave_sync();
    }
    if (MANY && UNIQUE && repeats >= DB_MANY) s_many = 1u;
  }
  __syncthreads();
  // many repeats: the kept entries before every 32 (where the lists were)
  uint16_t* s_pre = &s_list[0][0];
  static_assert(sizeof(s_list) >= 2 * (PS_THREADS + 1), "the counts fit");
  const bool many = MANY && UNIQUE && s_many != 0;  // (uniform)
  if (many) {
    const uint32_t c = (uint32_t)__popc(s_keep[t]), d = block_excl_scan<PS_THREADS>(c, s_tmp);
    s_pre[t] = (uint16_t)d;
    if (t == PS_THREADS - 1) s_pre[PS_THREADS] = (uint16_t)(d + c);
    __syncthreads();
  }
  // kept entries per quotient, and the thread's scan state: lp = kept +
  // max(quotient - kept entries before it) over the occupied quotients, four
  // quotients at a time (for an empty one the difference is no larger than
  // for the next occupied one; past the last occupied one, its index stands
  // for theirs)
  RS a = rs_none();
  {
    uint32_t n = sum;
    uint32_t last = 0;  // the last occupied quotient: the last whose count is not 0
    {
      uint32_t o[NW];
      words(o);
#pragma unroll
      for (uint32_t w = 0; w < NW; ++w) {
        const uint32_t c = ((o[w] >> 8) | ((w + 1 < NW ? o[w + 1] : sum) << 24)) - o[w];
        if (c) last = 4 * w + ((31u - (uint32_t)__builtin_clz(c)) >> 3);
      }
    }
    if (UNIQUE) {
      if (many) {
        // kept entries before position z of the group
        auto kept = [&](uint32_t z) { return s_pre[z >> 5] + (uint32_t)__popc(s_keep[z >> 5] & ((1u << (z & 31)) - 1u)); };
        const uint32_t k0 = kept(first);
        n = kept(first + sum) - k0;
#pragma unroll 1
        for (uint32_t w = 0; w < NW; ++w) {
          const uint32_t x = own[w];
          uint32_t y = 0;
#pragma unroll
          for (uint32_t b = 0; b < 4; ++b) y |= (kept(first + ((x >> (8 * b)) & 0xFFu)) - k0) << (8 * b);
          own[w] = y;
        }
      } else {
        // the offsets past every repeat fall by one (in LDS: a loop over them in
        // registers spilled 26, 330 MB of scratch at 53.7 M keys)
        for (uint32_t z0 = first & ~31u; z0 < first + sum; z0 += 32) {
          uint32_t lost = ~s_keep[z0 >> 5];
          if (z0 < first) lost &= ~0u << (first - z0);
          if (first + sum - z0 < 32) lost &= (1u << (first + sum - z0)) - 1u;
          for (; lost; lost &= lost - 1u) {
            const uint32_t z = z0 + (uint32_t)__builtin_ctz(lost) - first - (sum - n);  // its place among the kept so far
            const uint32_t s = z * 0x01010101u;
            // bytes of x above z
            auto fall = [&](uint32_t x) {
              const uint32_t lo = (x | 0x80808080u) - (s & 0x7F7F7F7Fu) - 0x01010101u;  // top bits: low 7 bits of x > those of s
              return x - ((((x & ~s) | (~(x ^ s) & lo)) & 0x80808080u) >> 7);
            };
            if constexpr (NW >= 4) {
#pragma unroll 1
              for (uint32_t h = NW / 4 * t; h < NW / 4 * t + NW / 4; ++h) {
                const uint4 x = c4[h];
                c4[h] = make_uint4(fall(x.x), fall(x.y), fall(x.z), fall(x.w));
              }
            } else {
              for (uint32_t w = 0; w < NW; ++w) own[w] = fall(own[w]);
            }
            --n;
          }
        }
      }
    }
    uint32_t o[NW];  // kept entries before each quotient, of the thread
    words(o);
    uint32_t kc[NW];
    int32_t mx = -256;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) {
      kc[w] = ((o[w] >> 8) | ((w + 1 < NW ? o[w + 1] : n) << 24)) - o[w];
#pragma unroll
      for (uint32_t b = 0; b < 4; ++b) {
        const uint32_t q = 4 * w + b < last ? 4 * w + b : last;
        const int32_t v = (int32_t)q - (int32_t)((o[w] >> (8 * b)) & 0xFFu);
        mx = v > mx ? v : mx;
      }
    }
    const uint32_t fq0 = (g << qb) + Q * t;
    if (n) a = RS{n, fq0 + (uint32_t)((int32_t)n + mx), fq0 + last + 1};
    put_words(counts + ((uint64_t)g << qb) + Q * t, kc);
  }
  RS ex;
  const RS all = rs_block_n<PS_THREADS / 64>(a, &ex, s_wave);
  if (Q * t % DB_Q == 0) th[(uint64_t)g * PS_THREADS + Q * t / DB_Q] = DbThread{ex.c, ex.lp};
  if (t == 0) agg[g] = rs_pack(all);
  if (UNIQUE && all.c != m) {  // (uniform) the kept bytes together: 32 keys per thread
    const uint4* s4 = reinterpret_cast<const uint4*>(s_rem);
    const uint4 x = s4[2 * t], y = s4[2 * t + 1];
    const uint32_t v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w}, keep = s_keep[t];
    uint32_t d = block_excl_scan<PS_THREADS>((uint32_t)__popc(keep), s_tmp);  // (all have read v)
    if (d != 32 * t || keep != ~0u) {
#pragma unroll
      for (uint32_t j = 0; j < 32; ++j) {
        if ((keep >> j) & 1u) rem8[d] = (uint8_t)(v[j >> 2] >> (8 * (j & 3)));
        d += (keep >> j) & 1u;
      }
    }
    __syncthreads();
  }
  uint4* d = reinterpret_cast<uint4*>(rems + (uint64_t)g * cap);
  for (uint32_t i = t; i < (all.c + 15) / 16; i += PS_THREADS) d[i] = reinterpret_cast<const uint4*>(s_rem)[i];
}

// ---------------------------------------------------------------- spills
// Boundary blockIdx.x + 1: the entries of the group before it that lie past
// its end (its spill) as run starts, bits from the boundary on; a spill longer
// than DB_SPILL, or one that the last 1024 quotients before the boundary do
// not hold, hands the build over.  (Nothing of the table is written yet.)
constexpr uint32_t DB_SPILL = 512, DB_SW = DB_SPILL / 32;
__device__ __forceinline__ uint32_t db_lp(const uint4* __restrict__ pre, uint32_t g, uint32_t ngroups,
                                          const uint32_t* __restrict__ ctr) {
  return g < ngroups ? rs_unpack(pre[g]).lp : ctr[CTR_MISC + 1];
}
[[maybe_unused]] static __global__ __launch_bounds__(256) void k_db_spill(const uint8_t* __restrict__ counts, uint32_t qb,
                                                                          const uint4* __restrict__ pre, uint32_t ngroups,
                                                                          uint32_t* __restrict__ spill,
                                                                          uint32_t* __restrict__ ctr) {
  __shared__ uint32_t s_tmp[4], s_bits[DB_SW];
  const uint32_t t = threadIdx.x, b = blockIdx.x + 1, q1 = b << qb;
  const uint32_t lp = db_lp(pre, b, ngroups, ctr);
  const uint32_t s = lp > q1 ? lp - q1 : 0u;
  if (t < DB_SW) s_bits[t] = 0u;
  if (s == 0 || s > DB_SPILL) {  // (uniform)
    if (t < DB_SW) spill[(uint64_t)b * DB_SW + t] = 0u;
    if (s && t == 0) ctr[CTR_MISC] = 1u;
    return;
  }
  const uint32_t c = *reinterpret_cast<const uint32_t*>(counts + q1 - 1024 + 4 * t);
  const uint32_t h = (c & 0x00FF00FFu) + ((c >> 8) & 0x00FF00FFu), sum = (h & 0xFFFFu) + (h >> 16);
  if (((c & 0xFFu) > DB_LONG) | ((c >> 8 & 0xFFu) > DB_LONG) | ((c >> 16 & 0xFFu) > DB_LONG) | (c >> 24 > DB_LONG)) ctr[CTR_MISC + 2] = 1u;
  const uint32_t before = block_excl_scan<256>(sum, s_tmp);
  __shared__ uint32_t s_all;
  if (t == 255) s_all = before + sum;
  __syncthreads();
  const uint32_t all = s_all;
  if (all < s && t == 0) ctr[CTR_MISC] = 1u;
  uint32_t at = before;
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t x = (c >> (8 * j)) & 0xFFu, start = s + at - all;  // wraps when before the boundary
    if (x && start < s) atomicOr(&s_bits[start >> 5], 1u << (start & 31));
    at += x;
  }
  __syncthreads();
  if (t < DB_SW) spill[(uint64_t)b * DB_SW + t] = s_bits[t];
}

// ---------------------------------------------------------------- table
// Both tables are written by slots: a group's workgroup owns the slots of its
// quotients [q0, q1) (the last group also its spill), with the spill of the
// groups before it at their front.  Bit planes in LDS over those slots --
// taken, run start -- come from the threads' quotients (in registers: 64 slots
// from the thread's first location on, longer reaches one by one); after a
// prefix count of the taken bits a thread writes 32 slots, whose remainders
// are consecutive bytes.  (Walking the keys of a thread's quotients takes
// every wave as many steps as its fullest lane: 157 us for 2^26 slots; this: 72 us,
// half of it the loads, which all workgroups issue at about the same time.)
constexpr uint32_t DB_PW = PS_THREADS + DB_SW + 2;  // words of a plane

// Calls write(word, taken, run starts, run ends, occupied quotients, unshifted
// ones, the thread's lp, remainder of the word's first entry) for the words of
// 32 slots of group g; the last group's: extra words more.
template <typename F>
__device__ __forceinline__ void db_table(uint32_t g, uint32_t qb, uint32_t ngroups, const uint32_t* __restrict__ gsize, uint32_t cap,
                                         const uint8_t* __restrict__ counts, const uint8_t* __restrict__ rems,
                                         const DbThread* __restrict__ th, const uint4* __restrict__ pre,
                                         const uint32_t* __restrict__ spill, uint32_t extra,
                                         const uint32_t* __restrict__ ctr, F write) {
  __shared__ __align__(16) uint32_t s_rem[(DB_SPILL + PS_TILE) / 4];  // the spill's bytes end where the group's begin
  __shared__ uint32_t s_f[DB_PW], s_r[DB_PW];
  __shared__ uint32_t s_tmp[PS_THREADS / 64], s_all;
  const uint32_t t = threadIdx.x, q0 = g << qb, nw = 1u << (qb - 5);
  const RS X = rs_unpack(pre[g]);
  const uint32_t s = X.lp > q0 ? X.lp - q0 : 0u;
  {
    const uint32_t m = gsize[g];
    const uint4* d = reinterpret_cast<const uint4*>(rems + (uint64_t)g * cap);
    for (uint32_t i = t; i < (m + 15) / 16; i += PS_THREADS) reinterpret_cast<uint4*>(s_rem)[DB_SPILL / 16 + i] = d[i];
    if (t < s) {
      const uint32_t kept = X.c - rs_unpack(pre[g - 1]).c;
      reinterpret_cast<uint8_t*>(s_rem)[DB_SPILL - s + t] = rems[(uint64_t)(g - 1) * cap + kept - s + t];
    }
  }
  uint4 c0 = make_uint4(0u, 0u, 0u, 0u), c1 = c0;
  uint32_t lp = 0;
  if (t < nw) {
    const uint4* p = reinterpret_cast<const uint4*>(counts + q0 + DB_Q * t);
    c0 = p[0];
    c1 = p[1];
    const DbThread x = th[(uint64_t)g * PS_THREADS + t];
    const uint32_t l = add_sat(X.lp, x.kept);
    lp = l > x.lp ? l : x.lp;
  }
  for (uint32_t i = t; i < DB_PW; i += PS_THREADS) {
    const uint32_t n = 32 * i >= s ? 0u : s - 32 * i;
    s_f[i] = n >= 32 ? ~0u : (1u << n) - 1u;
    s_r[i] = n ? spill[(uint64_t)g * DB_SW + i] : 0u;
  }
  __syncthreads();
  // the thread's runs
  const uint32_t fr0 = DB_Q * t, lr = lp > q0 ? lp - q0 : 0u;  // (slots from q0 on)
  const uint32_t base = lr > fr0 ? lr : fr0;
  uint32_t occ = 0, own = 0, loc = 0;
  uint64_t starts = 0, taken = 0;
  int32_t fr = (int32_t)fr0 - (int32_t)base;  // the quotient, from base
#pragma unroll 1
  for (uint32_t h = 0; h < 2; ++h) {
    const uint32_t c[4] = {c0.x, c0.y, c0.z, c0.w};
    c0 = c1;
    uint32_t o = 0, w = 0;
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
      const uint32_t x = (c[j >> 2] >> (8 * (j & 3))) & 0xFFu;
      const uint32_t nz = x ? 1u : 0u;
      const uint32_t at = (int32_t)loc > fr ? loc : (uint32_t)fr;
      o |= nz << j;
      w |= (at == (uint32_t)fr ? 1u : 0u) << j;
      starts |= (uint64_t)nz << (at & 63);
      // taken slots: one bit after each run less one at its start (nothing
      // when the run is empty)
      taken += (1ull << ((at + x) & 63)) - (1ull << (at & 63));
      loc = at + x;
      ++fr;
    }
    occ |= o << (16 * h);
    own |= w << (16 * h);
  }
  own &= occ;
  if (loc < 64) {
    if (occ) {
      const uint32_t w = base >> 5, sh = base & 31;
      auto put = [&](uint32_t* plane, uint64_t v) {
        const uint64_t lo = v << sh;
        const uint32_t hi = sh ? (uint32_t)(v >> (64 - sh)) : 0u;
        if ((uint32_t)lo && w < DB_PW) atomicOr(&plane[w], (uint32_t)lo);
        if ((uint32_t)(lo >> 32) && w + 1 < DB_PW) atomicOr(&plane[w + 1], (uint32_t)(lo >> 32));
        if (hi && w + 2 < DB_PW) atomicOr(&plane[w + 2], hi);
      };
      put(s_r, starts);
      put(s_f, taken);
    }
  } else {
    uint32_t next = base;
    for (uint32_t left = occ; left; left &= left - 1u) {
      const uint32_t j = (uint32_t)__builtin_ctz(left), x = counts[q0 + fr0 + j];
      const uint32_t at = next > fr0 + j ? next : fr0 + j;
      next = at + x;
      if ((at >> 5) < DB_PW) atomicOr(&s_r[at >> 5], 1u << (at & 31));
      for (uint32_t b = at; b < next && (b >> 5) < DB_PW; b = (b | 31u) + 1) {
        const uint32_t e = next < (b | 31u) + 1 ? next : (b | 31u) + 1;
        atomicOr(&s_f[b >> 5], (e - b == 32 ? ~0u : (1u << (e - b)) - 1u) << (b & 31));
      }
    }
    // unshifted quotients: the run starts at the quotient's own slot
    own = 0;
    next = base;
    for (uint32_t left = occ; left; left &= left - 1u) {
      const uint32_t j = (uint32_t)__builtin_ctz(left), x = counts[q0 + fr0 + j];
      if (next <= fr0 + j) {
        own |= 1u << j;
        next = fr0 + j;
      }
      next += x;
    }
  }
  __syncthreads();
  const uint32_t f = t < nw ? s_f[t] : 0u, n = (uint32_t)__popc(f);
  const uint32_t e = DB_SPILL - s + block_excl_scan<PS_THREADS>(n, s_tmp);
  const uint8_t* rem8 = reinterpret_cast<const uint8_t*>(s_rem);
  if (g + 1 < ngroups) extra = 0;
  if (t == nw - 1) s_all = e + n;
  if (extra) __syncthreads();  // (uniform)
  // 32 slots a thread, then the last group's spill
#pragma unroll 1
  for (uint32_t u = t, at = e; u < nw + extra; u += nw) {
    if (t >= nw) break;
    if (u >= nw) {
      occ = own = 0u;
      at = s_all;
      for (uint32_t i = nw; i < u; ++i) at += (uint32_t)__popc(s_f[i]);
    }
    const uint32_t tk = s_f[u], st = s_r[u];
    const uint32_t last = tk & ~((tk >> 1 | s_f[u + 1] << 31) & ~(st >> 1 | s_r[u + 1] << 31));
    write(u, tk, st, last, occ, own, lp, rem8 + at);
  }
}

// SQF slots.  occupied, continuation (not a run's first) and shifted (not in
// its quotient's own slot) bits from the planes.
template <int BPE>
__global__ __launch_bounds__(PS_THREADS, 8) void k_db_sqf(uint8_t* __restrict__ tb, uint32_t S,
                                                          const uint32_t* __restrict__ gsize, uint32_t cap,
                                                          uint32_t qb, const uint8_t* __restrict__ counts,
                                                          const uint8_t* __restrict__ rems,
                                                          const DbThread* __restrict__ th,
                                                          const uint4* __restrict__ pre,
                                                          const uint32_t* __restrict__ spill, uint32_t ngroups,
                                                          const uint32_t* __restrict__ ctr) {
  if (ctr[CTR_ERR] || ctr[CTR_MISC]) return;
  const uint32_t g = blockIdx.x;
  const bool vec = (reinterpret_cast<uintptr_t>(tb) & 15u) == 0;
  // the slots to write: the last group's end with its last entry
  uint32_t hi = (g + 1) << qb;
  if (g + 1 == ngroups && ctr[CTR_MISC + 3] > hi) hi = ctr[CTR_MISC + 3];
  if (hi > S) hi = S;
  db_table(g, qb, ngroups, gsize, cap, counts, rems, th, pre, spill, DB_SW, ctr,
           [&](uint32_t u, uint32_t tk, uint32_t st, uint32_t, uint32_t occ, uint32_t own, uint32_t, const uint8_t* rem) {
             const uint32_t s0 = (g << qb) + 32 * u;
             if (s0 >= hi) return;
             uint8_t* d = tb + (uint64_t)s0 * BPE;
             const uint32_t cont = tk & ~st, shifted = tk & ~own;
#pragma unroll
             for (uint32_t k = 0; k < 2 * BPE; ++k) {  // 16 bytes
               uint32_t x[4];
#pragma unroll
               for (uint32_t i = 0; i < 4; ++i) {
                 constexpr uint32_t PER = 4 / BPE;
                 const uint32_t j0 = (16 / BPE) * k + PER * i;
                 uint32_t v = 0;
#pragma unroll
                 for (uint32_t z = 0; z < PER; ++z) {
                   const uint32_t j = j0 + z, bit = (tk >> j) & 1u;
                   if (BPE == 1) {
                     v |= (bit ? (uint32_t)*rem << 3 : 0u) << (8 * z);
                   } else {
                     const uint32_t b = bit ? (uint32_t)*rem << 3 : 0u, o = (occ >> j) & 1u, n = (cont >> j) & 1u,
                                    h = (shifted >> j) & 1u, y = b | o << 2 | n << 1 | h;
                     v |= ((y & 0xFFu) << 8 | y >> 8) << (16 * z);
                   }
                   rem += bit;
                 }
                 if (BPE == 1) {
                   auto spread = [&](uint32_t m) { return __umul24((m >> j0) & 15u, 0x204081u) & 0x01010101u; };
                   v |= spread(occ) << 2 | spread(cont) << 1 | spread(shifted);
                 }
                 x[i] = v;
               }
               if (vec && s0 + 32 <= hi) {
                 reinterpret_cast<uint4*>(d)[k] = make_uint4(x[0], x[1], x[2], x[3]);
               } else {
#pragma unroll
                 for (uint32_t i = 0; i < 16; ++i)
                   if (s0 + (16 * k + i) / BPE < hi) d[16 * k + i] = (uint8_t)(x[i >> 2] >> (8 * (i & 3)));
               }
             }
           });
}

// RSQF blocks: R = 8, or 0 (rr bits, at most 7).  Even threads hold a
// block's first half.
template <int R>
__global__ __launch_bounds__(PS_THREADS, 8) void k_db_rsqf(uint8_t* __restrict__ meta, uint8_t* __restrict__ rem_base,
                                                           uint32_t rr, const uint32_t* __restrict__ gsize, uint32_t cap,
                                                           uint32_t qb, const uint8_t* __restrict__ counts,
                                                           const uint8_t* __restrict__ rems,
                                                           const DbThread* __restrict__ th,
                                                           const uint4* __restrict__ pre,
                                                           const uint32_t* __restrict__ spill, uint32_t ngroups,
                                                           const uint32_t* __restrict__ ctr) {
  if (ctr[CTR_ERR] || ctr[CTR_MISC]) return;
  const uint32_t g = blockIdx.x, q0 = g << qb;
  const uint32_t end = ctr[CTR_MISC + 1];
  db_table(g, qb, ngroups, gsize, cap, counts, rems, th, pre, spill, 2u, ctr,
           [&](uint32_t u, uint32_t tk, uint32_t, uint32_t last, uint32_t occ, uint32_t, uint32_t lp, const uint8_t* rem) {
             const uint32_t s0 = q0 + 32 * u;  // slot, and the first quotient
             const uint32_t occ1 = (uint32_t)__shfl_xor((int)occ, 1), last1 = (uint32_t)__shfl_xor((int)last, 1);
             const uint32_t lp0 = (uint32_t)__shfl_xor((int)lp, 1);
             uint4* mt = reinterpret_cast<uint4*>(meta + (uint64_t)(s0 >> 6) * 32);
             if ((u & 1) == 0) {
               mt[0] = make_uint4(occ, occ1, last, last1);
             } else {
               // slots of the block that entries of earlier quotients take
               const uint32_t l = u < (1u << (qb - 5)) ? lp0 : end, b0 = s0 & ~63u;
               mt[1] = make_uint4(l > b0 ? (l - b0) & 0xFFu : 0u, 0u, 0u, 0u);
             }
             if (R == 8) {
               uint4* d = reinterpret_cast<uint4*>(rem_base + s0);
#pragma unroll
               for (uint32_t k = 0; k < 2; ++k) {
                 uint32_t x[4];
#pragma unroll
                 for (uint32_t i = 0; i < 4; ++i) {
                   uint32_t v = 0;
#pragma unroll
                   for (uint32_t z = 0; z < 4; ++z) {
                     const uint32_t bit = (tk >> (16 * k + 4 * i + z)) & 1u;
                     v |= (bit ? (uint32_t)*rem : 0u) << (8 * z);
                     rem += bit;
                   }
                   x[i] = v;
                 }
                 d[k] = make_uint4(x[0], x[1], x[2], x[3]);
               }
             } else {
               uint32_t* d = reinterpret_cast<uint32_t*>(rem_base + (uint64_t)(s0 >> 5) * 4 * rr);
               uint64_t acc = 0;
               uint32_t fill = 0;
#pragma unroll 4
               for (uint32_t j = 0; j < 32; ++j) {
                 const uint32_t bit = (tk >> j) & 1u;
                 acc |= (uint64_t)(bit ? (uint32_t)*rem : 0u) << fill;
                 rem += bit;
                 fill += rr;
                 if (fill >= 32) {
                   *d++ = (uint32_t)acc;
                   acc >>= 32;
                   fill -= 32;
                 }
               }
             }
           });
}

// ---------------------------------------------------------------- host
static inline size_t ps_bytes(const PsPlan& p) {
  const size_t room = (size_t)p.ngroups * p.cap;
  return aligned_bytes(room * 4) + aligned_bytes(((size_t)p.ngroups + 1) * 4) + aligned_bytes((size_t)1 << (p.qb + p.gb)) +
         aligned_bytes(room) +
         aligned_bytes((size_t)p.ngroups * PS_THREADS * sizeof(DbThread)) + aligned_bytes((size_t)p.ngroups * 16) +
         aligned_bytes(((size_t)p.ngroups + 1) * DB_SW * 4) +
         aligned_bytes(((p.ngroups + RBS_PER - 1) / RBS_PER) * 16) + 2048;
}

// After a build: whether the stream's next one may expect few repeats -- three
// of four keys kept (NoDup), no run past DB_LONG entries among those that
// k_db_spill reads.  Until a build has shown it, many are expected: the form
// for many costs 1% on keys without, the other up to 60% on keys with.
static inline bool db_few(const DeviceState& ds, uint32_t n, bool done) {
  return done && (uint64_t)ds.h_pinned[CTR_COUNT] * 4 >= (uint64_t)n * 3 && ds.h_pinned[CTR_MISC + 2] == 0;
}

struct DbRuns {
  const uint32_t* gsize;
  uint8_t *counts, *rems;
  DbThread* th;
  uint4* agg;       // states before every group, after the scan
  uint32_t* spill;  // what reaches into every group
};
// Partition and runs of the raw keys; scans the locations (slots: the
// table's).  WIDE: fingerprints of more than 32 bits.  few: the keys are
// expected to hold few repeats (db_few).
template <bool WIDE>
static gqf_status db_runs(hipStream_t s, Arena& ar, const PsPlan& p, const uint32_t* keys, uint32_t fp_bits, uint32_t n,
                          uint32_t r, bool unique, bool few, uint64_t slots, uint32_t* ctr, DbRuns* o) {
  const uint32_t nd = p.ngroups, bits = p.shift + p.gb, hbits = bits > 32 ? bits - 32 : 0u;
  const size_t room = (size_t)nd * p.cap;
  uint32_t* mid = ar.take<uint32_t>(room);
  uint32_t* gsize = ar.take<uint32_t>(nd + 1);  // and whether one is past its room
  o->counts = ar.take<uint8_t>((size_t)1 << (p.qb + p.gb));
  o->rems = ar.take<uint8_t>(room);
  o->th = ar.take<DbThread>((size_t)nd * PS_THREADS);
  o->agg = ar.take<uint4>(nd);
  o->spill = ar.take<uint32_t>(((size_t)nd + 1) * DB_SW);
  if (ar.used > ar.cap) {
    set_error("internal: build workspace overflow");
    return GQF_ERR_INVALID;
  }
  o->gsize = gsize;
  GQF_LAUNCH(k_ps_reset, dim3(1), dim3(PS_THREADS), 0, s, gsize, nd + 1, ctr);
  GQF_LAUNCH_B((double)n * 8.0, (k_ps_scatter<WIDE, false>), dim3(p.wgs), dim3(PS_THREADS), 0, s, keys, n, fp_bits,
               p.shift, nd, hbits, p.tile, p.cap, gsize, mid, ctr, PsBack{});
  const double rb = (double)n * 5.0 + (double)((uint64_t)1 << (p.qb + p.gb));
#define GQF_DB_RUNS(U_, Q_, M_)                                                                                             \
  GQF_LAUNCH_B(rb, (k_db_runs<U_, Q_, M_>), dim3(nd), dim3(PS_THREADS), 0, s, mid, gsize, nd, p.cap, p.qb, r, o->counts, o->rems, \
               o->th, o->agg, ctr)
#define GQF_DB_RUNS_Q(U_)                          \
  do {                                             \
    if (p.qb == 15 && few) GQF_DB_RUNS(U_, 32, false); \
    else if (p.qb == 15) GQF_DB_RUNS(U_, 32, true);    \
    else if (p.qb == 14) GQF_DB_RUNS(U_, 16, true);    \
    else if (p.qb == 13) GQF_DB_RUNS(U_, 8, true);     \
    else GQF_DB_RUNS(U_, 4, true);                     \
  } while (0)
  static_assert(DB_QB == 15, "the quotients of a thread: 2^qb / 1024");
  if (unique) GQF_DB_RUNS_Q(true);
  else GQF_DB_RUNS_Q(false);
#undef GQF_DB_RUNS_Q
#undef GQF_DB_RUNS
  GQF_TRY(rb_scan(s, ar, o->agg, nd, slots, ctr, nullptr));
  GQF_LAUNCH(k_db_spill, dim3(nd), dim3(256), 0, s, o->counts, p.qb, o->agg, nd, o->spill, ctr);
  return GQF_OK;
}

}  // namespace gqf
