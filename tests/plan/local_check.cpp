// Host-only check of the localized updates' region code (sl_insert, sl_erase, SlPlanes)
// and of the rules that cut a sorted batch into regions: random canonical
// SQF tables, random sorted batches, the regions updated in a random order,
// the result compared with the canonical layout of the expected entries.
// Every table access is checked against the table's bounds and, per region,
// against the slots that region may write.  Built with hipcc for the host
// alone by tests/test_plans.py; prints "local ok" when nothing failed.
#include <algorithm>
#include <cstdio>
#include <random>
#include <set>
#include <vector>

#include "../../gpuquotientfilters_amd/csrc/gqf_rsqf_local.hpp"
#include "../../gpuquotientfilters_amd/csrc/gqf_sqf_local.hpp"

using namespace gqf;

static int fails = 0;
static void fail(const char* what, uint32_t a, uint32_t b) {
  if (++fails <= 10) std::printf("FAIL %s %u %u\n", what, a, b);
}

// The canonical table of sorted fingerprints; false if it does not fit.
static bool canon(const std::vector<uint32_t>& fps, uint32_t S, uint32_t r, std::vector<uint32_t>& t) {
  t.assign(S, 0u);
  int64_t loc = -1, last = -1;
  for (uint32_t f : fps) {
    const int64_t q = f >> r;
    loc = std::max(q, loc + 1);
    if (loc >= (int64_t)S) return false;
    t[(size_t)loc] |= ((f & ((1u << r) - 1u)) << 3) | (q == last ? 2u : 0u) | (loc != q ? 1u : 0u);
    if (q != last) t[(size_t)q] |= 4u;
    last = q;
  }
  return true;
}

struct Acc {
  std::vector<uint32_t>& t;
  uint32_t lo, hi;  // slots this region may write
  uint32_t get(uint32_t i) const {
    if (i >= t.size()) {
      if (i > t.size() + 1) fail("read far past the end", i, (uint32_t)t.size());
      return 0u;
    }
    return t[i];
  }
  void put(uint32_t i, uint32_t e) {
    if (i < lo || i > hi || i >= t.size()) return fail("write outside the region", i, lo);
    t[i] = e;
  }
};

// A window's planes from slot `base` on, and back.
template <int BPE>
struct Planes {
  std::vector<unsigned long long> occ, cont, shf, rem;
  SlPlanes<BPE> m;
  Planes(const std::vector<uint32_t>& t, uint32_t base) {
    const uint32_t nb = ((uint32_t)t.size() - base + 63) / 64;
    occ.assign(nb, 0);
    cont = shf = occ;
    rem.assign(nb * 8 * BPE, 0);
    m.occ = occ.data(), m.cont = cont.data(), m.shf = shf.data(), m.rem = rem.data();
    m.end = 64 * nb;
    m.dirty[0] = m.dirty[1] = 0;
    m.pend = 0;
    for (uint32_t s = base; s < t.size(); ++s) {
      const uint32_t i = s - base;
      occ[i >> 6] |= (uint64_t)((t[s] >> 2) & 1u) << (i & 63);
      cont[i >> 6] |= (uint64_t)((t[s] >> 1) & 1u) << (i & 63);
      shf[i >> 6] |= (uint64_t)(t[s] & 1u) << (i & 63);
      m.put_rem(i, t[s] >> 3);
    }
    if (t[base] & 1u) {
      uint32_t b = base;
      do {
        --b;
        m.pend += (t[b] & 4u ? 1u : 0u) - (t[b] & 2u ? 0u : 1u);
      } while (t[b] & 1u);
    }
  }
  uint32_t get(uint32_t i) const {
    return (m.get_rem(i) << 3) | (m.bit(m.occ, i) ? 4u : 0u) | (m.bit(m.cont, i) ? 2u : 0u) | (m.bit(m.shf, i) ? 1u : 0u);
  }
};

// The regions of `batch` (first keys at `heads`) in the order given: those
// that start before `base` on the elements, the others on the planes.
template <int BPE, bool INS>
static std::vector<uint32_t> on_planes(const std::vector<uint32_t>& t, const std::vector<uint32_t>& batch,
                                       const std::vector<uint32_t>& heads, const std::vector<uint32_t>& order, uint32_t r,
                                       uint32_t base) {
  const uint32_t S = (uint32_t)t.size(), rm = (1u << r) - 1u;
  std::vector<uint32_t> x(t);
  Planes<BPE> P(t, base);
  for (uint32_t i : order) {
    const uint32_t kb = i + 1 < heads.size() ? heads[i + 1] : (uint32_t)batch.size();
    Acc a{x, 0, S - 1};
    for (uint32_t k = heads[i]; k < kb; ++k) {
      const uint32_t fq = batch[k] >> r, fr = batch[k] & rm;
      if ((batch[heads[i]] >> r) < base) {
        if (INS) sl_insert(a, S, fq, fr);
        else sl_erase(a, S, fq, fr);
      } else {
        if (INS) P.m.insert(fq - base, fr);
        else P.m.erase(fq - base, fr);
      }
    }
  }
  for (uint32_t s = base; s < S; ++s) {
    const uint32_t e = P.get(s - base), b = (s - base) >> 6;
    if (e == t[s]) continue;
    if (b < 128 && !((P.m.dirty[b >> 6] >> (b & 63)) & 1ull)) fail("change outside the marked blocks", s, base);
    x[s] = e;
  }
  return x;
}

// RSQF: nb blocks, the canonical bits, remainders and offsets of sorted
// fingerprints (loc_i = max(fq_i, loc_{i-1} + 1)).
struct Rs {
  std::vector<unsigned long long> occ, ends, rem;
  std::vector<uint32_t> off;
  uint32_t nb, r;
  Rs(uint32_t nb_, uint32_t r_) : occ(nb_, 0), ends(nb_, 0), rem((size_t)nb_ * r_ + 1, 0), off(nb_, 0), nb(nb_), r(r_) {}
  bool fill(const std::vector<uint64_t>& fps) {
    int64_t loc = -1, last = -1;
    std::vector<int64_t> L(nb, -1);  // last location of a quotient below the block
    for (uint64_t f : fps) {
      const int64_t q = (int64_t)(f >> r);
      if (q != last && last >= 0) ends[(size_t)loc >> 6] |= 1ull << (loc & 63);
      loc = std::max(q, loc + 1);
      if (loc >= 64 * (int64_t)nb) return false;
      occ[(size_t)q >> 6] |= 1ull << (q & 63);
      for (uint32_t k = 0; k < r; ++k) {
        const uint64_t b = (uint64_t)loc * r + k;
        rem[b >> 6] |= (unsigned long long)((f >> k) & 1ull) << (b & 63);
      }
      for (size_t j = (size_t)(q >> 6) + 1; j < nb; ++j) L[j] = loc;
      last = q;
    }
    if (last >= 0) ends[(size_t)loc >> 6] |= 1ull << (loc & 63);
    for (uint32_t j = 0; j < nb; ++j) off[j] = L[j] >= 64 * (int64_t)j ? (uint32_t)(L[j] - 64 * (int64_t)j + 1) & 0xFFu : 0u;
    return true;
  }
  bool operator==(const Rs& o) const { return occ == o.occ && ends == o.ends && rem == o.rem && off == o.off; }
};

template <int R>
static void rsqf_case(std::mt19937& g, uint32_t r) {
  const uint32_t q = 6 + g() % 6, nb = (1u << q) / 64 + 1, S = 64 * nb;
  const uint32_t n = (uint32_t)(g() % 100 * (1u << q) / 100), m = 1 + g() % (1 + (1u << q) / 4);
  const uint64_t fm = (1ull << (q + r)) - 1;
  std::vector<uint64_t> base, batch;
  for (uint32_t i = 0; i < n; ++i) base.push_back(g() & fm);
  std::sort(base.begin(), base.end());
  for (uint32_t i = 0; i < m; ++i) batch.push_back(base.size() && g() % 2 ? base[g() % base.size()] : g() & fm);
  if (g() % 3 == 0)
    for (uint32_t i = 0; i < m; i += 1 + g() % 3) batch[i] = batch[0];
  std::sort(batch.begin(), batch.end());
  Rs t(nb, r);
  if (!t.fill(base)) return;
  // D at every slot, empty slots, boundaries
  std::vector<uint32_t> E(S + 1), D(S + 1), empties, lb(S);
  std::vector<unsigned long long> em(nb, 0);
  int32_t d = 0;
  for (uint32_t s = 0, l = 0; s < S; ++s) {
    E[s] = (uint32_t)empties.size();
    D[s] = (uint32_t)d;
    if (d == 0) l = s + 1;
    lb[s] = l;
    d += (int32_t)((t.occ[s >> 6] >> (s & 63)) & 1ull);
    if (d == 0) {
      empties.push_back(s);
      em[s >> 6] |= 1ull << (s & 63);
    }
    d -= (int32_t)((t.ends[s >> 6] >> (s & 63)) & 1ull);
  }
  auto run = [&](bool ins, const std::vector<uint32_t>& heads) {
    Rs x(t);
    std::vector<int32_t> off(nb, 0);
    RlPlanes<R> P;
    P.occ = x.occ.data(), P.ends = x.ends.data(), P.rem = x.rem.data(), P.empty = em.data(), P.off = off.data();
    P.end = S, P.r = r, P.dirty[0] = P.dirty[1] = 0;
    std::vector<uint32_t> order(heads.size());
    for (uint32_t i = 0; i < order.size(); ++i) order[i] = i;
    std::shuffle(order.begin(), order.end(), g);
    for (uint32_t i : order) {
      const uint32_t kb = i + 1 < heads.size() ? heads[i + 1] : m;
      const uint32_t a = (uint32_t)(batch[heads[i]] >> r);
      uint32_t e = a - 1;
      for (uint32_t k = heads[i]; k < kb; ++k) {
        const uint32_t fq = (uint32_t)(batch[k] >> r), fr = (uint32_t)batch[k] & ((1u << r) - 1u);
        if (ins) {
          e = P.next(em.data(), e + 1);
          P.insert(fq, fr, a, D[a], e);
        } else {
          P.erase(fq, fr, a, D[a]);
        }
      }
    }
    for (uint32_t j = 0; j < nb; ++j) {
      const bool changed = x.occ[j] != t.occ[j] || x.ends[j] != t.ends[j] || off[j] != 0;
      if (changed && !((P.dirty[j >> 6] >> (j & 63)) & 1ull)) fail("rsqf change outside the marked blocks", j, q);
      x.off[j] = (x.off[j] + (uint32_t)off[j]) & 0xFFu;
    }
    return x;
  };
  {
    std::vector<uint64_t> all(base);
    all.insert(all.end(), batch.begin(), batch.end());
    std::sort(all.begin(), all.end());
    std::vector<uint32_t> heads;
    bool fits = true;
    int64_t J = -1;
    for (uint32_t k = 0; k < m; ++k) {
      const int64_t e = E[batch[k] >> r];
      if (J < e) heads.push_back(k);
      J = std::max(J + 1, e);
      fits = fits && J < (int64_t)empties.size();
    }
    Rs want(nb, r);
    if (fits != want.fill(all)) fail("rsqf fits", q, r);
    if (fits && !(run(true, heads) == want)) fail("rsqf insert", q, r);
  }
  {
    std::multiset<uint64_t> ms(base.begin(), base.end());
    for (uint64_t b : batch) {
      auto p = ms.find(b);
      if (p != ms.end()) ms.erase(p);
    }
    std::vector<uint32_t> heads;
    for (uint32_t k = 0; k < m; ++k)
      if (k == 0 || lb[batch[k] >> r] > (uint32_t)(batch[k - 1] >> r) + 1) heads.push_back(k);
    Rs want(nb, r);
    (void)want.fill(std::vector<uint64_t>(ms.begin(), ms.end()));
    if (!(run(false, heads) == want)) fail("rsqf delete", q, r);
  }
}

int main() {
  std::mt19937 g(7);
  for (int it = 0; it < 1500; ++it) {
    rsqf_case<8>(g, 8);
    rsqf_case<0>(g, 1 + g() % 16);
  }
  for (int it = 0; it < 6000; ++it) {
    const uint32_t q = 3 + g() % 9, r = 1 + g() % 9;
    const uint32_t S = (uint32_t)((double)(1u << q) * 1.1);
    const uint32_t n = (uint32_t)(g() % 100 * (1u << q) / 100), m = 1 + g() % (1 + (1u << q) / 4);
    const bool dup = g() % 2;
    std::vector<uint32_t> base, batch, t, want;
    for (uint32_t i = 0; i < n; ++i) base.push_back(g() & ((1u << (q + r)) - 1u));
    std::sort(base.begin(), base.end());
    if (!dup) base.erase(std::unique(base.begin(), base.end()), base.end());
    for (uint32_t i = 0; i < m; ++i)
      batch.push_back(base.size() && g() % 2 ? base[g() % base.size()] : g() & ((1u << (q + r)) - 1u));
    if (g() % 3 == 0)  // one hot key
      for (uint32_t i = 0; i < m; i += 1 + g() % 3) batch[i] = batch[0];
    std::sort(batch.begin(), batch.end());
    if (!canon(base, S, r, t)) continue;
    // ---- insert
    {
      std::vector<uint32_t> all(base);
      for (uint32_t b : batch)
        if (!std::binary_search(all.begin(), all.end(), b)) all.insert(std::lower_bound(all.begin(), all.end(), b), b);
      std::vector<uint32_t> empties, E(S + 1, 0u);
      for (uint32_t s = 0; s < S; ++s) {
        E[s] = (uint32_t)empties.size();
        if ((t[s] & 7u) == 0) empties.push_back(s);
      }
      std::vector<uint32_t> J(m), heads;
      bool fits = true;
      for (uint32_t k = 0; k < m; ++k) {
        const uint32_t e = E[batch[k] >> r];
        J[k] = k && J[k - 1] + 1 > e ? J[k - 1] + 1 : e;
        fits = fits && J[k] < empties.size();
        if (k == 0 || J[k - 1] < e) heads.push_back(k);
      }
      if (fits) {
        if (!canon(all, S, r, want)) fail("fits", q, r);
        std::vector<uint32_t> x(t), order(heads.size());
        for (uint32_t i = 0; i < order.size(); ++i) order[i] = i;
        std::shuffle(order.begin(), order.end(), g);
        for (uint32_t i : order) {
          const uint32_t kb = i + 1 < heads.size() ? heads[i + 1] : m;
          Acc a{x, batch[heads[i]] >> r, empties[J[kb - 1]]};
          for (uint32_t k = heads[i]; k < kb; ++k) sl_insert(a, S, batch[k] >> r, batch[k] & ((1u << r) - 1u));
        }
        if (x != want) fail("insert", q, r);
        const uint32_t base = g() % 2 ? 0u : (g() % (1u << q)) & ~63u;
        if (r <= 5 && on_planes<1, true>(t, batch, heads, order, r, base) != want) fail("insert, planes", q, r);
        if (on_planes<2, true>(t, batch, heads, order, r, base) != want) fail("insert, 2-byte planes", q, r);
      }
    }
    // ---- delete
    {
      std::multiset<uint32_t> ms(base.begin(), base.end());
      for (uint32_t b : batch) {
        auto p = ms.find(b);
        if (p != ms.end()) ms.erase(p);
      }
      (void)canon(std::vector<uint32_t>(ms.begin(), ms.end()), S, r, want);
      std::vector<uint32_t> lb(S), heads;  // 1 + the last boundary at or before a slot
      for (uint32_t s = 0, l = 0; s < S; ++s) lb[s] = l = t[s] & 1u ? l : s + 1;
      for (uint32_t k = 0; k < m; ++k)
        if (k == 0 || lb[batch[k] >> r] > (batch[k - 1] >> r) + 1) heads.push_back(k);
      std::vector<uint32_t> x(t), order(heads.size());
      for (uint32_t i = 0; i < order.size(); ++i) order[i] = i;
      std::shuffle(order.begin(), order.end(), g);
      for (uint32_t i : order) {
        const uint32_t kb = i + 1 < heads.size() ? heads[i + 1] : m;
        uint32_t hi = batch[kb - 1] >> r;  // the region ends before the next boundary
        while (hi + 1 < S && (t[hi + 1] & 1u)) ++hi;
        Acc a{x, batch[heads[i]] >> r, hi};
        for (uint32_t k = heads[i]; k < kb; ++k) sl_erase(a, S, batch[k] >> r, batch[k] & ((1u << r) - 1u));
      }
      if (x != want) fail("delete", q, r);
      const uint32_t base = g() % 2 ? 0u : (g() % (1u << q)) & ~63u;
      if (r <= 5 && on_planes<1, false>(t, batch, heads, order, r, base) != want) fail("delete, planes", q, r);
      if (on_planes<2, false>(t, batch, heads, order, r, base) != want) fail("delete, 2-byte planes", q, r);
    }
  }
  // the window states' composition against the recurrence, key by key
  for (int it = 0; it < 2000; ++it) {
    LW p{0, 0, 0u, 0u};
    int64_t o = 0;
    for (int w = 0; w < 20; ++w) {
      const int32_t e = (int32_t)(g() % 40), nk = (int32_t)(g() % 30);
      std::vector<int32_t> E;
      for (int32_t k = 0; k < nk; ++k) E.push_back((int32_t)(g() % (uint32_t)(e + 1)));
      std::sort(E.begin(), E.end());
      int64_t c = o;
      int32_t M = 0;
      for (int32_t k = 0; k < nk; ++k) {
        c = std::max<int64_t>(c, E[(size_t)k]) + 1;
        M = std::max(M, E[(size_t)k] - k);
      }
      o = std::max<int64_t>(0, c - e);
      const int32_t a = nk - e;
      p = lw_combine(p, LW{a, std::max(0, nk ? M + a : 0), 0u, 0u});
      if (std::max(p.a, p.b) != o) fail("state", (uint32_t)w, (uint32_t)o);
    }
  }
  if (!fails) std::printf("local ok\n");
  return fails ? 1 : 0;
}
