// Host-only model of the RSQF's localized updates window by window: the plan's
// rules, the windows' scan and the apply kernel's limits (the blocks of the
// next window that a region may reach) over random and adversarial tables --
// stretches that are almost full right after a window's end, batches crowded
// at it, windows applied in a random order.  Every batch that the rules
// accept has to give the canonical table.  Region code, states and bounds are
// those of the kernels' headers.  Built with hipcc for the host alone by
// tests/test_local_windows.py; prints "windows ok" when nothing failed.
#include <algorithm>
#include <cstdio>
#include <random>
#include <set>
#include <vector>

#include "../../gpuquotientfilters_amd/csrc/gqf_rsqf_local.hpp"

using namespace gqf;

static int fails = 0;
static void fail(const char* what, uint32_t a, uint32_t b) {
  if (++fails <= 10) std::printf("FAIL %s %u %u\n", what, a, b);
}

using U = unsigned long long;
constexpr uint32_t r = 8;

// nb blocks: the canonical bits, remainders and offsets of sorted
// fingerprints (loc_i = max(fq_i, loc_{i-1} + 1)).
struct Table {
  std::vector<U> occ, ends, rem;
  std::vector<uint32_t> off;
  uint32_t nb;
  explicit Table(uint32_t nb_) : occ(nb_, 0), ends(nb_, 0), rem((size_t)nb_ * r, 0), off(nb_, 0), nb(nb_) {}
  bool fill(const std::vector<uint64_t>& fps) {
    int64_t loc = -1, last = -1;
    std::vector<int64_t> at(nb, -1);  // the last location of the quotients of each block
    for (uint64_t f : fps) {
      const int64_t q = (int64_t)(f >> r);
      if (q != last && last >= 0) ends[(size_t)loc >> 6] |= 1ull << (loc & 63);
      loc = std::max(q, loc + 1);
      if (loc >= 64 * (int64_t)nb) return false;
      occ[(size_t)q >> 6] |= 1ull << (q & 63);
      rem[((size_t)loc * r) >> 6] |= (U)(f & 0xFFu) << ((loc * r) & 63);
      at[(size_t)q >> 6] = loc;
      last = q;
    }
    if (last >= 0) ends[(size_t)loc >> 6] |= 1ull << (loc & 63);
    int64_t L = -1;
    for (uint32_t j = 0; j < nb; ++j) {
      off[j] = L >= 64 * (int64_t)j ? (uint32_t)(L - 64 * (int64_t)j + 1) & 0xFFu : 0u;
      L = std::max(L, at[j]);
    }
    return true;
  }
  bool operator==(const Table& o) const { return occ == o.occ && ends == o.ends && rem == o.rem && off == o.off; }
};

struct Plan {
  uint32_t W = 0;
  bool ok = true;
  std::vector<uint32_t> bstart, info, D, fb;
  std::vector<U> empty;
  std::vector<LW> st;
  std::vector<uint2> pre;
};

// k_rl_plan and the scan.
template <bool INS>
static Plan plan(const Table& t, const std::vector<uint64_t>& B, uint32_t min_heads) {
  Plan p;
  const uint32_t nb = t.nb, n = (uint32_t)B.size(), W = lw_windows((uint64_t)nb * 64);
  p.W = W;
  p.bstart.assign(W + 1, n);
  for (uint32_t w = 0; w <= W; ++w)
    p.bstart[w] = (uint32_t)(std::lower_bound(B.begin(), B.end(), ((uint64_t)w * LW_SLOTS) << r) - B.begin());
  p.info.assign(n, 0);
  p.D.assign(n, 0);
  p.fb.assign(W, 0);
  p.empty.assign(nb, 0);
  p.st.assign(W, LW{0, 0, 0u, 0u});
  // per slot: the empty slots, the boundaries, D
  std::vector<int32_t> D(64 * nb);
  std::vector<char> mask(64 * W, 0);
  mask.resize((size_t)W * LW_SLOTS, 0);
  int32_t d = 0;
  for (uint32_t s = 0; s < 64 * nb; ++s) {
    D[s] = d;
    if (!INS) mask[s] = d <= 0;
    d += (int32_t)((t.occ[s >> 6] >> (s & 63)) & 1);
    if (INS) mask[s] = d <= 0;
    d -= (int32_t)((t.ends[s >> 6] >> (s & 63)) & 1);
  }
  for (uint32_t w = 0; w < W; ++w) {
    const uint32_t b0 = p.bstart[w], nk = p.bstart[w + 1] - b0, base = w * LW_SLOTS;
    const bool after = w > 0 && p.bstart[w - 1] != b0;
    if (nk == 0 && !after) {
      p.st[w] = LW{-LW_SPILL, 0, base + 1, 0u};
      continue;
    }
    const char* m = mask.data() + base;
    uint32_t e = 0, first = LW_SLOTS, last = 0, end = 0;
    int32_t held = 0;
    for (uint32_t s = 0; s < LW_SLOTS; ++s)
      if (m[s]) {
        ++e;
        if (s < 64 * RL_HALO) ++held;
        if (first == LW_SLOTS) first = s;
        last = s + 1;
        if (INS) p.empty[(base + s) >> 6] |= 1ull << (s & 63);
      }
    bool bad = nk > LW_KEYS;
    if (INS) bad = bad || (w + 1 < W && e < (uint32_t)LW_SPILL);
    else bad = bad || first == LW_SLOTS;
    if (nb <= 64 * w + RL_HALO) held = 1 << 20;
    int32_t M = 0, fit = held - (int32_t)nk;
    uint32_t heads = 0;
    for (uint32_t k0 = 0; !bad && k0 < nk; k0 += 64) {
      bool any = false;
      for (uint32_t k = k0; k < std::min(nk, k0 + 64); ++k) {
        const uint32_t s = (uint32_t)(B[b0 + k] >> r) - base;
        p.D[b0 + k] = (uint32_t)D[base + s];
        bool head;
        if (INS) {
          const int32_t E = (int32_t)std::count(m, m + s, 1), v = E - (int32_t)k;
          p.info[b0 + k] = (uint32_t)E;
          head = v >= M;
          M = std::max(M, v);
          fit = std::max(fit, lw_fit(v, held, (int32_t)k));
        } else {
          uint32_t lb = 0;
          for (uint32_t z = 0; z <= s; ++z)
            if (m[z]) lb = z + 1;
          head = lb > (k ? (uint32_t)(B[b0 + k - 1] >> r) - base + 1 : 0u);
          p.info[b0 + k] = head;
          end = s + 1;
        }
        any |= head;
        heads += head;
      }
      if (k0 + 64 <= nk && !any) bad = true;
    }
    const int32_t a = INS ? (int32_t)nk - (int32_t)e : -2;
    int32_t b = INS ? (nk ? M + a : 0) : last <= end;
    if (b < 0) b = 0;
    if (bad) b = LW_BAD;
    p.st[w] = LW{a, b, INS ? lw_room(fit) : (last ? base + last : 0u) | (first > 64 * RL_HALO ? LW_FAR : 0u), heads};
    p.fb[w] = first;
  }
  p.pre.resize(W);
  LW acc{0, 0, 0u, 0u};
  for (uint32_t w = 0; w < W; ++w) {
    if (lw_put<INS>(acc, p.st[w], w, W, p.pre.data(), min_heads)) p.ok = false;
    acc = lw_combine(acc, p.st[w]);
  }
  return p;
}

// k_rl_apply for window w.
template <bool INS>
static void apply(Table& t, const Plan& p, const std::vector<uint64_t>& B, uint32_t w) {
  const uint32_t nb = t.nb, n = (uint32_t)B.size(), b0 = p.bstart[w], b1 = p.bstart[w + 1], nk = b1 - b0;
  if (nk == 0) return;
  const uint32_t base = w * LW_SLOTS, bw = w * 64;
  std::vector<uint32_t> head;
  int32_t M = (int32_t)p.pre[w].x;
  for (uint32_t k = 0; k < nk; ++k) {
    bool h;
    if (INS) {
      const int32_t v = (int32_t)p.info[b0 + k] - (int32_t)k;
      h = v >= M;
      M = std::max(M, v);
    } else {
      h = p.info[b0 + k] != 0;
      if (k == 0 && !h) h = b0 == 0 || p.pre[w].y > (uint32_t)(B[b0 - 1] >> r) + 1;
    }
    if (h) head.push_back(k);
  }
  if (head.empty()) return;
  uint32_t k1 = b1, hi = LW_SLOTS - 1;
  if (INS) {
    uint32_t need = w + 1 < p.W ? p.pre[w + 1].x : 0u;
    if (need) {
      uint32_t c = bw + 64;
      U em = c < nb ? p.empty[c] : 0ull;
      while ((uint32_t)__builtin_popcountll(em) < need && c + 1 < nb && c + 1 < bw + RL_BLOCKS) {
        need -= (uint32_t)__builtin_popcountll(em);
        em = p.empty[++c];
      }
      for (; need > 1; --need) em &= em - 1ull;
      for (;;) {
        while (em == 0 && c + 1 < nb && c + 1 < bw + RL_BLOCKS) em = p.empty[++c];
        if (em == 0) {
          fail("the region leaves the blocks held", w, p.pre[w + 1].x);
          break;
        }
        hi = 64 * (c - bw) + (uint32_t)__builtin_ctzll(em);
        em &= em - 1ull;
        if (k1 >= n || (uint32_t)(B[k1] >> r) > base + hi) break;
        ++k1;
      }
    }
  } else {
    uint32_t hp = (uint32_t)(B[b1 - 1] >> r);
    if (w + 1 < p.W && p.fb[w + 1] && p.pre[w + 1].y <= hp + 1) hi = LW_SLOTS + p.fb[w + 1] - 1;
    while (k1 < n) {
      const uint32_t h = (uint32_t)(B[k1] >> r), w2 = h / LW_SLOTS;
      if (h - w2 * LW_SLOTS >= p.fb[w2] || p.pre[w2].y > hp + 1) break;
      hp = h;
      ++k1;
    }
  }
  uint32_t held = hi / 64 + 1;
  if (held > RL_BLOCKS) {
    fail("blocks held", w, held);
    held = RL_BLOCKS;
  }
  std::vector<U> occ(held, 0), ends(held, 0), em(held, 0), rem((size_t)held * r + 1, 0);
  std::vector<int32_t> off(held, 0);
  for (uint32_t i = 0; i < held && bw + i < nb; ++i) {
    occ[i] = t.occ[bw + i];
    ends[i] = t.ends[bw + i];
    if (INS) em[i] = p.empty[bw + i];
    for (uint32_t z = 0; z < r; ++z) rem[(size_t)i * r + z] = t.rem[(size_t)(bw + i) * r + z];
  }
  RlPlanes<r> m;
  m.occ = occ.data(), m.ends = ends.data(), m.rem = rem.data(), m.empty = em.data(), m.off = off.data();
  m.end = 64 * held, m.r = r, m.dirty[0] = m.dirty[1] = 0;
  for (size_t ri = 0; ri < head.size(); ++ri) {
    const uint32_t ka = b0 + head[ri], kb = ri + 1 < head.size() ? b0 + head[ri + 1] : k1;
    const uint32_t a = (uint32_t)(B[ka] >> r) - base, D = p.D[ka];
    uint32_t e = a - 1;
    for (uint32_t k = ka; k < kb; ++k) {
      const uint32_t fq = (uint32_t)(B[k] >> r) - base, fr = (uint32_t)B[k] & 0xFFu;
      if (fq >= m.end) {
        fail("a key past the blocks held", w, fq);
        break;
      }
      if (INS) {
        e = m.next(em.data(), e + 1);
        m.insert(fq, fr, a, D, e);
      } else {
        m.erase(fq, fr, a, D);
      }
    }
  }
  const uint32_t lo = (INS ? p.pre[w].x > 0 : p.fb[w] > 0) ? (uint32_t)(B[b0 + head[0]] >> r) - base : 0u;
  for (uint32_t i = 0; i < held && bw + i < nb; ++i) {
    if (!((m.dirty[i >> 6] >> (i & 63)) & 1)) continue;
    U x = ~0ull;
    if (i == lo >> 6) x &= m.from(lo & 63);
    if (i == hi >> 6) x &= m.upto(hi & 63);
    t.occ[bw + i] ^= (t.occ[bw + i] ^ occ[i]) & x;
    t.ends[bw + i] ^= (t.ends[bw + i] ^ ends[i]) & x;
    t.off[bw + i] = (t.off[bw + i] + (uint32_t)off[i]) & 0xFFu;
    for (uint32_t s = 0; s < 64; ++s)
      if ((x >> s) & 1) {
        U& g = t.rem[((size_t)(bw + i) * 64 + s) * r / 64];
        const U v = rem[((size_t)i * 64 + s) * r / 64], z = 0xFFull << (s * r & 63);
        g ^= (g ^ v) & z;
      }
  }
}

template <bool INS>
static bool update(const Table& t, const std::vector<uint64_t>& B, std::mt19937& g, Table* out) {
  const Plan p = plan<INS>(t, B, 0);
  if (!p.ok) return false;
  std::vector<uint32_t> order(p.W);
  for (uint32_t w = 0; w < p.W; ++w) order[w] = w;
  std::shuffle(order.begin(), order.end(), g);
  *out = t;
  for (uint32_t w : order) apply<INS>(*out, p, B, w);
  return true;
}

static int accepted[2];
static void both(const std::vector<uint64_t>& base, const std::vector<uint64_t>& B, uint32_t nb, std::mt19937& g, uint32_t id) {
  Table t(nb), x(nb), want(nb);
  if (!t.fill(base)) return;
  std::vector<uint64_t> all(base);
  all.insert(all.end(), B.begin(), B.end());
  std::sort(all.begin(), all.end());
  const bool fits = want.fill(all);
  if (update<true>(t, B, g, &x)) {
    ++accepted[0];
    if (!fits) fail("insert accepted, does not fit", id, nb);
    else if (!(x == want)) fail("insert", id, nb);
  }
  std::multiset<uint64_t> ms(base.begin(), base.end());
  for (uint64_t b : B) {
    auto z = ms.find(b);
    if (z != ms.end()) ms.erase(z);
  }
  Table left(nb);
  (void)left.fill(std::vector<uint64_t>(ms.begin(), ms.end()));
  if (update<false>(t, B, g, &x)) {
    ++accepted[1];
    if (!(x == left)) fail("delete", id, nb);
  }
}

int main() {
  std::mt19937 g(11);
  auto u = [&](uint32_t n) { return (uint32_t)(g() % n); };
  // a region of x keys from the end of a window into one with 64 empty slots
  // in the blocks held, and c keys there that it takes with it
  for (uint32_t x = 60; x <= 66; ++x)
    for (uint32_t c : {0u, 1u, 2u, 4u, 7u, 20u})
      for (uint32_t spare : {0u, 1u, 4u, 30u}) {
        const uint32_t q = 14, nb = (1u << q) / 64 + 1;
        std::vector<uint64_t> base{(uint64_t)(LW_SLOTS - 1) << r}, B;
        for (uint32_t s = 0; s < 64 * RL_HALO; ++s)
          if (s % 45 || s / 45 >= 64) base.push_back((uint64_t)(LW_SLOTS + s) << r);
        for (uint32_t i = 0; i < spare; ++i) base.erase(base.begin() + 1 + 60 * i + 7);
        for (uint32_t i = 0; i < x; ++i) B.push_back((uint64_t)(LW_SLOTS - 1) << r | 5u);
        for (uint32_t i = 0; i < c; ++i) B.push_back((uint64_t)(LW_SLOTS + 1000 + 40 * i) << r | 9u);
        std::sort(base.begin(), base.end());
        std::sort(B.begin(), B.end());
        const int before = accepted[0];
        both(base, B, nb, g, 1000 * x + c);
        // (64 empty slots and `spare` more: the x keys and those taken along)
        const bool room = x <= 64 && (x + c <= 64 + spare || c == 0);
        if (room != (accepted[0] > before)) fail(room ? "handed over" : "accepted", 1000 * x + c, spare);
      }
  for (uint32_t it = 0; it < 700; ++it) {
    const uint32_t q = 12 + u(4), nb = (1u << q) / 64 + 1, N = 1u << q;
    std::vector<uint64_t> base, B;
    for (uint32_t i = 0, n = N / 100 * u(96); i < n; ++i) base.push_back((uint64_t)u(N) << r | u(256));
    // stretches from a window's end on, almost full
    for (uint32_t w = 0; w * LW_SLOTS < N; ++w) {
      if (u(3) == 0) continue;
      const uint32_t len = 1u << u(13), keep = 50 + u(50), from = w * LW_SLOTS - (w ? u(100) : 0u);
      base.erase(std::remove_if(base.begin(), base.end(), [&](uint64_t f) { return f >> r >= from && f >> r < from + len; }),
                 base.end());
      for (uint32_t s = from; s < from + len && s < N; ++s)
        if (u(100) < keep) base.push_back((uint64_t)s << r | u(256));
    }
    const uint32_t m = 1 + u(1 + N / 40);
    for (uint32_t i = 0; i < m; ++i) {
      uint32_t s = u(N);
      if (u(2)) s = (s & ~(LW_SLOTS - 1)) - 40 + u(80);  // crowded at the windows' ends
      if (s < N) B.push_back((uint64_t)s << r | (u(2) ? u(256) : u(3)));
    }
    if (!base.empty())
      for (uint64_t& b : B)
        if (u(3) == 0) b = base[u((uint32_t)base.size())];
    if (u(3) == 0 && !B.empty()) {
      const uint64_t hot = B[u((uint32_t)B.size())];
      for (uint32_t i = 0, k = u(64); i < k; ++i) B.push_back(hot);
    }
    std::sort(base.begin(), base.end());
    std::sort(B.begin(), B.end());
    if (!B.empty()) both(base, B, nb, g, it);
  }
  std::printf("accepted %d %d\n", accepted[0], accepted[1]);
  if (accepted[0] < 100 || accepted[1] < 100) fail("few batches were accepted", (uint32_t)accepted[0], (uint32_t)accepted[1]);
  if (!fails) std::printf("windows ok\n");
  return fails ? 1 : 0;
}
