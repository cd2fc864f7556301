// Seeding of one read by a group of G lanes (16 on the fast path, a whole
// wavefront for the reads that outgrow it): rounds 1 to 3 of the reference's
// seeding (preseedAndFilterV2, bwa/src/seed.cu:25-104 with 454-531; reseedV2,
// seed.cu:639-913; reseedThirdRound, seed.cu:1143-1190 with 1518-1550), whose
// results a host check compares with the same rounds on one thread.
//
// What bounds seeding in a small batch is the chain of dependent Occ fetches:
// each step of a search needs the interval of the step before (a full chip is
// bound by instructions, see k_seed).  A thread per read leaves the list entries of a backward step (about 6, up to 64) waiting one after
// another and most lanes of a load idle (11 of 64).  Here a list entry is a
// lane: entry e lives in register slot e / G of lane e % G, ends further
// right as e grows (longest match last), and a backward step is one pair of
// Occ fetches for all of them.  Two facts make the step free of list
// bookkeeping.  The entries are nested, so the ones that stop extending are
// the longest ones, and only the longest live entry can end as a match; and
// an entry whose interval equals the next longer one's can stay in the list,
// since it stops in the same step and is never the longest.
//
// Entries shorter than the k-mer table's K bases are not searched at all: an
// entry shorter than min_seed_len > K cannot be emitted, so nothing about it
// is needed before it has K bases, and then the table holds its interval.
// The K - 1 shortest ends of a list are looked up at once, a lane each, and
// the forward search starts from the table.  On a 100 Mbp text this removes
// about two thirds of the FM steps of rounds 1 and 2.
//
// Once a forward search has one occurrence its end is found by comparing the
// read with the text there, 32 bases a lane; the third round's passes, which
// nearly always cover exactly min_seed_len + 1 bases, run on the lanes at
// once and are kept up to the first that does not.
#pragma once
#include "g3a_lanes.h"

namespace g3a {

// A read in LDS: 2-bit codes, 16 bases a word, first base highest (0 past
// the end), and a mask of the bases that are N or past the end, 32 a word,
// first base highest.  Padded so that 32 bases can be read at any position.
constexpr int kPkWords = kMaxReadLen / 16 + 2, kNmWords = kMaxReadLen / 32 + 2;
struct PackedRead {
  uint32_t code[kPkWords], nm[kNmWords];
  G3A_LANE int base(int i) const {  // 0..3, or -1 for an N (0 <= i < len)
    const int c = (int)(code[i >> 4] >> (30 - 2 * (i & 15))) & 3;
    return (nm[i >> 5] << (i & 31)) >> 31 ? -1 : c;
  }
  G3A_LANE uint64_t bases32(int i) const {
    const int w = i >> 4, sh = 2 * (i & 15);
    const uint64_t v = (uint64_t)code[w] << 32 | code[w + 1];
    return sh ? v << sh | code[w + 2] >> (32 - sh) : v;
  }
  G3A_LANE uint32_t stop32(int i) const {
    const int w = i >> 5, sh = i & 31;
    return sh ? nm[w] << sh | nm[w + 1] >> (32 - sh) : nm[w];
  }
};

// The k-mer table of the layout that P computes in
G3A_LANE bool has_table_of(const DevIndex &x, uint32_t) { return x.kmer != nullptr; }
G3A_LANE bool has_table_of(const DevIndex &x, int64_t) { return x.kmer64 != nullptr; }
G3A_LANE void table_entry(const DevIndex &x, uint32_t code, uint32_t &k, uint32_t &l, uint32_t &s) {
  const uint32_t *e = x.kmer + 3 * (uint64_t)code;
  k = e[0];
  l = e[1];
  s = e[2];
}
G3A_LANE void table_entry(const DevIndex &x, uint32_t code, int64_t &k, int64_t &l, int64_t &s) {
  const int64_t *e = x.kmer64 + 3 * (uint64_t)code;
  k = e[0];
  l = e[1];
  s = e[2];
}

// Matches found by one backward search, in decreasing start order.
template <class P>
struct FoundList {
  P *k, *s;
  uint32_t *mn;
  int cap;
};
template <class P>
constexpr size_t seed_group_bytes(int cap) {
  return sizeof(PackedRead) + (size_t)cap * (2 * sizeof(P) + 4);
}
static_assert(sizeof(PackedRead) % 8 == 0, "64-bit found lists follow it");

template <class W, int G, int NS, class P, bool L>
struct SeedGroup {
  using I = IntvT<P>;
  const DevIndex &x;
  const Opt &o;
  PackedRead *q;
  FoundList<P> found;
  int gl, gb;  // this lane in the group, the group's first lane in the wavefront
  Intv *slot;
  int cap;      // intervals that fit slot
  int len, n;   // read length, intervals so far
  int64_t n_seed;
  uint32_t steps;
  int64_t *lc;
  // list entries
  P ek[NS], es[NS];
  int en[NS];

  G3A_LANE uint64_t ballot(bool p) const {
    const uint64_t m = W::ballot(p);
    return G == 64 ? m : (m >> gb) & ((1ull << G) - 1);
  }
  template <class T>
  G3A_LANE T from(T v, int lane) const { return W::from(v, gb + lane); }

  G3A_LANE void load(const uint8_t *p, int l) {
    len = l;
    n = 0;
    n_seed = 0;
    W::lds_sync();  // the group's earlier reads of its LDS are done
    uint16_t *nm16 = reinterpret_cast<uint16_t *>(q->nm);
    for (int w = gl; w < 2 * kNmWords; w += G) {
      const int left = l - 16 * w;
      uint32_t c = 0, m = 0xffff;
      if (left > 0) {
        // 16 codes from five aligned words (the buffer is padded)
        const uint8_t *a = p + 16 * w;
        const uint32_t *v = reinterpret_cast<const uint32_t *>(a - ((uintptr_t)a & 3));
        const uint32_t sh = 8 * (uint32_t)((uintptr_t)a & 3);
        m = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t y = sh ? v[t] >> sh | v[t + 1] << (32 - sh) : v[t];
          c = c << 8 | ((y & 3) << 6 | (y >> 8 & 3) << 4 | (y >> 16 & 3) << 2 | (y >> 24 & 3));
          m = m << 4 | ((y >> 2 & 1) << 3 | (y >> 10 & 1) << 2 | (y >> 18 & 1) << 1 | (y >> 26 & 1));
        }
        if (left < 16) {
          c &= ~0u << (32 - 2 * left);
          m |= 0xffffu >> left;
        }
      }
      if (w < kPkWords) q->code[w] = c;
      nm16[w ^ 1] = (uint16_t)m;
    }
    W::lds_sync();
  }

  // Interval of the group's next output, written by the lanes that call it
  G3A_LANE void put(int at, P k, P s, int m, int e) {
    if (at < cap) {
      Intv v;
      v.k = (int64_t)k;
      v.l = 0;  // nothing downstream reads it
      v.s = (int64_t)s;
      v.m = m;
      v.n = e;
      slot[at] = v;
    }
    n_seed += (int64_t)s > o.max_occ ? o.max_occ : (int64_t)s;
  }

  G3A_LANE bool add_entry(int &cnt, const I &v) {
    if (cnt == G * NS) return false;
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (cnt == k * G + gl) {
        ek[k] = v.k;
        es[k] = v.s;
        en[k] = v.n;
      }
    ++cnt;
    return true;
  }

  // How far a match that occurs once, at text position t - i + (its start),
  // continues from read position i at text position t
  G3A_LANE int run_on(int64_t t, int i) {
    int most = len - i;
    const int64_t lim = x.n - t;
    if (lim < most) most = (int)lim;
    for (int u0 = 0;; u0 += 32 * G) {
      const int u = u0 + 32 * gl;
      int f = 0;
      if (u < most) {
        const uint64_t d = text_word(x, t + u) ^ q->bases32(i + u);
        const uint32_t stop = q->stop32(i + u);
        f = d ? __builtin_clzll(d) >> 1 : 32;
        const int g = stop ? __builtin_clz(stop) : 32;
        f = g < f ? g : f;
        f = most - u < f ? most - u : f;
      }
      const uint64_t m = ballot(f < 32);
      if (m) {
        const int first = __builtin_ffsll((long long)m) - 1;
        return u0 + 32 * first + from(f, first);
      }
    }
  }

  // The list of a search that starts at x0 and keeps intervals of at least
  // `least` rows: entries with an end in [x0, ...), shortest first, of which
  // the first `low` (ends x0 .. x0 + low - 1) are pending until they have K
  // bases.  kq: K, or 1 when the table is not used.  Returns the number of
  // entries, or -1 when they do not fit; `end` is the longest one's end, and
  // ik.s is 0 when the text does not hold the base at x0.
  G3A_LANE int forward(int x0, P least, int &kq, int &low, int &end, I &ik) {
    const int K = kKmer;
    const int c0 = q->base(x0);
    intv_init(x, ik, c0);
    kq = has_table_of(x, P()) && o.min_seed_len > K && ik.s >= least ? K : 1;
    // the table's interval of the first K bases, where there is one (every
    // field gets a value on every path)
    P tk = 0, tl = 0, ts = 0;
    if (kq > 1 && (q->stop32(x0) >> (32 - K)) == 0) table_entry(x, (uint32_t)(q->bases32(x0) >> (64 - 2 * K)), tk, tl, ts);
    const bool jumped = kq > 1 && ts >= least;
    ik.k = jumped ? tk : ik.k;
    ik.l = jumped ? tl : ik.l;
    ik.s = jumped ? ts : ik.s;
    ik.m = x0;
    ik.n = jumped ? x0 + K - 1 : x0;
    low = jumped ? K - 1 : 0;
    int cnt = low;
    const bool keep = jumped || kq == 1;  // else every entry is shorter than K
    const bool text = least == 1 && (L && x.saf ? true : len - x0 > (2 << x.sa_shift));
    bool dead = false, full = false;
    for (int i = ik.n + 1; i < len; ++i) {
      if (text && ik.s == 1) {
        // one occurrence: every further step keeps s = 1 for as long as the
        // read matches the text (l, which nothing reads, is left stale)
        const int64_t at = L && x.saf ? (int64_t)x.saf[ik.k]
                           : sizeof(P) == 4 ? sa_value_n(x, (uint32_t)ik.k)
                                            : sa_value(x, (int64_t)ik.k, nullptr);
        const int run = run_on(at + (i - x0), i);
        if (L && gl == 0) {
          ++lc[2];
          lc[3] += run;
        }
        ik.n = i + run - 1;
        break;
      }
      const int c = q->base(i);
      if (c < 0) break;
      I ok = ik;
      forward_ext(x, ok, c);
      steps += gl == 0;
      if (ok.s != ik.s) {
        if (keep) full |= !add_entry(cnt, ik);
        if (full || ok.s < least) {
          dead = true;
          break;
        }
      }
      ik = ok;
      ik.n = i;
    }
    if (!dead && keep && ik.s >= least) full |= !add_entry(cnt, ik);
    end = ik.n;
    if (!keep) cnt = low = end - x0 + 1 < K - 1 ? end - x0 + 1 : K - 1;
    return full ? -1 : cnt;
  }

  // The first `low` entries: their intervals at K bases, which only ends
  // with K bases before them that hold no N and occur can reach; none at all
  // when the search cannot go back from x0 (`back`)
  G3A_LANE void look_up(int x0, int low, P least, bool back) {
    const int K = kKmer;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int e = k * G + gl;
      if (k * G >= low) break;
      if (e < low) {
        const int b = x0 + e - K + 1;
        P tk = 0, tl = 0, ts = 0;
        if (back && b >= 0 && (q->stop32(b) >> (32 - K)) == 0)
          table_entry(x, (uint32_t)(q->bases32(b) >> (64 - 2 * K)), tk, tl, ts);
        en[k] = x0 + e;
        ek[k] = tk;
        es[k] = ts >= least ? ts : 0;
      }
    }
  }

  // Extends the cnt entries backward from read position i; an entry goes on
  // while at least `least` rows hold it.  A match is found when the longest
  // entry stops (at a base, an N or the read's start) with at least
  // min_seed_len bases.  x0: the start of the list's pending entries.
  // Returns the number of matches found.
  G3A_LANE int backward(int x0, int i, int cnt, int kq, P least) {
    // slots past the list hold nothing
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (k * G + gl >= cnt) es[k] = 0;
    int top = -1, nf = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (k * G < cnt) {
        const uint64_t m = ballot(es[k] > 0);
        if (m) top = k * G + 63 - __builtin_clzll(m);
      }
    int c = i >= 0 ? q->base(i) : -1;
    while (top >= 0) {
      // while only pending entries are left, go to where the longest has K
      // bases (the bases between belong to its k-mer, which holds no N)
      if (top < kq - 1 && x0 + top - kq < i) {
        i = x0 + top - kq;
        c = i >= 0 ? q->base(i) : -1;
      }
      const int cn = i > 0 ? q->base(i - 1) : -1;
      int next = -1;
      bool out = false;
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        if (k * G <= top) {
          const bool act = es[k] > 0 && en[k] - i >= kq;
          P nk = ek[k], ns = c < 0 ? 0 : es[k];
          if (c >= 0 && act) {
            I v, w;
            v.k = nk;
            v.l = 0;
            v.s = ns;
            backward_ext_ks(x, v, c, w);
            ++steps;
            nk = w.k;
            ns = w.s >= least ? w.s : 0;
          }
          if (k * G + gl == top && act && ns == 0 && en[k] - i >= o.min_seed_len) {
            out = true;
            find(nf, ek[k], es[k], i + 1, en[k]);
          }
          ek[k] = nk;
          es[k] = ns;
          const uint64_t m = ballot(ns > 0);
          if (m) next = k * G + 63 - __builtin_clzll(m);
        }
      }
      if (next != top) {
        if (ballot(out)) ++nf;
        top = next;
      }
      --i;
      c = cn;
    }
    return nf;
  }

  G3A_LANE void find(int at, P k, P s, int m, int e) {
    if (at < found.cap) {
      found.k[at] = k;
      found.s[at] = s;
      found.mn[at] = (uint32_t)m | (uint32_t)e << 16;
    }
  }

  // Rounds 1 and 2, one search after another in one loop, so that the groups
  // of a wavefront share its code whichever round each is in.  Round 1
  // searches from the read's start and then from each base after the longest
  // match before (skipping N); round 2 (reseedV2, bwa/src/seed.cu:639-913)
  // searches again from the middle of each long match with few rows, for
  // matches with more.  False when a list or the output slots overflow.
  G3A_LANE bool searches() {
    const int split_len = (int)(o.min_seed_len * o.split_factor + .499);
    int x0 = 0, nsm = -1, at = 0;  // nsm: round 1's matches once it is done
    bool ok = true;
    while (ok) {
      int start = -1;
      P least = 1;
      if (nsm < 0) {
        while (x0 < len && q->base(x0) < 0) ++x0;
        if (x0 < len) {
          start = x0;
        } else {
          nsm = n;
          W::global_sync();  // round 1's intervals are read back by every lane
        }
      }
      if (nsm >= 0) {
        ok = nsm <= cap;
        while (ok && start < 0 && at < nsm) {
          const Intv v = slot[at++];
          const int pivot = (v.m + v.n + 1) >> 1;
          if (v.n - v.m + 1 >= split_len && v.s <= o.split_width && pivot <= 77 /* seed.cu:718 */ &&
              q->base(pivot) >= 0) {
            start = pivot;
            least = (P)(v.s + 1);
          }
        }
        if (start < 0) break;
      }
      I ik;
      int kq, low, end;
      const int cnt = forward(start, least, kq, low, end, ik);
      W::lds_sync();
      int nf = 0;
      if (cnt < 0) {
        ok = false;
      } else if (nsm < 0 && ik.s == 0) {
        // a base that the text does not hold: round 1 runs on to the end or
        // an N with no rows, and counts that as a match of none
        if (end - x0 + 1 >= o.min_seed_len) {
          find(0, ik.k, ik.s, x0, end);
          nf = 1;
        }
      } else {
        look_up(start, low, least, start > 0 && q->base(start - 1) >= 0);
        nf = backward(start, start - 1, cnt, kq, least);
        ok = nf <= found.cap;
      }
      W::lds_sync();
      if (ok) {
        // round 1's matches come in decreasing start (and end) order and are
        // output by end; round 2's in the order found
        for (int j = gl; j < nf; j += G) {
          const int f = nsm < 0 ? nf - 1 - j : j;
          put(n + j, found.k[f], found.s[f], (int)(found.mn[f] & 0xffff), (int)(found.mn[f] >> 16));
        }
        n += nf;
      }
      if (nsm < 0) x0 = end + 1;
    }
    return ok;
  }

  // One pass of the third round from m; returns the next start, sd.s > 0
  // when the pass emits.
  G3A_LANE int pass3(int m, I &sd) {
    const int K = kKmer, min_len = o.min_seed_len + 1;
    const int64_t max_intv = o.max_mem_intv;
    sd.s = 0;
    int base = q->base(m);
    if (base < 0) return m + 1;
    if (L && x.li_leaf && min_len <= 32 && m + min_len <= len && (q->stop32(m) >> (32 - min_len)) == 0) {
      // the pass emits at length min_len when fewer than max_intv rows hold
      // read[m, m + min_len): the learned index gives that interval directly
      const uint64_t key = q->bases32(m) & ~0ull << (64 - 2 * min_len);
      uint32_t kk, ss;
      ++lc[0];
      if (li_range(x, key, min_len, kk, ss, lc)) {
        if ((int64_t)ss < max_intv) {
          sd.k = (P)kk;
          sd.s = (P)ss;
          sd.m = m;
          sd.n = m + min_len - 1;
          return m + min_len;
        }
      } else {
        ++lc[1];
      }
    }
    I v;
    int i = m + 1;
    intv_init(x, v, base);
    if (has_table_of(x, P()) && min_len > K && (q->stop32(m) >> (32 - K)) == 0) {
      table_entry(x, (uint32_t)(q->bases32(m) >> (64 - 2 * K)), v.k, v.l, v.s);
      i = m + K;
    }
    for (; i < len; ++i) {
      base = q->base(i);
      if (base < 0) return i + 1;
      forward_ext(x, v, base);
      ++steps;
      if ((int64_t)v.s < max_intv && i - m + 1 >= min_len) {
        sd.k = v.k;
        sd.s = v.s;
        sd.m = m;
        sd.n = i;
        return i + 1;
      }
    }
    return len > m + 1 ? len : m + 1;
  }

  G3A_LANE void round3() {
    const int step = o.min_seed_len + 1;
    for (int m0 = 0; m0 < len;) {
      const int m = m0 + step * gl;
      I sd;
      sd.s = 0;
      int next = 0;
      if (m < len) next = pass3(m, sd);
      // the passes up to the first that does not end where the next began
      const uint64_t live = ballot(m < len), off = ballot(m < len && next != m + step);
      const int last = off ? __builtin_ffsll((long long)off) - 1 : 63 - __builtin_clzll(live);
      const bool emits = gl <= last && sd.s > 0;
      const uint64_t em = ballot(emits);
      if (emits) put(n + __builtin_popcountll(em & ((1ull << gl) - 1)), sd.k, sd.s, sd.m, sd.n);
      n += __builtin_popcountll(em);
      m0 = from(next, last);
    }
  }

  // Rounds 1 to 3 of the loaded read: false when a list or the output slots
  // overflow.  n and n_seed (the same on every lane) are the output's size.
  G3A_LANE bool run() {
    const bool ok = searches();
    if (ok) round3();
#pragma unroll
    for (int d = G / 2; d >= 1; d >>= 1) n_seed += W::from_xor(n_seed, d);
    return ok;
  }
};

}  // namespace g3a
