// The three seeding rounds on one thread, as the reference states them: what
// the group search of g3a_seed.h is checked against.  Host builds only; no
// kernel runs this code.
#pragma once
#include "g3a_dev.h"

namespace g3a {

template <class Q, class P>
G3A_HD IntvT<Q> intv_cast(const IntvT<P> &a) {
  IntvT<Q> r;
  r.k = (Q)a.k;
  r.l = (Q)a.l;
  r.s = (Q)a.s;
  r.m = a.m;
  r.n = a.n;
  return r;
}

// backwardExtBackward (fmindex.cu:162-180): k and s only
G3A_HD void backward_ext_b(const DevIndex &x, Intv &io, int base) {
  int64_t oa[4], ob[4];
  occ4_pair(x, io.k - 1, io.k + io.s - 1, oa, ob);
  io.k = pick4(x.count, base) + pick4(oa, base);
  io.s = pick4(ob, base) - pick4(oa, base);
}

// Number of leading positions u < maxlen with q[u] a base equal to the text
// symbol T[t + u], t + u < n: how far a match known to occur once, ending
// just before t, continues forward.
G3A_HD int text_run(const DevIndex &x, int64_t t, const uint8_t *q, int maxlen) {
  const int64_t lim = x.n - t;
  if (lim < maxlen) maxlen = (int)lim;
  int u = 0;
  while (u < maxlen) {
    const int c = maxlen - u < 32 ? maxlen - u : 32;
    uint64_t rw = 0;
    int v = 0;
    for (; v < c; ++v) {
      const int b = q[u + v];
      if (b > 3) break;
      rw |= (uint64_t)b << (62 - 2 * v);
    }
    const uint64_t tw = text_word(x, t + u);
    const uint64_t d = v ? (tw ^ rw) & (~0ULL << (64 - 2 * v)) : 0;
    if (d) return u + (__builtin_clzll(d) >> 1);
    u += v;
    if (v < c) return u;
  }
  return u;
}

// Output sink for one read's intervals: the first `cap` go to `slot`, the
// rest are only counted (the read is then redone with a bigger buffer).
struct IntvSink {
  Intv *slot;
  int cap, n;
  int64_t n_seed;  // sum over intervals of min(s, max_occ)
  int max_occ;
  template <class P>
  G3A_HD void push(const IntvT<P> &p) {
    if (n < cap) slot[n] = intv_cast<int64_t>(p);
    ++n;
    n_seed += (int64_t)p.s > max_occ ? max_occ : (int64_t)p.s;
  }
};

// Storage of the LEP and found lists.  LepWide keeps the whole interval;
// LepNarrow packs it into 16 bytes (one vector load or store per entry) and
// holds for texts of fewer than 2^32 rows.
// Each names the interval type its searches compute in (I).
struct LepWide {
  using I = Intv;
  static constexpr bool kNarrow = false;
  Intv v;
  static G3A_HD Intv get(const LepWide *p, int i) { return p[i].v; }
  static G3A_HD void put(LepWide *p, int i, const Intv &x) { p[i].v = x; }
};
struct alignas(16) LepNarrow {
  using I = IntvN;
  static constexpr bool kNarrow = true;
  uint32_t k, l, s;
  int16_t m, n;
  static G3A_HD IntvN get(const LepNarrow *p, int i) {
    const LepNarrow e = p[i];
    IntvN r;
    r.k = e.k;
    r.l = e.l;
    r.s = e.s;
    r.m = e.m;
    r.n = e.n;
    return r;
  }
  static G3A_HD void put(LepNarrow *p, int i, const IntvN &x) {
    LepNarrow e;
    e.k = x.k;
    e.l = x.l;
    e.s = x.s;
    e.m = (int16_t)x.m;
    e.n = (int16_t)x.n;
    p[i] = e;
  }
};

// Scratch for the LEP list and the found list.
// A list in a global slice of entries of type E.
template <class E>
struct GlobalList {
  using I = typename E::I;
  E *p;
  G3A_HD I get(int i) const { return E::get(p, i); }
  G3A_HD void put(int i, const I &v) const { E::put(p, i, v); }
};

// The LEP list a and the found list f of one thread, with their capacities.
template <class LA, class LF>
struct LepBuf {
  using I = typename LA::I;
  LA a;
  LF f;
  int cap, cap_f;
};
template <class E>
using GlobalBuf = LepBuf<GlobalList<E>, GlobalList<E>>;

// The backward steps of rounds 1 and 2, one list entry after another.  A
// step rebuilds its list in place (entry nc is written only after every
// entry j >= nc has been read) and returns the new length, or -1 when a list
// outgrows its capacity.
struct SerialBack {
  // Round 1 at read position i (base c, -1 past the read or at an N): an
  // entry that extends goes on, deduplicated by size; the first that does
  // not, when none before it did, is a new start, stored in `fl` when the
  // match is long enough to be emitted.
  template <class L, class LF>
  static G3A_HD int round1(const DevIndex &x, const Opt &o, const L &list, int np, int i, int c, const LF &fl,
                           int &nf, int cap, int cap_f, int &last_start, int64_t *steps) {
    using I = typename L::I;
    using P = decltype(I::s);
    int nc = 0;
    P last_s = 0;  // size of the last entry written (read only when nc > 0)
    for (int j = 0; j < np; ++j) {
      const I pj = list.get(j);
      I ok;
      bool ext_ok = false;
      if (c >= 0) {
        backward_ext_ks(x, pj, c, ok);
        if (steps) ++*steps;
        ext_ok = ok.s >= 1;
      }
      if (!ext_ok) {
        if (nc == 0 && i + 1 < last_start) {
          last_start = i + 1;
          if (pj.n - i >= o.min_seed_len) {
            I p = pj;
            p.m = i + 1;
            if (nf == cap_f) return -1;
            fl.put(nf++, p);
          }
        }
      } else if (nc == 0 || ok.s != last_s) {
        ok.m = pj.m;
        ok.n = pj.n;
        if (nc == cap) return -1;
        list.put(nc++, ok);
        last_s = ok.s;
      }
    }
    return nc;
  }
  // Round 2 at pivot-side position m (base = read[m - 1]): an extension at
  // least as large as the last kept one goes on; the first entry that falls
  // short, when long enough, becomes a seed.
  template <class L, class LF, class P>
  static G3A_HD int reseed(const DevIndex &x, const Opt &o, const L &leps, int num_old, int m, int base,
                           P min_seed_intv, const LF &seeds, int &ns, int cap_s, int64_t *steps) {
    using I = typename L::I;
    P curr = min_seed_intv;
    bool collected = false;
    int nl = 0;
    for (int j = 0; j < num_old; ++j) {
      I lep = leps.get(j), ext;
      backward_ext_ks(x, lep, base, ext);
      if (steps) ++*steps;
      if (ext.s >= curr) {
        ext.m = m - 1;
        ext.n = lep.n;
        leps.put(nl++, ext);
        curr = ext.s;
      } else if (!collected && lep.n - lep.m + 1 >= o.min_seed_len) {
        if (ns == cap_s) return -1;
        seeds.put(ns++, lep);
        collected = true;
      }
    }
    return nl;
  }
};

// Round 1 (preseedAndFilterV2, bwa/src/seed.cu:25-104 with
// preseedOnePos2Backward, seed.cu:454-531).  The reference keeps, for each
// end n, the longest match read[m(n)..n] and outputs it when it is right
// maximal; these are exactly the super-maximal exact matches of length >=
// min_seed_len.  They are found here with the bidirectional SMEM search
// (forward from a pivot collecting the points where the interval shrinks,
// then backward), which visits each read position a few times instead of
// once per end position.  Output order is by end position, as the
// reference's.  Returns false when a LEP list outgrows `buf`.
// The learned-index form is used when x.saf / x.li_leaf are set.
template <class B>
G3A_HD bool smem_round1(const DevIndex &x, const Opt &o, const uint8_t *q, int len, IntvSink &out, B &buf,
                        int64_t *steps, int64_t *lc = nullptr) {
  using I = typename B::I;
  using P = decltype(I::s);
  int x0 = 0;
  while (x0 < len) {
    if (q[x0] > 3) { ++x0; continue; }
    // the backward pass rebuilds the list in place: entry nc is written only
    // after entry j >= nc has been read
    const auto &prev = buf.a;
    int np = 0;
    I ik;
    intv_init(x, ik, q[x0]);
    ik.m = x0;
    ik.n = x0;
    int i = x0 + 1;
    if (x0 == 0 && x.kmer && len >= kKmer) {
      // the pass from 0 has no backward extensions: only its longest match
      // is used, so it may start from the k-mer table's interval of
      // read[0, kKmer) when that occurs (the shorter prefixes' entries
      // would never be read)
      uint32_t code = 0;
      int t = 0;
      for (; t < kKmer && q[t] < 4; ++t) code = code << 2 | q[t];
      if (t == kKmer) {
        const uint32_t *e = x.kmer + 3 * (uint64_t)code;
        if (e[2] > 0) {
          ik.k = (P)e[0];
          ik.l = (P)e[1];
          ik.s = (P)e[2];
          ik.n = kKmer - 1;
          i = kKmer;
        }
      }
    }
    for (; i < len; ++i) {
      if (x.saf && ik.s == 1) {
        // one occurrence, at saf[k]: the forward extensions keep s = 1 for
        // as long as the read matches the text after it, so compare the two
        // directly (only l, which nothing downstream reads, is left stale)
        const int run = text_run(x, (int64_t)x.saf[ik.k] + (i - x0), q + i, len - i);
        if (lc) {
          ++lc[2];
          lc[3] += run;
        }
        ik.n = i + run - 1;
        i += run;
        if (i < len) {
          if (np == buf.cap) return false;
          prev.put(np++, ik);
        }
        break;
      }
      if (q[i] < 4) {
        I ok = ik;
        forward_ext(x, ok, q[i]);
        if (steps) ++*steps;
        if (ok.s != ik.s) {
          if (np == buf.cap) return false;
          prev.put(np++, ik);
          if (ok.s < 1) break;
        }
        ik = ok;
        ik.n = i;
      } else {
        if (np == buf.cap) return false;
        prev.put(np++, ik);
        break;
      }
    }
    if (i == len) {
      if (np == buf.cap) return false;
      prev.put(np++, ik);
    }
    // longest first
    for (int a = 0, b = np - 1; a < b; ++a, --b) {
      const I ta = prev.get(a), tb = prev.get(b);
      prev.put(a, tb);
      prev.put(b, ta);
    }
    const int ret = prev.get(0).n + 1;
    // backward search; SMEMs are found in decreasing start order
    int nf = 0, last_start = len + 1;  // start of the last match found (none yet)
    const auto &fl = buf.f;
    for (i = x0 - 1; i >= -1; --i) {
      const int c = i < 0 ? -1 : (q[i] < 4 ? q[i] : -1);
      const int nc = SerialBack::round1(x, o, prev, np, i, c, fl, nf, buf.cap, buf.cap_f, last_start, steps);
      if (nc < 0) return false;
      if (nc == 0) break;
      np = nc;
    }
    // found in decreasing start (and end) order: emit them by end
    for (int j = nf - 1; j >= 0; --j) out.push(fl.get(j));
    x0 = ret;
  }
  return true;
}

// Round 1 by the reference's own per-end backward search; needs no scratch.
G3A_HD void smem_round1_per_end(const DevIndex &x, const Opt &o, const uint8_t *q, int len, IntvSink &out,
                                int64_t *steps) {
  int prev_m = -1, prev_valid = 0;
  Intv prev;
  prev.k = prev.l = prev.s = 0;
  prev.m = prev.n = 0;
  for (int n = 0; n < len; ++n) {
    int valid = 0;
    Intv cur;
    cur.k = cur.l = cur.s = 0;
    cur.m = cur.n = 0;
    if (n >= o.min_seed_len - 1 && q[n] < 4) {
      intv_init(x, cur, q[n]);
      int m = n;
      while (m > 0 && q[m - 1] < 4) {
        Intv t = cur;
        backward_ext_b(x, t, q[m - 1]);
        if (steps) ++*steps;
        if (t.s < 1) break;
        cur.k = t.k;
        cur.s = t.s;
        --m;
      }
      cur.m = m;
      cur.n = n;
      valid = n - m + 1 >= o.min_seed_len;
    }
    // previous end is kept unless this end extends the same start
    if (prev_valid && !(valid && cur.m == prev_m)) out.push(prev);
    prev = cur;
    prev_m = cur.m;
    prev_valid = valid;
  }
  if (prev_valid) out.push(prev);
}

// Round 2, reseedV2 (bwa/src/seed.cu:639-913), for one SMEM.  `leps` and
// `seeds` are scratch lists of capacities cap and cap_s.  Returns false on
// overflow.
template <class LA, class LF>
G3A_HD bool reseed_one(const DevIndex &x, const Opt &o, const uint8_t *q, int len, const Intv &smem,
                       const LA &leps, const LF &seeds, int cap, int cap_s, IntvSink &out, int64_t *steps) {
  using I = typename LA::I;
  using P = decltype(I::s);
  const int split_len = (int)(o.min_seed_len * o.split_factor + .499);
  const int slen = smem.n - smem.m + 1;
  if (slen < split_len || smem.s > o.split_width) return true;
  const P min_seed_intv = (P)(smem.s + 1);
  const int pivot = (smem.m + smem.n + 1) >> 1;
  if (pivot > 77) return true;  // seed.cu:718
  if (q[pivot] >= 4) return true;
  int nl = 0, ns = 0;
  I seed, old;
  intv_init(x, seed, q[pivot]);
  seed.m = pivot;
  seed.n = pivot;
  int n;
  for (n = pivot; n < len - 1; ++n) {
    old = seed;
    if (q[n + 1] >= 4) break;
    forward_ext(x, seed, q[n + 1]);
    if (steps) ++*steps;
    seed.n = n + 1;
    if (seed.s < old.s) {
      if (nl == cap) return false;
      leps.put(nl++, old);
      if (seed.s < min_seed_intv) break;
    }
  }
  if (seed.s >= min_seed_intv) {
    seed.n = n;
    if (nl == cap) return false;
    leps.put(nl++, seed);
  }
  for (int a = 0, b = nl - 1; a < b; ++a, --b) {
    const I ta = leps.get(a), tb = leps.get(b);
    leps.put(a, tb);
    leps.put(b, ta);
  }
  for (int m = pivot; m > 0; --m) {
    const int base = q[m - 1];
    if (base >= 4) break;
    nl = SerialBack::reseed(x, o, leps, nl, m, base, min_seed_intv, seeds, ns, cap_s, steps);
    if (nl < 0) return false;
    if (nl == 0) break;
  }
  if (nl > 0) {
    const I l0 = leps.get(0);
    if (l0.n - l0.m + 1 >= o.min_seed_len) {
      if (ns == cap_s) return false;
      seeds.put(ns++, l0);
    }
  }
  for (int j = 0; j < ns; ++j) out.push(seeds.get(j));
  return true;
}

// Round 3, reseedThirdRound (bwa/src/seed.cu:1143-1190) via reseedLastRound
// (seed.cu:1518-1550).  Every start m extends forward at least to length
// min_len before it can emit, so when the first kKmer bases hold no N their
// interval is read from the k-mer table instead of kKmer-1 forward steps.
template <class P>
G3A_HD void reseed_round3(const DevIndex &x, const Opt &o, const uint8_t *q, int len, IntvSink &out,
                          int64_t *steps, int64_t *lc = nullptr) {
  const int min_len = o.min_seed_len + 1;
  const int64_t max_intv = o.max_mem_intv;
  const bool table = x.kmer && min_len > kKmer;
  const bool learned = x.li_leaf && min_len <= 32;
  int m = 0;
  while (m < len) {
    int next_m = m + 1;
    int base = q[m];
    if (base < 4 && learned && m + min_len <= len) {
      // the pass emits at length min_len when fewer than max_intv rows hold
      // read[m, m + min_len): the learned index gives that interval directly
      uint64_t W = 0;
      int t = 0;
      for (; t < min_len && q[m + t] < 4; ++t) W |= (uint64_t)q[m + t] << (62 - 2 * t);
      uint32_t kk, ss;
      if (t == min_len) {
        if (lc) ++lc[0];
        if (li_range(x, W, min_len, kk, ss, lc)) {
          if ((int64_t)ss < max_intv) {
            if (ss > 0) {
              IntvT<P> sd;
              sd.k = (P)kk;
              sd.l = 0;
              sd.s = (P)ss;
              sd.m = m;
              sd.n = m + min_len - 1;
              out.push(sd);
            }
            m += min_len;
            continue;
          }
        } else if (lc) {
          ++lc[1];
        }
      }
    }
    if (base < 4) {
      IntvT<P> seed;
      int n0 = m + 1;
      uint32_t code = 0;
      bool jumped = false;
      if (table && m + kKmer <= len) {
        int k = 0;
        for (; k < kKmer && q[m + k] < 4; ++k) code = code << 2 | q[m + k];
        if (k == kKmer) {
          const uint32_t *e = x.kmer + 3 * (uint64_t)code;
          seed.k = (P)e[0];
          seed.l = (P)e[1];
          seed.s = (P)e[2];
          n0 = m + kKmer;
          next_m = n0;
          jumped = true;
        }
      }
      if (!jumped) intv_init(x, seed, base);
      for (int n = n0; n < len; ++n) {
        next_m = n + 1;
        base = q[n];
        if (base < 4) {
          forward_ext(x, seed, base);
          if (steps) ++*steps;
          if ((int64_t)seed.s < max_intv && (n - m + 1) >= min_len) {
            if (seed.s > 0) {
              seed.m = m;
              seed.n = n;
              out.push(seed);
            }
            break;
          }
        } else break;
      }
    }
    m = next_m;
  }
}

}  // namespace g3a
