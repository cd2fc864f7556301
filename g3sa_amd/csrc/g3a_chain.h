// Chaining of one read with many seeds by a wavefront: the seed sort, the
// B-tree chaining, the chain filter and the read's extension tasks, with the
// results of sort_seeds, chain_build, chain_filter and chain_window
// (g3a_dev.h), which run them on one thread.
//
// What bounds it on one thread is one dependent load after another: a tree
// descent a seed, the filter's pairs of chains, a walk of every chain for its
// weight and its window.  Here only the order of the seeds stays serial.  A
// node's keys are compared on the lanes at once, with the keys' positions in
// the node; the nodes and the first chains lie in LDS.  A chain's weight,
// window and length are kept up to date as seeds join it, and a seed knows its
// place in its chain, so nothing walks a chain; the sorts are counting sorts,
// the filter takes 64 chains at a time against the kept ones, and the tasks
// are written a seed a lane.
#pragma once
#include "g3a_lanes.h"

namespace g3a {

struct ChainNode {  // KbNode with the keys' positions
  int64_t pos[kKbN];
  uint16_t n, internal;
  uint16_t key[kKbN];
  uint16_t child[kKbN + 1];
  uint16_t pad[3];
};
static_assert(sizeof(ChainNode) == 144, "nodes follow each other");
constexpr int kChainIds = 1 << 16;  // chain and node numbers are 16 bits

// A chain under construction, 10 words; its positions on the text after the
// first are relative to that (a seed that joins is at most its distance on the
// read and the band further on: below 2^30 in all for bands of kChainMaxW).
struct ChainRec {
  int64_t first_rb;
  int32_t last_rb, end_r, lo, hi;  // end_r: end of its weight on the text; [lo, hi): its window
  uint32_t a;  // rid | first qbeg << 9 | last qbeg << 18
  uint32_t b;  // last len | end of its weight on the read << 9 | weight on the read << 18
  int32_t n, w_r;
};
static_assert(sizeof(ChainRec) == 40 && kMaxReadLen < 512, "read positions are 9 bits");
constexpr int kRecWords = sizeof(ChainRec) / 4, kChainMaxW = 1 << 13;

// Scratch of one read in memory, ns entries each (two for tmp), and LDS.
struct ChainMem {
  uint32_t *rec_a, *rec_b;  // words 0-5 and 6-9 of the records past the LDS
  int32_t *of, *order, *tmp;  // chain of a seed; chains in tree order; place of a seed in its chain | word per chain
  uint8_t *kept;
  ChainNode *nodes;
  int n_nodes;
};

// SORT: seeds sorted at most (2048, or fewer if no read has more), NODES, RECS:
// nodes and records in LDS, FILT: chains filtered at most (4096, or fewer)
template <int SORT, int NODES, int RECS, int FILT>
struct ChainStageL {
  static constexpr int kSort = SORT, kNodes = NODES, kRecs = RECS, kFilt = FILT;
  static constexpr int kFSort = FILT < 2048 ? FILT : 2048;  // chains sorted at most
  uint16_t idx[SORT];
  uint32_t rec[RECS * kRecWords];
  union {
    struct {
      uint32_t key[SORT], hist[512];
      uint16_t alt[SORT];
    } sort;
    ChainNode node[NODES];
    struct {
      uint32_t be[FILT], hist[512];
      uint16_t w[FILT], alt[kFSort], alt2[kFSort];
      uint64_t kept[FILT / 64];
    } filt;
  };
};

template <class W, class ST>
struct ChainGroup {
  const DevIndex &x;
  const Opt &o;
  ST *st;
  ChainMem g;
  const Seed *s;
  int ns, l_seq, read, lane;
  int n_sorted;  // seeds in sorted order; the rest stay in place
  int nch, root, nn;

  G3A_LANE int64_t get64(int64_t v, int l) const {
    return (int64_t)((uint64_t)(uint32_t)W::get((int)(uint32_t)v, l) |
                     (uint64_t)(uint32_t)W::get((int)(uint32_t)((uint64_t)v >> 32), l) << 32);
  }
  G3A_LANE const Seed &seed(int e) const { return s[e < n_sorted ? (int)st->idx[e] : e]; }
  G3A_LANE uint32_t rec_word(int c, int d) const {
    return c < ST::kRecs ? st->rec[c * kRecWords + d] : d < 6 ? g.rec_a[(int64_t)c * 6 + d] : g.rec_b[(int64_t)c * 4 + d - 6];
  }
  G3A_LANE void put_word(int c, int d, uint32_t v) {
    if (c < ST::kRecs) st->rec[c * kRecWords + d] = v;
    else if (d < 6) g.rec_a[(int64_t)c * 6 + d] = v;
    else g.rec_b[(int64_t)c * 4 + d - 6] = v;
  }
  G3A_LANE int64_t rec64(int c, int d) const { return (int64_t)((uint64_t)rec_word(c, d) | (uint64_t)rec_word(c, d + 1) << 32); }

  // Stable counting sort of m <= 2048 indices by key(i) < 512, src to dst
  template <class K>
  G3A_LANE void sort_by(const uint16_t *src, uint16_t *dst, int m, uint32_t *hist, K key) {
    W::lds_sync();
    for (int b = lane; b < 512; b += 64) hist[b] = 0;
    W::lds_sync();
    for (int e = lane; e < m; e += 64) W::lds_add(hist + key(src[e]), 1u);
    W::lds_sync();
    uint32_t v[8], sum = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      v[t] = hist[8 * lane + t];
      sum += v[t];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t u = W::from(incl, lane >= d ? lane - d : 0);
      incl += lane >= d ? u : 0;
    }
    uint32_t base = incl - sum;
    W::lds_sync();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      hist[8 * lane + t] = base;
      base += v[t];
    }
    W::lds_sync();
    for (int e0 = 0; e0 < m; e0 += 64) {
      const bool live = e0 + lane < m;
      const int i = live ? src[e0 + lane] : 0;
      const uint32_t k = live ? key(i) : 0;
      uint64_t peers = W::ballot(live);
#pragma unroll
      for (int b = 0; b < 9; ++b) {
        const uint64_t on = W::ballot(live && (k >> b & 1));
        peers &= k >> b & 1 ? on : ~on;
      }
      const int rank = __builtin_popcountll(peers & ((1ull << lane) - 1));
      const uint32_t at = live ? hist[k] + (uint32_t)rank : 0;
      W::lds_sync();
      if (live) {
        dst[at] = (uint16_t)i;
        if (rank == 0) hist[k] += (uint32_t)__builtin_popcountll(peers);
      }
      W::lds_sync();
    }
  }

  G3A_LANE void sort() {
    const int m = ns < 2048 ? ns : 2048;
    n_sorted = m;
    W::lds_sync();  // earlier reads of the LDS are done
    for (int e = lane; e < m; e += 64) {
      st->sort.key[e] = (uint32_t)s[e].qbeg | (uint32_t)s[e].len << 16;
      st->idx[e] = (uint16_t)e;
    }
    sort_by(st->idx, st->sort.alt, m, st->sort.hist, [&](int i) { return st->sort.key[i] >> 16; });
    sort_by(st->sort.alt, st->idx, m, st->sort.hist, [&](int i) { return st->sort.key[i] & 0xffff; });
  }

  // split child yi, the i-th of xi (kbtree_CUDA.cu:27-44)
  G3A_LANE void split(ChainNode *nd, int xi, int i, int yi, int zi) {
    ChainNode &X = nd[xi], &Y = nd[yi], &Z = nd[zi];
    const int n = X.n, in = Y.internal;
    const bool k5 = lane < kKbT - 1, kx = lane < n, cx = lane <= n;
    const int64_t zp = k5 ? Y.pos[kKbT + lane] : 0, xp = kx ? X.pos[lane] : 0, mp = Y.pos[kKbT - 1];
    const uint16_t zk = k5 ? Y.key[kKbT + lane] : 0, xk = kx ? X.key[lane] : 0, mk = Y.key[kKbT - 1];
    const uint16_t zc = in && lane < kKbT ? Y.child[kKbT + lane] : 0, xc = cx ? X.child[lane] : 0;
    W::global_sync();
    if (k5) {
      Z.pos[lane] = zp;
      Z.key[lane] = zk;
    }
    if (in && lane < kKbT) Z.child[lane] = zc;
    if (kx && lane >= i) {
      X.pos[lane + 1] = xp;
      X.key[lane + 1] = xk;
    }
    if (cx && lane > i) X.child[lane + 1] = xc;
    if (lane == 0) {
      Z.n = kKbT - 1;
      Z.internal = (uint16_t)in;
      Y.n = kKbT - 1;
      X.child[i + 1] = (uint16_t)zi;
      X.pos[i] = mp;
      X.key[i] = mk;
      X.n = (uint16_t)(n + 1);
    }
    W::global_sync();
  }
  // insert chain c at position p; false when the nodes run out
  G3A_LANE bool put(ChainNode *nd, int cap, int c, int64_t p) {
    if (nn + 2 > cap) return false;  // the root and one child may split before the next look
    if (nd[root].n == kKbN) {
      const int si = nn, old = root;
      nn += 2;
      if (lane == 0) {
        nd[si].n = 0;
        nd[si].internal = 1;
        nd[si].child[0] = (uint16_t)old;
      }
      W::global_sync();
      root = si;
      split(nd, si, 0, old, si + 1);
    }
    int xi = root;
    for (;;) {
      ChainNode &X = nd[xi];
      const int n = X.n, in = X.internal;
      const bool kx = lane < n;
      const int64_t xp = kx ? X.pos[lane] : 0;
      const uint16_t xk = kx ? X.key[lane] : 0;
      const uint64_t lt = W::ballot(kx && xp < p), eq = W::ballot(kx && xp == p);
      int i = __builtin_popcountll(lt) + (eq ? 1 : 0);  // after the first equal key
      if (!in) {
        W::global_sync();
        if (kx && lane >= i) {
          X.pos[lane + 1] = xp;
          X.key[lane + 1] = xk;
        }
        if (lane == 0) {
          X.pos[i] = p;
          X.key[i] = (uint16_t)c;
          X.n = (uint16_t)(n + 1);
        }
        W::global_sync();
        return true;
      }
      if (nd[X.child[i]].n == kKbN) {
        if (nn + 1 > cap) return false;
        split(nd, xi, i, X.child[i], nn++);
        if (p > X.pos[i]) ++i;
      }
      xi = X.child[i];
    }
  }

  // chain_build: chains and the seeds' places in them, the chains in tree
  // order in g.order; false when the nodes run out
  G3A_LANE bool build(ChainNode *nd, int cap) {
    W::global_sync();
    nch = root = 0;
    nn = 1;
    if (lane == 0) nd[0].n = nd[0].internal = 0;
    W::global_sync();
    for (int base = 0; base < ns; base += 64) {
      const bool live = base + lane < ns;
      const Seed v = live ? seed(base + lane) : Seed{};
      // the seed's window, relative to its place on the text
      const int tail = l_seq - v.qbeg - v.len;
      const int v_lo = -(v.qbeg + cal_max_gap(o, v.qbeg)), v_hi = v.len + (tail + cal_max_gap(o, tail));
      int my_c = -1, my_r = 0;
      const int cnt = ns - base < 64 ? ns - base : 64;
      for (int k = 0; k < cnt; ++k) {
        const int64_t rb = get64(v.rbeg, k);
        const int qb = W::get(v.qbeg, k), ln = W::get(v.len, k), rid = W::get(v.rid, k);
        const int lo = W::get(v_lo, k), hi = W::get(v_hi, k);
        bool merged = false;
        if (nch) {
          int low = -1, xi = root;
          for (;;) {
            const ChainNode &X = nd[xi];
            const int n = X.n, in = X.internal;
            const bool kx = lane < n;
            const int64_t xp = kx ? X.pos[lane] : 0;
            const int xk = kx ? X.key[lane] : 0, xc = lane <= n ? X.child[lane] : 0;
            const uint64_t lt = W::ballot(kx && xp < rb), eq = W::ballot(kx && xp == rb);
            const int b = __builtin_popcountll(lt);
            if (eq) {
              low = W::get(xk, b);
              break;
            }
            if (b > 0) low = W::get(xk, b - 1);
            if (!in) break;
            xi = W::get(xc, b);
          }
          if (low >= 0) {
            // test_and_merge (bwa/src/aux.cu:54-84)
            const int c = low;
            const int rw = lane < kRecWords ? (int)rec_word(c, lane) : 0;
            auto r64 = [&](int d) { return (int64_t)((uint64_t)(uint32_t)W::get(rw, d) | (uint64_t)(uint32_t)W::get(rw, d + 1) << 32); };
            const uint32_t a = (uint32_t)W::get(rw, 6), bb = (uint32_t)W::get(rw, 7);
            const int64_t first_rb = r64(0), last_rb = first_rb + W::get(rw, 2);
            const int c_rid = (int)(a & 511), first_qb = (int)(a >> 9 & 511), last_qb = (int)(a >> 18 & 511);
            const int last_ln = (int)(bb & 511);
            if (rid == c_rid) {
              if (qb >= first_qb && qb + ln <= last_qb + last_ln && rb >= first_rb && rb + ln <= last_rb + last_ln) {
                merged = true;  // contained in the chain: dropped
              } else if (!((last_rb < x.l_pac || first_rb < x.l_pac) && rb >= x.l_pac)) {
                const int64_t xd = qb - last_qb, yd = rb - last_rb;
                if (yd >= 0 && xd - yd <= o.w && yd - xd <= o.w && xd - last_ln < o.max_chain_gap &&
                    yd - last_ln < o.max_chain_gap) {
                  merged = true;
                  // the weights (mem_chain_weight, aux.cu:91-110) and the window go on
                  const int at = (int)(rb - first_rb), end_r = W::get(rw, 3), c_lo = W::get(rw, 4), c_hi = W::get(rw, 5);
                  int end_q = (int)(bb >> 9 & 511), w_q = (int)(bb >> 18), n = W::get(rw, 8), w_r = W::get(rw, 9);
                  if (qb >= end_q) w_q += ln;
                  else if (qb + ln > end_q) w_q += qb + ln - end_q;
                  end_q = end_q > qb + ln ? end_q : qb + ln;
                  if (at >= end_r) w_r += ln;
                  else if (at + ln > end_r) w_r += at + ln - end_r;
                  const int e2 = end_r > at + ln ? end_r : at + ln;
                  const int l2 = c_lo < at + lo ? c_lo : at + lo, h2 = c_hi > at + hi ? c_hi : at + hi;
                  if (lane == k) {
                    my_c = c;
                    my_r = n;
                  }
                  const uint32_t a2 = (a & 0x3ffff) | (uint32_t)qb << 18;
                  const uint32_t b2 = (uint32_t)ln | (uint32_t)end_q << 9 | (uint32_t)w_q << 18;
                  uint32_t nv = (uint32_t)at;
                  nv = lane == 3 ? (uint32_t)e2 : lane == 4 ? (uint32_t)l2 : lane == 5 ? (uint32_t)h2 : nv;
                  nv = lane == 6 ? a2 : lane == 7 ? b2 : lane == 8 ? (uint32_t)(n + 1) : lane == 9 ? (uint32_t)w_r : nv;
                  if (lane >= 2 && lane < kRecWords) put_word(c, lane, nv);
                  W::global_sync();
                }
              }
            }
          }
        }
        if (merged || rid < 0 || rid >= 455) continue;  // bwa/src/aux.cu:1799
        const int c = nch++;
        uint32_t nv = (uint32_t)rb;
        nv = lane == 1 ? (uint32_t)((uint64_t)rb >> 32) : lane == 2 ? 0u : lane == 3 ? (uint32_t)ln : nv;
        nv = lane == 4 ? (uint32_t)lo : lane == 5 ? (uint32_t)hi : nv;
        nv = lane == 6 ? (uint32_t)rid | (uint32_t)qb << 9 | (uint32_t)qb << 18 : nv;
        nv = lane == 7 ? (uint32_t)ln | (uint32_t)(qb + ln) << 9 | (uint32_t)ln << 18 : nv;
        nv = lane == 8 ? 1u : lane == 9 ? (uint32_t)ln : nv;
        if (lane < kRecWords) put_word(c, lane, nv);
        W::global_sync();
        if (!put(nd, cap, c, rb)) return false;
        if (lane == k) {
          my_c = c;
          my_r = 0;
        }
      }
      if (live) {
        g.of[base + lane] = my_c;
        g.tmp[base + lane] = my_r;
      }
    }
    if (nch == 0) return true;
    // in-order traversal: the nodes on the way down, and the next child of each, a lane each
    int k = 0, sp = 0, sn = lane == 0 ? root : 0, si = 0;
    while (sp >= 0) {
      const int xi = W::get(sn, sp), i = W::get(si, sp);
      const ChainNode &X = nd[xi];
      const int n = X.n;
      if (!X.internal) {
        if (lane < n) g.order[k + lane] = X.key[lane];
        k += n;
        --sp;
        continue;
      }
      if (i > 0 && i <= n) {
        if (lane == 0) g.order[k] = X.key[i - 1];
        ++k;
      }
      if (i > n) {
        --sp;
        continue;
      }
      if (lane == sp) si = i + 1;
      ++sp;
      if (lane == sp) {
        sn = X.child[i];
        si = 0;
      }
    }
    W::global_sync();
    return true;
  }

  // is a chain of (w, b | e << 16) dropped for a kept one before it, (wj, bej)?
  G3A_LANE bool drops(uint32_t wi, uint32_t bei, uint32_t wj, uint32_t bej) const {
    if ((int)wj - (int)wi < o.min_seed_len << 1) return false;
    const int bi = (int)(bei & 0xffff), ei = (int)(bei >> 16), bj = (int)(bej & 0xffff), ej = (int)(bej >> 16);
    const int b_max = bj > bi ? bj : bi, e_min = ej < ei ? ej : ei;
    if (e_min <= b_max) return false;
    const int li = ei - bi, lj = ej - bj, min_l = li < lj ? li : lj;
    return e_min - b_max >= min_l * o.mask_level && min_l < o.max_chain_gap && (int)wi < (int)wj * o.drop_ratio;
  }

  // chain_filter: the chains' output order in g.order, g.kept per chain of it
  G3A_LANE void filter() {
    const int n = nch;
    auto weight = [&](int c) {
      const int w_q = (int)(rec_word(c, 7) >> 18), w_r = (int)rec_word(c, 9);
      return (uint32_t)(uint16_t)(w_r < w_q ? w_r : w_q);
    };
    if (n > 4096) {  // neither sorted nor filtered
      for (int i = lane; i < n; i += 64) g.kept[i] = 1;
      W::global_sync();
      return;
    }
    auto &f = st->filt;
    W::lds_sync();  // the nodes are done with
    if (n <= 3072) {
      // stable, by decreasing weight (at most the read's length): the first 2048
      const int m = n < ST::kFSort ? n : ST::kFSort;
      for (int i = lane; i < m; i += 64) {
        f.w[i] = (uint16_t)weight(g.order[i]);
        f.alt[i] = (uint16_t)i;
      }
      sort_by(f.alt, f.alt2, m, f.hist, [&](int i) { return 511u - (uint32_t)f.w[i]; });
      for (int i0 = 0; i0 < m; i0 += 64) {
        const int c = i0 + lane < m ? g.order[f.alt2[i0 + lane]] : 0;
        if (i0 + lane < m) f.be[i0 + lane] = (uint32_t)c;
      }
      W::global_sync();
      for (int i = lane; i < m; i += 64) g.order[i] = (int32_t)f.be[i];
      W::global_sync();
    }
    for (int i = lane; i < n; i += 64) {
      const int c = g.order[i];
      const uint32_t a = rec_word(c, 6), b = rec_word(c, 7);
      f.w[i] = (uint16_t)weight(c);
      f.be[i] = (a >> 9 & 511) | ((a >> 18 & 511) + (b & 511)) << 16;
    }
    W::lds_sync();
    for (int t0 = 0; t0 < n; t0 += 64) {
      const int i = t0 + lane;
      const bool live = i < n;
      const uint32_t wi = live ? f.w[i] : 0xffff, bei = live ? f.be[i] : 0;
      bool drop = false;
      // against the kept chains of the tiles before
      for (int q = 0; q < t0 / 64; ++q)
        for (uint64_t m = f.kept[q]; m; m &= m - 1) {
          const int j = 64 * q + __builtin_ffsll((long long)m) - 1;
          drop = drop || (live && drops(wi, bei, f.w[j], f.be[j]));
        }
      // and of this one, in order
      uint64_t kept = 0;
      const int cnt = n - t0 < 64 ? n - t0 : 64;
      uint64_t out = W::ballot(drop);
      for (int j = 0; j < cnt; ++j) {
        if (out >> j & 1) continue;
        kept |= 1ull << j;
        const uint32_t wj = (uint32_t)W::get((int)wi, j), bej = (uint32_t)W::get((int)bei, j);
        out |= W::ballot(live && lane > j && drops(wi, bei, wj, bej));
      }
      if (lane == 0) f.kept[t0 / 64] = kept;
      if (live) g.kept[i] = (uint8_t)(kept >> lane & 1);
      W::lds_sync();
    }
    W::global_sync();
  }

  // the kept chains' tasks, in output order and chain order; returns their number
  G3A_LANE int tasks(Task *out) {
    int32_t *coff = g.tmp + ns;  // first task of a chain
    for (int c = lane; c < nch; c += 64) coff[c] = -1;
    W::global_sync();
    const int64_t l_pac = x.l_pac;
    int total = 0;
    for (int i0 = 0; i0 < nch; i0 += 64) {
      const bool on = i0 + lane < nch && g.kept[i0 + lane];
      const int c = on ? g.order[i0 + lane] : 0;
      const int len = on ? (int)rec_word(c, 8) : 0;
      int incl = len;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = W::from(incl, lane >= d ? lane - d : 0);
        incl += lane >= d ? u : 0;
      }
      if (on) {
        coff[c] = total + incl - len;
        // chain_window
        const int64_t mid = rec64(c, 0);
        int64_t rmax0 = mid + (int32_t)rec_word(c, 4), rmax1 = mid + (int32_t)rec_word(c, 5);
        rmax0 = rmax0 < l_pac << 1 ? rmax0 : l_pac << 1;
        rmax0 = rmax0 > 0 ? rmax0 : 0;
        rmax1 = rmax1 > 0 ? rmax1 : 0;
        rmax1 = rmax1 < l_pac << 1 ? rmax1 : l_pac << 1;
        if (rmax0 < l_pac && l_pac < rmax1) {
          if (mid < l_pac) rmax1 = l_pac;
          else rmax0 = l_pac;
        }
        int is_rev;
        const int rid = pos2rid(x, depos(x, mid, is_rev));
        int64_t far_beg = x.ctg_off[rid], far_end = far_beg + x.ctg_len[rid];
        if (is_rev) {
          const int64_t t = far_beg;
          far_beg = (l_pac << 1) - far_end;
          far_end = (l_pac << 1) - t;
        }
        rmax0 = rmax0 > far_beg ? rmax0 : far_beg;
        rmax1 = rmax1 < far_end ? rmax1 : far_end;
        put_word(c, 4, (uint32_t)(rmax0 - mid));
        put_word(c, 5, (uint32_t)(rmax1 - mid));
        put_word(c, 6, (uint32_t)rid);
      }
      total += W::get(incl, 63);
    }
    W::global_sync();
    for (int e = lane; e < ns; e += 64) {
      const int c = g.of[e];
      const int at = c >= 0 ? coff[c] : -1;
      if (at < 0) continue;
      const Seed &p = seed(e);
      Task tk;
      tk.rbeg = p.rbeg;
      const int64_t mid = rec64(c, 0);
      tk.rmax0 = mid + (int32_t)rec_word(c, 4);
      tk.rmax1 = mid + (int32_t)rec_word(c, 5);
      tk.qbeg = p.qbeg;
      tk.len = p.len;
      tk.read = read;
      tk.rid = (int32_t)rec_word(c, 6);
      out[at + g.tmp[e]] = tk;
    }
    return total;
  }

  // The whole read: the number of tasks, or -1 when the nodes run out (nothing
  // is written then)
  G3A_LANE int run(Task *out) {
    sort();
    if (!build(st->node, ST::kNodes) && !build(g.nodes, g.n_nodes)) return -1;
    if (nch == 0) return 0;
    filter();
    return tasks(out);
  }
};

}  // namespace g3a
