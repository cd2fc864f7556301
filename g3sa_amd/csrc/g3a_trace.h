// Global alignment of one kept region by a group of G lanes: the banded DP of
// global_dp, the walk of global_walk and the mismatch count of
// trace_and_finalize (g3a_dev.h, one thread), with the same results.
//
// What bounds it on one thread is a serial chain: 15 to 127 cells a row one
// after another, a walk of one dependent byte load a step, and a last pass
// over the read.  Here a lane (or two or four register slots of it) is a band
// column.  A row's F values depend on its M values only, so a row is one
// max-plus prefix scan over the lanes; E and the next row's H come from the
// lane itself or its neighbour.  A cell's direction is four bits, eight rows
// of a column share a 32-bit word in LDS, and the walk takes a run of matches
// eight rows at a time.
#pragma once
#include "g3a_lanes.h"

namespace g3a {

// Bands of at most kGapCols columns; wider ones run on one thread.
constexpr int kGapCols = 127, kGapW = kGapCols / 2;
// w is at least 3 more than the lengths differ by, so a band of half-width w
// spans at most kMaxReadLen + w - 3 rows
constexpr int kGapRows = (kMaxReadLen + kGapW - 3 + 3) & ~3;
struct GapStage {
  int8_t prof[5][kMaxReadLen];  // score of text base t against query column j
  uint8_t q[kMaxReadLen], t[kGapRows];
};
static_assert(sizeof(GapStage) % 4 == 0, "32-bit words follow it");
// 32-bit words of the direction bits of a band of w columns either side
G3A_HD int gap_cols(int qlen, int w) { return qlen < 2 * w + 1 ? qlen : 2 * w + 1; }
G3A_HD int gap_words(int qlen, int tlen, int w) { return ((tlen + 7) >> 3) * gap_cols(qlen, w); }

template <class W, int G, int NH>
struct GapGroup {
  const DevIndex &x;
  const Opt &o;
  GapStage *st;
  uint32_t *z;  // gap_words() words
  int gl, gb;   // this lane in the group, the group's first lane in the wavefront
  int qlen, tlen, w;

  G3A_LANE uint64_t ballot(bool p) const {
    const uint64_t m = W::ballot(p);
    return G == 64 ? m : (m >> gb) & ((1ull << G) - 1);
  }

  G3A_LANE void load(const uint8_t *query, int64_t rb) {
    W::lds_sync();  // the group's earlier reads of its LDS are done
    for (int j = gl; j < qlen; j += G) {
      const int c = query[j];
      st->q[j] = (uint8_t)c;
#pragma unroll
      for (int t = 0; t < 5; ++t) {
        const int v = c == 0 ? o.mat[5 * t] : c == 1 ? o.mat[5 * t + 1] : c == 2 ? o.mat[5 * t + 2]
                      : c == 3 ? o.mat[5 * t + 3] : o.mat[5 * t + 4];
        st->prof[t][j] = (int8_t)v;
      }
    }
    for (int i = 8 * gl; i < tlen; i += 8 * G) {
      const uint64_t v = text_word(x, rb + i);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (i + k < tlen) st->t[i + k] = (uint8_t)(v >> (62 - 2 * k) & 3);
    }
    W::lds_sync();
  }

  // value of column c of a row
  G3A_LANE int at(const int (&v)[NH], int c) const {
    int r = 0;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int u = W::from(v[h], gb + (c & (G - 1)));
      r = c / G == h ? u : r;
    }
    return r;
  }

  // global_dp: the direction bits into z; returns the score
  G3A_LANE int dp() {
    const int MINUS_INF = -0x40000000;
    const int oe_del = o.o_del + o.e_del, oe_ins = o.o_ins + o.e_ins;
    const int ncol = gap_cols(qlen, w);
    int hp[NH], ep[NH], beg_p = 0, n_p = 0;
    uint32_t zw[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      hp[h] = 0;
      ep[h] = MINUS_INF;
      zw[h] = 0;
    }
    for (int i = 0; i < tlen; ++i) {
      const int beg = i > w ? i - w : 0, end = i + w + 1 < qlen ? i + w + 1 : qlen, n = end - beg;
      const bool moved = beg != beg_p;  // by one column
      const int8_t *pr = st->prof[st->t[i]];
      int m[NH], pm[NH], ein[NH];
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int c = G * h + gl, j = beg + c;
        const bool act = c < n;
        const int sc = pr[act ? j : 0];
        // the column before in the row above, and this one
        const int left = h == 0 ? -(o.o_del + o.e_del * i) : W::from(hp[h - 1 < 0 ? 0 : h - 1], gb + G - 1);
        const int right = h + 1 < NH ? W::from(ep[h + 1 < NH ? h + 1 : h], gb) : MINUS_INF;
        const int hu = W::template before<G>(hp[h], left, gl), eu = W::template after<G>(ep[h], right, gl);
        int hd = moved ? hp[h] : hu;
        int e = moved ? eu : ep[h];
        e = c + (moved ? 1 : 0) >= n_p ? MINUS_INF : e;
        if (i == 0) {
          hd = j == 0 ? 0 : -(o.o_ins + o.e_ins * j);
          e = MINUS_INF;
        }
        ein[h] = e;
        m[h] = hd + sc;
        pm[h] = act ? m[h] - oe_ins + o.e_ins * (c + 1) : MINUS_INF;
      }
      int carry = MINUS_INF;
      const bool flush = (i & 7) == 7 || i == tlen - 1;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        int v = W::template max_scan<G>(pm[h], MINUS_INF - 0x20000000, gl);
        v = carry > v ? carry : v;
        int ex = W::template before<G>(v, carry, gl);
        ex = ex < MINUS_INF ? MINUS_INF : ex;
        if (h + 1 < NH) carry = W::from(v, gb + G - 1);
        const int c = G * h + gl;
        const int f = ex - c * o.e_ins;
        uint32_t dir = m[h] >= ein[h] ? 0 : 1;
        int hh = m[h] >= ein[h] ? m[h] : ein[h];
        dir = hh >= f ? dir : 2;
        hh = hh >= f ? hh : f;
        int tt = m[h] - oe_del, e2 = ein[h] - o.e_del;
        dir |= e2 > tt ? 4 : 0;
        e2 = e2 > tt ? e2 : tt;
        tt = m[h] - oe_ins;
        dir |= f - o.e_ins > tt ? 8 : 0;
        hp[h] = hh;
        ep[h] = e2;
        zw[h] = zw[h] >> 4 | dir << 28;
        if (flush && c < ncol) z[(i >> 3) * ncol + c] = zw[h] >> (4 * (7 - (i & 7)));
      }
      beg_p = beg;
      n_p = n;
    }
    W::global_sync();  // z may be global memory
    return at(hp, qlen - 1 - beg_p);
  }

  // global_walk, and the mismatches and gap bases of the alignment: the CIGAR
  // goes to core (room for qlen + tlen words); returns its operation count
  G3A_LANE int walk(uint32_t *core, int &nm) {
    const int ncol = gap_cols(qlen, w), room = qlen + tlen;
    int n = 0, which = 0, i = tlen - 1, k = (i + w + 1 < qlen ? i + w + 1 : qlen) - 1;
    int op = -1, len = 0, mism = 0, gap = 0;
    // operations come last first: the n-th goes to core[room - 1 - n]
    auto flush = [&]() {
      if (op < 0) return;
      if (gl == 0) core[room - 1 - n] = (uint32_t)(len << 4 | op);
      if (op == 0) {
        for (int u0 = 0; u0 < len; u0 += G) {
          const int u = u0 + gl;
          mism += __builtin_popcountll(ballot(u < len && st->q[k + 1 + u] != st->t[i + 1 + u]));
        }
      } else if (op == 1) {
        gap += len;
      } else if (n > 0 && (i >= 0 || k >= 0)) {
        gap += len;  // a deletion at either end is not counted
      }
      ++n;
    };
    auto push = [&](int what, int by) {
      if (what != op) {
        flush();
        op = what;
        len = 0;
      }
      len += by;
    };
    while (i >= 0 && k >= 0) {
      const int beg = i > w ? i - w : 0;
      const uint32_t v = z[(i >> 3) * ncol + (k - beg)];
      const int r = i & 7;
      if (which == 0) {
        // the matches from here up this column's word: along a diagonal the
        // band column stays the same while the band moves
        const uint32_t left = (v & 0x33333333u) << (4 * (7 - r));
        int run = left ? __builtin_clz(left) >> 2 : 8;
        run = run < r + 1 ? run : r + 1;
        if (i - w < run) run = i > w ? i - w : run < 1 ? run : 1;
        if (k + 1 < run) run = k + 1;
        if (run > 0) {
          push(0, run);
          i -= run;
          k -= run;
          continue;
        }
      }
      const uint32_t d = v >> (4 * r) & 15;
      which = which == 0 ? (int)(d & 3) : which == 1 ? (int)(d >> 2 & 1) : (int)(d >> 3 & 1) << 1;
      if (which == 0) {
        push(0, 1);
        --i;
        --k;
      } else if (which == 1) {
        push(2, 1);
        --i;
      } else {
        push(1, 1);
        --k;
      }
    }
    if (i >= 0) {
      const int by = i + 1;
      if (op != 2) {
        flush();
        op = 2;
        len = 0;
      }
      len += by;
      i = -1;
    }
    if (k >= 0) {
      const int by = k + 1;
      if (op != 1) {
        flush();
        op = 1;
        len = 0;
      }
      len += by;
      k = -1;
    }
    flush();
    nm = mism + gap;
    W::global_sync();
    // into place, a group's width at a time (the target is below the source)
    for (int a0 = 0; a0 < n && n < room; a0 += G) {
      const uint32_t v = a0 + gl < n ? core[room - n + a0 + gl] : 0;
      W::global_sync();
      if (a0 + gl < n) core[a0 + gl] = v;
    }
    return n;
  }
};

}  // namespace g3a
