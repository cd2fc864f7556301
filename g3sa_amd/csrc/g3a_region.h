// Region filter of one read by a wavefront, with the result of region_filter
// (g3a_dev.h): the redundancy filter, the secondary marks, the drop and the
// sort by score.
//
// What bounds it on one thread is the pairs: n^2 / 2 of them for reads of many
// regions, a load each.  The regions lie in LDS here, and a region is compared
// with 64 later ones at once.  The order of the one-thread code is kept: the
// first later region that removes this one stops it, those before it that this
// one removes are removed, those after it are not looked at.
#pragma once
#include "g3a_lanes.h"

namespace g3a {

// LDS of a read of at most N regions: 30 bytes a region
template <int N>
struct RegionStage {
  static constexpr int kMax = N;
  int64_t rb[N];
  int32_t rlen[N], score[N], rid[N];
  uint16_t qb[N], qe[N], len0[N];
  uint16_t sec[N];  // region that this one is secondary to, kNoSec if none
  uint16_t idx[N];  // the regions that are left
  uint64_t flag[N / 64];
};
constexpr uint32_t kNoSec = 0xffff;

template <class W, class ST>
struct RegionGroup {
  const Opt &o;
  ST *st;
  int lane;

  // a sorted-in-place read of n <= ST::kMax regions; returns the number kept
  G3A_LANE int run(Region *a, int n) {
    W::lds_sync();  // earlier reads of the LDS are done
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int i = i0 + lane;
      bool on = false;
      if (i < n) {
        const Region g = a[i];
        st->rb[i] = g.rb;
        st->rlen[i] = (int32_t)(g.re - g.rb);
        st->score[i] = g.score;
        st->rid[i] = g.rid;
        st->qb[i] = (uint16_t)g.qb;
        st->qe[i] = (uint16_t)g.qe;
        st->len0[i] = (uint16_t)g.seedlen0;
        on = g.score >= o.T;
      }
      const uint64_t m = W::ballot(on);
      if (lane == 0) st->flag[i0 / 64] = m;
    }
    W::lds_sync();
    const int tiles = (n + 63) / 64;
    // redundant regions
    for (int i = 0; i < n; ++i) {
      if (!(st->flag[i >> 6] >> (i & 63) & 1)) continue;
      const int64_t i_rb = st->rb[i], i_re = i_rb + st->rlen[i];
      const int i_rid = st->rid[i], i_qb = st->qb[i], i_qe = st->qe[i], i_score = st->score[i];
      for (int t = i >> 6; t < tiles; ++t) {
        uint64_t live = st->flag[t];
        if (t == i >> 6) live &= ~0ull << (i & 63) << 1;
        if (!live) continue;
        const int j = 64 * t + lane;
        bool red = false, lt = false;
        if (live >> lane & 1) {
          const int64_t j_rb = st->rb[j], j_re = j_rb + st->rlen[j];
          if (i_rid == st->rid[j] && !(i_rb < j_rb && i_re < j_rb) && !(j_rb < i_rb && j_re < i_rb)) {
            const int j_qb = st->qb[j], j_qe = st->qe[j];
            const int or_ = (int)(i_rb < j_rb ? i_re - j_rb : j_re - i_rb);
            const int oq = i_qb < j_qb ? i_qe - j_qb : j_qe - i_qb;
            const int rli = (int)(i_re - i_rb), rlj = (int)(j_re - j_rb);
            const int mr = rli < rlj ? rli : rlj;
            const int mq = i_qe - i_qb < j_qe - j_qb ? i_qe - i_qb : j_qe - j_qb;
            red = or_ > o.mask_level_redun * mr && oq > o.mask_level_redun * mq;
            lt = i_score < st->score[j];
          }
        }
        uint64_t gone = W::ballot(red);
        const uint64_t stop = W::ballot(red && lt);
        if (!gone) continue;
        if (stop) gone &= (stop & (0ull - stop)) - 1;  // those before the first that removes i
        W::lds_sync();
        if (lane == 0) {
          st->flag[t] &= ~gone;
          if (stop) st->flag[i >> 6] &= ~(1ull << (i & 63));
        }
        W::lds_sync();
        if (stop) break;
      }
    }
    // those left, in order
    int m = 0;
    for (int t = 0; t < tiles; ++t) {
      const uint64_t f = st->flag[t];
      if (f >> lane & 1) st->idx[m + __builtin_popcountll(f & ((1ull << lane) - 1))] = (uint16_t)(64 * t + lane);
      m += __builtin_popcountll(f);
    }
    for (int p = lane; p < m; p += 64) st->sec[p] = (uint16_t)kNoSec;
    W::lds_sync();
    // secondary marks, by place among those left
    for (int p = 0; p < m; ++p) {
      if (st->sec[p] != kNoSec) continue;
      const int i = st->idx[p], i_qb = st->qb[i], i_qe = st->qe[i], i_score = st->score[i];
      for (int q0 = p + 1; q0 < m; q0 += 64) {
        const int q = q0 + lane;
        bool ov = false, ge = false;
        if (q < m && st->sec[q] == kNoSec) {
          const int j = st->idx[q], j_qb = st->qb[j], j_qe = st->qe[j];
          const int qb_max = i_qb > j_qb ? i_qb : j_qb, qe_min = i_qe < j_qe ? i_qe : j_qe;
          if (qe_min > qb_max) {
            const int li = i_qe - i_qb, lj = j_qe - j_qb, min_l = li < lj ? li : lj;
            ov = qe_min - qb_max >= min_l * o.mask_level;
            ge = !(i_score > st->score[j]);
          }
        }
        uint64_t mark = W::ballot(ov);
        const uint64_t stop = W::ballot(ov && ge);
        if (!mark) continue;
        int by = -1;
        if (stop) {
          by = q0 + __builtin_ffsll((long long)stop) - 1;
          mark &= (stop & (0ull - stop)) - 1;
        }
        W::lds_sync();
        if (mark >> lane & 1) st->sec[q] = (uint16_t)p;
        if (stop && lane == 0) st->sec[p] = (uint16_t)by;
        W::lds_sync();
        if (stop) break;
      }
    }
    // the regions to output, in order
    int k = 0;
    if (!(o.flag & 0x8)) {
      for (int p0 = 0; p0 < m; p0 += 64) {
        const int p = p0 + lane;
        const bool on = p < m && st->sec[p] == kNoSec;
        const int i = on ? (int)st->idx[p] : 0;
        const uint64_t b = W::ballot(on);
        W::lds_sync();
        if (on) st->idx[k + __builtin_popcountll(b & ((1ull << lane) - 1))] = (uint16_t)i;
        W::lds_sync();
        k += __builtin_popcountll(b);
      }
      for (int p = lane; p < k; p += 64) st->sec[p] = (uint16_t)kNoSec;
      W::lds_sync();
    } else {
      // the one-thread code writes a kept region over an earlier place, and
      // later ones compare with what is there: places are followed one by one
      for (int p = 0; p < m; ++p) {
        const uint32_t sec = st->sec[p];
        const int i = st->idx[p];
        const bool drop = sec != kNoSec && st->score[i] < st->score[st->idx[sec]] * o.drop_ratio;
        W::lds_sync();
        if (!drop) {
          if (lane == 0) {
            st->idx[k] = (uint16_t)i;
            st->sec[k] = (uint16_t)sec;
          }
          ++k;
        }
        W::lds_sync();
      }
    }
    // by decreasing score, stable
    for (int p0 = 0; p0 < k; p0 += 64) {
      const int p = p0 + lane;
      const bool on = p < k;
      const int i = on ? (int)st->idx[p] : 0, sc = on ? st->score[i] : 0;
      int at = 0;
      for (int q = 0; q < k; ++q) {
        const int u = st->score[st->idx[q]];
        at += u > sc || (u == sc && q < p);
      }
      if (on) {
        Region g;
        g.rb = st->rb[i];
        g.re = g.rb + st->rlen[i];
        g.qb = st->qb[i];
        g.qe = st->qe[i];
        g.score = sc;
        g.rid = st->rid[i];
        g.seedlen0 = st->len0[i];
        g.secondary = st->sec[p] == kNoSec ? -1 : (int)st->sec[p];
        a[at] = g;
      }
    }
    return k;
  }
};

}  // namespace g3a
