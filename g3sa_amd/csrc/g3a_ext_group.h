// Banded local extension of one task by a group of 16 lanes, with the cell set
// and the result of the lane engine (g3a_ext.h) and the oracle's
// orc_ksw_extend.
//
// What bounds a task on one lane is its chain of columns: about 900 cycles a
// column of a 16-row strip, 0.5 ms for a side of a 150-base read, however few
// tasks there are.  Here a pass covers 128 target rows as a systolic array of
// 32 places of 4 rows: a lane holds two places in the halves of its registers
// (one packed operation computes two cells), and at step s place v is at
// column s - v.  The last row's H and E of a column reach the next place one
// step later, across lanes by DPP, from the last place to the first of the
// next pass through LDS.  A pass of a 107-base side is 138 steps instead of 8
// strips of 107 columns, and 122 of 138 steps' places are busy.
//
// A column that a place has not reached (j < 0) and those past the query
// score -8 on zeros and stay 0; the boundary (column -1) enters as the
// diagonal inputs of column 0.  The rules of the cell set (band, column limit,
// corner, quirk rows) are masks that only the steps where one can apply to
// some lane carry.  The best cell is kept as a 16-bit key, 4 H + (3 - row of
// the place), with its column, so that an equal score prefers the smaller row
// and then the later column.  When no cell exceeds h0 the position follows the
// reference's 32-lane residue rule, which needs a cell equal to h0 in every
// residue of the rows mod 32: a task in which that is possible is handed back.
//
// Exact pruning as in the lane engine, after each pass.  Extension of 100,000
// reads of 150 bases, 281,296 tasks: 10.1 ms on a wavefront per task, 2.9 ms.
#pragma once
#include "g3a_ext.h"
#include "g3a_lanes.h"

namespace g3a {

constexpr int kGrpPlaces = 32, kGrpRows = 4, kGrpPass = kGrpPlaces * kGrpRows;
constexpr int kGrpRun = 8;  // steps taken between looks at the rules
// columns past the query that steps touch: the places behind, the rest of a run
constexpr int kGrpCols = kExtQCap + kGrpPlaces + kGrpRun;
constexpr int kGrpQ = kGrpPlaces + kGrpCols;  // query codes from column -32 on
struct ExtGroupStage {
  uint32_t row[kGrpCols];  // H << 16 | E of the row above the pass
  uint32_t tab[6][16];                      // scores of a lane's 8 rows against each query code, 4 bits each
  uint8_t q[kGrpQ];
};
static_assert(sizeof(ExtGroupStage) % 4 == 0, "stages follow each other");

// A padding column must lose to the real column before it even through an
// insertion, and a padding row through a deletion.
G3A_HD bool ext_group_opt_ok(const Opt &o) {
  return ext_lane_opt_ok(o) && o.o_del + o.e_del > 0 && o.o_ins + o.e_ins > 0;
}

G3A_HD uint32_t p2_bits(P2 a) { return (uint32_t)(uint16_t)p2_lo(a) | (uint32_t)(uint16_t)p2_hi(a) << 16; }
G3A_HD P2 p2_of(uint32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
  P2 r;
  r.v = __builtin_bit_cast(g3a_s16x2, b);
  return r;
#else
  return p2((int16_t)(uint16_t)b, (int16_t)(uint16_t)(b >> 16));
#endif
}
// a's bits where m is set, b's elsewhere
G3A_HD P2 p2_pick(uint32_t m, P2 a, P2 b) { return p2_of((p2_bits(a) & m) | (p2_bits(b) & ~m)); }
G3A_HD P2 p2_and(uint32_t m, P2 a) { return p2_of(p2_bits(a) & m); }
// the low half of `own` as the high one, the high half of `from` as the low one
G3A_HD uint32_t pass_on(uint32_t own, uint32_t from) { return own << 16 | from >> 16; }
G3A_HD uint32_t halves(bool lo, bool hi) { return (lo ? 0xffffu : 0u) | (hi ? 0xffff0000u : 0u); }
// 0xffff in each half where a >= b (both >= 0)
G3A_HD uint32_t p2_ge(P2 a, P2 b) {
  const P2 one = p2(1, 1);
  return p2_bits(p2_sub(p2_min(p2_subsat(b, a), one), one));
}

struct ExtGroupOut {
  int score, qle, tle;
  bool exact;  // false: the residue rule may apply, nothing else is set
};

template <class W, bool SYM>
struct ExtGroup {
  const Opt &o;
  ExtGroupStage *st;
  int gl, gb;

  // the same value on the group's 16 lanes
  G3A_LANE int max16(int v) const {
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
      const int u = W::from_xor(v, d);
      v = u > v ? u : v;
    }
    return v;
  }
  G3A_LANE uint64_t max16(uint64_t v) const {
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
      const uint64_t u = W::from_xor(v, d);
      v = u > v ? u : v;
    }
    return v;
  }

  // qcode(j): query code of column j < qlen; rows8(i): target codes (0..3) of
  // rows i..i+7, two bits each, row i lowest (any for rows >= tlen)
  template <class Q, class T>
  G3A_LANE ExtGroupOut run(int qlen, Q qcode, int tlen, T rows8, int w, int h0) {
    const int oe_del = o.o_del + o.e_del, oe_ins = o.o_ins + o.e_ins, ms = mat_max(o);
    W::lds_sync();  // the group's earlier reads of its LDS are done
    for (int k = gl; k < kGrpQ; k += 16) {
      const int j = k - kGrpPlaces;
      st->q[k] = (uint8_t)(j >= 0 && j < qlen ? qcode(j) : kExtPad);
    }
    // row -1: H(-1, j) is the diagonal input of column j + 1
    for (int j = gl; j < kGrpCols; j += 16) {
      const int hv = h0 - oe_ins - j * o.e_ins;
      st->row[j] = j < qlen && hv > 0 ? (uint32_t)hv << 16 : 0;
    }
    const P2 oeP = p2(oe_del, oe_del), oiP = p2(oe_ins, oe_ins), edP = p2(o.e_del, o.e_del), eiP = p2(o.e_ins, o.e_ins);
    // scores of target code t against query codes 0..4, 4 bits each
    uint32_t mt[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      mt[t] = 0;
#pragma unroll
      for (int c = 0; c < 5; ++c) mt[t] |= (uint32_t)(o.mat[5 * t + c] & 15) << (4 * c);
    }
    uint64_t best = 0;  // score, row (smaller is more) and column of the best cell above h0
    uint32_t seen = 0;  // residues (mod 32) of rows whose place held a cell equal to h0
    for (int p0 = 0; p0 < tlen && p0 - w < qlen; p0 += kGrpPass) {  // later rows have no columns
      const int il = p0 + 8 * gl, ih = il + kGrpRows;  // first rows of this lane's two places
      {
        const uint32_t codes = rows8(il);
        uint32_t v[5] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const uint32_t t = codes >> (2 * r) & 3;
          uint32_t s = t & 1 ? (t & 2 ? mt[3] : mt[1]) : (t & 2 ? mt[2] : mt[0]);
          s = il + r < tlen ? s : 0x88888u;
#pragma unroll
          for (int c = 0; c < 5; ++c) v[c] |= (s >> (4 * c) & 15) << (4 * r);
        }
#pragma unroll
        for (int c = 0; c < 5; ++c) st->tab[c][gl] = v[c];
        st->tab[5][gl] = 0x88888888u;
      }
      W::lds_sync();
      // the boundary of the row above each row
      auto above = [&](int i) {
        const int b = h0 - o.o_del - o.e_del * i;
        return i == 0 ? h0 : b > 0 ? b : 0;
      };
      P2 bP[kGrpRows], hP[kGrpRows], fP[kGrpRows];
#pragma unroll
      for (int r = 0; r < kGrpRows; ++r) {
        bP[r] = p2(above(il + r), above(ih + r));
        hP[r] = fP[r] = p2(0, 0);
      }
      // columns [g0, j0) and from j1 on of a place need a rule.  Left of the
      // band a cell is 0 by itself as long as w + 1 deletions cost more than
      // h0 and the columns so far can give.
      const int spare = o.o_del + o.e_del * (w + 1) - h0, free_cols = ms > 0 && spare > 0 ? spare / ms : 0;
      auto plain = [&](int i0, int &g0, int &j0, int &j1) {
        g0 = free_cols;
        j0 = i0 + kGrpRows - 1 - w > 0 ? i0 + kGrpRows - 1 - w : 0;
        if (i0 + w + 1 < 30 - i0) {
          g0 = 0;
          j0 = j0 < 31 - i0 ? 31 - i0 : j0;
        }
        j1 = 32 * (i0 / 32 + 1) + w + 2;
        if (i0 >= 32 && (i0 & 31) == 0 && i0 + w + 2 < j1) j1 = i0 + w + 2;
      };
      int lg, l0, l1, ug, u0, u1;
      plain(il, lg, l0, l1);
      plain(ih, ug, u0, u1);
      // columns left of every row's band: nothing to do
      const int jb = p0 - w > 0 ? p0 - w : 0;
      // the boundary inputs' and the key's constants
      const P2 k0 = p2((h0 + 1) << 2, (h0 + 1) << 2);
      const uint32_t h0x = (uint32_t)h0 << 2 | (uint32_t)h0 << 18;
      P2 bk = k0, bj = p2(-1, -1), near = p2_of(0x7fff7fffu);
      P2 diag = p2(jb > 0 && gl == 0 ? (int)(st->row[jb - 1] >> 16) : 0, 0);
      uint32_t hl = 0, eo = 0;  // the last rows' H and E of the step before
      uint32_t tab_p = 0x88888888u;
      // place v is at column s - v at step s, from column jb on; before that
      // its cells are 0 as the query codes' padding and its inputs are
      const uint8_t *qs = st->q + (kGrpPlaces - 2 * gl);
      uint32_t tab_c = st->tab[2 * gl > 0 ? kExtPad : qs[jb]][gl];
      uint32_t code_n = 2 * gl > 1 ? (uint32_t)kExtPad : qs[jb + 1];
      uint32_t in_n = st->row[jb];
      const int s_end = qlen + kGrpPlaces - 1;
      auto step = [&](int s, auto general_tag, auto start_tag) {
        constexpr bool kGeneral = decltype(general_tag)::value, kStart = decltype(start_tag)::value;
        const int jl = s - 2 * gl, jh = jl - 1;
        const uint32_t X = (tab_c & 0xffffu) | (tab_p & 0xffff0000u);
        const uint32_t in_row = in_n;
        // the next step's loads
        tab_p = tab_c;
        tab_c = st->tab[code_n][gl];
        code_n = kStart && jl + 2 < jb ? (uint32_t)kExtPad : qs[s + 2];
        in_n = st->row[s + 1];
        const uint32_t h_in = pass_on(hl, (uint32_t)W::template before<16>((int)hl, (int)in_row, gl));
        const uint32_t e_in = pass_on(eo, (uint32_t)W::template before<16>((int)eo, (int)(in_row << 16), gl));
        P2 d0 = diag, e = p2_of(e_in);
        diag = p2_of(h_in);
        uint32_t ok[kGrpRows];
        if (kGeneral) {
          // the rules, for the rows of each half
          auto rows = [&](int i0, int j) -> uint32_t {
            int n = j + w - i0 + 1;  // band: row r <= j + w - i0
            n = n < 0 ? 0 : n > kGrpRows ? kGrpRows : n;
            if (j > 32 * (i0 / 32 + 1) + w + 1) n = 0;
            uint32_t m = (1u << n) - 1;
            int c = 31 - i0 - j < j - i0 - w - 1 ? 31 - i0 - j : j - i0 - w - 1;  // corner: rows below c are out
            c = c < 0 ? 0 : c > kGrpRows ? kGrpRows : c;
            return m & ~((1u << c) - 1);
          };
          const uint32_t ml = rows(il, jl), mh = rows(ih, jh);
#pragma unroll
          for (int r = 0; r < kGrpRows; ++r) ok[r] = halves(ml >> r & 1, mh >> r & 1);
          if (il >= 32 && (il & 31) == 0 && jl > il + w + 1) {  // quirk row: an injected diagonal and no E
            const int v = h0 - oe_ins - (jl - 1) * o.e_ins;
            d0 = p2(v > 0 ? v : 0, p2_hi(d0));
            e = p2_and(0xffff0000u, e);
          }
        }
        const uint32_t start = kStart ? halves(jl == 0, jh == 0) : 0;
#pragma unroll
        for (int r = kGrpRows - 1; r >= 0; --r) {
          P2 d = r ? hP[r - 1] : d0;
          if (kStart) d = p2_pick(start, bP[r], d);
          // M = 0 when the diagonal is 0: see g3a_ext.h
          hP[r] = p2_min(p2_add(d, p2_nibble(X, r)), p2_shl3(d));
        }
        P2 km = p2(0, 0);
#pragma unroll
        for (int r = 0; r < kGrpRows; ++r) {
          const P2 m = hP[r], f = fP[r];
          P2 h = p2_max(p2_max(m, e), f);
          const P2 td = p2_sub(m, oeP), ti = SYM ? td : p2_sub(m, oiP);
          e = p2_max(p2_subsat(e, edP), td);
          P2 f2 = p2_max(p2_subsat(f, eiP), ti);
          if (kGeneral) {
            h = p2_and(ok[r], h);
            e = p2_and(ok[r], e);
            f2 = p2_and(ok[r], f2);
          }
          hP[r] = h;
          fP[r] = f2;
          km = p2_max(km, p2_add(p2_add(p2_add(h, h), p2_add(h, h)), p2(kGrpRows - 1 - r, kGrpRows - 1 - r)));
        }
        hl = p2_bits(hP[kGrpRows - 1]);
        eo = p2_bits(e);
        const uint32_t ge = p2_ge(km, bk);
        bk = p2_max(bk, km);
        bj = p2_pick(ge, p2_of((uint32_t)(uint16_t)jl | (uint32_t)(uint16_t)jh << 16), bj);
        near = p2_min(near, p2_of((p2_bits(km) ^ h0x) & 0x7ffc7ffcu));
        if (gl == 15 && (!kStart || jh >= jb)) st->row[jh] = (hl & 0xffff0000u) | eo >> 16;
      };
      const int s_run = jb + kGrpPlaces;  // from here on every place is at or past column jb
      // kGrpRun steps at a time, on the form that all of them on all lanes
      // admit (the steps past s_end are at padding columns)
      for (int s = jb; s < s_end; s += kGrpRun) {
        const int jl = s - 2 * gl, jh = jl - 1, last = kGrpRun - 1;
        const bool gen = (jl < qlen && ((jl + last >= lg && jl < l0) || jl + last >= l1)) ||
                         (jh < qlen && ((jh + last >= ug && jh < u0) || jh + last >= u1));
        if (W::ballot(gen)) {
#pragma unroll 1
          for (int k = 0; k < kGrpRun; ++k) step(s + k, std::true_type(), std::true_type());
        } else if (W::ballot(s < s_run)) {
#pragma unroll 2
          for (int k = 0; k < kGrpRun; ++k) step(s + k, std::false_type(), std::true_type());
        } else {
#pragma unroll
          for (int k = 0; k < kGrpRun; ++k) step(s + k, std::false_type(), std::false_type());
        }
      }
      // the pass's best cells
      auto cand = [&](int key, int col, int i0) -> uint64_t {
        if (col < 0) return 0;
        const int row = i0 + kGrpRows - 1 - (key & 3);
        return (uint64_t)(uint32_t)(key >> 2) << 42 | (uint64_t)(0x1FFFFF - row) << 21 | (uint64_t)(uint32_t)col;
      };
      const uint64_t cl = cand(p2_lo(bk), p2_lo(bj), il), cu = cand(p2_hi(bk), p2_hi(bj), ih);
      best = cl > best ? cl : best;
      best = cu > best ? cu : best;
      seen |= (p2_lo(near) == 0 ? 15u << (il & 31) : 0) | (p2_hi(near) == 0 ? 15u << (ih & 31) : 0);
      W::lds_sync();
      const int i1 = p0 + kGrpPass;
      if (i1 >= tlen) break;
      // bound on every later cell: paths through the pass's last row, the
      // boundary of later rows, and the next quirk row's injections
      best = max16(best);
      const int top = best ? (int)(best >> 42) : h0;
      int ub = 0;
      for (int j = gl; j < qlen; j += 16) {
        const int h = (int)(st->row[j] >> 16), v = h + ms * (qlen - 1 - j);
        if (h > 0 && v > ub) ub = v;
      }
      ub = max16(ub);
      const int b = h0 - o.o_del - o.e_del * i1;
      if (b > 0 && b + ms * qlen > ub) ub = b + ms * qlen;
      const int iq = (i1 + 31) & ~31;
      if (iq + w + 2 <= qlen - 1) {
        const int dq = h0 - oe_ins - (iq + w + 1) * o.e_ins;
        const int bq = dq > 0 ? dq + ms * (qlen - iq - w - 2) : 0;
        ub = ub > bq ? ub : bq;
      }
      if (ub < top) break;
    }
    best = max16(best);
    ExtGroupOut r;
    r.score = h0;
    r.qle = r.tle = 0;
    r.exact = true;
    if (best) {
      r.score = (int)(best >> 42);
      r.tle = 0x1FFFFF - (int)(best >> 21 & 0x1FFFFF) + 1;
      r.qle = (int)(best & 0x1FFFFF) + 1;
    } else {
#pragma unroll
      for (int d = 8; d >= 1; d >>= 1) seen |= (uint32_t)W::from_xor((int)seen, d);
      r.exact = seen != 0xffffffffu;
    }
    return r;
  }
};

// Cells of the reference's cell set in row i
G3A_HD int ext_row_cells(int i, int qlen, int w) {
  const int jlim = 32 * (i / 32 + 1) + w + 1, lo = i - w > 0 ? i - w : 0, hi = qlen - 1 < jlim ? qlen - 1 : jlim;
  if (hi < lo) return 0;
  int n = hi - lo + 1;
  const int c0 = lo > i + w + 2 ? lo : i + w + 2, c1 = hi < 30 - i ? hi : 30 - i;  // corner cells
  if (c1 >= c0) n -= c1 - c0 + 1;
  return n;
}

}  // namespace g3a
