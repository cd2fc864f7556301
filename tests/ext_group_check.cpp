// The group extension of g3a_ext_group.h on the host, its lanes as fibers:
// score and position of random tasks against the oracle's banded extension
// (orc_ksw_extend), and the cells of a row against the oracle's count.
//   ext_group_check CASES SEED
// Prints the counts; exits non-zero on any mismatch.
#include "g3sa_amd/csrc/g3a_ext_group.h"
#include "tests/fibers.h"
extern "C" {
#include "oracle/oracle.h"
}
#include <cstring>
#include <random>
using namespace g3a;

template <bool SYM>
static ExtGroupOut group(Fibers &fb, const Opt &o, const std::vector<uint8_t> &q, int qlen, const std::vector<uint8_t> &t,
                         int tlen, int w, int h0) {
  static ExtGroupStage st;
  std::memset(&st, 0xa5, sizeof st);
  ExtGroupOut out[16];
  fb.run(16, [&](int lane) {
    ExtGroup<HostLanes, SYM> g{o, &st, lane, 0};
    out[lane] = g.run(
        qlen, [&](int j) { return (int)q[(size_t)j]; }, tlen,
        [&](int i) {
          uint32_t v = 0;
          for (int r = 0; r < 8; ++r) v |= (uint32_t)(i + r < tlen ? t[(size_t)(i + r)] : 1) << (2 * r);
          return v;
        },
        w, h0);
  });
  for (int l = 1; l < 16; ++l)
    if (out[l].score != out[0].score || out[l].qle != out[0].qle || out[l].tle != out[0].tle ||
        out[l].exact != out[0].exact) {
      std::printf("FAIL lanes disagree\n");
      std::exit(1);
    }
  return out[0];
}

int main(int argc, char **argv) {
  const int n = argc > 1 ? atoi(argv[1]) : 2000;
  std::mt19937_64 rng(argc > 2 ? strtoull(argv[2], 0, 10) : 1);
  auto U = [&](int lo, int hi) { return (int)(lo + rng() % (uint64_t)(hi - lo + 1)); };
  Fibers fb;
  long bad = 0, tested = 0, handed = 0, at_h0 = 0, narrow = 0, lng = 0;
  for (int it = 0; it < n; ++it) {
    Opt o;
    memset(&o, 0, sizeof o);
    o.a = it % 5 == 3 ? 2 : 1;
    o.b = it % 5 == 3 ? 3 : 4;
    o.o_del = o.o_ins = 6; o.e_del = o.e_ins = 1;
    if (rng() % 3 == 0) { o.o_del = U(0, 8); o.e_del = U(1, 2); o.o_ins = U(0, 8); o.e_ins = U(1, 2); }
    if (it % 50 == 7) { o.e_del = o.e_ins = 0; o.o_del = U(1, 4); o.o_ins = U(1, 4); }
    int k = 0;
    for (int i = 0; i < 4; ++i) { for (int j = 0; j < 4; ++j) o.mat[k++] = (int8_t)(i == j ? o.a : -o.b); o.mat[k++] = -1; }
    for (int j = 0; j < 5; ++j) o.mat[k++] = -1;
    int qlen = rng() % 4 == 0 ? U(1, 320) : U(1, 150);
    const int mode = U(0, 10);
    o.w = mode == 9 ? U(1, 40) : 100;
    int tlen = U(0, qlen + 2 * o.w + 20);
    int h0 = mode == 8 ? U(1, 3) : U(1, 320);
    std::vector<uint8_t> q((size_t)qlen), t((size_t)(tlen > 0 ? tlen : 1));
    for (auto &c : q) c = (uint8_t)U(0, 3);
    int sub = U(0, 20), pos = 0;
    for (int i = 0; i < tlen; ++i) {
      if (pos < qlen && mode < 7) {
        const int r = U(0, 999);
        t[(size_t)i] = r < sub * 5 ? (uint8_t)U(0, 3) : q[(size_t)pos];
        if (r >= 990) ++pos;
        else if (r >= 985) { --i; ++pos; continue; }
        ++pos;
      } else {
        t[(size_t)i] = (uint8_t)U(0, 3);
      }
    }
    if (U(0, 10) == 0) q[(size_t)U(0, qlen - 1)] = 4;
    if (mode == 10) {
      // the diagonal comes back to exactly h0 every few rows (see lane_check.cpp)
      qlen = U(100, 320);
      q.resize((size_t)qlen);
      for (auto &c : q) c = (uint8_t)U(0, 3);
      tlen = qlen;
      t.assign(q.begin(), q.end());
      const int per = 2 * U(1, 4) + 1, ph = U(0, per - 1);
      for (int i = ph; i < tlen; i += per) t[(size_t)i] = (uint8_t)((q[(size_t)i] + 1 + U(0, 2)) & 3);
      h0 = U(30, 200);
    }
    const int end_bonus = 5, w = ext_band_w(o, qlen, end_bonus);
    if (!ext_group_opt_ok(o) || !ext_lane_ok(o, qlen, w, h0)) continue;
    int qle, tle;
    int64_t cells = 0, mine = 0;
    const int sc = orc_ksw_extend(qlen, q.data(), tlen, t.data(), o.mat, o.o_del, o.e_del, o.o_ins, o.e_ins, o.w, end_bonus,
                                  h0, &qle, &tle, &cells);
    for (int i = 0; i < tlen; ++i) mine += ext_row_cells(i, qlen, w);
    const ExtGroupOut g = o.o_del + o.e_del == o.o_ins + o.e_ins ? group<true>(fb, o, q, qlen, t, tlen, w, h0)
                                                                  : group<false>(fb, o, q, qlen, t, tlen, w, h0);
    ++tested;
    at_h0 += sc == h0;
    narrow += w < 30;
    lng += qlen > 134;
    handed += !g.exact;
    const bool same = g.exact ? g.score == sc && g.qle == qle && g.tle == tle : sc == h0;
    if (!same || mine != cells) {
      if (bad++ < 10)
        std::printf("MISMATCH it=%d qlen=%d tlen=%d w=%d h0=%d: oracle (%d,%d,%d) group (%d,%d,%d) exact %d cells %lld/%lld\n",
                    it, qlen, tlen, w, h0, sc, qle, tle, g.score, g.qle, g.tle, g.exact, (long long)mine, (long long)cells);
    }
  }
  std::printf("tested=%ld bad=%ld handed_back=%ld at_h0=%ld narrow=%ld long=%ld\n", tested, bad, handed, at_h0, narrow, lng);
  return bad != 0;
}
