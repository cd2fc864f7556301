// The group alignment of g3a_trace.h on the host, its lanes as fibers: score,
// CIGAR and mismatch count of random banded alignments must equal those of
// the one-thread code (trace_and_finalize of g3a_dev.h).
//   trace_group_check CASES SEED
// Prints "ok key=value ..." or the first failure.
#include "g3sa_amd/csrc/g3a_trace.h"
#include "tests/fibers.h"

#include <cstring>
#include <random>

using namespace g3a;

template <int G, int NH>
static void group(Fibers &fb, const DevIndex &x, const Opt &o, const uint8_t *query, int64_t rb, int qlen, int tlen, int w,
                  std::vector<uint32_t> &cig, int &nw, int &nm) {
  GapStage st;
  std::memset(&st, 0xa5, sizeof st);
  std::vector<uint32_t> z((size_t)gap_words(qlen, tlen, w) + 1, 0xcdcdcdcd);
  std::vector<uint32_t> core((size_t)(qlen + tlen) + 1, 0xcdcdcdcd);
  int score[64], mm[64], n[64];
  fb.run(G, [&](int lane) {
    GapGroup<HostLanes, G, NH> g{x, o, &st, z.data(), lane, 0};
    g.qlen = qlen;
    g.tlen = tlen;
    g.w = w;
    g.load(query, rb);
    score[lane] = g.dp();
    n[lane] = g.walk(core.data(), mm[lane]);
  });
  for (int l = 1; l < G; ++l)
    if (score[l] != score[0] || mm[l] != mm[0] || n[l] != n[0]) {
      std::printf("FAIL lanes disagree\n");
      std::exit(1);
    }
  if (z.back() != 0xcdcdcdcd || core.back() != 0xcdcdcdcd) {
    std::printf("FAIL out of bounds\n");
    std::exit(1);
  }
  nw = score[0];
  nm = mm[0];
  cig.assign(core.begin(), core.begin() + n[0]);
}

int main(int argc, char **argv) {
  const int cases = argc > 1 ? std::atoi(argv[1]) : 1000;
  std::mt19937_64 rng(argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1);
  const int64_t l_pac = 5000;
  std::vector<uint8_t> pac(l_pac / 4 + 32, 0);
  for (int64_t i = 0; i < l_pac / 4; ++i) pac[(size_t)i] = (uint8_t)rng();
  DevIndex x;
  std::memset(&x, 0, sizeof x);
  x.n = 2 * l_pac;
  x.l_pac = l_pac;
  x.pac = pac.data();
  x.n_contigs = 1;
  const int64_t c_off = 0, c_len = l_pac;
  x.ctg_off = &c_off;
  x.ctg_len = &c_len;
  Fibers fb;
  int by[5] = {0, 0, 0, 0, 0}, gapped = 0;
  for (int it = 0; it < cases; ++it) {
    Opt o;
    std::memset(&o, 0, sizeof o);
    o.a = 1; o.b = 4; o.o_del = o.o_ins = 6; o.e_del = o.e_ins = 1; o.w = 100;
    if (it % 4 == 1) { o.a = 2; o.b = 3; o.o_del = 5; o.o_ins = 3; o.e_del = 2; o.e_ins = 1; }
    if (it % 4 == 2) { o.o_del = 0; o.o_ins = 1; o.e_del = 1; o.e_ins = 1; o.b = 1; }
    for (int t = 0; t < 5; ++t)
      for (int q = 0; q < 5; ++q) o.mat[5 * t + q] = (int8_t)(t == 4 || q == 4 ? -1 : t == q ? o.a : -o.b);
    int qlen = it % 9 == 0 ? 1 + (int)(rng() % 40) : it % 9 == 1 ? kMaxReadLen - (int)(rng() % 2) : 20 + (int)(rng() % 200);
    const int64_t rb = it % 5 == 4 ? l_pac + (int64_t)(rng() % (l_pac - 500)) : (int64_t)(rng() % (l_pac - 500));
    // a read with substitutions, N and indels of the text at rb
    std::vector<uint8_t> q;
    int64_t p = rb;
    const int kind = it % 7;
    while ((int)q.size() < qlen) {
      const int b = text_base(x, p++);
      const int u = (int)(rng() % 1000);
      if (u < 20) q.push_back((uint8_t)(rng() % 5));
      else if (u < 30 && kind) { p += 1 + (int)(rng() % (kind * 4)); q.push_back((uint8_t)b); }
      else if (u < 40 && kind) { for (int k = 1 + (int)(rng() % (kind * 4)); k > 0 && (int)q.size() < qlen; --k) q.push_back((uint8_t)(rng() % 4)); }
      else q.push_back((uint8_t)b);
    }
    int tlen = (int)(p - rb);
    if (it % 6 == 5) tlen = tlen + (int)(rng() % 9) - 4;
    if (tlen < 1) tlen = 1;
    if (tlen > qlen + 60) tlen = qlen + 60;
    if (tlen == qlen) ++tlen;
    q.resize((size_t)qlen + 40, 0);
    {
      // the ungapped pass, 32 bases at a time, against one base at a time
      Region g;
      std::memset(&g, 0, sizeof g);
      g.qe = qlen; g.rb = rb; g.re = rb + qlen; g.secondary = -1; g.score = qlen;
      std::vector<uint8_t> qq(q.begin(), q.begin() + qlen);
      qq.resize((size_t)qlen + 40, 0);
      if (it % 3 == 0) o.mat[4] = o.mat[9] = o.mat[14] = o.mat[19] = -3;
      if (it % 8 == 7) o.mat[7] = 2;  // no three-score matrix
      uint32_t cig[16];
      Aln a;
      trace_and_finalize(x, o, qq.data(), qlen, g, 0, EhArray{nullptr, nullptr}, nullptr, cig, 0, a);
      int nw = 0, nm = 0;
      for (int i = 0; i < qlen; ++i) {
        const int t = text_base(x, rb + i);
        nw += o.mat[5 * t + qq[(size_t)i]];
        nm += t != qq[(size_t)i];
      }
      if (a.nw_score != nw || a.nm != nm || a.n_core != 1) {
        std::printf("FAIL ungapped %d: %d/%d %d/%d\n", it, a.nw_score, nw, a.nm, nm);
        return 1;
      }
      if (it % 8 == 7) o.mat[7] = (int8_t)-o.b;
    }
    // a band that the score's rule could give, or any above the lengths' difference
    Region g;
    std::memset(&g, 0, sizeof g);
    g.qb = 0; g.qe = qlen; g.rb = rb; g.re = rb + tlen; g.secondary = -1;
    g.score = (int)(rng() % (qlen + 1));
    const int w = global_bw(o, qlen, tlen, g.score);
    if (w == 0 || w > kGapW) { ++by[4]; continue; }
    if (tlen > kMaxReadLen + w - 3) continue;
    std::vector<int32_t> eh((size_t)2 * (qlen + 2));
    std::vector<uint8_t> z((size_t)aln_z_size(qlen, tlen, w) + 16);
    std::vector<uint32_t> cig((size_t)aln_cigar_cap(qlen, tlen, w) + 8);
    Aln a;
    trace_and_finalize(x, o, q.data(), qlen, g, 0, EhArray{eh.data(), eh.data() + qlen + 2}, z.data(), cig.data(), 0, a);
    for (int form = 0; form < 4; ++form) {
      if ((form == 0 && w > 7) || (form == 1 && w > 15) || (form == 2 && w > 31)) continue;
      std::vector<uint32_t> got;
      int nw = 0, nm = 0;
      if (form == 0) group<16, 1>(fb, x, o, q.data(), rb, qlen, tlen, w, got, nw, nm);
      else if (form == 1) group<32, 1>(fb, x, o, q.data(), rb, qlen, tlen, w, got, nw, nm);
      else if (form == 2) group<64, 1>(fb, x, o, q.data(), rb, qlen, tlen, w, got, nw, nm);
      else group<64, 2>(fb, x, o, q.data(), rb, qlen, tlen, w, got, nw, nm);
      ++by[form];
      bool same = nw == a.nw_score && nm == a.nm && (int)got.size() == a.n_core;
      for (int k = 0; same && k < a.n_core; ++k) same = got[(size_t)k] == cig[(size_t)(a.core_off + k)];
      if (!same) {
        std::printf("FAIL case %d form %d q %d t %d w %d: score %d/%d nm %d/%d ops %zu/%d\n", it, form, qlen, tlen, w, nw,
                    a.nw_score, nm, a.nm, got.size(), a.n_core);
        return 1;
      }
      gapped += a.n_core > 1;
    }
  }
  std::printf("ok by16=%d by32=%d by64=%d by128=%d wide=%d gapped=%d\n", by[0], by[1], by[2], by[3], by[4], gapped);
  return 0;
}
