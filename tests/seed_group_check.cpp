// The group seeding of g3a_seed.h on the host: its lanes run as fibers that
// meet at each cross-lane operation, and its intervals (k, s, m, n) of every
// read must equal those of the one-thread code (smem_round1, reseed_one,
// reseed_round3 of g3a_seed_rounds.h).
//   seed_group_check PREFIX READS [MIN_SEED_LEN]
// Groups of 16 lanes with 64 entries (the fast path, which may give a read
// up) and of 64 lanes with 320 (which may not), in the narrow and the wide
// layout and with the full suffix array.  Prints "ok key=value ..." or the
// first failure; given_up_* and compared_* are the reads given up and the
// intervals compared of the 16-lane groups, by form.
#include "g3sa_amd/csrc/g3a_dev.h"
#include "g3sa_amd/csrc/g3a_index.h"
#include "g3sa_amd/csrc/g3a_layout.h"
#include "g3sa_amd/csrc/g3a_seed.h"
#include "tests/fibers.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <thread>
#include <vector>

using namespace g3a;

static int fail(const char *what, long long a, long long b, long long c) {
  std::printf("FAIL %s %lld %lld %lld\n", what, a, b, c);
  return 1;
}

template <int G, int NS, class P, bool L = false>
static bool group_read(Fibers &fb, const DevIndex &x, const Opt &o, const std::vector<uint8_t> &buf, int off, int len,
                       int cap, std::vector<Intv> &out, int64_t &n_seed, int64_t &steps) {
  PackedRead pk;
  std::memset(&pk, 0xa5, sizeof pk);
  const int fcap = G == 64 ? kMaxReadLen : 16;
  std::vector<P> fk((size_t)fcap), fs((size_t)fcap);
  std::vector<uint32_t> fmn((size_t)fcap);
  std::vector<Intv> slot((size_t)cap);
  bool ok[64];
  int n[64];
  int64_t ns[64], st[64];
  int64_t lc[64][6];
  fb.run(G, [&](int lane) {
    SeedGroup<HostLanes, G, NS, P, L> g{x, o, &pk, FoundList<P>{fk.data(), fs.data(), fmn.data(), fcap}, lane, 0};
    g.slot = slot.data();
    g.cap = cap;
    g.steps = 0;
    g.lc = lc[lane];
    for (int k = 0; k < NS; ++k) {
      g.ek[k] = (P)0xdeadbeef;
      g.es[k] = 7;
      g.en[k] = -1000;
    }
    g.load(buf.data() + off, len);
    ok[lane] = g.run();
    n[lane] = g.n;
    ns[lane] = g.n_seed;
    st[lane] = g.steps;
  });
  for (int l = 1; l < G; ++l)
    if (ok[l] != ok[0] || n[l] != n[0] || ns[l] != ns[0]) {
      std::printf("FAIL lanes disagree\n");
      std::exit(1);
    }
  for (int l = 0; l < G; ++l) steps += st[l];
  n_seed = ns[0];
  if (!ok[0] || n[0] > cap) return false;
  out.assign(slot.begin(), slot.begin() + n[0]);
  return true;
}

int main(int argc, char **argv) {
  if (argc < 3) return 2;
  const int n_reads = std::atoi(argv[2]);
  HostIndex h;
  std::string err;
  if (!load_index(argv[1], h, err)) {
    std::printf("load failed: %s\n", err.c_str());
    return 1;
  }
  unpack_bwt(h);
  h.pac.resize(h.pac.size() + 32, 0);
  DevIndex x;
  std::memset(&x, 0, sizeof x);
  std::vector<uint32_t> wide, narrow, sb;
  if (!build_occ_lines(h, wide, x.super) || !build_occ_narrow(h, narrow, sb)) {
    std::printf("layout failed\n");
    return 1;
  }
  x.occ = wide.data();
  x.occn = narrow.data();
  x.sbc = sb.data();
  x.primary = (int64_t)h.primary;
  x.n = (int64_t)h.seq_len;
  x.l_pac = h.l_pac;
  x.pac = h.pac.data();
  build_counts(h, x.count);
  if (h.sa_width == 4) x.sa32 = (const uint32_t *)h.sa.data();
  else x.sa64 = (const uint64_t *)h.sa.data();
  x.sa_shift = log2_exact(h.sa_intv);
  const int64_t n = x.n;
  std::vector<uint32_t> table((size_t)3 << (2 * kKmer));
  std::vector<int64_t> table64((size_t)3 << (2 * kKmer));
  {
    std::vector<std::thread> th;
    for (uint32_t t = 0; t < 8; ++t)
      th.emplace_back([&, t] {
        for (uint32_t c = t; c < (1u << (2 * kKmer)); c += 8) kmer_interval(x, c, &table64[3 * (size_t)c]);
      });
    for (auto &t : th) t.join();
  }
  for (size_t i = 0; i < table.size(); ++i) table[i] = (uint32_t)table64[i];
  x.kmer = table.data();
  DevIndex xw = x;  // the wide layout
  xw.occn = nullptr;
  xw.sbc = nullptr;
  xw.kmer = nullptr;
  xw.kmer64 = table64.data();
  std::vector<uint32_t> saf((size_t)n + 1);
  {
    std::vector<std::thread> th;
    for (int64_t t = 0; t < 8; ++t)
      th.emplace_back([&, t] {
        for (int64_t r = t; r <= n; r += 8) saf[(size_t)r] = (uint32_t)sa_value_n(x, (uint32_t)r);
      });
    for (auto &t : th) t.join();
  }
  DevIndex xl = x;  // the learned form's text comparison
  xl.saf = saf.data();
  Opt o;
  std::memset(&o, 0, sizeof o);
  o.a = 1; o.b = 4; o.o_del = o.o_ins = 6; o.e_del = o.e_ins = 1; o.w = 100; o.T = 30;
  o.pen_clip5 = o.pen_clip3 = 5; o.min_seed_len = argc > 3 ? std::atoi(argv[3]) : 19; o.split_width = 10;
  o.max_occ = 500; o.max_chain_gap = 10000; o.max_mem_intv = 20; o.split_factor = 1.5f; o.mask_level = 0.5f;
  o.drop_ratio = 0.5f; o.mask_level_redun = 0.95f;

  std::mt19937_64 rng(99);
  Fibers fb;
  int64_t n_iv = 0, given_up[3] = {0, 0, 0}, compared[3] = {0, 0, 0}, st1 = 0, st16 = 0, st64 = 0, stw = 0, stl = 0;
  for (int i = 0; i < n_reads; ++i) {
    // all lengths up to the limit, short ones and the limit more often
    int len = i % 7 == 0 ? (int)(rng() % 45) : i % 7 == 1 ? kMaxReadLen - (int)(rng() % 3) : 36 + (int)(rng() % 285);
    const int off = (int)(rng() % 4);  // reads start at any byte
    std::vector<uint8_t> buf((size_t)off + (size_t)len + 64, 3);
    uint8_t *q = buf.data() + off;
    if (i % 11 == 10 || len >= n) {
      for (int t = 0; t < len; ++t) q[t] = (uint8_t)(rng() % 4);
    } else {
      const int64_t p = (int64_t)(rng() % (uint64_t)(n - len));
      const bool two = i % 5 == 4;  // a read across two places
      const int64_t p2 = (int64_t)(rng() % (uint64_t)(n - len));
      for (int t = 0; t < len; ++t) q[t] = (uint8_t)text_base(x, (two && t > len / 2 ? p2 : p) + t);
      const int err_pm = i % 3 == 0 ? 0 : (i % 3 == 1 ? 10 : 50);  // per mille
      for (int t = 0; t < len; ++t) {
        if ((int)(rng() % 1000) < err_pm) q[t] = (uint8_t)((q[t] + 1 + rng() % 3) & 3);
        if (i % 2 && rng() % 200 == 0) q[t] = 4;
      }
    }
    if (i % 29 == 28)
      for (int t = 0; t < len; ++t) q[t] = (uint8_t)(t % (1 + i % 3));  // repeats of one to three bases
    // the one-thread code
    std::vector<Intv> slot(4096), ref;
    std::vector<LepNarrow> la(400), lf(400);
    IntvSink sink{slot.data(), 4096, 0, 0, o.max_occ};
    GlobalBuf<LepNarrow> lb{GlobalList<LepNarrow>{la.data()}, GlobalList<LepNarrow>{lf.data()}, 400, 400};
    if (!smem_round1(x, o, q, len, sink, lb, &st1)) return fail("one-thread overflow", i, len, 0);
    const int nsm = sink.n;
    for (int k = 0; k < nsm; ++k)
      if (!reseed_one(x, o, q, len, slot[(size_t)k], GlobalList<LepNarrow>{la.data()},
                      GlobalList<LepNarrow>{lf.data()}, 400, 400, sink, &st1))
        return fail("one-thread reseed overflow", i, len, 0);
    reseed_round3<uint32_t>(x, o, q, len, sink, &st1);
    ref.assign(slot.begin(), slot.begin() + sink.n);
    n_iv += sink.n;
    for (int form = 0; form < 6; ++form) {
      std::vector<Intv> got;
      int64_t ns = 0;
      bool ok = form == 0   ? group_read<16, 4, uint32_t>(fb, x, o, buf, off, len, 64, got, ns, st16)
                : form == 1 ? group_read<64, 5, uint32_t>(fb, x, o, buf, off, len, 4096, got, ns, st64)
                : form == 2 ? group_read<16, 4, int64_t>(fb, xw, o, buf, off, len, 64, got, ns, stw)
                : form == 3 ? group_read<64, 5, int64_t>(fb, xw, o, buf, off, len, 4096, got, ns, stw)
                : form == 4 ? group_read<16, 4, uint32_t, true>(fb, xl, o, buf, off, len, 64, got, ns, stl)
                            : group_read<64, 5, uint32_t, true>(fb, xl, o, buf, off, len, 4096, got, ns, stl);
      if (!ok) {
        if (form & 1) return fail("wavefront group gave up", i, len, form);
        ++given_up[form / 2];
        continue;
      }
      if (got.size() != ref.size()) return fail("intervals", i, form, (long long)got.size() - (long long)ref.size());
      if (ns != sink.n_seed) return fail("n_seed", i, form, ns - sink.n_seed);
      for (size_t k = 0; k < ref.size(); ++k) {
        const Intv &u = ref[k], &v = got[k];
        if (u.k != v.k || u.s != v.s || u.m != v.m || u.n != v.n) return fail("interval", i, form, (long long)k);
      }
      if (!(form & 1)) compared[form / 2] += (int64_t)ref.size();
    }
  }
  std::printf("ok reads=%d intervals=%lld", n_reads, (long long)n_iv);
  const char *name[3] = {"narrow", "wide", "text"};
  for (int f = 0; f < 3; ++f)
    std::printf(" given_up_%s=%lld compared_%s=%lld", name[f], (long long)given_up[f], name[f], (long long)compared[f]);
  std::printf(" steps_thread=%lld steps_16=%lld steps_64=%lld steps_wide=%lld steps_text=%lld\n", (long long)st1,
              (long long)st16, (long long)st64, (long long)stw, (long long)stl);
  return 0;
}
