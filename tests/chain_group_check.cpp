// The wavefront chaining of g3a_chain.h on the host, its lanes as fibers: the
// tasks of random reads must equal those of the one-thread code (sort_seeds,
// chain_build, chain_filter, chain_window of g3a_dev.h).
//   chain_group_check READS SEED
// Seed lists of 1 to 6000 with repeated positions, several contigs and both
// strands; the stages of the two size classes, and one whose nodes and
// records do not fit the LDS.  Prints "ok key=value ..." or the first failure.
#include "g3sa_amd/csrc/g3a_chain.h"
#include "tests/fibers.h"

#include <cstring>
#include <memory>
#include <random>

using namespace g3a;

template <class ST>
static int group(Fibers &fb, const DevIndex &x, const Opt &o, const std::vector<Seed> &s, int l_seq, std::vector<Task> &out) {
  const int ns = (int)s.size();
  std::unique_ptr<ST> st(new ST);
  std::memset((void *)st.get(), 0xa5, sizeof(ST));
  std::vector<uint32_t> ra((size_t)ns * 6, 0xcdcdcdcd), rb((size_t)ns * 4, 0xcdcdcdcd);
  std::vector<int32_t> of((size_t)ns, 77), order((size_t)ns, 77), tmp((size_t)ns * 2, 77);
  std::vector<uint8_t> kept((size_t)ns, 9);
  std::vector<ChainNode> nodes((size_t)(ns + 32) / 4);
  out.resize((size_t)ns + 1);
  int n[64];
  fb.run(64, [&](int lane) {
    ChainGroup<HostLanes, ST> g{x, o, st.get(), ChainMem{ra.data(), rb.data(), of.data(), order.data(), tmp.data(), kept.data(), nodes.data(), (int)nodes.size()}};
    g.s = s.data();
    g.ns = ns;
    g.l_seq = l_seq;
    g.read = 7;
    g.lane = lane;
    n[lane] = g.run(out.data());
  });
  for (int l = 1; l < 64; ++l)
    if (n[l] != n[0]) {
      std::printf("FAIL lanes disagree\n");
      std::exit(1);
    }
  return n[0];
}

int main(int argc, char **argv) {
  const int reads = argc > 1 ? std::atoi(argv[1]) : 100;
  std::mt19937_64 rng(argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1);
  auto U = [&](int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); };
  DevIndex x;
  std::memset(&x, 0, sizeof x);
  const int64_t l_pac = 300000;
  const int64_t off[3] = {0, 100000, 220000}, len[3] = {100000, 120000, 80000};
  x.l_pac = l_pac;
  x.n = 2 * l_pac;
  x.n_contigs = 3;
  x.ctg_off = off;
  x.ctg_len = len;
  Fibers fb;
  long n_tasks = 0, big = 0;
  for (int it = 0; it < reads; ++it) {
    Opt o;
    std::memset(&o, 0, sizeof o);
    o.a = 1; o.b = 4; o.o_del = o.o_ins = 6; o.e_del = o.e_ins = 1; o.w = it % 3 ? 100 : 10; o.min_seed_len = 19;
    o.max_chain_gap = it % 4 == 3 ? 50 : 10000; o.mask_level = 0.5f; o.drop_ratio = 0.5f;
    const int l_seq = (int)U(36, 320);
    const int ns = it % 5 == 0 ? (int)U(1, 130) : it % 5 < 3 ? (int)U(120, 512) : it % 5 == 3 ? (int)U(500, 2500) : (int)U(2000, 6000);
    std::vector<Seed> s((size_t)ns);
    std::vector<int64_t> places;
    const int np = (int)U(1, it % 2 ? 400 : 20);
    for (int k = 0; k < np; ++k) places.push_back(U(0, 2 * l_pac - 400));
    for (auto &v : s) {
      v.len = (int32_t)U(10, l_seq < 60 ? l_seq : 60);
      if (rng() % 9 == 0) v.len = (int32_t)U(10, l_seq);
      v.qbeg = (int32_t)U(0, l_seq - v.len);
      const int64_t p = places[rng() % places.size()];
      const int kind = (int)(rng() % 8);
      v.rbeg = kind < 4 ? p + v.qbeg : kind < 6 ? p + v.qbeg + U(-5, 5) : kind == 6 ? p : U(0, 2 * l_pac - 400);
      if (v.rbeg < 0) v.rbeg = 0;
      v.rid = (int32_t)intv2rid(x, v.rbeg, v.rbeg + v.len);
      v.pad = 0;
    }
    if (it % 6 == 5)  // repeats of one unit: many seeds at the same few positions
      for (auto &v : s) v.rbeg = 5000 + 3 * (int64_t)(rng() % 40), v.rid = 0;
    // the one-thread code
    std::vector<Seed> sorted = s, tmp((size_t)ns);
    sort_seeds(sorted.data(), ns, tmp.data());
    std::vector<ChainTmp> ch((size_t)ns);
    std::vector<int32_t> nxt((size_t)ns), order((size_t)ns), tmpi((size_t)ns * 2);
    std::vector<KbNode> nodes((size_t)(ns + 32) / 4);
    std::vector<uint16_t> w16((size_t)ns);
    std::vector<uint8_t> kept((size_t)ns);
    const int nch = chain_build(x, o, sorted.data(), ns, ch.data(), nxt.data(), nodes.data(), (int)nodes.size(), order.data());
    const int nk = chain_filter(o, sorted.data(), nxt.data(), ch.data(), order.data(), nch, w16.data(), tmpi.data(), kept.data());
    std::vector<Task> want;
    for (int c = 0; c < nk; ++c) {
      const ChainTmp &cc = ch[(size_t)order[(size_t)c]];
      int64_t r0, r1;
      int rid;
      chain_window(x, o, sorted.data(), nxt.data(), cc, l_seq, r0, r1, rid);
      for (int j = cc.head; j >= 0; j = nxt[(size_t)j])
        want.push_back(Task{sorted[(size_t)j].rbeg, r0, r1, sorted[(size_t)j].qbeg, sorted[(size_t)j].len, 7, rid});
    }
    for (int form = 0; form < 3; ++form) {
      if (form == 0 && ns > 512) continue;
      std::vector<Task> got;
      const int n = form == 0   ? group<ChainStageL<512, 108, 128, 512>>(fb, x, o, s, l_seq, got)
                    : form == 1 ? group<ChainStageL<2048, 290, 400, 4096>>(fb, x, o, s, l_seq, got)
                                : group<ChainStageL<2048, 3, 2, 4096>>(fb, x, o, s, l_seq, got);
      bool same = n == (int)want.size();
      for (size_t k = 0; same && k < want.size(); ++k)
        same = got[k].rbeg == want[k].rbeg && got[k].rmax0 == want[k].rmax0 && got[k].rmax1 == want[k].rmax1 &&
               got[k].qbeg == want[k].qbeg && got[k].len == want[k].len && got[k].rid == want[k].rid && got[k].read == 7;
      if (!same) {
        std::printf("FAIL read %d form %d: %d seeds, %d chains, tasks %d/%zu\n", it, form, ns, nch, n, want.size());
        return 1;
      }
    }
    n_tasks += (long)want.size();
    big += ns > 2048;
  }
  std::printf("ok reads=%d tasks=%ld big=%ld\n", reads, n_tasks, big);
  return 0;
}
