// The wavefront region filter of g3a_region.h on the host, its lanes as
// fibers, against region_filter (g3a_dev.h), field by field.
//   region_group_check READS SEED
#include "g3sa_amd/csrc/g3a_region.h"
#include "tests/fibers.h"

#include <cstring>
#include <memory>
#include <random>

using namespace g3a;

template <class ST>
static int group(Fibers &fb, const Opt &o, std::vector<Region> &a) {
  std::unique_ptr<ST> st(new ST);
  std::memset((void *)st.get(), 0xa5, sizeof(ST));
  int n[64];
  fb.run(64, [&](int lane) {
    RegionGroup<HostLanes, ST> g{o, st.get(), lane};
    n[lane] = g.run(a.data(), (int)a.size());
  });
  return n[0];
}

int main(int argc, char **argv) {
  const int reads = argc > 1 ? std::atoi(argv[1]) : 100;
  std::mt19937_64 rng(argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1);
  auto U = [&](int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); };
  Fibers fb;
  long kept = 0, sec = 0;
  for (int it = 0; it < reads; ++it) {
    Opt o;
    std::memset(&o, 0, sizeof o);
    o.T = it % 3 ? 30 : 0;
    o.mask_level = 0.5f; o.drop_ratio = it % 5 == 4 ? 0.9f : 0.5f; o.mask_level_redun = 0.95f;
    o.flag = it % 2 ? 0x8 : 0;
    const int n = it % 4 == 0 ? (int)U(1, 70) : it % 4 < 3 ? (int)U(60, 512) : (int)U(500, 2000);
    const int places = (int)U(1, it % 3 == 1 ? 8 : 600), l_seq = (int)U(40, 320);
    std::vector<Region> a((size_t)n);
    for (auto &g : a) {
      const int64_t p = 10000 + 1000 * U(0, places);
      g.qb = (int32_t)U(0, l_seq - 30);
      g.qe = (int32_t)U(g.qb + 19, l_seq);
      if (rng() % 3) { g.qb = 0; g.qe = l_seq; }
      g.rb = p + g.qb + U(-2, 2) * (rng() % 5 == 0);
      g.re = g.rb + (g.qe - g.qb) + U(-2, 2) * (rng() % 5 == 0);
      g.score = (int32_t)U(10, g.qe - g.qb);
      if (rng() % 2) g.score = g.qe - g.qb;
      g.rid = (int32_t)(p / 200000);
      g.seedlen0 = (int32_t)U(19, 320);
      g.secondary = 0;
    }
    std::vector<Region> ref = a;
    std::vector<uint8_t> flag((size_t)n);
    std::vector<int32_t> s((size_t)n);
    const int m = region_filter(o, ref.data(), n, flag.data(), s.data());
    for (int form = 0; form < 2; ++form) {
      if (form == 0 && n > 512) continue;
      std::vector<Region> b = a;
      const int k = form == 0 ? group<RegionStage<512>>(fb, o, b) : group<RegionStage<2048>>(fb, o, b);
      bool same = k == m;
      for (int i = 0; same && i < m; ++i)
        same = b[i].rb == ref[i].rb && b[i].re == ref[i].re && b[i].qb == ref[i].qb && b[i].qe == ref[i].qe &&
               b[i].score == ref[i].score && b[i].rid == ref[i].rid && b[i].seedlen0 == ref[i].seedlen0 &&
               b[i].secondary == ref[i].secondary;
      if (!same) {
        std::printf("FAIL read %d form %d: %d regions, kept %d/%d\n", it, form, n, k, m);
        return 1;
      }
    }
    kept += m;
    for (int i = 0; i < m; ++i) sec += ref[i].secondary >= 0;
  }
  std::printf("ok reads=%d kept=%ld secondary=%ld\n", reads, kept, sec);
  return 0;
}
