// The copying threads of g3a_copy.h against plain copies, with a transfer that
// moves a slot's bytes only when it is awaited (as late as a DMA may), and one
// that fails part way; and a crew that finds no memory for its threads.
#include "g3sa_amd/csrc/g3a_copy.h"

#include <cstdio>
#include <cstdlib>
#include <new>

using namespace g3a;

static bool no_memory = false;
void *operator new(size_t n) {
  void *p = no_memory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

int main() {
  {
    CopyCrew none;  // it is asked from C entry points: nothing may be thrown
    no_memory = true;
    const bool ready = none.ready();
    no_memory = false;
    if (ready) return std::printf("FAIL ready without memory\n"), 1;
  }
  CopyCrew crew;
  if (!crew.ready()) return 2;
  const size_t chunk = 4096;
  std::vector<uint8_t> slots(CopyCrew::kSlots * chunk);
  auto slot = [&](size_t i) { return slots.data() + i % CopyCrew::kSlots * chunk; };
  int runs = 0;
  for (size_t bytes : {(size_t)1, chunk - 1, chunk, chunk + 1, 7 * chunk, 16 * chunk, 17 * chunk, 24 * chunk + 5, 25 * chunk,
                       100 * chunk + 77, 1000 * chunk + 1}) {
    for (int rep = 0; rep < 8; ++rep, ++runs) {
      std::vector<uint8_t> user(bytes), dev(bytes, 0xee), back(bytes, 0xdd);
      for (size_t i = 0; i < bytes; ++i) user[i] = (uint8_t)(rand() >> 4);
      size_t at_[CopyCrew::kSlots], m_[CopyCrew::kSlots], moved = 0, sent = 0;
      // transfers run in order: awaiting one moves all up to it
      auto move = [&](size_t i, bool in) {
        for (; moved <= i; ++moved) {
          const size_t k = moved % CopyCrew::kSlots;
          if (in) std::memcpy(dev.data() + at_[k], slot(moved), m_[k]);
          else std::memcpy(slot(moved), dev.data() + at_[k], m_[k]);
        }
      };
      auto issue = [&](size_t i, size_t at, size_t m) {
        at_[i % CopyCrew::kSlots] = at;
        m_[i % CopyCrew::kSlots] = m;
        sent = i + 1;
        return 0;
      };
      int rc = crew.in(user.data(), bytes, chunk, slot, issue, [&](size_t i) { move(i, true); return 0; });
      if (sent) move(sent - 1, true);
      if (rc || dev != user) return std::printf("FAIL in %zu\n", bytes), 1;
      moved = sent = 0;
      rc = crew.out(back.data(), bytes, chunk, slot, issue, [&](size_t i) { move(i, false); return 0; });
      if (rc || back != user) return std::printf("FAIL out %zu\n", bytes), 1;
      // an error ends the transfer with every helper away
      moved = sent = 0;
      const size_t bad = bytes / chunk / 2;
      rc = crew.out(back.data(), bytes, chunk, slot, issue, [&](size_t i) { move(i, false); return i == bad ? 5 : 0; });
      if (rc != 5) return std::printf("FAIL error %zu %d\n", bytes, rc), 1;
      moved = sent = 0;
      rc = crew.in(user.data(), bytes, chunk, slot, [&](size_t i, size_t at, size_t m) { return i == bad ? 6 : issue(i, at, m); },
                   [&](size_t i) { move(i, true); return 0; });
      if (rc != 6) return std::printf("FAIL error in %zu %d\n", bytes, rc), 1;
    }
  }
  std::printf("ok runs=%d\n", runs);
  return 0;
}
