// The lanes of a group as fibers, for host checks of code that is written for
// the lanes of a wavefront.
#pragma once
#include <ucontext.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <vector>

// G fibers, resumed in lane order between cross-lane operations
struct Fibers {
  static constexpr size_t kStack = 256 << 10;
  int n = 0, cur = 0;
  ucontext_t main_ctx, ctx[64];
  std::vector<std::vector<char>> stack = std::vector<std::vector<char>>(64, std::vector<char>(kStack));
  bool done[64];
  int64_t box[2][64];
  bool in[2][64];
  int phase[64];
  std::function<void(int)> body;
  static Fibers *self;
  static void entry(int lane) {
    self->body(lane);
    self->done[lane] = true;
    swapcontext(&self->ctx[lane], &self->main_ctx);
  }
  // every live lane leaves a value; returns when all have
  const int64_t *meet(int64_t v) {
    const int l = cur, p = phase[l]++ & 1;
    box[p][l] = v;
    in[p][l] = true;
    swapcontext(&ctx[l], &main_ctx);
    return box[p];
  }
  void run(int lanes, std::function<void(int)> f) {
    self = this;
    n = lanes;
    body = std::move(f);
    for (int l = 0; l < n; ++l) {
      done[l] = false;
      phase[l] = 0;
      getcontext(&ctx[l]);
      ctx[l].uc_stack.ss_sp = stack[(size_t)l].data();
      ctx[l].uc_stack.ss_size = kStack;
      ctx[l].uc_link = nullptr;
      makecontext(&ctx[l], (void (*)())entry, 1, l);
    }
    for (;;) {
      int live = 0;
      for (cur = 0; cur < n; ++cur)
        if (!done[cur]) {
          swapcontext(&main_ctx, &ctx[cur]);
          live += !done[cur];
        }
      if (!live) return;
      if (live != n) {
        std::printf("FAIL lanes parted\n");
        std::exit(1);
      }
      for (int l = 1; l < n; ++l)
        if (phase[l] != phase[0]) {
          std::printf("FAIL lanes out of step\n");
          std::exit(1);
        }
    }
  }
};
Fibers *Fibers::self = nullptr;

struct HostLanes {
  static uint64_t ballot(bool p) {
    const int64_t *b = Fibers::self->meet(p);
    uint64_t m = 0;
    for (int l = 0; l < Fibers::self->n; ++l) m |= (uint64_t)(b[l] != 0) << l;
    return m;
  }
  template <class T>
  static T from(T v, int lane) {
    return (T)Fibers::self->meet((int64_t)v)[lane];
  }
  template <class T>
  static T from_xor(T v, int d) {
    const int l = Fibers::self->cur;
    return (T)Fibers::self->meet((int64_t)v)[l ^ d];
  }
  static int get(int v, int l) { return (int)Fibers::self->meet(v)[l]; }
  static void lds_add(uint32_t *p, uint32_t v) { *p += v; }
  template <int G>
  static int before(int v, int edge, int gl) {
    const int64_t *b = Fibers::self->meet(v);
    return gl ? (int)b[gl - 1] : edge;
  }
  template <int G>
  static int after(int v, int edge, int gl) {
    const int64_t *b = Fibers::self->meet(v);
    return gl < G - 1 ? (int)b[gl + 1] : edge;
  }
  template <int G>
  static int max_scan(int v, int, int gl) {
    const int64_t *b = Fibers::self->meet(v);
    for (int l = 0; l < gl; ++l) v = b[l] > v ? (int)b[l] : v;
    return v;
  }
  static void lds_sync() { Fibers::self->meet(0); }
  static void global_sync() { Fibers::self->meet(0); }
};
