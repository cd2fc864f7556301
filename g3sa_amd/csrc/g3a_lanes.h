// Cross-lane operations of the kernels that give a read or an alignment to a
// group of G lanes (16, 32 or 64) of a wavefront.  Their code takes the lanes
// as a type, so that a host test can run it on lanes of its own.
#pragma once
#include "g3a_dev.h"

#if defined(__HIPCC__)
#define G3A_LANE __device__ __forceinline__
#else
#define G3A_LANE inline
#endif

namespace g3a {

#if defined(__HIPCC__)
struct WaveLanes {
  static G3A_LANE uint64_t ballot(bool p) { return __ballot(p); }
  template <class T>
  static G3A_LANE T from(T v, int lane) { return __shfl(v, lane); }
  template <class T>
  static G3A_LANE T from_xor(T v, int d) { return __shfl_xor(v, d); }
  // v of lane l, the same l on every lane
  static G3A_LANE int get(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
  static G3A_LANE void lds_add(uint32_t *p, uint32_t v) { atomicAdd(p, v); }
  // v of the lane before (after) this one in the group, gl its place there;
  // the first (last) lane gets `edge`
  template <int G>
  static G3A_LANE int before(int v, int edge, int gl) {
    if (G == 16) return __builtin_amdgcn_update_dpp(edge, v, 0x111 /* row_shr:1 */, 0xf, 0xf, false);
    const int u = __builtin_amdgcn_update_dpp(edge, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
    return G == 64 ? u : gl == 0 ? edge : u;
  }
  template <int G>
  static G3A_LANE int after(int v, int edge, int gl) {
    if (G == 16) return __builtin_amdgcn_update_dpp(edge, v, 0x101 /* row_shl:1 */, 0xf, 0xf, false);
    const int u = __builtin_amdgcn_update_dpp(edge, v, 0x130 /* wave_shl:1 */, 0xf, 0xf, false);
    return G == 64 ? u : gl == G - 1 ? edge : u;
  }
  // maximum over the group's lanes up to this one; `least` is below every v
  template <int G>
  static G3A_LANE int max_scan(int v, int least, int) {
    int u;
    u = __builtin_amdgcn_update_dpp(least, v, 0x111 /* row_shr:1 */, 0xf, 0xf, false);
    v = u > v ? u : v;
    u = __builtin_amdgcn_update_dpp(least, v, 0x112, 0xf, 0xf, false);
    v = u > v ? u : v;
    u = __builtin_amdgcn_update_dpp(least, v, 0x114, 0xf, 0xf, false);
    v = u > v ? u : v;
    u = __builtin_amdgcn_update_dpp(least, v, 0x118, 0xf, 0xf, false);
    v = u > v ? u : v;
    if (G >= 32) {
      u = __builtin_amdgcn_update_dpp(least, v, 0x142 /* row_bcast:15 */, 0xa, 0xf, false);
      v = u > v ? u : v;
    }
    if (G >= 64) {
      u = __builtin_amdgcn_update_dpp(least, v, 0x143 /* row_bcast:31 */, 0xc, 0xf, false);
      v = u > v ? u : v;
    }
    return v;
  }
  // the wavefront's LDS stores are seen by its lanes
  static G3A_LANE void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // its global stores are seen by its lanes
  static G3A_LANE void global_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
};
#endif

}  // namespace g3a
