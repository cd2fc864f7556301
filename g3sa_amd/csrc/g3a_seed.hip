// Seeding kernels for MI355X (gfx950, wave64):
//   k_seed       16 lanes per read: SMEM + reseed + third-round intervals
//   k_seed_slow  wavefront per read, for reads whose lists outgrew the fast
//                path's
// The search itself is in g3a_seed.h.
#include "g3a_kernels.h"
#include "g3a_seed.h"

#include <hip/hip_runtime.h>

namespace g3a {

// What bounds it once the chip is full of searches is integer VALU issue (19
// instructions a step, 89% of the cycles), with loads pending on the L1 behind
// it most of the time (two 16-byte Occ lines a step at random places, 0.59 of
// them from memory at 1 Gbp: 2.1 TB/s); in a small batch the chain of steps of
// one read.  Before, a thread per read; now, at 16 lanes a read (150 bp, 1%
// substitutions, 100 Mbp): 250,000 reads 4.6 -> 3.0 ms, 200 reads 2.96 -> 0.20
// ms; in the wide layout 10.5 -> 3.6 ms; on 1 Gbp 1,000,000 reads 27.5 -> 16.0
// ms, 10,000,000 190 -> 143 ms.  The learned form takes 14% fewer steps but is
// no faster (10,000,000 reads 176 -> 152 ms): a model lookup is a chain of
// dependent loads that one lane of a group waits for.
// Persistent grid: each group of kSeedLanes lanes takes the next read from a
// device counter (one atomic per wavefront and turn), so that a group held up
// by a long read takes fewer.  The superblock counts (narrow: 16 B per 2^21
// rows, at most 32 KB; wide: 128 B) are copied to LDS, so a narrow Occ lookup
// costs one 16-byte global load; after them come the groups' packed reads and
// found lists.
constexpr int kSeedLanes = 16, kSeedSlots = kLepCap / kSeedLanes;
// 16-byte pieces of the superblock counts
template <class P>
__host__ __device__ __forceinline__ int seed_super_lines(const DevIndex &x) {
  return sizeof(P) == 4 ? (int)(((uint64_t)x.n + 1) >> 21) + 1 : 8;
}
// L: the learned-index form (text comparison at the full SA's positions, the
// model's intervals in the last round); a separate kernel, so that the
// FM-only one keeps its registers
template <class P, bool L>
__global__ void __launch_bounds__(1024) k_seed(SeedArgs a) {
  extern __shared__ uint4 sb_lds[];
  const int n_sb = seed_super_lines<P>(a.idx);
  {
    const uint4 *src = sizeof(P) == 4 ? (const uint4 *)a.idx.sbc : (const uint4 *)a.idx.super_dev;
    for (int k = threadIdx.x; k < n_sb; k += blockDim.x) sb_lds[k] = src[k];
    __syncthreads();
    if (sizeof(P) == 4) a.idx.sbc = (const uint32_t *)sb_lds;
    else a.idx.super_dev = (const int64_t *)sb_lds;
  }
  const int lane = threadIdx.x & 63, gl = lane % kSeedLanes, gb = lane - gl;
  uint8_t *mine =
      (uint8_t *)(sb_lds + n_sb) + (threadIdx.x / kSeedLanes) * seed_group_bytes<P>(kFoundCap);
  P *fk = (P *)(mine + sizeof(PackedRead)), *fs = fk + kFoundCap;
  int64_t lc[6] = {0, 0, 0, 0, 0, 0};
  SeedGroup<WaveLanes, kSeedLanes, kSeedSlots, P, L> g{
      a.idx, a.opt, (PackedRead *)mine, FoundList<P>{fk, fs, (uint32_t *)(fs + kFoundCap), kFoundCap}, gl, gb};
  g.cap = a.slot_cap;
  g.steps = 0;
  g.lc = lc;
  for (;;) {
    const uint64_t lead = __ballot(gl == 0);
    const int first = __ffsll((unsigned long long)lead) - 1;
    int i = 0;
    if (lane == first) i = atomicAdd(a.next_read, __popcll(lead));
    i = __shfl(i, first) + __popcll(lead & ((1ull << gb) - 1));
    if (i >= a.n_reads) break;
    const int r = a.order ? a.order[i] : i;
    const int off = a.off[r], len = a.off[r + 1] - off;
    bool ok = true;
    int n = 0;
    int64_t n_seed = 0;
    if (len <= kMaxReadLen) {  // longer reads stay unaligned (documented limit)
      g.slot = a.intv + (int64_t)r * a.slot_cap;
      g.load(a.seq + off, len);
      ok = g.run() && g.n <= a.slot_cap;
      n = g.n;
      n_seed = g.n_seed;
    }
    if (gl == 0) {
      a.slow[r] = ok ? 0 : 1;
      a.n_intv[r] = ok ? n : 0;
      a.n_seed[r] = ok ? n_seed : 0;
    }
  }
  if (a.fm_steps) {  // one atomic per wavefront
    uint32_t steps = g.steps;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) steps += __shfl_xor(steps, o);
    if (lane == 0 && steps) atomicAdd((unsigned long long *)a.fm_steps, (unsigned long long)steps);
  }
  if (L && a.li_stats) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      int64_t v = lc[k];
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
      if (lane == 0 && v) atomicAdd((unsigned long long *)a.li_stats + k, (unsigned long long)v);
    }
  }
}

// Slow path for the reads listed in `list`, a wavefront per read: a group of
// 64 lanes, whose 320 entries no list of a read of <= 320 bases can outgrow.
// Pass 0 counts and keeps the first kSlowScratch intervals in the read's
// scratch; pass 1 puts all intervals at the pool offsets computed from the
// counts, copying them from the scratch when it still holds them all
// (`from_scratch`: every slow read had its own scratch in pass 0) and
// searching again otherwise.
template <class P, bool L>
__global__ void __launch_bounds__(64) k_seed_slow(SeedArgs a, const int32_t *list, int n_list, const int32_t *n_dev,
                                                  int c0, Intv *scratch, const int64_t *pool_off, Intv *pool, int pass,
                                                  int from_scratch) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  __shared__ PackedRead read;
  __shared__ P fk[kMaxReadLen], fs[kMaxReadLen];
  __shared__ uint32_t fmn[kMaxReadLen];
  const int t = blockIdx.x, lane = threadIdx.x;
  int nv = n_list;
  if (n_dev) {
    const int m = *n_dev - c0;
    nv = m < 0 ? 0 : m < n_list ? m : n_list;
  }
  if (t >= nv) return;  // the whole wavefront
  const int r = list[t];
  const int off = a.off[r], len = a.off[r + 1] - off;
  Intv *sc = scratch + (int64_t)t * kSlowScratch;
  if (pass && from_scratch && a.n_intv[r] <= kSlowScratch) {
    Intv *dst = pool + pool_off[t];
    for (int k = lane, n = a.n_intv[r]; k < n; k += 64) dst[k] = sc[k];
    return;
  }
  int64_t lc[6] = {0, 0, 0, 0, 0, 0};
  SeedGroup<WaveLanes, 64, kMaxReadLen / 64, P, L> g{
      a.idx, a.opt, &read, FoundList<P>{fk, fs, fmn, kMaxReadLen}, lane, 0};
  g.slot = pass ? pool + pool_off[t] : sc;
  g.cap = pass ? (int)(pool_off[t + 1] - pool_off[t]) : kSlowScratch;
  g.steps = 0;
  g.lc = lc;
  g.load(a.seq + off, len);
  g.run();
  if (lane == 0) {
    a.n_intv[r] = g.n;
    a.n_seed[r] = g.n_seed;
  }
}

// the narrow layout is in use (texts below 2^32 rows, unless the context
// was set to the wide layout): decided by the index, not by the text size
static bool seed_narrow(const DevIndex &x) { return x.occn != nullptr && x.sbc != nullptr; }
void launch_seed(const SeedArgs &a, int n_cu, int blocks_per_cu, int block, hipStream_t s) {
  if (!a.n_reads) return;
  // a batch that leaves compute units idle in blocks of this size runs in
  // smaller ones (200 reads fill 4 blocks of 1024 threads, or 50 of one
  // wavefront, each on a compute unit of its own); blocks_per_cu holds for them
  // too, so just below 2048, 4096, ... 16,384 reads (on 256 compute units) half
  // as many groups as reads are in flight and they take two turns
  const int64_t threads = (int64_t)a.n_reads * kSeedLanes;
  while (block > 64 && threads < (int64_t)n_cu * block) block = block / 2 / 64 * 64 > 64 ? block / 2 / 64 * 64 : 64;
  const bool narrow = seed_narrow(a.idx);
  void (*kern)(SeedArgs) = narrow ? (a.idx.saf ? k_seed<uint32_t, true> : k_seed<uint32_t, false>)
                                  : k_seed<int64_t, false>;
  const size_t groups = (size_t)block / kSeedLanes;
  const size_t lds = narrow ? (size_t)seed_super_lines<uint32_t>(a.idx) * 16 +
                                  groups * seed_group_bytes<uint32_t>(kFoundCap)
                            : (size_t)seed_super_lines<int64_t>(a.idx) * 16 +
                                  groups * seed_group_bytes<int64_t>(kFoundCap);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds) != hipSuccess || per_cu < 1)
    per_cu = 1;
  // no more blocks than the compute units hold at once
  if (blocks_per_cu > 0 && blocks_per_cu < per_cu) per_cu = blocks_per_cu;
  const int64_t need = (threads + block - 1) / block, have = (int64_t)n_cu * per_cu;
  hipLaunchKernelGGL(kern, dim3((unsigned)(need < have ? need : have)), dim3(block), lds, s, a);
}
void launch_seed_slow(const SeedArgs &a, const int32_t *list, int n_list, const int32_t *n_dev, int c0, Intv *scratch,
                      const int64_t *pool_off, Intv *pool, int pass, int from_scratch, hipStream_t s) {
  if (!n_list) return;
  auto kern = seed_narrow(a.idx) ? (a.idx.saf ? k_seed_slow<uint32_t, true> : k_seed_slow<uint32_t, false>)
                                 : k_seed_slow<int64_t, false>;
  hipLaunchKernelGGL(kern, dim3(n_list), dim3(64), 0, s, a, list, n_list, n_dev, c0, scratch, pool_off, pool, pass,
                     from_scratch);
}

}  // namespace g3a
