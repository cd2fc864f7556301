// Traceback kernels for MI355X (gfx950, wave64):
//   k_tb_count, k_tb_order  alignments by class of band
//   k_tb_gap                a group of lanes per gapped alignment (g3a_trace.h)
//   k_traceback             thread per alignment: the ungapped ones, the
//                           widest bands, and every alignment's final record
#include "g3a_kernels.h"
#include "g3a_trace.h"

#include <hip/hip_runtime.h>

namespace g3a {

constexpr int kQMax = kMaxReadLen + 2;

// Tiles of kTilePer * 256 elements for the classifying kernels: a tile
// counts its members in LDS and reserves its places with one global atomic a
// counter.
constexpr int kTilePer = 16;

__device__ __forceinline__ int64_t dcount(const int64_t *dev, int64_t cap) {
  if (!dev) return cap;
  const int64_t v = *dev;
  return v < cap ? v : cap;
}

// Classes by band: 0: at most 16 columns, 1: at most 32, 2: wider, 3:
// ungapped (w = 0).
__device__ __forceinline__ int tb_class(const TbArgs &a, int64_t t) {
  const Region g = a.aln_reg[t];
  const int w = global_bw(a.opt, g.qe - g.qb, g.re - g.rb, g.score);
  return w == 0 ? 3 : w <= 7 ? 0 : w <= 15 ? 1 : 2;
}
// tb_ctr[0..2]: alignments of classes 0..2 (tiles of kTilePer * 256)
__global__ void __launch_bounds__(256) k_tb_count(TbArgs a) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  __shared__ int32_t cnt[3];
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t tile = (int64_t)blockIdx.x * (256 * kTilePer);
  const int64_t n = dcount(a.n_dev, a.n_alns);
  int c3[3] = {0, 0, 0};
#pragma unroll
  for (int i = 0; i < kTilePer; ++i) {
    const int64_t t = tile + i * 256 + threadIdx.x;
    const int c = t < n ? tb_class(a, t) : 3;
#pragma unroll
    for (int k = 0; k < 3; ++k) c3[k] += c == k;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (c3[k]) atomicAdd(&cnt[k], c3[k]);
  __syncthreads();
  if (threadIdx.x < 3 && cnt[threadIdx.x]) atomicAdd(a.tb_ctr + threadIdx.x, cnt[threadIdx.x]);
}
// The list holds classes 0, 1, 2 in turn from the front and class 3 from the
// back; tb_ctr[4..7] are the placement cursors (tiles of kTilePer * 256).
__global__ void __launch_bounds__(256) k_tb_order(TbArgs a) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  __shared__ int32_t cnt[4], base[4];
  if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t tile = (int64_t)blockIdx.x * (256 * kTilePer);
  const int64_t n_alns = dcount(a.n_dev, a.n_alns);
  int cls[kTilePer], at[kTilePer];
#pragma unroll
  for (int i = 0; i < kTilePer; ++i) {
    const int64_t t = tile + i * 256 + threadIdx.x;
    cls[i] = t < n_alns ? tb_class(a, t) : -1;
    at[i] = cls[i] >= 0 ? atomicAdd(&cnt[cls[i]], 1) : -1;
  }
  __syncthreads();
  if (threadIdx.x < 4) base[threadIdx.x] = cnt[threadIdx.x] ? atomicAdd(a.tb_ctr + 4 + threadIdx.x, cnt[threadIdx.x]) : 0;
  __syncthreads();
  const int64_t base1 = a.tb_ctr[0], base2 = base1 + a.tb_ctr[1];
#pragma unroll
  for (int i = 0; i < kTilePer; ++i) {
    const int c = cls[i];
    if (c < 0) continue;
    const int r = base[c] + at[i];
    const int64_t pos = c == 0 ? r : c == 1 ? base1 + r : c == 2 ? base2 + r : n_alns - 1 - r;
    a.tb_order[pos] = (int32_t)(tile + i * 256 + threadIdx.x);
  }
}

// Both for a few alignments in one block, with the zero before them: three
// launches less of 4 to 5 us.
constexpr int kTbSmall = 1 << 14, kTbThreads = 1024;
__global__ void __launch_bounds__(kTbThreads) k_tb_small(TbArgs a) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  __shared__ int32_t cnt[4], cur[4];
  const int tid = threadIdx.x;
  if (tid < 4) cnt[tid] = cur[tid] = 0;
  __syncthreads();
  const int n = (int)dcount(a.n_dev, a.n_alns);
  uint32_t cls = 0;  // two bits an alignment
  for (int k = 0, t = tid; t < n; ++k, t += kTbThreads) {
    const int c = tb_class(a, t);
    cls |= (uint32_t)c << (2 * k);
    atomicAdd(&cnt[c], 1);
  }
  __syncthreads();
  for (int k = 0, t = tid; t < n; ++k, t += kTbThreads) {
    const int c = cls >> (2 * k) & 3, r = atomicAdd(&cur[c], 1);
    const int pos = c == 0 ? r : c == 1 ? cnt[0] + r : c == 2 ? cnt[0] + cnt[1] + r : n - 1 - r;
    a.tb_order[pos] = t;
  }
  if (tid < 3) a.tb_ctr[tid] = cnt[tid];
}
static_assert(kTbSmall / kTbThreads * 2 <= 32, "an alignment's class is two bits of a word");
// One gapped alignment by a group: the CIGAR, the score and the mismatch
// count, which k_traceback takes into the final record.
template <int G, int NH>
__device__ __forceinline__ void gap_one(const TbArgs &a, int64_t t, uint8_t *lds, int lds_bytes) {
  const int lane = threadIdx.x & 63, gl = lane % G, gb = lane - gl;
  uint8_t *mine = lds + gb / G * (lds_bytes * G / 64);
  const int r = a.aln_read[t];
  const Region g = a.aln_reg[t];
  GapGroup<WaveLanes, G, NH> gg{a.idx, a.opt, reinterpret_cast<GapStage *>(mine),
                                reinterpret_cast<uint32_t *>(mine + sizeof(GapStage)), gl, gb};
  gg.qlen = g.qe - g.qb;
  gg.tlen = (int)(g.re - g.rb);
  gg.w = global_bw(a.opt, gg.qlen, gg.tlen, g.score);
  // direction bits that the LDS does not hold go to the alignment's bytes in
  // memory (only wide bands of long reads; four bits a cell there too)
  if (gap_words(gg.qlen, gg.tlen, gg.w) * 4 > lds_bytes * G / 64 - (int)sizeof(GapStage))
    gg.z = reinterpret_cast<uint32_t *>(a.z + a.z_off[t]);
  gg.load(a.seq + a.off[r] + g.qb, g.rb);
  const int nw = gg.dp();
  int nm;
  const int n = gg.walk(a.cigar + a.cig_off[t] + aln_core_at(gg.qlen, gg.tlen, gg.w), nm);
  if (gl == 0) {
    a.alns[t].nw_score = nw;
    a.alns[t].nm = nm;
    a.alns[t].n_core = n;
  }
}
// What bounds it: the chain of one alignment's rows (about 40 instructions
// each) while a batch does not fill the chip, VALU issue after.  On one thread
// (a band's cells one after another, then a dependent byte load a step) the
// five kernels this replaces took 2.0 ms for any batch of 4,000 to 250,000
// reads of 150 bp, because the slowest alignment did; traceback in all, 10,000
// reads 2.23 -> 0.29 ms, 250,000 reads 2.6 -> 0.65 ms.  16 lanes suit 94% of the
// gapped alignments and shift by row DPP; the LDS of four such alignments
// (20 KB, the class's bound at 320 bases) leaves 8 blocks a compute unit.
// A persistent grid of one-wavefront blocks: a unit is one alignment of
// class 2, two of class 1 (32 lanes each) or four of class 0 (16 lanes each),
// the longest-running class first.
constexpr int kGapSlice = (int)sizeof(GapStage) + 4 * 41 * 16;  // class 0: 324 rows of at most 15 columns
static_assert(kGapSlice * 2 >= (int)sizeof(GapStage) + 4 * 42 * 31, "class 1: 332 rows of at most 31 columns");
__global__ void __launch_bounds__(64) k_tb_gap(TbArgs a) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  __shared__ __align__(16) uint8_t lds[kGapSlice * 4];
  const int lane = threadIdx.x;
  const int64_t n0 = a.tb_ctr[0], n1 = a.tb_ctr[1], n2 = a.tb_ctr[2];
  const int64_t u1 = (n1 + 1) / 2, u0 = (n0 + 3) / 4;
  for (int64_t u = blockIdx.x; u < n2 + u1 + u0; u += gridDim.x) {
    if (u < n2) {
      const int64_t t = a.tb_order[n0 + n1 + u];
      const Region g = a.aln_reg[t];
      const int w = global_bw(a.opt, g.qe - g.qb, g.re - g.rb, g.score);
      if (w <= 31) gap_one<64, 1>(a, t, lds, (int)sizeof lds);
      else if (w <= kGapW) gap_one<64, 2>(a, t, lds, (int)sizeof lds);
      // else k_traceback's
    } else if (u < n2 + u1) {
      const int64_t e = (u - n2) * 2 + lane / 32;
      if (e < n1) gap_one<32, 1>(a, a.tb_order[n0 + e], lds, (int)sizeof lds);
    } else {
      const int64_t e = (u - n2 - u1) * 4 + lane / 16;
      if (e < n0) gap_one<16, 1>(a, a.tb_order[e], lds, (int)sizeof lds);
    }
  }
}

__global__ void __launch_bounds__(64) k_traceback(TbArgs a) {
  if (a.stop && *a.stop) return;  // a capacity check before this kernel failed: the batch is redone
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nthreads = (int64_t)gridDim.x * blockDim.x;
  int32_t *eh_h = a.eh_pool + gtid * 2 * kQMax, *eh_e = eh_h + kQMax;
  const int64_t n_alns = dcount(a.n_dev, a.n_alns);
  for (int64_t e = gtid; e < n_alns; e += nthreads) {
    const int64_t t = a.tb_order[e];
    const int r = a.aln_read[t];
    const int off = a.off[r], l_seq = a.off[r + 1] - off;
    const Region g = a.aln_reg[t];
    const int w = global_bw(a.opt, g.qe - g.qb, g.re - g.rb, g.score);
    Aln out;
    trace_and_finalize(a.idx, a.opt, a.seq + off, l_seq, g, a.aln_rank[t], EhArray{eh_h, eh_e}, a.z + a.z_off[t],
                       a.cigar + a.cig_off[t], a.cig_off[t], out, w > 0 && w <= kGapW ? a.alns + t : nullptr);
    a.alns[t] = out;
  }
}

int traceback_grid_threads(int n_cu) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_traceback, 64, 0) != hipSuccess || per_cu < 1)
    per_cu = 16;
  return n_cu * per_cu * 64;
}
int64_t traceback_pool_words(int n_threads) { return (int64_t)n_threads * 2 * kQMax; }
void launch_traceback(const TbArgs &a, int n_threads, int n_cu, hipStream_t s) {
  if (!a.n_alns) return;
  if (a.n_alns <= kTbSmall) {
    hipLaunchKernelGGL(k_tb_small, dim3(1), dim3(kTbThreads), 0, s, a);
  } else {
    launch_fill_i32(a.tb_ctr, 8, 0, s);
    const dim3 gt((unsigned)((a.n_alns + 256 * kTilePer - 1) / (256 * kTilePer)));
    hipLaunchKernelGGL(k_tb_count, gt, dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_tb_order, gt, dim3(256), 0, s, a);
  }
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_tb_gap, 64, 0) != hipSuccess || per_cu < 1) per_cu = 4;
  const int64_t all = (int64_t)n_cu * per_cu;
  hipLaunchKernelGGL(k_tb_gap, dim3((unsigned)(a.n_alns < all ? a.n_alns : all)), dim3(64), 0, s, a);
  // the pool has a slice for each of the n_threads threads
  const int64_t need = (a.n_alns + 63) / 64, have = n_threads / 64;
  hipLaunchKernelGGL(k_traceback, dim3((unsigned)(need < have ? need : have)), dim3(64), 0, s, a);
}

}  // namespace g3a
