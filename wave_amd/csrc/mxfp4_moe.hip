// Token alignment in front of the grouped (MoE) GEMM: sort the (token, slot)
// entries of a top-k routing table by expert, keep their original order inside
// an expert, pad every expert's run to a multiple of the block size.  Integer
// work on a few thousand to a few hundred thousand entries: one workgroup of
// sixteen waves does it in one launch (count, scan, place), everything but the
// ids themselves in LDS.
#include "mxfp4_common.h"
#include "mxfp4_group_table.h"

namespace wave_mxfp4 {

namespace {

constexpr int kAlignWaves = 16;
constexpr int kAlignThreads = kAlignWaves * 64;
// Steps of 64 entries whose places a wave keeps in registers between the count and the placement: 16 steps x 16
// waves = 16384 entries, read and ranked once.  A longer table is ranked a second time when it is placed.
constexpr int kRegSteps = 16;

// The place of every lane's entry among the entries of its expert that the wave has met so far, and the count of them
// moved on: `row[e]` before this step plus the lanes of the same expert below this one.  The lanes of one expert are
// found with one ballot per bit of the id (`bits` of them) and not with a turn per expert that occurs, which left a
// chain of 28 dependent turns per 64 entries at 32 experts.  The wave's LDS operations complete in their order, so
// the steps need no wait in between: the leader's addition follows every lane's read, the next step's read follows it.
__device__ __forceinline__ int rank_in_expert(int e, bool valid, int bits, int lane, int *row) {
  uint64_t same = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool one = (e >> b) & 1;
    const uint64_t ones = __ballot(one);
    same &= one ? ones : ~ones;
  }
  const int below = __popcll(same & ((1ull << lane) - 1));
  int before = 0;
  if (valid) before = __hip_atomic_load(row + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (valid && below == 0)
    __hip_atomic_fetch_add(row + e, __popcll(same), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  return before + below;
}

// Bound by latency: one round trip for the ids, the ranks of a wave's steps (about 45 vector instructions per 64
// entries at 32 experts), two barriers, one store.  MI355X, a whole expert MLP with it (us, a turn per expert that
// occurs -> ballots): 8452 entries of 32 experts 417 -> 374 (the kernel alone took 59 of them), 3672 of 32 207 -> 188,
// 192 of 32 128.4 -> 124.8, 8192 of 8 experts 810 -> 808.  The kernel alone at 8192 of 8 experts: 14.7 with every step's ids
// loaded behind a branch, 11.2 with the loads in flight together.
template <typename IdT>
__global__ void __launch_bounds__(kAlignThreads) moe_align_kernel(const IdT *__restrict__ topk_ids, int n, int num_experts,
                                                                  int block_size, int32_t *__restrict__ sorted_ids,
                                                                  int sorted_len, int32_t *__restrict__ expert_ids,
                                                                  int expert_ids_len, int32_t *__restrict__ total_out,
                                                                  int32_t *__restrict__ offsets_out) {
  extern __shared__ int lds[];
  int *cnt = lds;                                // [kAlignWaves][E]: entries of expert e in wave w's segment, later
                                                 // the first (a long table: the next) position for them
  int *wave_sums = lds + kAlignWaves * num_experts;  // [kAlignWaves]
  int *starts = wave_sums + kAlignWaves;             // [E + 1]: first position of every expert's run, then the total
  int *counts = starts + num_experts + 1;            // [E]: entries of every expert
  const int E = num_experts;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int bits = E > 1 ? 32 - __clz(E - 1) : 0;
  int *row = cnt + wave * E;

  // wave w owns the contiguous segment [seg0, seg1) of the flat table
  const int per_wave = ((n + kAlignWaves - 1) / kAlignWaves + 63) & ~63;
  const int seg0 = min(n, wave * per_wave), seg1 = min(n, seg0 + per_wave);
  const bool in_regs = per_wave <= kRegSteps * 64;

  // (all steps' ids are fetched together, lanes beyond the segment its last one: a step at a time, and a step behind a
  // branch, would pay a memory round trip each)
  int id[kRegSteps], place[kRegSteps];
  auto fetch_and_rank = [&](int base) {
#pragma unroll
    for (int s = 0; s < kRegSteps; ++s) {
      const int i = base + s * 64 + lane;
      const int64_t v = (int64_t)topk_ids[min(i, seg1 - 1)];
      id[s] = i < seg1 && v >= 0 && v < E ? (int)v : -1;
    }
#pragma unroll
    for (int s = 0; s < kRegSteps; ++s)
      if (base + s * 64 < seg1) place[s] = rank_in_expert(id[s], id[s] >= 0, bits, lane, row);
  };
  for (int i = t; i < kAlignWaves * E; i += kAlignThreads) cnt[i] = 0;
  __syncthreads();
  for (int base = seg0; base < seg1; base += kRegSteps * 64) fetch_and_rank(base);
  __syncthreads();

  // thread e: the expert's count, padded count and first position
  int count = 0;
  if (t < E) {
    for (int w = 0; w < kAlignWaves; ++w) count += cnt[w * E + t];
  }
  const int blocks = (count + block_size - 1) / block_size, padded = blocks * block_size;
  const int end = block_inclusive_scan(padded, wave_sums, lane, wave);  // also the total, in the last thread
  const int start = end - padded;
  if (t < E) {
    int run = start;
    for (int w = 0; w < kAlignWaves; ++w) {
      const int c = cnt[w * E + t];
      cnt[w * E + t] = run;
      run += c;
    }
    starts[t] = start;
    counts[t] = count;
    if (offsets_out) offsets_out[t] = start;
  }
  if (t == kAlignThreads - 1) starts[E] = end;
  __syncthreads();

  // place
  if (in_regs) {
#pragma unroll
    for (int s = 0; s < kRegSteps; ++s) {
      if (seg0 + s * 64 >= seg1) break;
      if (id[s] >= 0) {
        const int pos = row[id[s]] + place[s];
        if (pos < sorted_len) sorted_ids[pos] = seg0 + s * 64 + lane;
      }
    }
  } else {
    for (int base = seg0; base < seg1; base += kRegSteps * 64) {
      fetch_and_rank(base);
#pragma unroll
      for (int s = 0; s < kRegSteps; ++s)
        if (id[s] >= 0 && place[s] < sorted_len) sorted_ids[place[s]] = base + s * 64 + lane;
    }
  }

  const int total = starts[E];
  if (t == 0) {
    total_out[0] = total;
    if (offsets_out) offsets_out[E] = total;
  }
  for (int i = total + t; i < sorted_len; i += kAlignThreads) sorted_ids[i] = n;  // past the padded total
  // every run's padding (fewer than block_size entries): one wave per expert, a lane per entry
  for (int e = wave; e < E; e += kAlignWaves) {
    const int from = starts[e] + counts[e], to = min(starts[e + 1], sorted_len);
    for (int i = from + lane; i < to; i += 64) sorted_ids[i] = n;
  }
  // the expert of every block: a wave per expert fills the blocks of its run (an empty expert has none)
  for (int e = wave; e < E; e += kAlignWaves) {
    const int from = starts[e] / block_size, to = min(starts[e + 1] / block_size, expert_ids_len);
    for (int b = from + lane; b < to; b += 64) expert_ids[b] = e;
  }
}

// The M tile table of a grouped GEMM (mxfp4_group_table.h) by a launch of its own: a thread per group, one wave for up to 64
// of them, whose barriers then cost nothing (8 groups, kernel trace: 6.8 -> 5.0 us).
template <int NT>
__global__ void __launch_bounds__(NT) grouped_tile_table_kernel(const GroupTableArgs g) {
  __shared__ int wave_sums[NT / 64];
  __shared__ int carry[2];
  build_group_tile_table<NT>(g, wave_sums, carry);
}

}  // namespace

hipError_t launch_grouped_tile_table(const int32_t *offsets, int num_groups, int bm, int short_rows, int64_t total_rows,
                                     int32_t *table, hipStream_t stream) {
  const GroupTableArgs g{offsets, num_groups, bm, short_rows, (int)total_rows, table};
  if (num_groups <= 64) grouped_tile_table_kernel<64><<<1, 64, 0, stream>>>(g);
  else grouped_tile_table_kernel<kAlignThreads><<<1, kAlignThreads, 0, stream>>>(g);
  return hipGetLastError();
}

hipError_t launch_moe_align(const void *topk_ids, int ids_int64, int64_t n, int num_experts, int block_size,
                            int32_t *sorted_ids, int64_t sorted_len, int32_t *expert_ids, int64_t expert_ids_len,
                            int32_t *total, int32_t *offsets, hipStream_t stream) {
  const size_t lds = (size_t)(kAlignWaves * num_experts + kAlignWaves + 2 * num_experts + 1) * sizeof(int);
  static LdsAttrOnce once[2];
  const void *fn = ids_int64 ? (const void *)moe_align_kernel<int64_t> : (const void *)moe_align_kernel<int32_t>;
  const hipError_t e = allow_dynamic_lds(
      once[ids_int64 ? 1 : 0], fn, (int)((kAlignWaves * kMoeMaxExperts + kAlignWaves + 2 * kMoeMaxExperts + 1) * sizeof(int)));
  if (e != hipSuccess) return e;
  if (ids_int64)
    moe_align_kernel<int64_t><<<1, kAlignThreads, lds, stream>>>((const int64_t *)topk_ids, (int)n, num_experts, block_size,
                                                                 sorted_ids, (int)sorted_len, expert_ids,
                                                                 (int)expert_ids_len, total, offsets);
  else
    moe_align_kernel<int32_t><<<1, kAlignThreads, lds, stream>>>((const int32_t *)topk_ids, (int)n, num_experts, block_size,
                                                                 sorted_ids, (int)sorted_len, expert_ids,
                                                                 (int)expert_ids_len, total, offsets);
  return hipGetLastError();
}

}  // namespace wave_mxfp4
