// Sharded ray queues and the per-ray walk with lane refill, shared by the single-scene renderer
// and the batch renderer.
#pragma once
#include "device_trace.h"

namespace nova_hip {

// A ray queue is cut into 2^shard_bits shards. Workgroup b works on shard b mod 2^shard_bits: its
// first rays and its claims come from that shard, its survivors go to the same shard of the
// next queue, and each shard's counters have a cache line of their own. Atomics on one address
// run at 11.4 ns each on this chip, whatever the number of waves: with one counter the claims
// (one per 56 rays) bound the camera walk of a one-sample 1080p frame (0.50 -> 0.34 ms; the
// frame 2.11 -> 1.90 ms, six frames at 1021x577 of a scene with many misses 2.33 -> 1.84), and
// long walks could not refill more often (64 samples at 1080p: 47.5 -> 45.8 ms). One shard per
// XCD: 16 take 46.1 ms there, 32 take 46.4.
//
// The first queue is linear (entry = path id): shard k holds every 2^shard_bits-th chunk of
// kQueueChunk entries, so all shards move through the image together. Later queues give shard k
// the entries [k * seg, (k + 1) * seg), seg being what the shard holds at the start.
constexpr uint32_t kQueueChunk = 256;
constexpr uint32_t kMaxShardBits = 3;
constexpr uint32_t kCounterStride = 32;  // words between two shards' counters
// Entries of share k of S of a linear queue of n entries, its runs of kRun dealt out in turn.
template <uint32_t kRun>
NOVA_HD uint32_t linear_share_count(uint32_t n, uint32_t S, uint32_t k) {
  const uint32_t runs = n / kRun, rest = n % kRun, last = runs % S;
  return (runs / S + (k < last ? 1u : 0u)) * kRun + (k == last ? rest : 0u);
}
// Entry i of shard k of a linear queue.
NOVA_HD uint32_t linear_shard_pos(uint32_t bits, uint32_t k, uint32_t i) { return (((i / kQueueChunk) << bits) + k) * kQueueChunk + i % kQueueChunk; }

// The workgroup's shard and its place among the workgroups of that shard.
__device__ __forceinline__ uint32_t block_shard(uint32_t bits) { return blockIdx.x & ((1u << bits) - 1); }
__device__ __forceinline__ uint32_t shard_blocks(uint32_t bits, uint32_t k) { return (gridDim.x + (1u << bits) - 1 - k) >> bits; }

// Entries of a whole queue, the same value in every lane.
__device__ __forceinline__ uint32_t queue_total(const uint32_t *shard_n, uint32_t bits) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t mine = lane < (1u << bits) ? shard_n[lane * kCounterStride] : 0u;
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < (1 << kMaxShardBits); k++) n += (uint32_t)__builtin_amdgcn_readlane((int)mine, k);
  return n;
}

#ifndef NOVA_TRACE_REFILL
// idle lanes that trigger a refill of the per-ray walk (64 samples at 1080p: 48.3 ms at 60, 47.5
// at 56, 46.2 at 40, 45.8 at 24, 47.2 at 8)
#define NOVA_TRACE_REFILL 24
#endif
// The per-ray walk of a queue by a whole grid: one traversal step per loop turn; a lane whose
// ray has ended takes the next unclaimed ray as soon as NOVA_TRACE_REFILL lanes of its wave are
// idle (one atomic per refill for the wave), so lanes do not wait for the wave's longest ray.
// The queue comes in shares with a claim counter each; a wave claims from its own share only
// (the shares are statistically alike, and taking over another's rays cost the loop 18
// registers). A share's first rays go one per lane by thread index, without an atomic: a launch
// over a nearly empty queue (the last bounces) then makes no claims at all. fetch(p, o, d) gives
// the ray at place p of the queue (and may point tc at the ray's scene), store(p, st) takes its
// finished state.
template <uint32_t kRun>
struct WalkShare {
  uint32_t n;            // its entries
  uint32_t first, step;  // the place of its entry 0, and from a run of kRun entries to its next
  uint32_t begin;        // the entry of this workgroup's first lane
  uint32_t handed;       // entries handed out by thread index
  __device__ __forceinline__ uint32_t pos(uint32_t i) const { return first + (i / kRun) * step + i % kRun; }
};
// The share of a bounce's queue that this workgroup works on, its shard: the first queue is linear.
__device__ __forceinline__ WalkShare<kQueueChunk> shard_share(const uint32_t *shard_n, uint32_t bits, uint32_t seg, bool linear) {
  const uint32_t k = block_shard(bits), n = shard_n[k * kCounterStride];
  return {n, linear ? k * kQueueChunk : k * seg, linear ? kQueueChunk << bits : kQueueChunk, (blockIdx.x >> bits) * (uint32_t)kTraceBlock,
          shard_blocks(bits, k) * (uint32_t)kTraceBlock};
}
// Every workgroup a share of its own of a linear queue: runs of a wave's entries dealt out in
// turn, short ones so that a share mixes many parts of the queue (normals of the 1080p scene of
// 1,048,576 triangles: 0.52 ms with runs of 256, 0.47 with 64, 0.53 with 32).
constexpr uint32_t kShareRun = 64;
__device__ __forceinline__ WalkShare<kShareRun> workgroup_share(uint32_t n) {
  return {linear_share_count<kShareRun>(n, gridDim.x, blockIdx.x), blockIdx.x * kShareRun, kShareRun * gridDim.x, 0, kTraceBlock};
}
struct WalkCounts {
  uint32_t nodes = 0, tests = 0, wave_turns = 0, lane_turns = 0, tri_rounds = 0;  // instrumented launches only
};

template <bool kCount, bool kAhead = false, class Share, class Fetch, class Store, class TieOf = TieFromCtx>
__device__ __forceinline__ void refill_walk(const TraceCtx &tc, LdsStack &stk, const Share &share, uint32_t *claims, Fetch fetch, Store store,
                                            WalkCounts &c, TieOf tie_of = TieOf()) {
  const uint32_t lane = threadIdx.x & 63, n = share.n, handed = share.handed;
  TraceState ts;
  NodeWords words;
  bool have = false, exhausted = handed >= n;
  uint32_t ray = 0;
  for (uint32_t turns = 0; turns < (1u << 30); turns++) {
    const uint64_t idle = __ballot(!have);
    uint32_t base = share.begin + threadIdx.x - lane;  // first turn: every lane idle, a ray per lane
    bool fill = turns == 0;
    if (!fill && !exhausted && __popcll(idle) >= NOVA_TRACE_REFILL) {
      const int leader = __builtin_ffsll((long long)idle) - 1;
      if ((int)lane == leader) base = handed + atomicAdd(claims, (uint32_t)__popcll(idle));
      base = __shfl(base, leader, 64);
      if (base >= n) exhausted = true;
      fill = true;
    }
    if (fill && !have) {
      const uint32_t i = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0));
      if (i < n) {
        const uint32_t p = share.pos(i);
        f3 o, d;
        fetch(p, o, d);
        trace_init(ts, o, d);
        if (kAhead) load_node(tc, ts.node, words);
        ray = p;
        have = true;
      }
    }
    const uint64_t busy = __ballot(have);
    if (busy == 0) break;
    if (kCount && (threadIdx.x & 63) == 0) {
      c.wave_turns++;
      c.lane_turns += (uint32_t)__popcll(busy);
    }
    if (have && trace_step<kCount>(tc, stk, ts, 0.000001f, c.nodes, c.tests, tie_of, kAhead ? &words : nullptr)) {
      store(ray, ts);
      have = false;
      if (kCount) c.tri_rounds += ts.tri_rounds;
    }
  }
}

// A finished ray's record: (prim id bits, t, u, v).
__device__ __forceinline__ float4 hit_record(const TraceState &st) {
  return make_float4(__builtin_bit_cast(float, (int32_t)(st.best)), st.tbest, st.bu, st.bv);
}

// How a batch's queues are cut: 2^bits shards of at least 4,096 paths each.
struct QueueShape {
  uint32_t bits, seg;
  size_t entries;  // of one queue: the shards' room, a little more than the paths
};
static QueueShape queue_shape(size_t paths, uint32_t max_bits) {
  QueueShape q{0, (uint32_t)paths, paths};
  while (q.bits < max_bits && (paths >> (q.bits + 1)) >= 4096) q.bits++;
  if (q.bits == 0) return q;
  const size_t chunks = (paths + kQueueChunk - 1) / kQueueChunk, S = (size_t)1 << q.bits;
  q.seg = (uint32_t)((chunks + S - 1) / S * kQueueChunk);
  q.entries = (size_t)q.seg * S;
  return q;
}

}  // namespace nova_hip
