// Unordered SSSP/BFS rounds of a middle-sized graph in one launch.
//
// A round of such a graph is a chain of latencies: launched as a tile and a
// drain kernel it took 33 us on RMAT-16 (65536 vertices, 2^20 arcs), most of
// it with a few thousand arcs to do.  Here all rounds run in one launch of at
// most kRoundWgs workgroups that meet at a barrier (5 us for a round of a few
// arcs, 10 for some tens of thousands, 80 for RMAT-17's largest with 1.9
// million, where the loads and atomics of dist bind), and the chain is cut
// down:
// - A workgroup keeps what it queues in LDS, each entry with its vertex, first
//   arc and the number of queued arcs before it, and then takes its place in
//   the next queue with one 64-bit atomic on (entries, arcs).  The queue is so
//   sorted by arcs: its length, its arcs and an entry's first arc are known
//   without another pass or scan.
// - Every workgroup takes an equal share of the round's arcs, whatever the
//   degrees: no chunk queue, no claims.
// - What crosses workgroups is stored and read device-coherent and each wave
//   waits for its stores before the barrier, so the barrier needs no L2
//   write-back or invalidate.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"
#include "grid_barrier.h"
#include "lds_sssp.h"
#include "smdp_internal.h"

namespace smdp {

constexpr int kRoundWgs = 256;       // most workgroups (a launch has at most three quarters of the CUs)
constexpr int kRoundThreads = 1024;
constexpr int kRoundOut = 8192;      // entries a workgroup keeps before they go to the queue
constexpr int kRoundIlp = 2;         // arcs per thread and step
constexpr int kTriedBits = 11;       // of the slots for candidates that a workgroup has tried

// A workgroup's part of a queue: arcs before it and first entry in the high
// and low half of at, entries in count.  Found with the queue's counters, it
// saves a search of the whole queue for the first entry of a share.
struct RoundPart {
  uint64_t at, count;
};

struct RoundCtl {
  uint32_t bar[kBarLines * 32];
  uint64_t queued[4 * 16];  // (entries << 32 | arcs) of round r at [(r & 3) * 16]
  int32_t many[2];          // the last round of each parity whose queue holds several parts of one workgroup
  int32_t pad[30];
  RoundPart part[2][kRoundWgs];
};
static_assert(sizeof(RoundCtl) <= 4 * sizeof(Ctl), "kept in the graph's control blocks");

// How a launch ended (Counters::done).
constexpr int kRoundsCapped = 1, kRoundsRetry = 2;

struct RoundArgs {
  const int32_t* __restrict__ row;
  const int32_t* __restrict__ col;
  const int32_t* __restrict__ w;
  int32_t* dist;
  int32_t* stamp;     // nullptr: BFS
  RoundEntry* queue;  // [2][qcap]
  RoundCtl* ctl;
  Counters* cnt;
  int32_t n;
  int32_t qcap;
  int32_t rmax;
  unsigned long long* rlog;  // profiling: per round (queue length, arcs), then the rounds' starting clocks, or nullptr
};

template <typename T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_rounds_init(RoundArgs a, int32_t inf, int32_t src) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * blockDim.x) {
    a.dist[i] = i == src ? 0 : inf;
    if (a.stamp) a.stamp[i] = -1;
  }
  if (blockIdx.x == 0) {
    int32_t* c = reinterpret_cast<int32_t*>(a.ctl);
    for (int i = threadIdx.x; i < (int)(sizeof(RoundCtl) / 4); i += blockDim.x) c[i] = 0;
    unsigned long long* k = reinterpret_cast<unsigned long long*>(a.cnt);
    for (int i = threadIdx.x; i < (int)(kCntParts * sizeof(Counters) / 8); i += blockDim.x) k[i] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
      const int st = a.row[src];
      a.queue[0] = RoundEntry{(uint64_t)(uint32_t)st << 32 | (uint32_t)src, 0};
      a.ctl->queued[0] = 1ull << 32 | (uint32_t)(a.row[src + 1] - st);
      a.ctl->part[0][0] = RoundPart{0, 1};
    }
  }
}

// grid_barrier without its fences: the caller's stores that others read are
// device-coherent, and complete before the arrival.
__device__ __forceinline__ bool coherent_barrier(uint32_t* bar, uint32_t epoch, int* s_ok) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t nwg = gridDim.x, grp = blockIdx.x & 7;
    const uint32_t members = (nwg - grp + 7) / 8;  // workgroups g < nwg with g % 8 == grp
    const uint32_t ngroups = nwg < 8 ? nwg : 8;
    if (atomicAdd(&bar[32 * grp], 1u) + 1 == epoch * members && atomicAdd(&bar[32 * 8], 1u) + 1 == epoch * ngroups)
      agent_store(&bar[32 * 9], epoch);
    int ok = 1;
    for (int spins = 0; agent_load(&bar[32 * 9]) < epoch;) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins > kBarSpinLimit) {
        ok = 0;
        break;
      }
    }
    *s_ok = ok;
  }
  __syncthreads();
  return *s_ok != 0;
}

struct RoundShared {
  int of[kRoundThreads];   // the window's entries: queued arcs before, INT32_MAX past the share
  int st[kRoundThreads];   // first arc less of
  int du[kRoundThreads];
  int nent[2];             // entries of the window that are in the share (by the window's parity)
  unsigned long long out;  // (entries << 32 | arcs) queued in this round
  unsigned long long base; // what the next queue held before them
  int count;               // the entries among them
  int ok;
  uint64_t tried[1 << kTriedBits];  // vertex << 32 | candidate, at the vertex's tried_slot
  int v[kRoundOut], start[kRoundOut], before[kRoundOut];  // what the workgroup queued
};

__device__ __forceinline__ uint32_t tried_slot(int v) { return (uint32_t)v * 2654435761u >> (32 - kTriedBits); }

struct RoundCount {
  uint32_t tries = 0, wins = 0, pushes = 0;
};

// A round's arcs read their targets before any of its atomics lands, so where
// many lead to one vertex nearly all of them tried to lower it, one after
// another: 200000 arcs into one vertex took BFS 1107 us and SSSP 603, into 64
// vertices 468 and 293.  So of the lanes of a wave that want to lower the same
// vertex only one with the lowest candidate stays, and every workgroup keeps
// what it has tried: 59 and 76 us, 152 and 260.  (A vertex in RoundShared::tried
// is only skipped for candidates that are no lower than one whose atomic was
// issued, in this round or before.)
// The first lanes' targets are looked at as long as kSameTarget lanes or more
// share them: once, where they do not.  A round of fewer than kCrowdedArcs arcs
// does without, since it costs 0.15 us of the 5 that such a round takes.
constexpr int kSameTarget = 4;
constexpr int kCrowdedArcs = 8192;
__device__ __forceinline__ bool lowest_of_target(bool want, int v, int alt) {
  for (uint64_t m = ballot(want); m;) {
    const int target = __builtin_amdgcn_readlane(v, first_lane(m));
    const bool same = want && v == target;
    const uint64_t s = ballot(same);
    if (__popcll(s) < kSameTarget) break;
    m &= ~s;
    const int lowest = __builtin_amdgcn_readlane(wave_min_dpp(same ? alt : INT32_MAX), SMDP_WAVE - 1);
    if (same) want = lane_id() == first_lane(ballot(same && alt == lowest));
  }
  return want;
}

// Relaxes the window's arcs jb + K * thread + k below jend, K per thread.
// Wave-uniform.  A thread's arcs follow one another, so one search finds them
// all.  Two of them measured best: RMAT-17 x 16 382 us, three 388, four 392,
// six 396; BFS on a tree of 4M 114, 121, 132, 153, on RMAT-20 322, 325, 341,
// 334 (four arcs kRoundThreads apart, each with its search: 406, 113, 382).
template <bool BFS, int K>
__device__ __forceinline__ void round_arcs(const RoundArgs& a, RoundShared& sh, int jb, int jend, int top, int r,
                                           bool crowded, RoundCount& n) {
  const int lane = lane_id();
  int j[K], own[K], v[K], alt[K], seen[K];
  const int j0 = jb + (int)threadIdx.x * K;
#pragma unroll
  for (int k = 0; k < K; ++k) j[k] = min(j0 + k, jend - 1);
  own[0] = 0;
  for (int step = top; step; step >>= 1) {
    const int i = own[0] + step;
    if (i < kRoundThreads && sh.of[min(i, kRoundThreads - 1)] <= j[0]) own[0] = i;
  }
#pragma unroll
  for (int k = 1; k < K; ++k) {
    own[k] = own[k - 1];
    // every queued vertex has an arc, so the next arc is this entry's or the next's
    if (own[k] + 1 < kRoundThreads && sh.of[min(own[k] + 1, kRoundThreads - 1)] <= j[k]) ++own[k];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int e = sh.st[own[k]] + j[k];
    v[k] = a.col[e];
    alt[k] = BFS ? r + 1 : sh.du[own[k]] + a.w[e];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) seen[k] = agent_load(a.dist + v[k]);
  // Only the atomic is under a condition: loads in a branch were waited for
  // there, slot after slot.  A lane without a candidate loads vertex 0's words.
  int old[K], stamp[K], st[K], deg[K], wants[K];
  uint64_t tried[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    wants[k] = j0 + k < jend && alt[k] < seen[k] ? 1 : 0;
    tried[k] = ~0ull;
  }
  if (crowded) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      wants[k] = lowest_of_target(wants[k] != 0, v[k], alt[k]) ? 1 : 0;
      tried[k] = __hip_atomic_load(&sh.tried[tried_slot(v[k])], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint64_t t = tried[k];
    const bool want = wants[k] && ((int)(t >> 32) != v[k] || (int)(uint32_t)t > alt[k]);
    if (want && crowded)
      __hip_atomic_store(&sh.tried[tried_slot(v[k])], (uint64_t)(uint32_t)v[k] << 32 | (uint32_t)alt[k],
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    old[k] = INT32_MIN;
    if (want) old[k] = atomicMin(&a.dist[v[k]], alt[k]);
    v[k] = want ? v[k] : 0;
    n.tries += want;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    stamp[k] = BFS ? 0 : agent_load(a.stamp + v[k]);
    st[k] = a.row[v[k]];
    deg[k] = a.row[v[k] + 1];
  }
  // the first of the round's improvements of v queues it; the flags stay in
  // vector registers (K masks more spilled the scalar ones: 40 % slower)
  int push[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    deg[k] -= st[k];
    const int won = old[k] != INT32_MIN && alt[k] < old[k] ? 1 : 0;
    n.wins += won;
    push[k] = deg[k] > 0 && (BFS || stamp[k] != r + 1) ? won : 0;
    asm("" : "+v"(push[k]));
    if (!BFS && push[k]) stamp[k] = atomicExch(&a.stamp[v[k]], r + 1);
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool push_k = push[k] && (BFS || stamp[k] != r + 1);
    const uint64_t m = ballot(push_k);
    if (!m) continue;
    const int incl = wave_scan_dpp(push_k ? deg[k] : 0);
    const int arcs = __builtin_amdgcn_readlane(incl, SMDP_WAVE - 1);
    unsigned long long at = 0;
    if (lane == 0) at = atomicAdd(&sh.out, (unsigned long long)__popcll(m) << 32 | (uint32_t)arcs);
    const int before = __builtin_amdgcn_readfirstlane((int)(uint32_t)at);
    const int pos = __builtin_amdgcn_readfirstlane((int)(at >> 32)) + mbcnt(m);
    n.pushes += push_k;
    if (push_k) {
      sh.v[pos] = v[k];
      sh.start[pos] = st[k];
      sh.before[pos] = before + incl - deg[k];
    }
  }
}

// What the workgroup has queued goes to the queue of round r + 1 (all
// threads); last: the round's last time.
__device__ __forceinline__ void round_flush(const RoundArgs& a, RoundShared& sh, int r, bool last) {
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long out = sh.out;
    sh.out = 0;
    sh.base = out ? atomicAdd(reinterpret_cast<unsigned long long*>(&a.ctl->queued[((r + 1) & 3) * 16]), out) : 0;
    sh.count = (int)(out >> 32);
    if (last) {
      RoundPart* mine = &a.ctl->part[(r + 1) & 1][blockIdx.x];
      agent_store(&mine->at, (uint64_t)(sh.base << 32 | sh.base >> 32));
      agent_store(&mine->count, (uint64_t)(out >> 32));
    } else {
      agent_store(&a.ctl->many[(r + 1) & 1], r + 1);
    }
  }
  __syncthreads();
  const uint32_t arc0 = (uint32_t)sh.base;
  RoundEntry* q = a.queue + (int64_t)((r + 1) & 1) * a.qcap + (sh.base >> 32);
  for (int i = threadIdx.x; i < sh.count; i += kRoundThreads) {
    agent_store(&q[i].x, (uint64_t)(uint32_t)sh.start[i] << 32 | (uint32_t)sh.v[i]);
    agent_store(&q[i].y, (uint64_t)(arc0 + (uint32_t)sh.before[i]));
  }
  if (!last) __syncthreads();
}

template <bool BFS>
__global__ __launch_bounds__(kRoundThreads) void k_rounds(RoundArgs a, int32_t inf) {
  __shared__ RoundShared sh;
  const int lane = lane_id(), tid = threadIdx.x, b = blockIdx.x, G = gridDim.x;
  RoundCount n;
  unsigned long long edges = 0, verts = 0;
  for (int i = tid; i < 1 << kTriedBits; i += kRoundThreads) sh.tried[i] = ~0ull;
  if (tid == 0) {
    sh.out = 0;
    sh.nent[0] = sh.nent[1] = 0;
  }
  __syncthreads();
  int r = 0, end = 0, windows = 0;
  for (;; ++r) {
    const uint64_t q = agent_load(&a.ctl->queued[(r & 3) * 16]);
    // the last part that begins at or before this share
    uint64_t at[kRoundWgs / SMDP_WAVE];
    int have[kRoundWgs / SMDP_WAVE];
    const RoundPart* part = a.ctl->part[r & 1];
#pragma unroll
    for (int k = 0; k < kRoundWgs / SMDP_WAVE; ++k) {
      const int i = k * SMDP_WAVE + lane;
      at[k] = i < G ? agent_load(&part[i].at) : 0;
      have[k] = i < G ? (int)agent_load(&part[i].count) : 0;
    }
    const bool many = agent_load(&a.ctl->many[r & 1]) == r;
    const int L = (int)(q >> 32), A = (int)(uint32_t)q;
    if (a.rlog && b == 0 && tid == 0 && r < kRoundLogCap) {
      a.rlog[2 * r] = (unsigned long long)L;
      a.rlog[2 * r + 1] = (unsigned long long)A;
      a.rlog[2 * kRoundLogCap + r] = wall_clock64();
    }
    if (r >= a.rmax) {  // the last round, which finds no work, counts too
      end = kRoundsCapped;
      break;
    }
    if (L == 0) break;
    if (b == 0 && tid == 0) {
      agent_store(&a.ctl->queued[((r + 2) & 3) * 16], (uint64_t)0);  // nobody uses it before round r + 1
      edges += A;
      verts += L;
    }
    const int j0 = (int)((int64_t)A * b / G), j1 = (int)((int64_t)A * (b + 1) / G);
    const RoundEntry* qin = a.queue + (int64_t)(r & 1) * a.qcap;
    if (j0 < j1) {
      int before = 0, p = 0, cnt = 0;  // of the part: arcs before, first entry, entries
#pragma unroll
      for (int k = 0; k < kRoundWgs / SMDP_WAVE; ++k)
        if (have[k] && (int)(at[k] >> 32) <= j0 && (int)(at[k] >> 32) >= before) {
          before = (int)(at[k] >> 32);
          p = (int)(uint32_t)at[k];
          cnt = have[k];
        }
      // parts with entries have arcs, so the one with most arcs before it has the highest entry
      const int most = ~__builtin_amdgcn_readlane(wave_min_dpp(cnt ? ~p : INT32_MAX), SMDP_WAVE - 1);
      cnt = __builtin_amdgcn_readlane(cnt, first_lane(ballot(cnt && p == most)));
      p = most;
      if (many) {
        p = 0;
        cnt = L;
      }
      // the share's first entry is among the kRoundThreads / 2 from p on
      while (cnt > kRoundThreads / 2) {
        const int step = (cnt + SMDP_WAVE - 1) / SMDP_WAVE;
        const bool le = lane * step < cnt && (int)agent_load(&qin[p + min(lane * step, cnt - 1)].y) <= j0;
        const int to = (__popcll(ballot(le)) - 1) * step;
        p += to;
        cnt = min(step, cnt - to);
      }
      int room = kRoundOut;  // entries that surely fit: an arc queues one at most
      for (int jb = j0; jb < j1; ++windows) {
        const int i = p + tid;
        RoundEntry e{0, 0};
        if (i < L) {
          e.x = agent_load(&qin[i].x);
          e.y = agent_load(&qin[i].y);
        }
        const int of = (int)(uint32_t)e.y;
        const bool in = i < L && of < j1;
        sh.of[tid] = in ? of : INT32_MAX;
        sh.st[tid] = (int)(e.x >> 32) - of;
        if (!BFS && in) sh.du[tid] = agent_load(a.dist + (uint32_t)e.x);
        const uint64_t m = ballot(in);
        if (lane == 0 && m) atomicMax(&sh.nent[windows & 1], tid + __popcll(m));
        if (tid == 0) sh.nent[(windows + 1) & 1] = 0;
        __syncthreads();
        const int nent = sh.nent[windows & 1];
        // a full window's last entry only ends it
        const int jend = nent == kRoundThreads ? sh.of[kRoundThreads - 1] : j1;
        const int top = 1 << (31 - __builtin_clz(nent));
        while (jb < jend) {
          if (room < kRoundIlp * kRoundThreads) {
            __syncthreads();
            room = kRoundOut - (int)(sh.out >> 32);
            __syncthreads();
            if (room < kRoundIlp * kRoundThreads) {
              round_flush(a, sh, r, false);
              room = kRoundOut;
            }
          }
          room -= min(jend - jb, kRoundIlp * kRoundThreads);
          if (jend - jb > kRoundThreads) {
            round_arcs<BFS, kRoundIlp>(a, sh, jb, jend, top, r, A >= kCrowdedArcs, n);
            jb += kRoundIlp * kRoundThreads;
          } else {
            round_arcs<BFS, 1>(a, sh, jb, jend, top, r, A >= kCrowdedArcs, n);
            jb += kRoundThreads;
          }
        }
        jb = jend;
        p += kRoundThreads - 1;
        if (jb < j1) __syncthreads();  // the next window is written over this one
      }
    }
    round_flush(a, sh, r, true);
    if (!coherent_barrier(a.ctl->bar, (uint32_t)r + 1, &sh.ok)) {
      end = kRoundsRetry;
      break;
    }
  }
  // out-arcs of the reached vertices
  unsigned long long reached = 0;
  if (!end)
    for (int64_t i = (int64_t)b * kRoundThreads + tid; i < a.n; i += (int64_t)G * kRoundThreads)
      if (agent_load(a.dist + i) != inf) reached += (unsigned long long)(a.row[i + 1] - a.row[i]);
  reached = wave_sum(reached);
  const uint32_t tries = wave_total_dpp(n.tries), wins = wave_total_dpp(n.wins), pushes = wave_total_dpp(n.pushes);
  Counters* c = cnt_of(a.cnt);
  if (lane == 0 && reached) atomicAdd(&c->reached, reached);
  if (lane == SMDP_WAVE - 1) {
    if (tries) atomicAdd(&c->atom_try, (unsigned long long)tries);
    if (wins) atomicAdd(&c->atom_win, (unsigned long long)wins);
    if (pushes) atomicAdd(&c->push[0], (unsigned long long)pushes);
  }
  if (tid == 0) {
    if (edges) atomicAdd(&c->edges, edges);
    if (verts) atomicAdd(&c->verts, verts);
    if (b == 0) atomicMax(&c->rounds, (unsigned long long)r);
    if (end) atomicMax(&c->done, (unsigned long long)end);
  }
}

}  // namespace smdp
