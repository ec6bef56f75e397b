// SSSP and BFS of one graph whose distances stay in LDS for the whole solve:
// by one workgroup (up to kLdsVerts vertices) or by a cluster of k workgroups
// that own kLdsVerts vertices each at most and exchange relaxations of each
// other's vertices through message buffers.
//
// The reference runs every round of a solve as kernels over the whole device
// (apps/sssp/src/sssp_wrapper.cu:147-302).  A round of a small graph is then a
// chain of dependent memory steps (queue entry, offsets, arc, distance,
// atomic, stamp, queue append: 12-20 us on this device, most of them beyond
// L2) that its few arcs cannot hide.  Here distances and the frontier are in
// LDS, and only offsets and arcs are read from memory.
//
// Order.  A round takes the active vertices within `window` of the smallest
// active distance instead of all of them (a sliding delta-stepping bucket).
// The window is 7 * mean weight / mean degree: on uniform graphs of degree
// 4-32 rounds stay about as many and relaxed arcs fall from 2.1-3.6 to
// 1.01-1.14 per arc; on RMAT-10..15 the time is flat in the window (factors
// of 5 to 10 within 5%; 2.6 costs 15-80% more rounds).  The smallest active
// distance is final, so a round settles at least one vertex: at most n rounds
// with work.  Weights must be in [0, 2^30); a solve that reads another one
// ends with kLdsWeight and is left to the unordered rounds.
//
// A vertex is one word x: 2 d + 1 while active, 2 d once expanded, 2^31 when
// unreached.  A candidate d' competes as 2 d' + 1, so one LDS minimum lowers
// the distance and marks the vertex active, a candidate equal to an expanded
// distance loses, and an expansion claims the vertex and reads its distance
// with one LDS and.
//
// Work split.  What bounds a round with many vertices is instruction issue (a
// CU issues about one wave instruction per clock), so the loops are counted
// in instructions per 64 arcs or vertices.  A wave scans every 16th block of
// 256 vertices (four per lane and load), takes the selected ones 64 at a time
// and lays their arcs end to end: a bit per arc marks where a vertex's arcs
// begin, so an arc finds its vertex by counting the marks before it (a binary
// search over offsets was 10 LDS reads per arc).  Vertices of kLdsHeavy arcs
// or more become chunks that all waves share after a barrier; those that find
// no room in a round's list stay active for the next round, which takes only
// the smallest distance, so that it settles a vertex.  (Expanded by the wave
// that found them, they left 15 waves idle: complete graph of 600 vertices 204
// us, now 118; star of 500000 leaves on a cluster of 16 2634, now 448; hub of 4
// million arcs 20.9 ms, now 2.8.)  Graphs of few scan blocks share vertices
// from kLdsHeavyFew arcs on: 255 vertices of 255 arcs 160 us, now 51.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"
#include "smdp_internal.h"

namespace smdp {

constexpr int kLdsThreads = 1024;
constexpr int kLdsWaves = kLdsThreads / SMDP_WAVE;
constexpr int kLdsVerts = 32768;  // vertices of one workgroup: 128 KB of distances
constexpr int kLdsBlock = 256;    // vertices a wave scans at once
constexpr int kLdsIlp = 4;        // arcs per lane and step
constexpr int kLdsStep = kLdsIlp * SMDP_WAVE;
constexpr int kLdsHeavy = 256;    // arcs from which a vertex is cut into chunks for all waves
constexpr int kLdsHeavyFew = 64;  // the same where the scan blocks are too few for the waves: kLdsFew vertices
constexpr int kLdsFew = 4 * kLdsBlock;
constexpr int kLdsChunks = 512;   // such chunks per round
constexpr int kLdsPieces = 128;   // chunks of one vertex, about, at most: of kLdsStep arcs below 32768 arcs, longer above
constexpr int kLdsChunkBits = 17; // of a chunk's arcs
constexpr int kLdsSeg = 2048;     // arcs whose begin bits a wave holds at once
constexpr int kLdsList = SMDP_WAVE + kLdsBlock;  // selected vertices a wave holds
constexpr int kLdsMaxCluster = 16;
constexpr int kLdsSpinLimit = 1 << 21;  // polls before a cluster barrier gives up (about a second)
constexpr float kLdsWindow = 7.0f;
constexpr int32_t kLdsWeightLimit = 1 << 30;
static_assert(kLdsVerts % kLdsBlock == 0 && kLdsVerts <= 65536, "whole blocks, 16-bit local ids");
static_assert(kLdsVerts <= 1 << (32 - kLdsChunkBits), "a chunk's vertex and arcs share a word");
static_assert(kLdsSeg % kLdsStep == 0 && kLdsSeg / 32 == SMDP_WAVE, "one mark word per lane, whole steps");

struct LdsGraph {
  const int32_t* __restrict__ row;  // n + 1 offsets into col and w (row[n] - row[0] < 2^28)
  const int32_t* __restrict__ col;
  const int32_t* __restrict__ w;    // BFS: unused
  int32_t n;
  int32_t src;
  int32_t* out;                     // n distances
  // cluster of k workgroups: workgroup i owns vertices [i * block, (i + 1) * block)
  int32_t block;
  uint32_t inv;                     // ceil(2^32 / block): v * inv >> 32 is v / block or one more
  uint64_t* msg;                    // messages (target << 32 | candidate word), both parities
  const int64_t* moff;              // [k][k]: first message of the pair (sender, receiver), parity 0
  int64_t mtotal;                   // messages of one parity
  uint64_t* flags;                  // [2][k][k]: epoch << 55 | messages << 31 | smallest distance
  // profiling: per counted round (vertices, arcs), then the rounds' starting clocks and the end's (zeroed), or nullptr
  unsigned long long* rlog;
};

struct LdsShared {
  uint32_t x[kLdsVerts];
  int2 ent[kLdsWaves][SMDP_WAVE];        // per entry with arcs: (4 * (first arc - its offset), word)
  uint32_t mark[kLdsWaves][kLdsSeg / 32];
  uint16_t list[kLdsWaves][kLdsList];
  int2 chunk[kLdsChunks];                // (4 * first arc, vertex << kLdsChunkBits | arcs)
  // Round r uses slot r % 3: written during it, read after its last barrier.
  // Fast waves may be a round ahead of the last reader, never two, so slot
  // (r + 1) % 3 is cleared as round r starts.
  int32_t smin[3];                       // smallest active distance left
  int32_t nchunk[3];
  int32_t work[3];                       // one workgroup: a wave relaxed arcs of its own vertices
  int32_t bad[3];                        // a weight outside [0, 2^30) was read
  int32_t mn;                            // cluster: smallest distance anywhere
  int32_t mcnt[kLdsMaxCluster];          // cluster: messages queued for each workgroup this round
  int32_t got[kLdsMaxCluster];           // cluster: messages received from each
  uint64_t* mbase[2][kLdsMaxCluster];    // cluster: message buffers to each, by parity
};
static_assert(sizeof(LdsShared) <= 160 * 1024, "the LDS of a CU");

struct LdsCount {
  uint32_t verts = 0, wins = 0;    // of the wave (the same on every lane)
  unsigned long long edges = 0;    // of the wave
  unsigned long long reached = 0;  // of the lane
};

// Results of a solve below 0.
constexpr int kLdsRoundCap = -1, kLdsTimeout = -2, kLdsWeight = -3;

// Smallest x of the wave, in lane 63.
__device__ __forceinline__ int wave_min_dpp(int x) {
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x111, 0xF, 0xF, false));
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x112, 0xF, 0xF, false));
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x114, 0xF, 0xF, false));
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x118, 0xF, 0xF, false));
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x142, 0xA, 0xF, false));
  x = min(x, __builtin_amdgcn_update_dpp(INT32_MAX, x, 0x143, 0xC, 0xF, false));
  return x;
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lanes [0, cnt) of a wave, for any cnt.
__device__ __forceinline__ uint64_t low_lanes(int cnt) {
  return cnt >= SMDP_WAVE ? ~0ull : cnt <= 0 ? 0ull : (1ull << cnt) - 1;
}

// p[off / 4] with a 32-bit byte offset (scalar base, one vector register).
__device__ __forceinline__ int load_at(const int32_t* p, uint32_t off) {
  return *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(p) + off);
}

// The workgroup of a cluster that owns vertex v < 2^20.
__device__ __forceinline__ int lds_owner(uint32_t v, int32_t block, uint32_t inv) {
  const uint32_t d = (uint32_t)(((uint64_t)v * inv) >> 32);
  return (int)d - (d * (uint32_t)block > v ? 1 : 0);
}

template <bool BFS, bool CL>
struct LdsSolver {
  LdsShared& sh;
  const LdsGraph& g;
  LdsCount& c;
  const int32_t* col;  // at the graph's first arc
  const int32_t* w;
  const int rank, k, lo, nl, lane, wave, row0;
  int rest;       // per lane: smallest word left active, rotated (see round_pass)
  uint32_t low;   // per lane: smallest candidate word that lowered a vertex
  int slot = 0;   // round % 3
  int rounds = 0; // one workgroup: rounds that relaxed an arc, and the first
  int parity = 0;

  __device__ __forceinline__ LdsSolver(LdsShared& s, const LdsGraph& gg, LdsCount& cc, int rank_, int k_)
      : sh(s), g(gg), c(cc), rank(rank_), k(k_), lo(CL ? rank_ * gg.block : 0),
        nl(CL ? max(0, min(gg.block, gg.n - rank_ * gg.block)) : gg.n), lane(lane_id()),
        wave(__builtin_amdgcn_readfirstlane((int)threadIdx.x / SMDP_WAVE)), row0(gg.row[0]) {
    col = gg.col + row0;
    w = BFS ? nullptr : gg.w + row0;
  }

  // Lanes of m offer candidate words a to local vertices lv whose words they
  // read larger: the vertices fall this round, here or through another lane.
  __device__ __forceinline__ void lower(uint64_t m, int lv, uint32_t a) {
    if (!m) return;
    c.wins += __popcll(m);
    if (__builtin_amdgcn_inverse_ballot_w64(m)) {
      __hip_atomic_fetch_min(&sh.x[lv], a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      low = min(low, a);
    }
  }

  // Relaxes a step: lane l's arc t lies at byte offset q[t] (always a valid
  // one) and leaves a vertex whose word is from[t]; it exists if bit l of
  // ok[t] is set.
  __device__ __forceinline__ void step(const uint32_t (&q)[kLdsIlp], const uint32_t (&from)[kLdsIlp],
                                       const uint64_t (&ok)[kLdsIlp]) {
    int v[kLdsIlp];
    uint32_t a[kLdsIlp], cur[kLdsIlp];
#pragma unroll
    for (int t = 0; t < kLdsIlp; ++t) v[t] = load_at(col, q[t]);
    if (BFS) {
#pragma unroll
      for (int t = 0; t < kLdsIlp; ++t) a[t] = from[t] + 2;
    } else {
      int wt[kLdsIlp];
#pragma unroll
      for (int t = 0; t < kLdsIlp; ++t) wt[t] = load_at(w, q[t]);
      int all = 0;
#pragma unroll
      for (int t = 0; t < kLdsIlp; ++t) {
        all |= wt[t];
        a[t] = from[t] + 2 * (uint32_t)wt[t];
      }
      if ((uint32_t)all >= (uint32_t)kLdsWeightLimit) sh.bad[slot] = 1;
    }
#pragma unroll
    for (int t = 0; t < kLdsIlp; ++t) {
      v[t] -= lo;
      if (CL) cur[t] = (uint32_t)v[t] < (uint32_t)nl ? sh.x[v[t]] : 0u;
      else cur[t] = sh.x[v[t]];
    }
#pragma unroll
    for (int t = 0; t < kLdsIlp; ++t) lower(__builtin_amdgcn_ballot_w64(a[t] < cur[t]) & ok[t], v[t], a[t]);
    if (CL) send(v, a, ok);
  }

  // Messages of a cluster: candidates for other workgroups' vertices.  Every
  // lane takes its own place in its receiver's buffer (a loop over the
  // receivers present, one LDS atomic each, cost 16 of them per 64 arcs in a
  // cluster of 16).
  __device__ __forceinline__ void send(const int (&lv)[kLdsIlp], const uint32_t (&a)[kLdsIlp],
                                       const uint64_t (&ok)[kLdsIlp]) {
    uint64_t m[kLdsIlp];
    int at[kLdsIlp], dest[kLdsIlp];
#pragma unroll
    for (int t = 0; t < kLdsIlp; ++t) {
      // (a candidate at or beyond the unreached word lowers nothing)
      m[t] = __builtin_amdgcn_ballot_w64((uint32_t)lv[t] >= (uint32_t)nl && a[t] < (uint32_t)SMDP_SSSP_INF * 2) & ok[t];
      dest[t] = at[t] = 0;
      if (__builtin_amdgcn_inverse_ballot_w64(m[t])) {
        low = min(low, a[t]);
        dest[t] = lds_owner((uint32_t)(lv[t] + lo), g.block, g.inv);
        at[t] = __hip_atomic_fetch_add(&sh.mcnt[dest[t]], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
#pragma unroll
    for (int t = 0; t < kLdsIlp; ++t)
      if (__builtin_amdgcn_inverse_ballot_w64(m[t]))
        __hip_atomic_store(sh.mbase[parity][dest[t]] + at[t], (uint64_t)(uint32_t)(lv[t] + lo) << 32 | a[t],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // Expands the last `cnt` (<= 64) entries of the wave's list of length `n`.
  __device__ __forceinline__ void expand(int n, int cnt) {
    wave_lds_sync();
    int s = 0, deg = 0, u = 0;
    uint32_t x = 0;
    if (lane < cnt) {
      u = sh.list[wave][n - cnt + lane];
      s = load_at(g.row, 4 * (uint32_t)(lo + u));
      deg = load_at(g.row, 4 * (uint32_t)(lo + u) + 4) - s;
      s -= row0;
      // claims the vertex: lowered from here on it is active again
      x = __hip_atomic_fetch_and(&sh.x[u], ~1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    bool back = false;
    if (deg >= (nl <= kLdsFew ? kLdsHeavyFew : kLdsHeavy)) {
      const int steps = (deg + kLdsStep - 1) / kLdsStep;
      constexpr int kMost = ((1 << kLdsChunkBits) - 1) / kLdsStep;
      const int each = steps <= kLdsPieces ? 1 : min((steps + kLdsPieces - 1) / kLdsPieces, kMost);
      const int nch = each == 1 ? steps : (steps + each - 1) / each, len = each * kLdsStep;
      const int at = __hip_atomic_fetch_add(&sh.nchunk[slot], nch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (at + nch <= kLdsChunks) {
        for (int i = 0; i < nch; ++i)
          sh.chunk[at + i] =
              make_int2(4 * (s + i * len), (int)((uint32_t)u << kLdsChunkBits) | min(len, deg - i * len));
      } else {
        // no room: active again, and the slots below the limit stay empty
        for (int i = at; i < kLdsChunks; ++i) sh.chunk[i] = make_int2(4 * s, 0);
        __hip_atomic_fetch_or(&sh.x[u], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        low = min(low, x | 1u);
        back = true;
      }
      deg = 0;
    }
    c.verts += cnt - __popcll(__builtin_amdgcn_ballot_w64(back));
    const int incl = wave_scan_dpp(deg);
    const int off = incl - deg;
    const int T = __builtin_amdgcn_readlane(incl, SMDP_WAVE - 1);
    c.edges += T;
    const bool has = deg > 0;
    if (has) sh.ent[wave][mbcnt(__builtin_amdgcn_ballot_w64(has))] = make_int2(4 * (s - off), (int)x);
    // An entry's begin is marked one place early (the first one's not at
    // all), so the entry of arc j is the number of marks before j.
    for (int seg = 0; seg < T; seg += kLdsSeg) {
      sh.mark[wave][lane] = 0;
      wave_lds_sync();
      const int at = off - 1 - seg;
      const bool begins = has && off > 0;
      if (begins && (uint32_t)at < (uint32_t)kLdsSeg)
        __hip_atomic_fetch_or(&sh.mark[wave][at >> 5], 1u << (at & 31), __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_WORKGROUP);
      int first = __popcll(__builtin_amdgcn_ballot_w64(begins && at < 0));  // marks before the window
      wave_lds_sync();
      const int send_ = min(T, seg + kLdsSeg);
      for (int p = seg; p < send_; p += kLdsStep) {
        uint32_t q[kLdsIlp], from[kLdsIlp];
        uint64_t ok[kLdsIlp], mk[kLdsIlp];
#pragma unroll
        for (int t = 0; t < kLdsIlp; ++t)
          mk[t] = *reinterpret_cast<const uint64_t*>(&sh.mark[wave][(p - seg) / 32 + 2 * t]);
#pragma unroll
        for (int t = 0; t < kLdsIlp; ++t) {
          const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)mk[t]) |
                             (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(mk[t] >> 32)) << 32;
          const int2 en = sh.ent[wave][first + mbcnt(m)];
          first += __popcll(m);
          ok[t] = low_lanes(send_ - p - t * SMDP_WAVE);
          q[t] = (uint32_t)en.x + 4 * (uint32_t)min(p + t * SMDP_WAVE + lane, T - 1);
          from[t] = (uint32_t)en.y;
        }
        step(q, from, ok);
      }
      wave_lds_sync();  // mark and ent are read before they are written again
    }
  }

  // The wave's vertices: expands the active ones below thr.  Rotated right by
  // one bit a word is d - 2^31 when active and not negative when not, so one
  // signed compare selects.
  __device__ __forceinline__ void round_pass(int thr) {
    const int lim = (int)((uint32_t)thr ^ 0x80000000u);
    int n = 0, b = wave * kLdsBlock;
    // (one call of expand(): inlined at several places its code did not stay
    // in the instruction cache)
    for (;;) {
      for (; b < nl && n <= SMDP_WAVE; b += kLdsWaves * kLdsBlock) {
        const uint4 xx = *reinterpret_cast<const uint4*>(&sh.x[b + 4 * lane]);
        const uint32_t x[4] = {xx.x, xx.y, xx.z, xx.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = (int)__builtin_amdgcn_alignbit(x[i], x[i], 1);
          const bool sel = r < lim;
          const uint64_t sm = __builtin_amdgcn_ballot_w64(sel);
          rest = min(rest, sel ? INT32_MAX : r);
          if (sm) {
            if (sel) sh.list[wave][n + mbcnt(sm)] = (uint16_t)(b + 4 * lane + i);
            n += __popcll(sm);
          }
        }
      }
      if (!n) break;
      const int cnt = min(n, SMDP_WAVE);
      expand(n, cnt);
      n -= cnt;
    }
  }

  // Chunks of the round's heavy vertices, one wave each.
  __device__ __forceinline__ void chunk_pass(int nch) {
    for (int h = wave; h < nch; h += kLdsWaves) {
      const int2 ch = sh.chunk[h];
      const int len = __builtin_amdgcn_readfirstlane(ch.y & ((1 << kLdsChunkBits) - 1));
      if (!len) continue;
      const uint32_t x = sh.x[(uint32_t)ch.y >> kLdsChunkBits] | 1u;
      c.edges += len;
      for (int o = 0; o < len; o += kLdsStep) {
        uint32_t q[kLdsIlp], from[kLdsIlp];
        uint64_t ok[kLdsIlp];
#pragma unroll
        for (int t = 0; t < kLdsIlp; ++t) {
          ok[t] = low_lanes(len - o - t * SMDP_WAVE);
          q[t] = (uint32_t)ch.x + 4 * (uint32_t)min(o + t * SMDP_WAVE + lane, len - 1);
          from[t] = x;
        }
        step(q, from, ok);
      }
    }
  }

  // The smallest active distance this wave knows of, into the round's slot.
  __device__ __forceinline__ void publish_min() {
    const int a = rest < 0 ? (int)((uint32_t)rest ^ 0x80000000u) : INT32_MAX;
    const int m = wave_min_dpp(min(a, (int)(low >> 1)));
    if (lane == SMDP_WAVE - 1 && m != INT32_MAX)
      __hip_atomic_fetch_min(&sh.smin[slot], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    rest = INT32_MAX;
    low = UINT32_MAX;
  }

  // Window of the solve: the mean of 1024 weights spread over the arcs.
  __device__ __forceinline__ int window(int* s_sum) {
    if (BFS) return 1;
    const int m = g.row[g.n] - row0;
    if (m <= 0) return 1;
    // summed in two halves: weights go up to 2^30 (a mean held to 2^20 made the
    // window of larger ones so narrow that uniform 16384 x 8 with weights up to
    // 2^28 took 1300 us, against 470 in unordered rounds and 127 now)
    const int x = max(0, min(w[(int64_t)m * threadIdx.x / kLdsThreads], kLdsWeightLimit));
    const int high = wave_scan_dpp(x >> 12), part = wave_scan_dpp(x & 0xFFF);
    if (lane == SMDP_WAVE - 1) s_sum[wave] = __float_as_int((float)high * 4096.f + (float)part);
    __syncthreads();
    float mean = 0.f;
    for (int i = 0; i < kLdsWaves; ++i) mean += __int_as_float(s_sum[i]) / (float)kLdsThreads;
    __syncthreads();
    return (int)fminf(fmaxf(kLdsWindow * mean * (float)g.n / (float)m, 1.f), (float)kLdsWeightLimit);
  }

  // Cluster: publishes this round's message counts and smallest distance,
  // waits for the others', and applies the messages sent here.  Returns the
  // smallest distance anywhere, or -1 when a workgroup did not come.
  // Messages and flags are stored and read device-coherent, and each wave
  // waits for its stores before the flags are written, so no agent-scope
  // fence is needed.  A parity's buffers are written again two rounds later,
  // after every receiver stored the flags of the round between.
  __device__ __forceinline__ int exchange(int r, int mn) {
    const uint64_t epoch = (uint64_t)((r + 1) & 511);
    uint64_t* f = g.flags + parity * k * k;
    if (wave == 0) {
      if (lane < k)
        __hip_atomic_store(f + rank * k + lane, epoch << 55 | (uint64_t)(uint32_t)sh.mcnt[lane] << 31 | (uint64_t)mn,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      uint64_t v = 0;
      bool ok = true;
      for (int spins = 0;;) {
        v = lane < k ? __hip_atomic_load(f + lane * k + rank, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                     : epoch << 55;
        if (__builtin_amdgcn_ballot_w64(v >> 55 != epoch) == 0) break;
        __builtin_amdgcn_s_sleep(1);
        if (++spins > kLdsSpinLimit) {
          ok = false;
          break;
        }
      }
      const int m = wave_min_dpp(lane < k ? (int)(v & 0x7FFFFFFF) : INT32_MAX);
      if (lane < k) {
        sh.got[lane] = (int)((v >> 31) & 0xFFFFFF);
        sh.mcnt[lane] = 0;
      }
      if (lane == SMDP_WAVE - 1) sh.mn = ok ? m : -1;
    }
    __syncthreads();
    const int gmin = sh.mn;
    if (gmin < 0 || gmin == INT32_MAX) return gmin;
    for (int j = 0; j < k; ++j) {
      if (j == rank) continue;
      const int cnt = sh.got[j];
      const uint64_t* in = g.msg + parity * g.mtotal + g.moff[j * k + rank];
      for (int b = 0; b < cnt; b += kLdsIlp * kLdsThreads) {
        uint64_t ms[kLdsIlp];
#pragma unroll
        for (int t = 0; t < kLdsIlp; ++t)
          ms[t] = __hip_atomic_load(in + min(b + t * kLdsThreads + (int)threadIdx.x, cnt - 1), __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int t = 0; t < kLdsIlp; ++t) {
          const int lv = (int)(ms[t] >> 32) - lo;
          const uint32_t a = (uint32_t)ms[t];  // (a repeated last message changes nothing)
          lower(__builtin_amdgcn_ballot_w64(a < sh.x[lv]), lv, a);
        }
      }
    }
    low = UINT32_MAX;  // the senders counted these candidates
    __syncthreads();
    parity ^= 1;
    return gmin;
  }

  // Profiling: the wave's part of the last counted round (one without arcs
  // joins the one before).
  __device__ __forceinline__ void log_round(uint32_t verts0, unsigned long long edges0) {
    if (rounds > kRoundLogCap || lane != 0) return;
    const unsigned long long by[2] = {c.verts - verts0, c.edges - edges0};
    for (int i = 0; i < 2; ++i)
      if (by[i])
        __hip_atomic_fetch_add(&g.rlog[2 * (rounds - 1) + i], by[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ void log_clock() {
    if (rounds < kRoundLogCap && threadIdx.x == 0 && !g.rlog[2 * kRoundLogCap + rounds])
      g.rlog[2 * kRoundLogCap + rounds] = wall_clock64();
  }

  // The solve; returns the rounds run or a result below 0.
  __device__ __forceinline__ int solve() {
    const int tid = threadIdx.x;
    const uint32_t inf = (uint32_t)SMDP_SSSP_INF * 2;
    // whole blocks: the words past nl stay unreached
    for (int i = tid; i < (nl + kLdsBlock - 1) / kLdsBlock * kLdsBlock; i += kLdsThreads) sh.x[i] = inf;
    if (tid < kLdsMaxCluster) sh.mcnt[tid] = 0;
    if (CL && tid < k) {
      sh.mbase[0][tid] = g.msg + g.moff[rank * k + tid];
      sh.mbase[1][tid] = sh.mbase[0][tid] + g.mtotal;
    }
    if (tid < 3) {
      sh.smin[tid] = INT32_MAX;
      sh.nchunk[tid] = 0;
      sh.work[tid] = 0;
      sh.bad[tid] = 0;
    }
    const int win = window(sh.got);
    __syncthreads();
    if (tid == 0 && (uint32_t)(g.src - lo) < (uint32_t)nl) sh.x[g.src - lo] = 1;  // distance 0, active
    __syncthreads();
    int thr = win;  // the source's distance is 0
    rest = INT32_MAX;
    low = UINT32_MAX;
    int r = 0;
    for (;; ++r) {
      // rounds that settle a vertex number at most n; after each there may be
      // one that overflowed the list of chunks, or in a cluster one that found
      // only candidates that lowered nothing
      if (r > (CL ? 4 : 2) * g.n + 2) return kLdsRoundCap;
      slot = r % 3;
      if (tid == 0) {
        const int next = (r + 1) % 3;
        sh.smin[next] = INT32_MAX;
        sh.nchunk[next] = 0;
        sh.work[next] = 0;
      }
      const uint32_t verts0 = c.verts;
      const unsigned long long edges0 = c.edges;
      if (!CL && g.rlog) log_clock();
      round_pass(thr);
      if (!CL && c.edges != edges0) sh.work[slot] = 1;
      publish_min();
      if (CL) __builtin_amdgcn_s_waitcnt(0);  // this wave's messages are stored
      __syncthreads();
      const int listed = sh.nchunk[slot];
      if (listed) {
        chunk_pass(min(listed, kLdsChunks));
        publish_min();
        if (CL) __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
      }
      if (!CL) {
        // (vertices without arcs are not queued in rounds of other kinds, and make no round here)
        if (r == 0 || listed || sh.work[slot]) ++rounds;
        if (g.rlog) log_round(verts0, edges0);
      }
      int mn = sh.smin[slot];
      if (!BFS && !CL && sh.bad[slot]) return kLdsWeight;  // (clusters are given weights in range)
      if (CL) {
        mn = exchange(r, mn);
        if (mn < 0) return kLdsTimeout;
      }
      if (mn == INT32_MAX) break;
      thr = min(mn + (listed > kLdsChunks ? 1 : win), SMDP_SSSP_INF);
    }
    if (!CL && g.rlog) log_clock();
    for (int i = tid; i < nl; i += kLdsThreads) {
      const uint32_t x = sh.x[i];
      g.out[lo + i] = x == inf ? (BFS ? SMDP_BFS_UNDEF : SMDP_SSSP_INF) : (int)(x >> 1);
      if (x != inf) c.reached += (unsigned long long)(g.row[lo + i + 1] - g.row[lo + i]);
    }
    return r + 1;
  }
};

}  // namespace smdp
