// Merge-path CSR SpMV, the tuned solution of y = A x.
//
// The rows' end offsets and the nonzeros form one merged sequence of n + m
// items (a row end comes before nonzero j when the row ends at or before j).
// Every workgroup takes kMpItems consecutive items of it, so the work per
// workgroup is the same whatever the row lengths: no row is too long for a
// workgroup and no workgroup waits on one long row.  This is the published
// merge-based SpMV (Merrill and Garland, "Merge-based parallel sparse matrix-
// vector multiplication", SC16), built here for 64-lane waves:
//
//  * the tile's nonzeros are multiplied with all x gathers of a thread in
//    flight and the products (with their rounding errors) staged in LDS,
//  * each thread walks kMpT items of the tile with a compensated sum,
//  * a row crossing threads is finished by the thread that reaches its end,
//    which merges the partial sums of the threads before it in thread order,
//  * a row crossing tiles is finished by k_merge_fixup, which merges the tile
//    partials in tile order.
//
// Every row is summed in an order fixed by the matrix alone, so results are
// identical from run to run.  Replaces csr_spmv_* (SpMV_kernel.cu:81-403) for
// the tuned solution.
//
// A PageRank iteration over the plain in-CSR is the same reduction without
// values (k_pr_merge): the tile's row sums go to LDS, the epilogue of its rows
// runs coalesced, and the last workgroup finishes the rows that cross tiles
// and applies the stop rule, so an iteration is one launch.  It replaces
// pagerank_* (pagerank_kernel.cu:95-601) on graphs below the binned layout's
// size.

#include <algorithm>
#include <vector>

#include "rowreduce.h"

namespace smdp {
namespace {

constexpr int kMpNT = 256;                // threads per workgroup
// Merge items per thread of a product: kMpBig where the tiles fill the device
// many times over, kMpSmall where they would not (see items_per_thread).
constexpr int kMpBig = 16;
constexpr int kMpSmall = 4;

struct MergePlan {
  int32_t items = 0;             // merge items per tile
  int32_t* tstart = nullptr;     // ntiles + 1: row ends before each tile's first item
  int32_t* pcol = nullptr;       // m: the columns renumbered by falling in-degree (ties by id)
  int32_t* perm = nullptr;       // n: renumbered column -> original column
  float* xp = nullptr;           // n: x in the renumbered order, of the columns that occur
  int32_t ncols = 0;             // columns that occur in the matrix (the first ncols renumbered ids)
  float2* carry = nullptr;       // per tile: partial sum of the row open at its end
  float2* head = nullptr;        // per tile: its part of a row begun in an earlier tile and ended in it
  int32_t* head_row = nullptr;   // per tile: that row, or -1
  double2* part = nullptr;       // PageRank, per tile: (residual, dangling)
  int32_t ntiles = 0;
  int32_t n = -1;
  int32_t m = -1;
};

struct MArgs {
  const int32_t* __restrict__ row;
  const int32_t* __restrict__ col;
  const float* __restrict__ val;
  const float* __restrict__ x;
  float* y;
  const int32_t* __restrict__ tstart;
  float2* carry;
  float2* head;
  int32_t* head_row;
  Counters* cnt;
  int32_t n, m, ntiles, items;
};

// Items per thread of a matrix with `total` = n + m merge items.  A tile of
// kMpSmall * 256 items has a quarter of the serial work of a kMpBig one but
// pays the tile's fixed steps four times as often: SpMV on 900K items (220 or
// 880 tiles on 256 CUs) took 87.8 us a call with kMpBig and 83.7 with kMpSmall;
// on 17.8M items kMpBig is the faster (0.102 against 0.136 ms).  The line is
// two kMpBig tiles per CU.
int items_per_thread(int64_t total, int cus) {
  return total <= (int64_t)cus * kMpNT * kMpBig * 2 ? kMpSmall : kMpBig;
}

// The same for a PageRank iteration, which every workgroup ends with a fence
// and a ticket, so fewer and larger tiles pay earlier.  Microseconds an
// iteration with 4, 8, 16 and 32 items: 74K items 13.5, 13.9, 17.1, 23.2; 147K
// 14.9, 14.6, 17.8, 24.2; 279K 18.7, 16.3, 17.7, 23.7; 557K 27.6, 21.6, 19.9,
// 24.4; 1.11M 52.8, 34.7, 25.5, 27.2; 2.23M 99.7, 62.9, 37.8, 34.0; 4.46M 153,
// 121, 79.7, 60.8.
int items_per_thread_pr(int64_t total, int cus) {
  if (total <= 550 * (int64_t)cus) return 4;
  if (total <= 1600 * (int64_t)cus) return 8;
  return total <= 5000 * (int64_t)cus ? 16 : 32;
}

// Number of row ends among the first d merge items: the smallest i with
// end(i) > d - i - 1, searched in [max(0, d - nz), min(d, nr)].
template <typename End>
__device__ __forceinline__ int64_t merge_search(End end, int64_t d, int64_t nr, int64_t nz) {
  int64_t lo = d - nz > 0 ? d - nz : 0;
  int64_t hi = d < nr ? d : nr;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (end(mid) <= d - mid - 1) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__global__ void k_merge_starts(const int32_t* __restrict__ row, int32_t n, int32_t m, int32_t ntiles,
                               int32_t items, int32_t* tstart) {
  const int64_t total = (int64_t)n + m;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t <= ntiles; t += gridDim.x * blockDim.x) {
    const int64_t d = (int64_t)t * items < total ? (int64_t)t * items : total;
    tstart[t] = (int32_t)merge_search([&](int64_t i) { return (int64_t)row[i + 1]; }, d, n, m);
  }
}

// Inclusive segmented scan of the threads' open sums: every thread gets the
// sum of its row's partials (rows are the keys, which do not decrease from
// thread to thread, so the threads ending inside one row are consecutive)
// from the first of those threads up to itself: six shuffle steps in the
// wave, then the tails of at most three earlier waves.  The combination order
// is fixed.  All threads; the three arrays hold one entry per wave.
__device__ __forceinline__ CSum open_row_scan(int key, CSum sc, int32_t* s_hk, int32_t* s_tk, float2* s_tv) {
  const int lane = lane_id(), wave = threadIdx.x / SMDP_WAVE;
#pragma unroll
  for (int d = 1; d < SMDP_WAVE; d <<= 1) {
    const int k2 = __shfl_up(key, d);
    CSum o;
    o.s = __shfl_up(sc.s, d);
    o.c = __shfl_up(sc.c, d);
    if (lane >= d && k2 == key) {
      o.merge(sc);
      sc = o;
    }
  }
  if (lane == 0) s_hk[wave] = key;
  if (lane == SMDP_WAVE - 1) {
    s_tk[wave] = key;
    s_tv[wave] = make_float2(sc.s, sc.c);
  }
  __syncthreads();
  if (key == s_hk[wave]) {
    int v = wave;
    while (v > 0 && s_tk[v - 1] == key) {
      --v;
      if (s_hk[v] != key) break;
    }
    if (v < wave) {
      CSum pre;
      for (int u = v; u < wave; ++u) {
        CSum o;
        o.s = s_tv[u].x;
        o.c = s_tv[u].y;
        pre.merge(o);
      }
      pre.merge(sc);
      sc = pre;
    }
  }
  return sc;
}

// Sum of row r (below 0: none), which began before tile t and ends in it: the
// partials of the tiles it crosses, in tile order, then tile t's part.  All
// lanes of a wave, a row each.  The row's first arc is merge item r + row[r],
// which names the first of those tiles.  A row over more than kCross of them is
// merged by the whole wave, in an order that depends on the matrix alone; by one
// lane, which waited for one partial after another and to find the first, twice
// (a row of 10^6 nonzeros in tiles of 1024 items took 236 us a product, now
// 44; PageRank with a row of 4 x 10^6 131 us an iteration, now 33).
constexpr int kCross = 16;
__device__ __forceinline__ CSum crossing_row(const int32_t* row, int64_t items, const float2* carry,
                                             const float2* head, int t, int r) {
  auto part = [](float2 v) {
    CSum o;
    o.s = v.x;
    o.c = v.y;
    return o;
  };
  const int k = r >= 0 ? (int)((r + (int64_t)row[r]) / items) : t;
  const bool far = t - k > kCross;
  CSum tot;
  if (!far && k < t) {
    float2 v[kCross];
#pragma unroll
    for (int u = 0; u < kCross; ++u) v[u] = carry[min(k + u, t - 1)];
#pragma unroll
    for (int u = 0; u < kCross; ++u)
      if (k + u < t) tot.merge(part(v[u]));
  }
  for (uint64_t m = ballot(far); m; m &= m - 1) {
    const int l = first_lane(m);
    const int q0 = __shfl(k, l), q1 = __shfl(t, l);
    CSum sum;
    for (int q = q0 + lane_id(); q < q1; q += kCross * SMDP_WAVE) {
      float2 v[kCross];
#pragma unroll
      for (int u = 0; u < kCross; ++u) v[u] = carry[min(q + u * SMDP_WAVE, q1 - 1)];
#pragma unroll
      for (int u = 0; u < kCross; ++u)
        if (q + u * SMDP_WAVE < q1) sum.merge(part(v[u]));
    }
    sum = wave_csum_dpp(sum);
    if (lane_id() == l) tot = sum;
  }
  if (r >= 0) tot.merge(part(head[t]));
  return tot;
}

template <int kMpT>
__global__ __launch_bounds__(kMpNT) void k_spmv_merge(MArgs a) {
  constexpr int kMpItems = kMpNT * kMpT;
  // The tile's nr row ends and nz nonzeros fill its kMpItems merge items, so
  // one array holds both: slot k < nr the end of row i0 + k (in tile nonzero
  // positions, as int bits in .x), slot nr + j the product of nonzero j and
  // its rounding error.  At 16 items per thread, 34 KB of LDS per workgroup: 4 workgroups per CU.
  __shared__ float2 s_item[kMpItems];
  __shared__ float2 s_cs[kMpNT];       // per thread: partial sum of its open row, scanned over the row's threads
  __shared__ int32_t s_hk[kMpNT / SMDP_WAVE], s_tk[kMpNT / SMDP_WAVE];  // per wave: open row of lanes 0 and 63
  __shared__ float2 s_tv[kMpNT / SMDP_WAVE];                           // per wave: scanned sum of lane 63
  const int tid = threadIdx.x;
  const int t = blockIdx.x;
  const int64_t d0 = (int64_t)t * kMpItems;
  const int64_t dn = (int64_t)a.n + a.m;
  const int64_t d1 = d0 + kMpItems < dn ? d0 + kMpItems : dn;
  const int i0 = a.tstart[t], i1 = a.tstart[t + 1];
  const int j0 = (int)(d0 - i0), j1 = (int)(d1 - i1);
  const int nr = i1 - i0, nz = j1 - j0;
  // the tile's first row began in an earlier tile
  const bool mid_row = i0 < a.n && a.row[i0] < j0;
  if (tid == 0) {
    a.head_row[t] = (mid_row && nr > 0) ? i0 : -1;
    Counters* c = cnt_of(a.cnt);
    if (nz) atomicAdd(&c->edges, (unsigned long long)nz);
    if (nr) atomicAdd(&c->verts, (unsigned long long)nr);
  }
  // Every load of the tile is issued before the first one is used.  Loads go
  // to clamped positions inside the tile (the branches on nz and nr are the
  // same for the whole workgroup): a load under a per-lane condition would
  // make the compiler wait for it before the other lanes' default value is
  // written to the same register.
  if (nz > 0) {
    int c[kMpT], re[kMpT];
    float v[kMpT], xv[kMpT];
#pragma unroll
    for (int u = 0; u < kMpT; ++u) {
      const int k = min(tid + u * kMpNT, nz - 1);
      c[u] = stream_load(a.col + j0 + k);
      v[u] = stream_load(a.val + j0 + k);
    }
    if (nr > 0) {
#pragma unroll
      for (int u = 0; u < kMpT; ++u) re[u] = a.row[i0 + min(tid + u * kMpNT, nr - 1) + 1];
    }
#pragma unroll
    for (int u = 0; u < kMpT; ++u) xv[u] = a.x[c[u]];
    if (nr > 0) {
#pragma unroll
      for (int u = 0; u < kMpT; ++u) {
        const int k = tid + u * kMpNT;
        if (k < nr) s_item[k].x = __int_as_float(re[u] - j0);
      }
    }
#pragma unroll
    for (int u = 0; u < kMpT; ++u) {
      const int k = tid + u * kMpNT;
      if (k < nz) {
#pragma clang fp contract(off)
        const float p = v[u] * xv[u];
        s_item[nr + k] = make_float2(p, __builtin_fmaf(v[u], xv[u], -p));
      }
    }
  } else if (nr > 0) {
    int re[kMpT];
#pragma unroll
    for (int u = 0; u < kMpT; ++u) re[u] = a.row[i0 + min(tid + u * kMpNT, nr - 1) + 1];
#pragma unroll
    for (int u = 0; u < kMpT; ++u) {
      const int k = tid + u * kMpNT;
      if (k < nr) s_item[k].x = __int_as_float(re[u] - j0);
    }
  }
  __syncthreads();

  const int dl = min(tid * kMpT, nr + nz), dr = min(dl + kMpT, nr + nz);
  int ri;
  {
    int lo = max(0, dl - nz), hi = min(dl, nr);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (__float_as_int(s_item[mid].x) <= dl - mid - 1) lo = mid + 1;
      else hi = mid;
    }
    ri = lo;
  }
  int zi = dl - ri;
  const int rfirst = ri;
  CSum acc, fpart;
  bool fdone = false;
  for (int q = dl; q < dr; ++q) {
    if (ri < nr && __float_as_int(s_item[ri].x) <= zi) {
      if (ri == rfirst) {
        fpart = acc;
        fdone = true;
      } else {
        a.y[i0 + ri] = acc.value();
      }
      acc = CSum();
      ++ri;
    } else {
      const float2 pe = s_item[nr + zi];
      acc.add(pe.x);
      acc.c += pe.y;
      ++zi;
    }
  }
  const CSum sc = open_row_scan(ri, acc, s_hk, s_tk, s_tv);
  s_cs[tid] = make_float2(sc.s, sc.c);
  __syncthreads();

  if (fdone) {
    // thread tid - 1 ended inside rfirst: its scanned sum holds every earlier
    // thread's part of the row
    CSum tot;
    if (tid > 0) {
      tot.s = s_cs[tid - 1].x;
      tot.c = s_cs[tid - 1].y;
    }
    tot.merge(fpart);
    if (rfirst == 0 && mid_row) a.head[t] = make_float2(tot.s, tot.c);
    else a.y[i0 + rfirst] = tot.value();
  }
  if (tid == kMpNT - 1) {
    a.carry[t] = make_float2(sc.s, sc.c);
  }
}

// Column renumbering.  RMAT columns are heavy-tailed: on RMAT-20 the 8192
// most frequent columns (32 KB of x) take 48.5% of the nonzeros and 48% of
// the columns never occur.  Numbered by falling in-degree, the frequent x
// values share a few cache lines that stay in each CU's L1, instead of one
// line each.  Every product and every row's order are unchanged, so y is
// bit for bit the same as with the original columns.
__global__ void k_col_degree(const int32_t* __restrict__ col, int64_t m, int32_t* deg) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += (int64_t)gridDim.x * blockDim.x)
    __hip_atomic_fetch_add(deg + col[e], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_renumber_cols(const int32_t* __restrict__ col, int64_t m, const int32_t* __restrict__ inv,
                                int32_t* __restrict__ pcol) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += (int64_t)gridDim.x * blockDim.x)
    pcol[e] = inv[col[e]];
}

// xp[i] = x[perm[i]] for the ncols columns that occur; workgroup 0 also clears
// the counters that the product adds to.
__global__ void k_permute_x(const float* __restrict__ x, const int32_t* __restrict__ perm, int32_t ncols,
                            float* __restrict__ xp, Counters* cnt) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ncols; i += gridDim.x * blockDim.x) xp[i] = x[perm[i]];
  if (blockIdx.x == 0) {
    unsigned long long* c = reinterpret_cast<unsigned long long*>(cnt);
    for (int i = threadIdx.x; i < (int)(kCntParts * sizeof(Counters) / 8); i += blockDim.x) c[i] = 0;
  }
}

// Rows that began in an earlier tile (whole waves, see crossing_row).
__global__ void k_merge_fixup(MArgs a) {
  for (int t0 = blockIdx.x * blockDim.x; t0 < a.ntiles; t0 += gridDim.x * blockDim.x) {
    const int t = t0 + threadIdx.x;
    const int r = t < a.ntiles ? a.head_row[t] : -1;
    const CSum tot = crossing_row(a.row, a.items, a.carry, a.head, t, r);
    if (r >= 0) a.y[r] = tot.value();
  }
}

// One PageRank iteration: tiles of the merged sequence of the in-CSR's row
// ends and arcs, grid-stride over the launch (the ticket that ends an
// iteration is one address, so the launch is held to a few workgroups per
// CU).  The tile's arcs gather their sources' contributions; rows' sums are
// collected in LDS and their epilogue (rank, contribution, FP64 residual and
// dangling mass) runs one row per thread with the old ranks and degrees
// loaded at the tile's start.
//
// What bounds it below 2^20 arcs is the chain of one tile (row ends, columns,
// gathers, walk, scan, epilogue) and the launch, not bytes: 262K arcs and 16K
// rows take 16 us an iteration.  The row-tile kernel it replaces took 157 us
// there: 64 tiles of 256 rows on 64 of the 256 CUs, with each row of 64 or
// more arcs summed by one wave after another.  A drop-in PageRank of RMAT-14
// went from 2.55 to 0.43 ms.
template <int kMpT>
__global__ __launch_bounds__(kMpNT) void k_pr_merge(RArgs a, MArgs p, int k) {
  if (a.st->done) return;
  constexpr int kMpItems = kMpNT * kMpT;
  __shared__ int32_t s_item[kMpItems];  // slots < nr: row ends; then the arcs' contributions (float bits)
  __shared__ float s_sum[kMpItems];     // row sums of the tile
  __shared__ float2 s_cs[kMpNT];
  __shared__ int32_t s_hk[kMpNT / SMDP_WAVE], s_tk[kMpNT / SMDP_WAVE];
  __shared__ float2 s_tv[kMpNT / SMDP_WAVE];
  __shared__ double2 s_red2[kMpNT / SMDP_WAVE];
  __shared__ int s_last;
  const float base = iteration_base(a, k);
  const int tid = threadIdx.x;
  const int64_t dn = (int64_t)p.n + p.m;
  unsigned long long edges = 0, rows = 0;
  for (int t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    const int64_t d0 = (int64_t)t * kMpItems;
    const int64_t d1 = d0 + kMpItems < dn ? d0 + kMpItems : dn;
    const int i0 = p.tstart[t], i1 = p.tstart[t + 1];
    const int j0 = (int)(d0 - i0), j1 = (int)(d1 - i1);
    const int nr = i1 - i0, nz = j1 - j0;
    const bool mid_row = i0 < p.n && a.row[i0] < j0;
    edges += nz;
    rows += nr;
    if (tid == 0) p.head_row[t] = (mid_row && nr > 0) ? i0 : -1;
    float rold[kMpT];
    int od[kMpT];
    // every load at a clamped position, issued before the first use
    if (nr > 0) {
      int re[kMpT];
#pragma unroll
      for (int u = 0; u < kMpT; ++u) {
        const int q = i0 + min(tid + u * kMpNT, nr - 1);
        re[u] = a.row[q + 1];
        rold[u] = a.rold[q];
        od[u] = a.outdeg[q];
      }
#pragma unroll
      for (int u = 0; u < kMpT; ++u) {
        const int q = tid + u * kMpNT;
        if (q < nr) s_item[q] = re[u] - j0;
      }
    }
    if (nz > 0) {
      int c[kMpT];
      float xv[kMpT];
#pragma unroll
      for (int u = 0; u < kMpT; ++u) c[u] = a.col[j0 + min(tid + u * kMpNT, nz - 1)];
#pragma unroll
      for (int u = 0; u < kMpT; ++u) xv[u] = a.x[c[u]];
#pragma unroll
      for (int u = 0; u < kMpT; ++u) {
        const int q = tid + u * kMpNT;
        if (q < nz) s_item[nr + q] = __float_as_int(xv[u]);
      }
    }
    __syncthreads();

    const int dl = min(tid * kMpT, nr + nz), dr = min(dl + kMpT, nr + nz);
    int ri;
    {
      int lo = max(0, dl - nz), hi = min(dl, nr);
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s_item[mid] <= dl - mid - 1) lo = mid + 1;
        else hi = mid;
      }
      ri = lo;
    }
    int zi = dl - ri;
    const int rfirst = ri;
    CSum acc, fpart;
    bool fdone = false;
    for (int q = dl; q < dr; ++q) {
      if (ri < nr && s_item[ri] <= zi) {
        if (ri == rfirst) {
          fpart = acc;
          fdone = true;
        } else {
          s_sum[ri] = acc.value();
        }
        acc = CSum();
        ++ri;
      } else {
        acc.add(__int_as_float(s_item[nr + zi]));
        ++zi;
      }
    }
    const CSum sc = open_row_scan(ri, acc, s_hk, s_tk, s_tv);
    s_cs[tid] = make_float2(sc.s, sc.c);
    __syncthreads();
    if (fdone) {
      CSum tot;
      if (tid > 0) {
        tot.s = s_cs[tid - 1].x;
        tot.c = s_cs[tid - 1].y;
      }
      tot.merge(fpart);
      if (rfirst == 0 && mid_row) p.head[t] = make_float2(tot.s, tot.c);
      else s_sum[rfirst] = tot.value();
    }
    if (tid == kMpNT - 1) {
      p.carry[t] = make_float2(sc.s, sc.c);
    }
    __syncthreads();
    double res = 0.0, dang = 0.0;
    if (nr > 0) {
#pragma unroll
      for (int u = 0; u < kMpT; ++u) {
        const int q = tid + u * kMpNT;
        if (q < nr && !(q == 0 && mid_row)) pr_epilogue(a, i0 + q, s_sum[q], base, rold[u], od[u], res, dang);
      }
    }
    const double2 part = wg_sum2<kMpNT>(make_double2(res, dang), s_red2);
    if (tid == 0) a.tile_part[t] = part;
  }
  if (tid == 0) {
    Counters* c = cnt_of(a.cnt);
    if (edges) atomicAdd(&c->edges, edges);
    if (rows) atomicAdd(&c->verts, rows);
  }
  if (arrive_last(a.st, &s_last)) {
    double res = 0.0, dang = 0.0;
    for (int t0 = 0; t0 < p.ntiles; t0 += kMpNT) {
      const int t = t0 + tid;
      const int r = t < p.ntiles ? p.head_row[t] : -1;
      const CSum tot = crossing_row(a.row, kMpItems, p.carry, p.head, t, r);
      if (r >= 0) epilogue<true>(a, r, tot.value(), base, res, dang);
    }
    finish_pass<true>(a, k, make_double2(res, dang), s_red2);
  }
}

}  // namespace

void merge_free(void* p) {
  MergePlan* mp = static_cast<MergePlan*>(p);
  if (!mp) return;
  void* ptrs[] = {mp->tstart, mp->carry, mp->head, mp->head_row, mp->pcol, mp->perm, mp->xp, mp->part};
  for (void* q : ptrs)
    if (q) (void)hipFree(q);
  delete mp;
}

// Renumbers the columns by falling in-degree (ties by id): degrees counted
// on the device, a counting sort by degree on the host, the renumbered
// column array written on the device.  Once per matrix.
static int renumber_columns(smdp_graph* g, MergePlan* mp, hipStream_t s) {
  const int64_t n = g->n, m = g->m;
  const int grid = std::max(1, g->ctx->cus * 8);
  DeviceScratch<int32_t> tmp;
  SMDP_CHECK(alloc_once(&tmp.p, n));
  int32_t* deg = tmp.p;
  SMDP_HIP(hipMemsetAsync(deg, 0, sizeof(int32_t) * n, s));
  hipLaunchKernelGGL(k_col_degree, dim3(grid), dim3(256), 0, s, g->col, m, deg);
  std::vector<int32_t> hd((size_t)n);
  SMDP_HIP(hipMemcpyAsync(hd.data(), deg, sizeof(int32_t) * n, hipMemcpyDeviceToHost, s));
  SMDP_HIP(hipStreamSynchronize(s));
  int32_t dmax = 0;
  for (int64_t v = 0; v < n; ++v) dmax = std::max(dmax, hd[(size_t)v]);
  // start of each degree's run, highest degree first
  std::vector<int64_t> at((size_t)dmax + 2, 0);
  for (int64_t v = 0; v < n; ++v) ++at[(size_t)(dmax - hd[(size_t)v]) + 1];
  for (size_t d = 1; d < at.size(); ++d) at[d] += at[d - 1];
  std::vector<int32_t> perm((size_t)n), inv((size_t)n);
  for (int64_t v = 0; v < n; ++v) {
    const int64_t k = at[(size_t)(dmax - hd[(size_t)v])]++;
    perm[(size_t)k] = (int32_t)v;
    inv[(size_t)v] = (int32_t)k;
  }
  int64_t ncols = 0;
  for (int64_t v = 0; v < n; ++v) ncols += hd[(size_t)v] > 0;
  SMDP_CHECK(alloc_once(&mp->pcol, m));
  SMDP_CHECK(alloc_once(&mp->perm, n));
  SMDP_CHECK(alloc_once(&mp->xp, std::max<int64_t>(1, ncols)));
  // deg's memory holds inv while the columns are renumbered
  SMDP_HIP(hipMemcpyAsync(deg, inv.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  SMDP_HIP(hipMemcpyAsync(mp->perm, perm.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_renumber_cols, dim3(grid), dim3(256), 0, s, g->col, m, deg, mp->pcol);
  SMDP_HIP(hipGetLastError());
  SMDP_HIP(hipStreamSynchronize(s));
  mp->ncols = (int32_t)ncols;
  return SMDP_OK;
}

// The plan of g's CSR in *slot, built on first use; `spmv` adds the column
// renumbering, else the per-tile partials of PageRank.
static int ensure_merge(smdp_graph* g, void** slot, bool spmv, hipStream_t s, MergePlan** out) {
  MergePlan* mp = static_cast<MergePlan*>(*slot);
  if (mp && mp->n == g->n && mp->m == g->m) {
    *out = mp;
    return SMDP_OK;
  }
  merge_free(mp);
  *slot = nullptr;
  mp = new MergePlan();
  *slot = mp;
  const int64_t total = (int64_t)g->n + g->m;
  mp->items = kMpNT * (spmv ? items_per_thread(total, g->ctx->cus) : items_per_thread_pr(total, g->ctx->cus));
  mp->ntiles = (int32_t)((total + mp->items - 1) / mp->items);
  const int64_t nt = std::max<int64_t>(1, mp->ntiles);
  SMDP_CHECK(alloc_once(&mp->tstart, nt + 1));
  SMDP_CHECK(alloc_once(&mp->carry, nt));
  SMDP_CHECK(alloc_once(&mp->head, nt));
  SMDP_CHECK(alloc_once(&mp->head_row, nt));
  if (!spmv) SMDP_CHECK(alloc_once(&mp->part, nt));
  hipLaunchKernelGGL(k_merge_starts, dim3((mp->ntiles + 256) / 256), dim3(256), 0, s, g->row, g->n, g->m, mp->ntiles,
                     mp->items, mp->tstart);
  SMDP_HIP(hipGetLastError());
  if (spmv && g->m > 0) SMDP_CHECK(renumber_columns(g, mp, s));
  mp->n = g->n;
  mp->m = g->m;
  *out = mp;
  return SMDP_OK;
}

static MArgs merge_args(smdp_graph* g, const MergePlan* mp) {
  MArgs a{};
  a.row = g->row;
  a.col = g->col;
  a.val = g->val;
  a.x = g->x;
  a.y = g->y;
  a.tstart = mp->tstart;
  a.carry = mp->carry;
  a.items = mp->items;
  a.head = mp->head;
  a.head_row = mp->head_row;
  a.cnt = g->cnt;
  a.n = g->n;
  a.m = g->m;
  a.ntiles = mp->ntiles;
  return a;
}

int merge_spmv(smdp_graph* g, void** slot, hipStream_t s, int* launches) {
  if (g->n <= 0 || (int64_t)g->n + g->m > (int64_t)INT32_MAX - kMpNT * kMpBig) return SMDP_ERR_ARG;
  MergePlan* mp = nullptr;
  SMDP_CHECK(ensure_merge(g, slot, true, s, &mp));
  MArgs a = merge_args(g, mp);
  prof_mark(g->ctx, 0);
  // x in the renumbered order (part of the timed product); without arcs only
  // the counters are cleared
  hipLaunchKernelGGL(k_permute_x, dim3(std::max(1, std::min((mp->ncols + 255) / 256, g->ctx->cus * 8))), dim3(256), 0,
                     s, g->x, mp->perm, mp->ncols, mp->xp, g->cnt);
  if (mp->pcol) {
    a.col = mp->pcol;
    a.x = mp->xp;
  }
  if (mp->items == kMpNT * kMpSmall)
    hipLaunchKernelGGL(k_spmv_merge<kMpSmall>, dim3(mp->ntiles), dim3(kMpNT), 0, s, a);
  else
    hipLaunchKernelGGL(k_spmv_merge<kMpBig>, dim3(mp->ntiles), dim3(kMpNT), 0, s, a);
  prof_mark(g->ctx, 0);
  prof_mark(g->ctx, 1);
  hipLaunchKernelGGL(k_merge_fixup, dim3((mp->ntiles + 255) / 256), dim3(256), 0, s, a);
  prof_mark(g->ctx, 1);
  *launches += 3;
  SMDP_HIP(hipGetLastError());
  return SMDP_OK;
}

// The last tile of the largest kind still ends within 32-bit positions.
bool merge_pagerank_fits(int64_t n, int64_t m) { return n + m <= (int64_t)INT32_MAX - kMpNT * 32; }

int merge_pagerank_ensure(smdp_graph* g, void** slot, RArgs* a) {
  MergePlan* mp = nullptr;
  SMDP_CHECK(ensure_merge(g, slot, false, g->ctx->stream, &mp));
  a->tile_part = mp->part;
  a->ntiles = mp->ntiles;
  return SMDP_OK;
}

void merge_pagerank_pass(smdp_graph* g, void* slot, int grid, const RArgs& a, int k, int* launches) {
  const MergePlan* mp = static_cast<const MergePlan*>(slot);
  const MArgs p = merge_args(g, mp);
  const dim3 gd(std::max(1, std::min(grid, mp->ntiles)));
  prof_mark(g->ctx, 0);
  hipStream_t s = g->ctx->stream;
  switch (mp->items / kMpNT) {
    case 4: hipLaunchKernelGGL(k_pr_merge<4>, gd, dim3(kMpNT), 0, s, a, p, k); break;
    case 8: hipLaunchKernelGGL(k_pr_merge<8>, gd, dim3(kMpNT), 0, s, a, p, k); break;
    case 16: hipLaunchKernelGGL(k_pr_merge<16>, gd, dim3(kMpNT), 0, s, a, p, k); break;
    default: hipLaunchKernelGGL(k_pr_merge<32>, gd, dim3(kMpNT), 0, s, a, p, k); break;
  }
  prof_mark(g->ctx, 0);
  ++*launches;
}

}  // namespace smdp
