// fz_nblist.hip -- cell (column) binning and cluster-pair neighbour list.
//
// Replaces the reference's CellBuild/CellUpdate/CellClean and
// nbbuild_exclbitvec/nbbuild_excllist (src/cell_based_kernels.cu:198-399,
// 1048-1493) and the host-side rebuild branch of SingleStep
// (src/dynamics.cu:727-737).  Design:
//   * positions are 64-bit fixed-point fractions of the box, so binning is an
//     exact integer mulhi and every test below is bit-reproducible;
//   * atoms are binned into x-y columns, sorted by (z, atom id) inside each
//     column, and cut into clusters of 8 consecutive atoms;
//   * a cluster pair (I <= J) enters the list iff the periodic gap between the
//     two clusters' bounding boxes is below the pair-list distance; the gap is
//     formed in integers and squared in FP64 without contraction;
//   * each list entry carries a 64-bit mask, one bit per lane of the 8x8 wave64
//     pair tile, clearing padding, the lower triangle of self pairs and
//     excluded (1-2, 1-3, 1-4) pairs;
//   * the rebuild decision is taken on the device (displacement since the
//     last build > half the skin), so a step never waits on the host.
#include "fz_device.h"
#include "fz_launch.h"

namespace fz {

#define SYS_FROM(pre)                                  \
  const int s_ = block_sys(pre, nsys, blockIdx.x);        \
  const SysDev& d = S[s_];                             \
  const int lb = blockIdx.x - block_base(pre, nsys, s_);                 \
  (void)lb;

// ---------------------------------------------------------------------------
// rebuild trigger: any atom moved more than half the skin since the last build
// (reference CoordsUpdate, src/mdcuda.cu:453-458)
__global__ __launch_bounds__(256) void k_check(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  SYS_FROM(pre);
  const int i = lb * 256 + threadIdx.x;
  bool move = false;
  if (i < d.n_atoms) {
    double dx = fx_d(d.rx[i], d.ux[i], d.sc[0]);
    double dy = fx_d(d.ry[i], d.uy[i], d.sc[1]);
    double dz = fx_d(d.rz[i], d.uz[i], d.sc[2]);
    move = dx * dx + dy * dy + dz * dz > d.skin2;
  }
  if (__any(move) && (threadIdx.x & 63) == 0) d.flags[F_REBUILD] = 1;
}

__device__ __forceinline__ bool skip_build(const SysDev& d) {
  return d.flags[F_REBUILD] == 0 || d.flags[F_OVERFLOW] != 0;
}
// The same answer for every wave of the block.  The pair search and the fill raise
// F_OVERFLOW themselves: waves that each read it would leave one by one, and those
// left behind pass the barriers (an ended wave no longer counts) without the words in
// LDS that the others owe them.
__device__ __forceinline__ bool skip_build_block(const SysDev& d) {
  __shared__ int skip;
  if (threadIdx.x == 0) skip = skip_build(d);
  __syncthreads();
  return skip != 0;
}

// Last block done: each of the system's nblocks blocks takes a ticket once its
// device-scope atomics are performed; the block that draws the last ticket sees every
// other block's atomics, if it reads them with agent_load (past its own caches), and
// runs the system's single-block step (no block ever waits for another).  The counter
// is left at zero for the next launch.
// Only atomics: a wave's s_waitcnt waits until its atomics have been performed where
// agent_load reads, which holds for this target and not for the language's memory
// model; plain stores stay in the XCD's L2.  A step that reads plain stores needs a
// release fence before the ticket, which writes that L2 back, of the order of 0.5 us per
// block and XCD (50,000 atoms: 25 us for the count with it, 6 without).
__device__ __forceinline__ bool last_block_of_atomics(unsigned* ctr, int nblocks) {
  __shared__ int last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    last = atomicAdd(ctr, 1u) == (unsigned)(nblocks - 1);
    if (last) atomicExch(ctr, 0u);
  }
  __syncthreads();
  return last != 0;
}
__device__ __forceinline__ int agent_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int column_of(const SysDev& d, int i) {
  int cx = (int)__umul64hi(d.ux[i], (unsigned long long)d.ncx);
  int cy = (int)__umul64hi(d.uy[i], (unsigned long long)d.ncy);
  return cy * d.ncx + cx;
}

// Column histograms are formed in LDS per block of 256 atoms (consecutive atoms
// are mostly neighbours, so a block touches few columns) and added to the
// global counts once per touched column: the global atomics no longer queue
// up by the hundred on each column's counter.  Systems with more columns than
// the LDS table holds use global atomics directly.
constexpr int BIN_LDS = 4096;

// clusters per column, exclusive scan, capacity checks (one block of 256 threads)
__device__ void col_scan_block(const SysDev& d) {
  constexpr int NT = 256;
  __shared__ int part[NT];
  __shared__ int bad;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  const int n = d.ncol;
  const int per = (n + NT - 1) / NT;
  const int c0 = threadIdx.x * per, c1 = min(n, c0 + per);
  int sum = 0;
  for (int c = c0; c < c1; c++) {
    const int cnt = agent_load(d.col_count + CNT_LINE * c);
    if (cnt > MAX_COLUMN_ATOMS) bad = 1;
    sum += (cnt + CLUSTER - 1) / CLUSTER;
  }
  part[threadIdx.x] = sum;
  __syncthreads();
  for (int o = 1; o < NT; o <<= 1) {  // Hillis-Steele inclusive scan
    int v = threadIdx.x >= o ? part[threadIdx.x - o] : 0;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  int run = part[threadIdx.x] - sum;
  for (int c = c0; c < c1; c++) {
    d.col_clu0[c] = run;
    d.col_fill[CNT_LINE * c] = 0;
    run += (agent_load(d.col_count + CNT_LINE * c) + CLUSTER - 1) / CLUSTER;
  }
  if (threadIdx.x == NT - 1) {
    int total = part[NT - 1];
    d.col_clu0[n] = total;
    *d.n_clusters = total;
    int ov = 0;
    if (bad) ov |= OV_COLUMN;
    if (total > d.n_clusters_cap || total * CLUSTER > d.n_slots_cap) ov |= OV_SLOTS;
    if (ov) atomicOr(d.flags + F_OVERFLOW, ov);
  }
}

// Binning count.  FUSED: the block that finishes last (ticket) also runs the
// column scan.  The tickets are drawn one after the other, 11 ns each, so launches of
// many blocks use the separate k_col_scan instead.
template <bool FUSED>
__global__ __launch_bounds__(256) void k_bin_count(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  SYS_FROM(pre);
  if (skip_build(d)) return;
  __shared__ int hist[BIN_LDS];
  const bool lds = d.ncol <= BIN_LDS;  // uniform over the block
  const int i = lb * 256 + threadIdx.x;
  if (lds) {
    for (int k = threadIdx.x; k < d.ncol; k += 256) hist[k] = 0;
    __syncthreads();
  }
  if (i < d.n_atoms) {
    const int c = column_of(d, i);
    d.atom_col[i] = c;
    if (lds) atomicAdd(hist + c, 1);
    else atomicAdd(d.col_count + CNT_LINE * c, 1);
  }
  // clear the counts of the coming pair search and group build
  const int ntile = (d.n_clusters_cap + 63) >> 6, nb = pre[s_ + 1] - pre[s_];
  for (int k = lb * 256 + threadIdx.x; k < ntile; k += nb * 256) d.tile_cnt[CNT_LINE * k] = 0;
  if (lb == 0 && threadIdx.x == 0) *d.pg_n = 0ull;
  if (lds) {
    __syncthreads();
    for (int k = threadIdx.x; k < d.ncol; k += 256) {
      const int v = hist[k];
      if (v) atomicAdd(d.col_count + CNT_LINE * k, v);
    }
  }
  if (FUSED && last_block_of_atomics(d.tick + 0, pre[s_ + 1] - pre[s_])) col_scan_block(d);
}

// one block per system
__global__ __launch_bounds__(256) void k_col_scan(const SysDev* __restrict__ S, int nsys) {
  const SysDev& d = S[blockIdx.x];
  if (skip_build(d)) return;
  col_scan_block(d);
}

// places each atom in its column's range of bin_tmp (order inside a column is
// arbitrary here; k_col_sort fixes it)
__global__ __launch_bounds__(256) void k_bin_scatter(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  SYS_FROM(pre);
  if (skip_build(d)) return;
  __shared__ int hist[BIN_LDS];
  const bool lds = d.ncol <= BIN_LDS;
  const int i = lb * 256 + threadIdx.x;
  if (lds) {
    for (int k = threadIdx.x; k < d.ncol; k += 256) hist[k] = 0;
    __syncthreads();
  }
  int c = -1, r = 0;
  if (i < d.n_atoms) {
    c = d.atom_col[i];
    r = lds ? atomicAdd(hist + c, 1) : atomicAdd(d.col_fill + CNT_LINE * c, 1);
  }
  if (lds) {
    __syncthreads();
    for (int k = threadIdx.x; k < d.ncol; k += 256) {
      const int v = hist[k];
      if (v) hist[k] = atomicAdd(d.col_fill + CNT_LINE * k, v);  // this block's base in column k
    }
    __syncthreads();
    if (c >= 0) r += hist[c];
  }
  if (c >= 0) d.bin_tmp[d.col_clu0[c] * CLUSTER + r] = i;
}

// One block per column: sort by (u_z, id), lay out slots, snapshot positions,
// cluster bounding boxes.  What bounds it is the latency of dependent loads and
// barriers.  Columns of up to COL_RANK atoms (the default grids have about a hundred)
// read everything an atom needs in one go, rank it by counting the atoms before it,
// and store its slot from registers; longer ones sort in LDS (bitonic, 28 barriers at
// 100 atoms) and read the atoms again.  12 -> 7.4 us at 1,000 atoms, 17 -> 12 at
// 19,000, 19 -> 12 at 50,000; 42-49 either way at 227,000, where the scattered stores
// of the snapshot bound it.
constexpr int COL_RANK = 512;

__global__ __launch_bounds__(256) void k_col_sort(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  SYS_FROM(pre);
  if (skip_build(d)) return;
  const int c = lb;
  __shared__ unsigned long long key[MAX_COLUMN_ATOMS];
  __shared__ int ids[MAX_COLUMN_ATOMS];
  const int n = d.col_count[CNT_LINE * c];
  const int clu0 = d.col_clu0[c];
  const int nclu = d.col_clu0[c + 1] - clu0;
  const int base = clu0 * CLUSTER;
  const int nsc = d.n_slots_cap;
  auto put_slot = [&](int k, int a, unsigned long long x, unsigned long long y, unsigned long long z, double q, int t) {
    d.slot_atom[base + k] = a;
    if (a >= 0) {
      d.atom_slot[a] = base + k;
      d.rx[a] = x;
      d.ry[a] = y;
      d.rz[a] = z;
    }
    d.su[base + k] = x;
    d.su[nsc + base + k] = y;
    d.su[2 * nsc + base + k] = z;
    store_slot(d, base + k, x, y, z, q, t);  // the pair kernel's copy (kept current by k_step_first)
  };
  if (n <= COL_RANK) {
    constexpr int PER = COL_RANK / 256;
    unsigned* hx = (unsigned*)(ids + COL_RANK);  // top words in sorted order; key: z
    unsigned* hy = hx + COL_RANK;
    int a[PER], t[PER], rank[PER];
    unsigned long long x[PER], y[PER], z[PER];
    double q[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int k = threadIdx.x + 256 * e;
      a[e] = k < n ? d.bin_tmp[base + k] : -1;
    }
#pragma unroll
    for (int e = 0; e < PER; e++)
      if (a[e] >= 0) {
        x[e] = d.ux[a[e]];
        y[e] = d.uy[a[e]];
        z[e] = d.uz[a[e]];
        q[e] = d.q[a[e]];
        t[e] = d.type[a[e]];
        key[COL_RANK + threadIdx.x + 256 * e] = z[e];
        ids[threadIdx.x + 256 * e] = a[e];
      }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; e++)
      if (a[e] >= 0) {
        int r = 0;
#pragma unroll 8
        for (int k = 0; k < n; k++) {
          const unsigned long long zk = key[COL_RANK + k];
          r += (zk < z[e]) | ((zk == z[e]) & (ids[k] < a[e]));
        }
        rank[e] = r;
        key[r] = z[e];
        hx[r] = (unsigned)(x[e] >> 32);
        hy[r] = (unsigned)(y[e] >> 32);
      }
#pragma unroll
    for (int e = 0; e < PER; e++)
      if (a[e] >= 0) put_slot(rank[e], a[e], x[e], y[e], z[e], q[e], t[e]);
    for (int k = n + threadIdx.x; k < nclu * CLUSTER; k += 256) put_slot(k, -1, 0ull, 0ull, 0ull, 0.0, 0);
    __syncthreads();
    // eight lanes per cluster
    for (int k = threadIdx.x; k < nclu * CLUSTER; k += 256) {
      const int at = min(k, n - 1);  // the last cluster's padding repeats its last atom
      unsigned lo[3] = {hx[at], hy[at], (unsigned)(key[at] >> 32)}, hi[3];
#pragma unroll
      for (int e = 0; e < 3; e++) {
        hi[e] = lo[e];
#pragma unroll
        for (int o = 1; o < CLUSTER; o <<= 1) {
          lo[e] = min(lo[e], (unsigned)__shfl_xor((int)lo[e], o, 64));
          hi[e] = max(hi[e], (unsigned)__shfl_xor((int)hi[e], o, 64));
        }
      }
      if ((k & (CLUSTER - 1)) == 0) {
        const int m = clu0 + k / CLUSTER;
        d.bb[2 * (size_t)m] = make_uint4(lo[0], lo[1], lo[2], 0u);
        d.bb[2 * (size_t)m + 1] = make_uint4(hi[0], hi[1], hi[2], 0u);
        d.clu_col[m] = c;
      }
    }
  } else {
    int P = 1;
    while (P < n) P <<= 1;
    for (int k = threadIdx.x; k < P; k += 256) {
      if (k < n) {
        int a = d.bin_tmp[base + k];
        ids[k] = a;
        key[k] = d.uz[a];
      } else {
        ids[k] = 0x7fffffff;
        key[k] = ~0ull;
      }
    }
    __syncthreads();
    // bitonic sort of (key, id) ascending
    for (int size = 2; size <= P; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int t = threadIdx.x; t < P / 2; t += 256) {
          int lo = 2 * t - (t & (stride - 1));
          int hi = lo + stride;
          bool up = (lo & size) == 0;
          unsigned long long ka = key[lo], kb = key[hi];
          int ia = ids[lo], ib = ids[hi];
          bool gt = ka > kb || (ka == kb && ia > ib);
          if (gt == up) {
            key[lo] = kb; key[hi] = ka;
            ids[lo] = ib; ids[hi] = ia;
          }
        }
        __syncthreads();
      }
    }
    for (int k = threadIdx.x; k < nclu * CLUSTER; k += 256) {
      const int a = k < n ? ids[k] : -1;
      if (a >= 0) put_slot(k, a, d.ux[a], d.uy[a], key[k], d.q[a], d.type[a]);
      else put_slot(k, -1, 0ull, 0ull, 0ull, 0.0, 0);
    }
    for (int m = threadIdx.x; m < nclu; m += 256) {
      unsigned lo[3] = {~0u, ~0u, ~0u}, hi[3] = {0u, 0u, 0u};
      for (int k = m * CLUSTER; k < min(n, (m + 1) * CLUSTER); k++) {
        int a = ids[k];
        const unsigned v[3] = {(unsigned)(d.ux[a] >> 32), (unsigned)(d.uy[a] >> 32), (unsigned)(key[k] >> 32)};
#pragma unroll
        for (int e = 0; e < 3; e++) {
          lo[e] = v[e] < lo[e] ? v[e] : lo[e];
          hi[e] = v[e] > hi[e] ? v[e] : hi[e];
        }
      }
      uint4* b = d.bb + 2 * (size_t)(clu0 + m);
      b[0] = make_uint4(lo[0], lo[1], lo[2], 0u);
      b[1] = make_uint4(hi[0], hi[1], hi[2], 0u);
      d.clu_col[clu0 + m] = c;
    }
  }
  // z-window tables: the clusters' z bounds are non-decreasing along the column
  // (atoms are sorted by z), so each table entry is a binary search
  const int nzb = d.nzb;
  for (int bz = threadIdx.x; bz <= nzb; bz += 256) {
    int lo = 0, hi = nclu;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const unsigned long long zu = key[min(mid * CLUSTER + CLUSTER - 1, n - 1)];
      if ((int)__umul64hi(zu, (unsigned long long)nzb) >= bz) hi = mid; else lo = mid + 1;
    }
    d.zt_hi[(size_t)c * (nzb + 1) + bz] = lo;
    lo = 0; hi = nclu;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const unsigned long long zl = key[mid * CLUSTER];
      if ((int)__umul64hi(zl, (unsigned long long)nzb) >= bz) hi = mid; else lo = mid + 1;
    }
    d.zt_lo[(size_t)c * (nzb + 1) + bz] = lo;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    d.col_count[CNT_LINE * c] = 0;
    d.col_fill[CNT_LINE * c] = 0;
  }
}

// ---------------------------------------------------------------------------
// Lower bound of the periodic gap, in Angstrom, between two intervals given by the
// top words of their ends (an end lies anywhere in its word).  sc: Angstrom per word.
__device__ __forceinline__ float axis_gap(unsigned alo, unsigned ahi, unsigned blo, unsigned bhi, float sc) {
  const unsigned g = min(blo - ahi, alo - bhi) - 1u;  // wraps where they overlap
  return (float)((alo > bhi || blo > ahi) ? g : 0u) * sc;
}

__device__ __forceinline__ bool is_excluded(const SysDev& d, int a, int b) {
  if (!d.use_excl_list) {
    int off = b - a;
    if (off < -32 || off > 31) return false;
    return (d.excl_bits[a] >> (off + 32)) & 1ull;
  }
  int lo = d.excl_off[a], hi = d.excl_off[a + 1];
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    int v = d.excl_list[mid];
    if (v < b) lo = mid + 1; else hi = mid;
  }
  return lo < d.excl_off[a + 1] && d.excl_list[lo] == b;
}

// FP32 atom-pair distance of the list test: 32-bit top words of the fixed-point
// positions, products and sums rounded one by one (no contraction), so the
// oracle restates it bit for bit.  The threshold carries a 1e-6 relative margin
// over rl^2, so every pair with r < rl is kept whatever the rounding.
__device__ __forceinline__ float r2_list32(const SysDev& d, unsigned ax, unsigned ay, unsigned az, unsigned bx,
                                           unsigned by, unsigned bz) {
#pragma clang fp contract(off)
  const float dx = (float)(int)(bx - ax) * d.sc32[0];
  const float dy = (float)(int)(by - ay) * d.sc32[1];
  const float dz = (float)(int)(bz - az) * d.sc32[2];
  float r2 = dx * dx;
  r2 = r2 + dy * dy;
  r2 = r2 + dz * dz;
  return r2;
}

// bit 8 k set where byte k of m is not zero
__device__ __forceinline__ unsigned long long byte_any(unsigned long long m) {
  m |= m >> 4;
  m |= m >> 2;
  m |= m >> 1;
  return m & 0x0101010101010101ull;
}

// One wave per I cluster.
//  1. Candidate columns (those at or after I's own, column-gap prefilter), one per
//     lane; per column, the z-window tables give the (at most two) ranges of clusters
//     whose z bounds can come within the pair-list distance of I's z bounds.
//  2. Those ranges (J >= I) are packed 64 to a block; each lane tests its J's
//     bounding box (a lower bound of the periodic gap, from the top words).
//  3. The hits queue in LDS and are tested eight at a time, lane (h, j) holding slot j
//     of the h-th against the eight atoms of I in scalar registers: one gather per
//     eight hits, and the lanes' bytes are the entries' masks.  A pair is kept when
//     both slots hold atoms, it is not excluded, i < j inside a self pair, and the FP32
//     list distance is below the threshold.  An entry without a pair is dropped.  The
//     next group's atoms are loaded while one is tested.
//  The distance of step 3 is the expanded square |b|^2 + (|a|^2 - 2 a.b) about I's
//  first atom, three fused multiply-adds and an addition per pair; a group with a pair
//  closer to the threshold than its rounding (about 1 % of them) is done again as
//  r2_list32 has it, so the list is that test's to the bit.  It needs the nearest image
//  of b about that atom to be the nearest about all of them: rl plus I's extent within
//  half the box, else every group is tested the second way.  Exclusions are looked up
//  only in groups with an atom among the indexes of I's partners.
//  With split > 1, split consecutive waves share one I cluster, each taking an equal
//  share of the candidates (of the columns, when there are more than 64) and writing
//  its own buffer part; the fill concatenates the parts in order, which is the order
//  one wave would have produced.
// What bounds it: VALU issue on large systems (170 of 236 us at 227,000 atoms), memory
// latency on small ones.  Hit by hit, with I's and J's atoms in lanes (i, j), every
// entry in a store of its lane and an atomic per wave, a build's search took 461 us at
// 227,000 atoms, 130 at 50,000, 82 at 19,000 and 17 at 1,000; this 236, 75, 35 and 12.
// Of the 48 us gained at 19,000 the atomics were the larger part: one per wave on three
// lines of counters, done one after the other (CNT_LINE).
__device__ __forceinline__ float uniform_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

constexpr int HIT_RING = 128;
__global__ __launch_bounds__(256, 5) void k_pair_search(
    const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre, int split_cap) {
  SYS_FROM(pre);
  if (skip_build_block(d)) return;
  __shared__ int block_cnt[2];  // entries, waves done
  if (threadIdx.x == 0) block_cnt[0] = block_cnt[1] = 0;
  __syncthreads();
  // a private copy of the descriptor: the entry stores below cannot alias it,
  // so its fields stay in registers instead of being reloaded per hit
  const SysDev dv = d;
  const int lane = threadIdx.x & 63;
  const int jl = lane & 7, hl = lane >> 3;
  const int split = search_split(dv.search_parts, split_cap);
  const int gw = lb * 4 + (threadIdx.x >> 6);
  const int I = gw / split, part = gw - I * split;
  if (I >= *dv.n_clusters) return;
  const int pcap = dv.search_parts * SEARCH_TMP_CAP / split;  // entries per part
  const int nsc = dv.n_slots_cap;
  // global-address-space views: global_* loads and stores, which wait on the
  // vector memory counter only (generic ones also wait on the LDS counter)
  const FZ_GLOBAL unsigned* su32 = (const FZ_GLOBAL unsigned*)dv.su;  // high words at odd indices
  const FZ_GLOBAL int* slot_atom = (const FZ_GLOBAL int*)dv.slot_atom;
  typedef unsigned word4 __attribute__((ext_vector_type(4)));
  const FZ_GLOBAL word4* bbg = (const FZ_GLOBAL word4*)dv.bb;
  // The I cluster's atoms, one to lanes i, 8 + i, ...: their positions relative to
  // its first atom as the terms of the expanded square, in scalar registers.
  const int ai = slot_atom[I * CLUSTER + jl];
  const unsigned long long wa = (ai >= 0 && !dv.use_excl_list) ? dv.excl_bits[ai] : 0ull;
  const unsigned vix = su32[2 * (I * CLUSTER + jl) + 1], viy = su32[2 * (nsc + I * CLUSTER + jl) + 1],
                 viz = su32[2 * (2 * nsc + I * CLUSTER + jl) + 1];
  const unsigned imask = (unsigned)__ballot(ai >= 0) & 0xffu;
  const unsigned ox = (unsigned)__builtin_amdgcn_readfirstlane((int)vix),
                 oy = (unsigned)__builtin_amdgcn_readfirstlane((int)viy),
                 oz = (unsigned)__builtin_amdgcn_readfirstlane((int)viz);
  float ax[8], ay[8], az[8], na[8];
  int iw[8];      // first index of atom i's excluded partners
  unsigned span;  // the widest range of partners of one atom, 0: none
  bool expand;
  float margin;
  {
    const float ux = ai >= 0 ? (float)(int)(vix - ox) * dv.sc32[0] : 0.0f;
    const float uy = ai >= 0 ? (float)(int)(viy - oy) * dv.sc32[1] : 0.0f;
    const float uz = ai >= 0 ? (float)(int)(viz - oz) * dv.sc32[2] : 0.0f;
    const float n2 = ux * ux + uy * uy + uz * uz;
    float top = n2;
    const int w0 = wa ? __ffsll((long long)wa) - 1 : 0, w1 = wa ? 64 - __clzll((long long)wa) : 0;
    int wide = w1 - w0;
    const int first = wa ? ai - 32 + w0 : -0x40000000;
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
      top = fmaxf(top, __shfl_xor(top, o, 64));
      wide = max(wide, __shfl_xor(wide, o, 64));
    }
    top = uniform_f(top, 0);
    span = (unsigned)__builtin_amdgcn_readfirstlane(wide);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      ax[i] = uniform_f(-2.0f * ux, i);
      ay[i] = uniform_f(-2.0f * uy, i);
      az[i] = uniform_f(-2.0f * uz, i);
      na[i] = uniform_f(n2, i);
      iw[i] = __builtin_amdgcn_readlane(first, i);
    }
    const float ext = sqrtf(top), rl = sqrtf(dv.rl2f), reach = rl + 2.0f * ext;
    margin = uniform_f(4e-6f * (reach * reach + dv.rl2f), 0);
    const float half = 0.49999f * 4294967296.0f * fminf(dv.sc32[0], fminf(dv.sc32[1], dv.sc32[2]));
    expand = __builtin_amdgcn_readfirstlane((int)(rl + ext < half)) != 0;
  }
  const size_t obase = (size_t)I * dv.search_parts * SEARCH_TMP_CAP + (size_t)part * pcap;
  FZ_GLOBAL unsigned long long* mout = (FZ_GLOBAL unsigned long long*)(dv.search_mtmp + obase);
  FZ_GLOBAL int* out = (FZ_GLOBAL int*)(dv.search_tmp + obase);
  const word4 blo = bbg[2 * (size_t)I], bhi = bbg[2 * (size_t)I + 1];
  const int cI = dv.clu_col[I];
  const int cx = cI % dv.ncx, cy = cI / dv.ncx;
  const unsigned wx = (unsigned)(dv.colw_x >> 32), wy = (unsigned)(dv.colw_y >> 32);
  const bool allx = 2 * dv.kx_range + 1 >= dv.ncx, ally = 2 * dv.ky_range + 1 >= dv.ncy;
  // rows of columns at or after I's own (clusters of the others come before I): the
  // first ny0 wrap below row 0
  const int ny0 = ally ? 0 : max(0, dv.ky_range - cy);
  const int ny = ny0 + (ally ? dv.ncy - cy : min(dv.ky_range, dv.ncy - 1 - cy) + 1);
  const int nxv = allx ? dv.ncx : 2 * dv.kx_range + 1;
  // z window [w0, w1] on the 2^64 circle
  const int nzb = dv.nzb;
  const unsigned long long R = dv.zwin;
  const unsigned long long binw = ~0ull / (unsigned long long)nzb;
  const unsigned long long z0 = (unsigned long long)blo.z << 32, z1 = ((unsigned long long)bhi.z << 32) | 0xffffffffull;
  const bool zfull = R >= (1ull << 61) || z1 - z0 >= ~0ull - 2 * R - binw;
  const unsigned long long w0 = z0 - R, w1 = z1 + R;
  const bool zwrap = !zfull && w0 > w1;
  const int b0 = (int)__umul64hi(w0, (unsigned long long)nzb);
  const int b1 = (int)__umul64hi(w1, (unsigned long long)nzb);

  int count = 0;
  int cand = 0, fill = 0;
  __shared__ int ring_s[4][HIT_RING];
  __shared__ int outj_s[4][HIT_RING];
  __shared__ unsigned outm_s[4][HIT_RING][2];
  int* ring = ring_s[threadIdx.x >> 6];
  int* outj = outj_s[threadIdx.x >> 6];
  unsigned(*outm)[2] = outm_s[threadIdx.x >> 6];
  int head = 0, tail = 0, stored = 0;

  // entries wait in LDS and are stored 64 at a time: full lines, and the loads in
  // flight do not queue behind a store per group
  auto store_entries = [&]() {
    const int e = stored + lane;
    if (e < count && e < pcap) {
      const unsigned* m = outm[e & (HIT_RING - 1)];
      out[e] = outj[e & (HIT_RING - 1)];
      mout[e] = ((unsigned long long)m[1] << 32) | m[0];
    }
    stored += 64;
  };

  // lane (h, j) of a group of eight hits: the h-th hit's slot j
  struct Hit { int J, b; unsigned x, y, z; };
  auto load_hits = [&](int first) {
    Hit t;
    t.J = first + hl < tail ? ring[(first + hl) & (HIT_RING - 1)] : -1;
    t.b = -1;
    t.x = t.y = t.z = 0u;
    if (t.J >= 0) {
      const int slot = t.J * CLUSTER + jl;
      t.b = slot_atom[slot];
      t.x = su32[2 * slot + 1];
      t.y = su32[2 * (nsc + slot) + 1];
      t.z = su32[2 * (2 * nsc + slot) + 1];
    }
    return t;
  };
  auto test_hits = [&](const Hit& t) {
    unsigned m8 = 0u;  // bit i: atom i of I near this lane's
    unsigned off = ~0u;
    float clear = __builtin_inff();
#pragma unroll
    for (int i = 0; i < 8; i++) off = min(off, (unsigned)(t.b - iw[i]));
    if (expand) {
      const float ux = (float)(int)(t.x - ox) * dv.sc32[0], uy = (float)(int)(t.y - oy) * dv.sc32[1],
                  uz = (float)(int)(t.z - oz) * dv.sc32[2];
      const float nb = fmaf(ux, ux, fmaf(uy, uy, fmaf(uz, uz, -dv.rl2f)));
#pragma unroll
      for (int i = 7; i >= 0; i--) {
        const float r = fmaf(ax[i], ux, fmaf(ay[i], uy, fmaf(az[i], uz, nb + na[i])));  // r^2 - rl^2
        m8 = __builtin_amdgcn_alignbit(m8, __float_as_uint(r), 31);                      // 2 m8 + (r < 0)
        clear = fminf(clear, fabsf(r));
      }
    }
    if (!expand || __ballot(clear < margin)) {
      m8 = 0u;
      for (int i = 7; i >= 0; i--)
        m8 = 2u * m8 + (r2_list32(dv, (unsigned)__builtin_amdgcn_readlane((int)vix, i),
                                  (unsigned)__builtin_amdgcn_readlane((int)viy, i),
                                  (unsigned)__builtin_amdgcn_readlane((int)viz, i), t.x, t.y, t.z) < dv.rl2f
                            ? 1u
                            : 0u);
    }
    m8 &= t.b >= 0 ? imask : 0u;
    if (t.J == I) m8 &= (1u << jl) - 1u;  // i < j inside a self pair
    if (dv.use_excl_list) {
      for (int i = 0; i < 8; i++) {
        const int a = __builtin_amdgcn_readlane(ai, i);
        if ((m8 >> i) & 1u)
          if (is_excluded(dv, a, t.b)) m8 &= ~(1u << i);
      }
    } else if (__ballot(off < span)) {  // some atom may be a partner: few groups
      for (int i = 0; i < 8; i++) {
        const unsigned sh = (unsigned)(t.b - __builtin_amdgcn_readlane(ai, i) + 32);
        const unsigned long long w =
            ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(wa >> 32), i) << 32) |
            (unsigned)__builtin_amdgcn_readlane((int)(unsigned)wa, i);
        if (sh < 64u && ((w >> (sh & 63u)) & 1ull)) m8 &= ~(1u << i);
      }
    }
    // entries of the hits with a pair: bytes j of the mask, four to a word
    const unsigned long long pairs = __ballot(m8 != 0u), kept = byte_any(pairs);
    if (!kept) return;
    int w = (int)(m8 << (8 * (jl & 3)));
    w |= __builtin_amdgcn_mov_dpp(w, 0xB1, 0xf, 0xf, true);  // lane ^ 1
    w |= __builtin_amdgcn_mov_dpp(w, 0x4E, 0xf, 0xf, true);  // lane ^ 2
    const bool mine = (kept >> (8 * hl)) & 1ull;
    const int pos = count + __builtin_popcountll(kept & ((1ull << (8 * hl)) - 1ull));
    if (mine && (jl & 3) == 0) outm[pos & (HIT_RING - 1)][jl >> 2] = (unsigned)w;
    if (mine && jl == 0) outj[pos & (HIT_RING - 1)] = t.J;
    count += __builtin_popcountll(kept);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (count - stored >= 64) store_entries();
  };
  // hits in the ring in groups of eight, the next group's atoms loaded before a
  // group is tested; a last group of fewer when asked for
  auto drain = [&](int least) {
    if (tail - head < least) return;
    Hit t = load_hits(head);
    while (true) {
      head += 8;
      const bool more = tail - head >= least;
      Hit n = t;
      if (more) n = load_hits(head);
      test_hits(t);
      if (!more) break;
      t = n;
    }
    head = min(head, tail);
  };
  auto test_cands = [&](int least) {
    bool hit = false;
    if (lane < fill) {
      const word4 clo = bbg[2 * (size_t)cand], chi = bbg[2 * (size_t)cand + 1];
      const float gx = axis_gap(blo.x, bhi.x, clo.x, chi.x, dv.sc32[0]), gy = axis_gap(blo.y, bhi.y, clo.y, chi.y, dv.sc32[1]),
                  gz = axis_gap(blo.z, bhi.z, clo.z, chi.z, dv.sc32[2]);
      hit = gx * gx + gy * gy + gz * gz < dv.rl2f;
    }
    const unsigned long long bal = __ballot(hit);
    if (hit)
      ring[(tail + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u))) &
           (HIT_RING - 1)] = cand;
    tail += __builtin_popcountll(bal);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    drain(least);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  const int nq = ny * nxv;
  // parts: equal shares of the candidates of up to 64 columns, else of the columns
  const bool by_cand = nq <= 64;
  const int q0 = by_cand ? 0 : part * nq / split, q1 = by_cand ? nq : (part + 1) * nq / split;
  for (int g = q0; g < q1; g += 64) {
    // per lane: one candidate column and its (up to two) cluster ranges
    int r0a = 0, r0e = 0, r1a = 0, r1e = 0;
    const int q = g + lane;
    if (q < q1) {
      const int iy = q / nxv, ix = q - iy * nxv;
      int yy = iy < ny0 ? dv.ncy + cy - dv.ky_range + iy : cy + iy - ny0, xx = allx ? ix : cx + ix - dv.kx_range;
      xx += xx < 0 ? dv.ncx : xx >= dv.ncx ? -dv.ncx : 0;
      // (a column's words: its edges are c 2^32 / ncx, of which wx is the whole part)
      const float gx = axis_gap(blo.x, bhi.x, xx * wx, xx == dv.ncx - 1 ? ~0u : (xx + 1) * (wx + 1u), dv.sc32[0]);
      const float gy = axis_gap(blo.y, bhi.y, yy * wy, yy == dv.ncy - 1 ? ~0u : (yy + 1) * (wy + 1u), dv.sc32[1]);
      if (gx * gx + gy * gy < dv.rl2f) {
        const int C = yy * dv.ncx + xx;
        const FZ_GLOBAL int* clu0 = (const FZ_GLOBAL int*)dv.col_clu0;
        const int j0 = clu0[C], nc = clu0[C + 1] - j0;
        const FZ_GLOBAL int* th = (const FZ_GLOBAL int*)dv.zt_hi + (size_t)C * (nzb + 1);
        const FZ_GLOBAL int* tl = (const FZ_GLOBAL int*)dv.zt_lo + (size_t)C * (nzb + 1);
        if (zfull) {
          r0a = 0; r0e = nc;
        } else if (!zwrap) {
          r0a = th[b0]; r0e = tl[b1 + 1];
        } else {
          const int e1 = tl[b1 + 1], s0 = th[b0];
          if (s0 <= e1) { r0a = 0; r0e = nc; }
          else { r0a = 0; r0e = e1; r1a = s0; r1e = nc; }
        }
        r0a += j0; r0e += j0; r1a += j0; r1e += j0;
        r0a = max(r0a, I); r1a = max(r1a, I);
      }
    }
    // The group's candidates in order (column by column, each column's first
    // range then its second) are numbered by an inclusive scan of the per-lane
    // counts; each free slot of the 64-candidate block finds its column by a
    // binary search over the scan (lane permutes), so the block fills without
    // a scalar loop over columns.
    const int l0 = max(r0e - r0a, 0), l1 = max(r1e - r1a, 0);
    int incl = l0 + l1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    const int total = __builtin_amdgcn_readlane(incl, 63);
    const int last = by_cand ? (part + 1) * total / split : total;
    for (int base = by_cand ? part * total / split : 0; base < last;) {
      const int m = min(last - base, 64 - fill);
      // every lane takes part in the permutes; lanes outside [fill, fill + m) discard
      const int p = base + lane - fill;
      int lo = 0;
#pragma unroll
      for (int step = 32; step >= 1; step >>= 1) {  // first k with incl[k] > p
        const int v = __shfl(incl, lo + step - 1, 64);
        if (v <= p) lo += step;
      }
      const int k = min(lo, 63);
      const int off = p - (__shfl(incl, k, 64) - __shfl(l0 + l1, k, 64));
      const int c0 = __shfl(r0a, k, 64), n0 = __shfl(l0, k, 64), c1 = __shfl(r1a, k, 64);
      if (lane >= fill && lane < fill + m) cand = off < n0 ? c0 + off : c1 + (off - n0);
      fill += m;
      base += m;
      if (fill == 64) { test_cands(8); fill = 0; }
    }
  }
  test_cands(1);
  store_entries();
  if (lane == 0) {
    const int kept = count < pcap ? count : pcap;
    dv.search_cnt[I * split + part] = kept;
    // one add per block: the block's last wave (64 split is a multiple of its four waves: one tile)
    atomicAdd(block_cnt, kept);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    if (atomicAdd(block_cnt + 1, 1) == min(4, *dv.n_clusters * split - 4 * lb) - 1) {
      const int sum = atomicAdd(block_cnt, 0);
      if (sum) atomicAdd(dv.tile_cnt + CNT_LINE * (I >> 6), sum);
    }
    if (I == 0) dv.n_clusters[1] = split;
    if (count > pcap) atomicOr(dv.flags + F_OVERFLOW, OV_SEARCH);
  }
}

// ---------------------------------------------------------------------------
// Pair groups and work items from the entries, one wave per pair of clusters
// (I0 = 2 s, I1 = 2 s + 1; almost always neighbours along one column, with most
// of their j slots in common).
//
// The j slots of the pair of clusters are split into three runs: B, near an atom
// of both; A0, near I0 only; A1, near I1 only.  A group of B gives the pair kernel
// two tiles for one gather, one j reduction and one j-force atomic; a group of A0
// or A1 one.  The tiles are as many as with a list per cluster (each run's last
// group is padded: under 1 %), the groups, hence the atomics' cache lines, 0.6 of
// them.
//
// The entries of I1 are hashed by J in LDS and those of I0 looked up there; a
// first pass counts the runs, one atomic per block reserves the groups and the
// work items, a second pass writes them.  Where a pair of clusters lands depends
// on the order in which blocks get there, but a work item never crosses from one
// pair of clusters to the next, so the sums a wave forms do not depend on it.
// A wave keeps its entries in registers between the passes (FILL_REG rounds of 64
// per cluster; longer lists are read again), and reads a cluster's parts as one
// sequence, so the whole build is a handful of memory round trips: 1,000 atoms
// 9 us, where reading part by part in both passes took 32.
constexpr int FILL_HASH = 1024;  // slots of a wave's table; lists of I1 over three quarters of it are not merged
constexpr int FILL_REG = 5;

// entry e of a cluster's list: its parts one after the other (cnt: their counts, first: the first part's buffer)
struct FillList {
  int cnt[4], total;
  size_t first;
  int pcap;
  __device__ __forceinline__ size_t at(int e) const {
    int p = 0;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (p == k && e >= cnt[k]) { e -= cnt[k]; p = k + 1; }
    return first + (size_t)p * pcap + e;
  }
};

__device__ __forceinline__ FillList fill_list(const SysDev& d, int I, bool live, int split) {
  FillList l;
  l.pcap = d.search_parts * SEARCH_TMP_CAP / split;
  l.first = (size_t)I * d.search_parts * SEARCH_TMP_CAP;
  l.total = 0;
#pragma unroll
  for (int p = 0; p < 4; p++) {
    l.cnt[p] = live && p < split ? d.search_cnt[I * split + p] : 0;
    l.total += l.cnt[p];
  }
  return l;
}

struct FillEntry { int J; unsigned long long m; };

// slot of J in a wave's table, or of the first free one on its way
__device__ __forceinline__ int fill_find(const int* key, int J) {
  int at = (int)((unsigned)J * 2654435761u >> 22);
  while (key[at] != -1 && (key[at] & 0x7fffffff) != J) at = (at + 1) & (FILL_HASH - 1);
  return at;
}

// Both clusters' entries, 64 at a time, I0's first: f(J, m0, m1) per lane, called
// by the whole wave (zero masks where a lane has no entry).  With merge, I0's entry
// takes I1's mask along and marks it, and I1's marked entries are left out.
template <class F>
__device__ __forceinline__ void fill_scan(const SysDev& d, const FillList (&l)[2], const FillEntry (&reg)[2][FILL_REG], bool merge,
                                          int* key, const unsigned long long* val, F&& f) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    auto round = [&](FillEntry e) {
      unsigned long long m0 = h == 0 ? e.m : 0ull, m1 = h == 0 ? 0ull : e.m;
      if (merge && e.m) {
        const int at = fill_find(key, e.J);
        if (key[at] != -1) {
          if (h == 0) {
            m1 = val[at];
            key[at] = e.J | (int)0x80000000;
          } else if (key[at] < 0) {
            m1 = 0ull;
          }
        }
      }
      f(e.J, m0, m1);
    };
#pragma unroll
    for (int r = 0; r < FILL_REG; r++)
      if (r * 64 < l[h].total) round(reg[h][r]);
    for (int k = FILL_REG * 64; k < l[h].total; k += 64) {
      FillEntry e = {0, 0ull};
      if (k + lane < l[h].total) {
        const size_t at = l[h].at(k + lane);
        e.J = d.search_tmp[at];
        e.m = d.search_mtmp[at];
      }
      round(e);
    }
  }
}

// The entries of the clusters I0 and I0 + 1 of an entry list into place: offset, the
// counts of the 64-cluster tiles before theirs and of the clusters before I0 inside it.
__device__ __forceinline__ void fill_entries(const SysDev& d, int I0, int n, int split) {
  const int lane = threadIdx.x & 63;
  if (I0 >= n) return;
  const FillList l[2] = {fill_list(d, I0, true, split), fill_list(d, I0 + 1, I0 + 1 < n, split)};
  const int t = I0 >> 6, nt = (n + 63) >> 6;
  long long before = 0, total = 0;
  for (int k = lane; k < nt; k += 64) {
    const long long v = d.tile_cnt[CNT_LINE * k];
    total += v;
    if (k < t) before += v;
  }
  for (int k = (t << 6) * split + lane; k < I0 * split; k += 64) before += d.search_cnt[k];
  before = wave_sum(before);
  total = wave_sum(total);
  if (I0 == 0 && lane == 0) {
    if (total > d.n_pairs_cap) atomicOr(d.flags + F_OVERFLOW, OV_PAIRS);
    else d.flags[F_NBUILD] += 1;
    *d.n_pairs = total > d.n_pairs_cap ? 0 : total;
  }
  if (total > d.n_pairs_cap) return;
  const int n0 = l[0].total, n01 = n0 + l[1].total;
#pragma unroll 4
  for (int k = lane; k < n01; k += 64) {
    const size_t at = k < n0 ? l[0].at(k) : l[1].at(k - n0);
    const int J = d.search_tmp[at];
    const unsigned long long m = d.search_mtmp[at];
    d.pl_ij[before + k] = make_int2(k < n0 ? I0 : I0 + 1, J);
    d.pl_mask[before + k] = m;
  }
}

__global__ __launch_bounds__(256) void k_pair_fill(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre,
                                                   int split_cap) {
  SYS_FROM(pre);
  if (skip_build_block(d)) return;
  __shared__ int4 keys[4][FILL_HASH / 4];
  __shared__ unsigned long long vals[4][FILL_HASH];
  __shared__ bool fits;
  __shared__ unsigned long long need[4];  // groups (low 40 bits) and items of each wave, then their offsets
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int n = *d.n_clusters;
  const int I0 = 2 * (lb * 4 + wv);
  if (2 * (lb * 4) >= n) return;  // the whole block
  const bool live = I0 < n, two = I0 + 1 < n;
  const int split = search_split(d.search_parts, split_cap);
  if (d.entry_list) {
    fill_entries(d, I0, n, split);
    return;
  }
  const FillList l[2] = {fill_list(d, I0, live, split), fill_list(d, I0 + 1, two, split)};
  long long total = 0;
  for (int k = threadIdx.x; k < (n + 63) >> 6; k += 256) total += d.tile_cnt[CNT_LINE * k];
  FillEntry reg[2][FILL_REG];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int r = 0; r < FILL_REG; r++) {
      reg[h][r] = FillEntry{0, 0ull};
      if (r * 64 + lane < l[h].total) {
        const size_t at = l[h].at(r * 64 + lane);
        reg[h][r].J = d.search_tmp[at];
        reg[h][r].m = d.search_mtmp[at];
      }
    }
  int* key = (int*)keys[wv];
  unsigned long long* val = vals[wv];
  const bool merge = l[0].total > 0 && l[1].total > 0 && l[1].total <= FILL_HASH / 4 * 3;
  if (merge) {
#pragma unroll
    for (int k = 0; k < FILL_HASH / 256; k++) keys[wv][k * 64 + lane] = make_int4(-1, -1, -1, -1);
  }
  total = wave_sum(total);
  if (lane == 0) need[wv] = (unsigned long long)total;
  __syncthreads();
  total = (long long)(need[0] + need[1] + need[2] + need[3]);
  if (total > d.n_pairs_cap) {  // every block
    if (I0 == 0 && lane == 0) {
      atomicOr(d.flags + F_OVERFLOW, OV_PAIRS);
      *d.n_pairs = 0;
    }
    return;
  }
  if (I0 == 0 && lane == 0) {
    *d.n_pairs = total;
    atomicAdd(d.flags + F_NBUILD, 1);
  }
  __syncthreads();
  if (merge) {
    auto insert = [&](FillEntry e) {
      if (!e.m) return;  // a kept entry has a mask
      int at = (int)((unsigned)e.J * 2654435761u >> 22);
      while (atomicCAS(&key[at], -1, e.J) != -1) at = (at + 1) & (FILL_HASH - 1);
      val[at] = e.m;
    };
#pragma unroll
    for (int r = 0; r < FILL_REG; r++) insert(reg[1][r]);
    for (int k = FILL_REG * 64 + lane; k < l[1].total; k += 64) {
      const size_t at = l[1].at(k);
      insert(FillEntry{d.search_tmp[at], d.search_mtmp[at]});
    }
  }
  __syncthreads();
  int nB = 0, n0 = 0, n1 = 0;  // per lane, then of the wave
  fill_scan(d, l, reg, merge, key, val, [&](int, unsigned long long m0, unsigned long long m1) {
    const unsigned long long a = byte_any(m0), b = byte_any(m1);
    nB += __popcll(a & b);
    n0 += __popcll(a & ~b);
    n1 += __popcll(b & ~a);
  });
  nB = wave_sum(nB);
  n0 = wave_sum(n0);
  n1 = wave_sum(n1);
  const int gB = (nB + 7) >> 3, g0 = (n0 + 7) >> 3, g1 = (n1 + 7) >> 3;
  const int tiles = 2 * gB + g0 + g1;
  const int items = (tiles + d.item_tiles - 1) / d.item_tiles;
  if (lane == 0) need[wv] = (unsigned long long)(gB + g0 + g1) | ((unsigned long long)items << 40);
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long all = need[0] + need[1] + need[2] + need[3];
    unsigned long long run = atomicAdd(d.pg_n, all);
    fits = (long long)((run + all) & ((1ull << 40) - 1)) <= d.n_groups_cap;
    // more groups than there is room for: as with more entries, no build to count
    if (!fits && !(atomicOr(d.flags + F_OVERFLOW, OV_PAIRS) & OV_PAIRS)) atomicSub(d.flags + F_NBUILD, 1);
    for (int k = 0; k < 4; k++) {
      const unsigned long long v = need[k];
      need[k] = run;
      run += v;
    }
  }
  __syncthreads();
  if (!fits) return;  // the whole block
  const long long gofs = (long long)(need[wv] & ((1ull << 40) - 1));
  int4* it = d.pg_item + (need[wv] >> 40);
  // items of about equal tiles: tile t lies in group t / 2 of B or in A0, A1 after it
  for (int k = lane; k < items; k += 64) {
    const int t0 = (int)((long long)tiles * k / items), t1 = (int)((long long)tiles * (k + 1) / items);
    const int q0 = t0 < 2 * gB ? t0 >> 1 : t0 - gB, q1 = t1 < 2 * gB ? t1 >> 1 : t1 - gB;
    it[k] = make_int4((int)(gofs + q0), q1 - q0, I0, two ? I0 + 1 : I0);
  }
  unsigned* out = d.pg_j + 8 * gofs;
  unsigned char* mk = (unsigned char*)(d.pg_mask + gofs);
  auto put = [&](int pos, unsigned off, unsigned b0, unsigned b1) {
    out[pos] = off;
    unsigned char* m = mk + (size_t)(pos >> 3) * 16 + (pos & 7);
    m[0] = (unsigned char)b0;
    m[8] = (unsigned char)b1;
  };
  int pB = 0, p0 = 8 * gB, p1 = 8 * (gB + g0);
  fill_scan(d, l, reg, merge, key, val, [&](int J, unsigned long long m0, unsigned long long m1) {
    const unsigned long long a = byte_any(m0), b = byte_any(m1);
    // the three runs' counts in one scan, ten bits each (at most 512 in a wave)
    const int c = __popcll(a & b) | (__popcll(a & ~b) << 10) | (__popcll(b & ~a) << 20);
    int incl = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    const int x = incl - c;
    int qB = pB + (x & 1023), q0 = p0 + ((x >> 10) & 1023), q1 = p1 + (x >> 20);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const unsigned b0 = (unsigned)(m0 >> (8 * j)) & 0xffu, b1 = (unsigned)(m1 >> (8 * j)) & 0xffu;
      if (b0 | b1) {
        const int pos = b0 && b1 ? qB : b0 ? q0 : q1;
        qB += b0 && b1;
        q0 += b0 && !b1;
        q1 += !b0;
        put(pos, (unsigned)(J * CLUSTER + j) * SLOT_BYTES, b0, b1);
      }
    }
    const int all = __builtin_amdgcn_readlane(incl, 63);
    pB += all & 1023;
    p0 += (all >> 10) & 1023;
    p1 += all >> 20;
  });
  // padding: an existing slot with no lane of its own
  const unsigned pad = (unsigned)(I0 * CLUSTER) * SLOT_BYTES;
  if (lane < 8 * gB - nB) put(nB + lane, pad, 0u, 0u);
  if (lane < 8 * g0 - n0) put(8 * gB + n0 + lane, pad, 0u, 0u);
  if (lane < 8 * g1 - n1) put(8 * (gB + g0) + n1 + lane, pad, 0u, 0u);
}

// The entries of the last build in list order, from the search buffers (for
// inspection): one wave per I cluster, offsets as in k_pair_fill.
__global__ __launch_bounds__(256) void k_pair_entries(const SysDev* __restrict__ S, int2* __restrict__ pairs,
                                                      unsigned long long* __restrict__ masks) {
  const SysDev& d = S[0];
  const int lane = threadIdx.x & 63;
  const int I = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (I >= d.n_clusters[0]) return;
  const int split = d.n_clusters[1];
  const int pcap = d.search_parts * SEARCH_TMP_CAP / split;
  const int t = I >> 6;
  long long off = 0;
  for (int k = lane; k < t; k += 64) off += d.tile_cnt[CNT_LINE * k];
  for (int k = (t << 6) * split + lane; k < I * split; k += 64) off += d.search_cnt[k];
  off = wave_sum(off);
  for (int p = 0; p < split; p++) {
    const int cnt = d.search_cnt[I * split + p];
    const size_t base = (size_t)I * d.search_parts * SEARCH_TMP_CAP + (size_t)p * pcap;
    for (int k = lane; k < cnt; k += 64) {
      pairs[off + k] = make_int2(I, d.search_tmp[base + k]);
      masks[off + k] = d.search_mtmp[base + k];
    }
    off += cnt;
  }
}

void launch_pair_entries(const Launch& L, int2* pairs, unsigned long long* masks) {
  hipLaunchKernelGGL(k_pair_entries, dim3(L.w_clus.total), dim3(256), 0, L.stream, L.d_sys, pairs, masks);
}

// ---------------------------------------------------------------------------
void launch_nblist(const Launch& L, bool check) {
  if (check) hipLaunchKernelGGL(k_check, dim3(L.w_atoms.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
  if (L.w_atoms.total <= 512) {
    hipLaunchKernelGGL(k_bin_count<true>, dim3(L.w_atoms.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
  } else {
    hipLaunchKernelGGL(k_bin_count<false>, dim3(L.w_atoms.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    hipLaunchKernelGGL(k_col_scan, dim3(L.nsys), dim3(256), 0, L.stream, L.d_sys, L.nsys);
  }
  hipLaunchKernelGGL(k_bin_scatter, dim3(L.w_atoms.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
  hipLaunchKernelGGL(k_col_sort, dim3(L.w_cols.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_cols.pre);
  hipLaunchKernelGGL(k_pair_search, dim3(L.w_search.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_search.pre,
                     L.search_cap);
  hipLaunchKernelGGL(k_pair_fill, dim3(L.w_fill.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_fill.pre,
                     L.search_cap);
}

}  // namespace fz
