// fz_pme.hip -- smooth PME (order 4): spread, 3-D FFT, reciprocal convolution,
// force gather.
//
// Replaces the reference's lattice lists + ChargeSpread_small/_medium
// (src/cell_based_kernels.cu:1557-1765, src/pme_kernels.cu:20-380), the two
// cuFFT C2C transforms (src/mdcuda.cu:748,780), BCMultiply
// (src/cell_based_kernels.cu:1770) and PMEForce_medium/_large
// (src/pme_kernels.cu:381-773).  Differences by design: closed-form cardinal
// B-splines instead of the 1001-sample table (defect B2); atom-centric spread
// with order-independent accumulation (int64 fixed point in the mixed form);
// an own LDS FFT for 2,3,5-smooth sizes with real-to-complex / complex-to-real
// x passes, so only the half spectrum is stored and moved; the convolution,
// reciprocal energy and virial are fused into the z pass, which transforms
// forward, multiplies and transforms back while the line is in LDS.
//
// Conventions: Q(k) = sum_i q_i M4(u_x - k_x) M4(u_y - k_y) M4(u_z - k_z),
// u_d = K_d * frac_d; Qhat = unnormalised forward DFT; G(m) = CC/(pi V)
// exp(-pi^2 m^2 / beta^2) / m^2 * B(m), |b_d|^2 = 9 / (2 + cos(2 pi j / K_d))^2;
// E = 1/2 sum_m G |Qhat|^2; phi = unnormalised inverse DFT of G Qhat;
// F_i = -q_i sum_k grad(theta_i) phi(k).
#include "fz_device.h"
#include "fz_fft.h"
#include "fz_launch.h"

namespace fz {

// The weights are computed with no contraction into fused multiply-adds, so
// that every spread path (atomic, bricks, planes) forms bitwise the same values
// whatever code the compiler inlines them into.
template <class R>
__device__ __forceinline__ void bspline4(R f, R* th, R* dth) {
#pragma clang fp contract(off)
  const R f2 = f * f, f3 = f2 * f, g = R(1) - f;
  th[0] = g * g * g * R(1.0 / 6.0);
  th[1] = (R(3) * f3 - R(6) * f2 + R(4)) * R(1.0 / 6.0);
  th[2] = (R(-3) * f3 + R(3) * f2 + R(3) * f + R(1)) * R(1.0 / 6.0);
  th[3] = f3 * R(1.0 / 6.0);
  if (dth) {
    dth[0] = R(-0.5) * g * g;
    dth[1] = R(0.5) * (R(3) * f2 - R(4) * f);
    dth[2] = R(0.5) * (R(-3) * f2 + R(2) * f + R(1));
    dth[3] = R(0.5) * f2;
  }
}

// grid index (first of 4) and spline fraction from a 64-bit fixed-point fraction
template <class R>
__device__ __forceinline__ int spline_pos(unsigned long long u, int K, R& f) {
  const unsigned long long hi = __umul64hi(u, (unsigned long long)K);
  const unsigned long long lo = u * (unsigned long long)K;
  if (sizeof(R) == 4) f = (R)(float)(unsigned)(lo >> 40) * R(5.9604644775390625e-08);  // 2^-24
  else f = (R)(double)(lo >> 11) * R(1.1102230246251565e-16);                         // 2^-53
  int g = (int)hi - 3;
  return g < 0 ? g + K : g;
}

// weight k (0..3) of the order-4 cardinal B-spline at fraction f
template <class R>
__device__ __forceinline__ R bspline4_k(R f, int k) {
#pragma clang fp contract(off)
  const R f2 = f * f, f3 = f2 * f, g = R(1) - f;
  const R w0 = g * g * g, w1 = R(3) * f3 - R(6) * f2 + R(4), w2 = R(-3) * f3 + R(3) * f2 + R(3) * f + R(1);
  const R w = k == 0 ? w0 : k == 1 ? w1 : k == 2 ? w2 : f3;
  return w * R(1.0 / 6.0);
}

// ---------------------------------------------------------------------------
// Charge spreading with global atomics, for launches over few atoms, where the
// brick pipeline's four launches cost more than the contention they remove.
// One atom per wave iteration, one of its 4x4x4 grid points per lane: the 64
// atomics of an instruction fall on 16 rows of 4 consecutive x points.  Atoms
// are visited with a multiplier coprime to their count, so that concurrent
// waves work on distant atoms; the kernel reads no cluster slots and can run
// before the list build.  The wave's 64 atoms are read and placed on the grid
// in parallel first (lane k: the k-th atom).
// Qacc must be zero before; the x pass of the FFT clears it after reading.
// The mixed-form grid is the same integer sum as the brick path's.
__device__ __forceinline__ float bcast(float v, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k)); }
__device__ __forceinline__ double bcast(double v, int k) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k), __builtin_amdgcn_readlane(__double2loint(v), k));
}

template <bool MIXED>
__global__ __launch_bounds__(256) void k_spread_atomic(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int lane = threadIdx.x & 63;
  const int t0 = ((blockIdx.x - block_base(pre, nsys, s_)) * 4 + (threadIdx.x >> 6)) * 64;
  const int na = d.n_atoms;
  const unsigned long long mult = d.spread_mult;
  const int K0 = d.K[0], K1 = d.K[1], K2 = d.K[2];
  const int ca = lane & 3, cb = (lane >> 2) & 3, cc = lane >> 4;
  R q = R(0), fx = R(0), fy = R(0), fz = R(0);
  int gx0 = 0, gy0 = 0, gz0 = 0;
  bool has = false;
  if (t0 + lane < na) {
    const int a = (int)(((unsigned long long)(t0 + lane) * mult) % (unsigned long long)na);
    q = (R)d.q[a];
    has = q != R(0);
    gx0 = spline_pos<R>(d.ux[a], K0, fx);
    gy0 = spline_pos<R>(d.uy[a], K1, fy);
    gz0 = spline_pos<R>(d.uz[a], K2, fz);
  }
  unsigned long long bal = __ballot(has);
  while (bal) {
    const int k = __ffsll((long long)bal) - 1;
    bal &= bal - 1ull;
    int gx = __builtin_amdgcn_readlane(gx0, k) + ca;
    int gy = __builtin_amdgcn_readlane(gy0, k) + cb;
    int gz = __builtin_amdgcn_readlane(gz0, k) + cc;
    gx -= gx >= K0 ? K0 : 0;
    gy -= gy >= K1 ? K1 : 0;
    gz -= gz >= K2 ? K2 : 0;
    const R v = bcast(q, k) * bspline4_k<R>(bcast(fx, k), ca) * bspline4_k<R>(bcast(fy, k), cb) *
                bspline4_k<R>(bcast(fz, k), cc);
    const size_t g = ((size_t)gz * K1 + gy) * K0 + gx;
    if (MIXED) atomicAdd((unsigned long long*)d.Qacc + g, fixed_f32((float)v));
    else unsafeAtomicAdd((double*)d.Qacc + g, (double)v);
  }
}

// ---------------------------------------------------------------------------
// Charge spreading by bricks.  The grid is cut into bricks of 8^3 points; an
// atom belongs to the brick holding the first point of its 4^3 stencil, so its
// stencil lies inside the brick's (8+3)^3 block.  Per step:
//   count    atoms per brick (rank of each atom inside its brick),
//   scan     brick offsets (and the counts cleared for the next step),
//   scatter  per atom a record: stencil weights along x, y, z, charge, and the
//            stencil's first point inside the block,
//   spread   one workgroup per brick sums its atoms' 64 weights each into the
//            block in LDS (int64 fixed point at 2^32 per charge unit in the
//            mixed form, FP64 in the FP64 form) and stores the block,
//   reduce   every grid point adds the blocks that overlap it (at most 2 per
//            axis): the first transform's lines do, as they are read.
// No global atomics: the grid is an integer sum in the mixed form, the same
// for any order of the atoms, and bitwise equal to adding the 64 weights of
// every atom into the grid one by one.

constexpr int BRK = 8;          // brick edge (grid points)
constexpr int BRH = BRK + 3;    // block edge: brick + the stencil's reach
constexpr int BRV = BRH * BRH * BRH;

// Atoms, not cluster slots, are visited, so the spread needs nothing from the
// list build.  Consecutive atoms are mostly bonded neighbours, so the lanes of
// a wave fall into few bricks: one atomic per distinct brick of the wave,
// ranks in lane order after it.
template <bool MIXED>
__global__ __launch_bounds__(256) void k_brick_count(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int a = (blockIdx.x - block_base(pre, nsys, s_)) * 256 + threadIdx.x;
  const bool inside = a < d.n_atoms;
  int h = -1;
  if (inside) {
    if ((R)d.q[a] != R(0)) {
      R f;
      const int gx = spline_pos<R>(d.ux[a], d.K[0], f);
      const int gy = spline_pos<R>(d.uy[a], d.K[1], f);
      const int gz = spline_pos<R>(d.uz[a], d.K[2], f);
      h = (gx >> 3) + d.nbr[0] * ((gy >> 3) + d.nbr[1] * (gz >> 3));
    }
  }
  // the wave's groups of one brick first, then one atomic by the leaders of all: a
  // returning atomic per group, one after the other, took 12.6 us at 227,000 atoms (this 6.0)
  const int lane = threadIdx.x & 63;
  int leader = lane, rank = 0, count = 0;
  unsigned long long todo = __ballot(h >= 0);
  while (todo) {
    const int first = __ffsll((long long)todo) - 1;
    const unsigned long long m = __ballot(h == __builtin_amdgcn_readlane(h, first));
    if ((m >> lane) & 1ull) {
      leader = first;
      rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    }
    if (lane == first) count = __popcll(m);
    todo &= ~m;
  }
  const int base = count ? atomicAdd(d.br_cnt + h, count) : 0;
  rank += __shfl(base, leader, 64);
  if (inside) d.br_atom[a] = make_int2(h, rank);
}

// one block per system
__global__ __launch_bounds__(1024) void k_brick_scan(const SysDev* __restrict__ S, int nsys) {
  const SysDev& d = S[blockIdx.x];
  __shared__ int part[16];
  const int n = d.n_bricks, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per = (n + 1023) / 1024;
  const int c0 = threadIdx.x * per, c1 = min(n, c0 + per);
  int sum = 0;
#pragma unroll 8
  for (int c = c0; c < c1; c++) sum += d.br_cnt[c];
  int incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int below = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 16; w++) {
    below += w < wave ? part[w] : 0;
    total += part[w];
  }
  int run = below + incl - sum;
#pragma unroll 8
  for (int c = c0; c < c1; c++) {
    d.br_off[c] = run;
    run += d.br_cnt[c];
    d.br_cnt[c] = 0;
  }
  if (threadIdx.x == 0) d.br_off[n] = total;
}

template <bool MIXED>
__global__ __launch_bounds__(256) void k_brick_scatter(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int a = (blockIdx.x - block_base(pre, nsys, s_)) * 256 + threadIdx.x;
  if (a >= d.n_atoms) return;
  const int2 r = d.br_atom[a];
  if (r.x < 0) return;
  R fx, fy, fz;
  const int gx = spline_pos<R>(d.ux[a], d.K[0], fx);
  const int gy = spline_pos<R>(d.uy[a], d.K[1], fy);
  const int gz = spline_pos<R>(d.uz[a], d.K[2], fz);
  R* rec = (R*)d.br_rec + (size_t)(d.br_off[r.x] + r.y) * 16;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    rec[k] = bspline4_k<R>(fx, k);
    rec[4 + k] = bspline4_k<R>(fy, k);
    rec[8 + k] = bspline4_k<R>(fz, k);
  }
  rec[12] = (R)d.q[a];
  rec[13] = (R)((gx & 7) + BRH * ((gy & 7) + BRH * (gz & 7)));  // exact integer
}

// One workgroup per brick; a wave adds one atom's stencil per iteration, lane
// l holding point (l & 3, (l >> 2) & 3, l >> 4) of it.
template <bool MIXED>
__global__ __launch_bounds__(256) void k_brick_spread(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using A = typename std::conditional<MIXED, unsigned long long, double>::type;
  __shared__ A blk[BRV];
  __shared__ R rec[64 * 16];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int b = blockIdx.x - block_base(pre, nsys, s_);
  const int a0 = d.br_off[b], a1 = d.br_off[b + 1];
  A* out = (A*)d.br_part + (size_t)b * BRV;
  if (a0 == a1) {
    for (int i = threadIdx.x; i < BRV; i += 256) out[i] = A(0);
    return;
  }
  for (int i = threadIdx.x; i < BRV; i += 256) blk[i] = A(0);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ca = lane & 3, cb = (lane >> 2) & 3, cc = lane >> 4;
  const int lofs = ca + BRH * (cb + BRH * cc);
  const R* src = (const R*)d.br_rec;
  for (int base = a0; base < a1; base += 64) {
    const int n = min(64, a1 - base);
    __syncthreads();  // block cleared / previous records consumed
    for (int i = threadIdx.x; i < n * 16; i += 256) rec[i] = src[(size_t)base * 16 + i];
    __syncthreads();
    for (int k = wv; k < n; k += 4) {
      const R* r = rec + k * 16;
      const R v = r[12] * r[ca] * r[4 + cb] * r[8 + cc];
      const int loc = (int)r[13] + lofs;
      if (MIXED) atomicAdd((unsigned long long*)&blk[loc], fixed_f32((float)v));
      else atomicAdd((double*)&blk[loc], (double)v);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < BRV; i += 256) out[i] = blk[i];
}

// Block points over grid index x along one axis.  Blocks span the unwrapped
// coordinates [0, 8 nb + 3); every X = x + m K in that range is point X & 7 of
// brick X >> 3 (when that brick exists) and, when X & 7 < 3, point (X & 7) + 8
// of the brick before.  At most 4 entries for any K >= 4.
__device__ __forceinline__ int brick_cover(int x, int K, int nb, int* br, int* loc) {
  int n = 0;
  for (int X = x; X < BRK * nb + 3; X += K) {
    const int h = X >> 3, l = X & 7;
    if (h < nb) { br[n] = h; loc[n] = l; n++; }
    if (l < 3 && h >= 1) { br[n] = h - 1; loc[n] = l + BRK; n++; }
  }
  return n;
}

// The charge sums of nl lines of the grid along x, (y, z) from line l0 on, out of the
// blocks that overlap them, into q in LDS: per line the block rows over (y, z), per x
// the points of a row (both in the order z, y, x).
struct BrickCover {
  int row[64][16], rows[64];  // offsets into br_part
  int point[256][4];          // -1: none
};
template <class R, class A>
__device__ __forceinline__ void brick_lines(const SysDev& d, int l0, int nl, BrickCover& bc, R* q) {
  const int K0 = d.K[0], K1 = d.K[1], nb0 = d.nbr[0], nb1 = d.nbr[1];
  for (int x = threadIdx.x; x < K0; x += 256) {
    int c[4], l[4];
    const int n = brick_cover(x, K0, nb0, c, l);
#pragma unroll
    for (int i = 0; i < 4; i++) bc.point[x][i] = i < n ? c[i] * BRV + l[i] : -1;
  }
  for (int t = threadIdx.x; t < nl; t += 256) {
    const int z = (l0 + t) / K1, y = l0 + t - z * K1;
    int cy[4], ly[4], cz[4], lz[4];
    const int ny = brick_cover(y, K1, nb1, cy, ly), nz = brick_cover(z, d.K[2], d.nbr[2], cz, lz);
    int n = 0;
    for (int k = 0; k < nz; k++)
      for (int j = 0; j < ny; j++) bc.row[t][n++] = nb0 * (cy[j] + nb1 * cz[k]) * BRV + BRH * (ly[j] + BRH * lz[k]);
    bc.rows[t] = n;
  }
  __syncthreads();
  const A* part = (const A*)d.br_part;
  const unsigned m_k0 = fdiv_magic(K0);
  for (int t = threadIdx.x; t < nl * K0; t += 256) {
    const int line = fdiv(t, K0, m_k0), x = t - line * K0;
    const int n = bc.rows[line], p0 = bc.point[x][0], p1 = bc.point[x][1];
    A sum = A(0);
    if (n <= 4 && bc.point[x][2] < 0) {  // all but grids a few bricks across
      A v[4][2];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        v[r][0] = v[r][1] = A(0);
        if (r < n) {
          const int o = bc.row[line][r];
          v[r][0] = part[o + p0];
          if (p1 >= 0) v[r][1] = part[o + p1];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; r++) sum = (sum + v[r][0]) + v[r][1];
    } else {
      for (int r = 0; r < n; r++)
        for (int i = 0; i < 4 && bc.point[x][i] >= 0; i++) sum += part[bc.row[line][r] + bc.point[x][i]];
    }
    q[line * K0 + x] = sizeof(R) == 4 ? (R)from_fixed_acc((unsigned long long)sum) : (R)sum;
  }
}

void launch_spread(const Launch& L) {
  dim3 b(256);
  if (!L.spread_bricks) {
    if (L.mixed) hipLaunchKernelGGL(k_spread_atomic<true>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    else hipLaunchKernelGGL(k_spread_atomic<false>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    return;
  }
  if (L.mixed) {
    hipLaunchKernelGGL(k_brick_count<true>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    hipLaunchKernelGGL(k_brick_scan, dim3(L.nsys), dim3(1024), 0, L.stream, L.d_sys, L.nsys);
    hipLaunchKernelGGL(k_brick_scatter<true>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    hipLaunchKernelGGL(k_brick_spread<true>, dim3(L.w_bricks.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_bricks.pre);
  } else {
    hipLaunchKernelGGL(k_brick_count<false>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    hipLaunchKernelGGL(k_brick_scan, dim3(L.nsys), dim3(1024), 0, L.stream, L.d_sys, L.nsys);
    hipLaunchKernelGGL(k_brick_scatter<false>, dim3(L.w_atoms.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
    hipLaunchKernelGGL(k_brick_spread<false>, dim3(L.w_bricks.total), b, 0, L.stream, L.d_sys, L.nsys, L.w_bricks.pre);
  }
}

// ---------------------------------------------------------------------------
// grid passes: NL lines per workgroup (fz_fft.h); LDS: two line buffers and the
// axis' twiddles

// the axis' twiddles (K entries) into LDS after the two line buffers
template <class C>
__device__ __forceinline__ const C* stage_tw(C* lds, const C* __restrict__ tw, int K) {
  for (int k = threadIdx.x; k < K; k += blockDim.x) lds[k] = tw[k];
  return lds;
}

// x pass, forward: real grid -> half spectrum.  BRICKS: the grid's lines are summed out
// of the bricks' blocks first (as a kernel of its own, through the grid: 39 + 15 us at
// 144^3; this 46, without the launch between); otherwise the grid is read and cleared,
// as the next atomic spread needs it.
template <bool MIXED, bool BRICKS>
__global__ __launch_bounds__(256) void k_fft_x_r2c(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre, int NL) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  using A = typename std::conditional<MIXED, unsigned long long, double>::type;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int lb = blockIdx.x - block_base(pre, nsys, s_);
  const int K0 = d.K[0], nlines = d.K[1] * d.K[2], Kxh = d.Kxh, LS = fft_line(K0, 1, sizeof(C));
  C* b0 = (C*)smem;
  C* b1 = b0 + NL * LS;
  const int l0 = lb * NL, nl = min(NL, nlines - l0);
  const C* twl = stage_tw(b1 + NL * LS, (const C*)d.tw, K0);
  R* q = (R*)b1;
  if (BRICKS) {
    __shared__ BrickCover bc;
    brick_lines<R, A>(d, l0, nl, bc, q);
  }
  __syncthreads();
  C* Qc = (C*)d.Qc;
  fft_lines<C, R, false>(
      nl, K0, 1, twl, R(-1), b0, b1, LS,
      [&](int line, int x) {
        C v;
        v.y = R(0);
        if (BRICKS) {
          v.x = q[line * K0 + x];
          return v;
        }
        const size_t g = (size_t)(l0 + line) * K0 + x;
        A* Q = (A*)d.Qacc;
        v.x = MIXED ? (R)from_fixed_acc((unsigned long long)Q[g]) : (R)Q[g];
        Q[g] = A(0);
        return v;
      },
      [&](int line, int kx, C v, C*) {
        if (kx < Kxh) Qc[(size_t)(l0 + line) * Kxh + kx] = v;
      });
}

// y pass (either direction): lines along y for NL consecutive kx at fixed z
template <bool MIXED>
__global__ __launch_bounds__(256) void k_fft_y(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre, int NL, int dirv) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int lb = blockIdx.x - block_base(pre, nsys, s_);
  const int K1 = d.K[1], Kxh = d.Kxh, LS = fft_line(K1, 1, sizeof(C));
  const int ng = (Kxh + NL - 1) / NL;
  const int z = lb / ng, kx0 = (lb - z * ng) * NL;
  C* b0 = (C*)smem;
  C* b1 = b0 + NL * LS;
  const C* twl = stage_tw(b1 + NL * LS, (const C*)d.tw + d.K[0], K1);
  __syncthreads();
  C* Q = (C*)d.Qc + (size_t)z * K1 * Kxh + kx0;
  fft_lines<C, R, true>(
      min(NL, Kxh - kx0), K1, 1, twl, R(dirv), b0, b1, LS, [&](int l, int y) { return Q[(size_t)y * Kxh + l]; },
      [&](int l, int y, C v, C*) { Q[(size_t)y * Kxh + l] = v; });
}

// G(m) of grid point (kx, y, z) and |m|^2 from the per-axis tables, with no
// contraction into fused multiply-adds: the table below and the z pass form
// bitwise the same value.  (kx, y, z) = 0 is not evaluated here.
__device__ __forceinline__ double pme_G(const double* __restrict__ mt, const double* __restrict__ ex,
                                        const double* __restrict__ bsp, double pre, int K0, int K1, int kx, int y, int z,
                                        double& m2) {
#pragma clang fp contract(off)
  const double mx = mt[kx], my = mt[K0 + y], mz = mt[K0 + K1 + z];
  m2 = mx * mx + my * my + mz * mz;
  return pre * ex[kx] * ex[K0 + y] * ex[K0 + K1 + z] * bsp[kx] * bsp[K0 + y] * bsp[K0 + K1 + z] / m2;
}

// G(m) over the half spectrum ([z][y][kx], G(0) = 0) for a fixed box, once
// per system: the z pass reads it instead of forming it per point
__global__ __launch_bounds__(256) void k_pme_gtable(double* __restrict__ G, const double* __restrict__ mt,
                                                    const double* __restrict__ ex, const double* __restrict__ bsp,
                                                    double pre, int K0, int K1, int K2, int Kxh) {
  const size_t n = (size_t)K2 * K1 * Kxh;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const int kx = (int)(i % Kxh), y = (int)((i / Kxh) % K1), z = (int)(i / ((size_t)Kxh * K1));
    double m2;
    G[i] = (kx == 0 && y == 0 && z == 0) ? 0.0 : pme_G(mt, ex, bsp, pre, K0, K1, kx, y, z, m2);
  }
}

void launch_pme_gtable(const SysDev& d, hipStream_t st) {
  const size_t n = (size_t)d.K[2] * d.K[1] * d.Kxh;
  const int blocks = (int)std::min<size_t>(4096, (n + 255) / 256);
  hipLaunchKernelGGL(k_pme_gtable, dim3(blocks), dim3(256), 0, st, d.pme_g, d.pme_m, d.pme_ex, d.pme_bsp, d.pme_pre,
                     d.K[0], d.K[1], d.K[2], d.Kxh);
}

// z pass: forward FFT, multiply by G(m) (mode 0) or 1 (mode 1), energy and
// virial, inverse FFT.  G comes from the system's table when it has one (fixed
// box) and is formed per point otherwise (barostat: the box changes every step).
template <bool MIXED, bool EV>
__global__ __launch_bounds__(256) void k_fft_z_conv(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre, int NL, int mode) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int lb = blockIdx.x - block_base(pre, nsys, s_);
  const int K0 = d.K[0], K1 = d.K[1], K2 = d.K[2], Kxh = d.Kxh, LS = fft_line(K2, 1, sizeof(C));
  const int ng = (Kxh + NL - 1) / NL;
  const int y = lb / ng, kx0 = (lb - y * ng) * NL, nl = min(NL, Kxh - kx0);
  C* b0 = (C*)smem;
  C* b1 = b0 + NL * LS;
  const C* twz = stage_tw(b1 + NL * LS, (const C*)d.tw + K0 + K1, K2);
  __syncthreads();
  const size_t zs = (size_t)K1 * Kxh;
  C* Q = (C*)d.Qc + (size_t)y * Kxh + kx0;
  const double* Gt = !EV && mode == 0 && d.pme_g ? d.pme_g + (size_t)y * Kxh + kx0 : nullptr;
  C* res = fft_lines<C, R, true>(
      nl, K2, 1, twz, R(-1), b0, b1, LS, [&](int l, int z) { return Q[z * zs + l]; },
      [&](int l, int z, C v, C* out) {
        if (Gt) {
          const double G = Gt[z * zs + l];
          v.x = (R)(v.x * G);
          v.y = (R)(v.y * G);
        }
        out[l * LS + z] = v;
      });
  __syncthreads();
  if (!Gt) {  // G formed per point, energies
    double ev[10];
#pragma unroll
    for (int k = 0; k < 10; k++) ev[k] = 0.0;
    const unsigned m_k2 = fdiv_magic(K2);
    for (int e = threadIdx.x; e < nl * K2; e += 256) {
      const int l = fdiv(e, K2, m_k2), z = e - l * K2;
      const int kx = kx0 + l;
      C v = res[l * LS + z];
      double G = 1.0;
      if (mode == 0) {
        if (kx == 0 && y == 0 && z == 0) {
          G = 0.0;
        } else {
          double m2;
          G = pme_G(d.pme_m, d.pme_ex, d.pme_bsp, d.pme_pre, K0, K1, kx, y, z, m2);
          if (EV) {
            const double mx = d.pme_m[kx], my = d.pme_m[K0 + y], mz = d.pme_m[K0 + K1 + z];
            const double wgt = (kx == 0 || 2 * kx == K0) ? 1.0 : 2.0;
            const double Em = 0.5 * wgt * G * ((double)v.x * v.x + (double)v.y * v.y);
            const double fac = 2.0 * (1.0 + d.pi2_beta2 * m2) / m2;
            ev[0] += Em;
            const double mm[3] = {mx, my, mz};
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
              for (int b = 0; b < 3; b++) ev[1 + 3 * a + b] += Em * ((a == b ? 1.0 : 0.0) - fac * mm[a] * mm[b]);
          }
        }
      }
      v.x = (R)(v.x * G);
      v.y = (R)(v.y * G);
      res[l * LS + z] = v;
    }
    __syncthreads();
    if (EV && mode == 0) {
      const int slots[10] = {A_PME, A_VIR + 0, A_VIR + 1, A_VIR + 2, A_VIR + 3, A_VIR + 4,
                             A_VIR + 5, A_VIR + 6, A_VIR + 7, A_VIR + 8};
      block_acc_fixed<10>(ev, d.acc, slots);
    }
  }
  fft_lines<C, R, true>(
      nl, K2, 1, twz, R(1), res == b0 ? b1 : b0, res, LS, [&](int l, int z) { return res[l * LS + z]; },
      [&](int l, int z, C v, C*) { Q[z * zs + l] = v; });
}

// x pass, inverse: half spectrum -> real potential grid
template <bool MIXED>
__global__ __launch_bounds__(256) void k_fft_x_c2r(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre, int NL) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int lb = blockIdx.x - block_base(pre, nsys, s_);
  const int K0 = d.K[0], nlines = d.K[1] * d.K[2], Kxh = d.Kxh, LS = fft_line(K0, 1, sizeof(C));
  C* b0 = (C*)smem;
  C* b1 = b0 + NL * LS;
  const int l0 = lb * NL;
  const C* twl = stage_tw(b1 + NL * LS, (const C*)d.tw, K0);
  __syncthreads();
  const C* Q = (const C*)d.Qc + (size_t)l0 * Kxh;
  R* phi = (R*)d.phi + (size_t)l0 * K0;
  fft_lines<C, R, false>(
      min(NL, nlines - l0), K0, 1, twl, R(1), b0, b1, LS,
      [&](int line, int k) {
        const bool up = k >= Kxh;  // conjugate half
        C v = Q[line * Kxh + (up ? K0 - k : k)];
        v.y = up ? -v.y : v.y;
        return v;
      },
      [&](int line, int x, C v, C*) { phi[line * K0 + x] = v.x; });
}

// ---------------------------------------------------------------------------
// Plane kernels, for systems of up to a few ten thousand atoms whose grid
// plane fits in LDS: one workgroup per z plane.
//
// Forward: the plane's charge sum, then its x (real to half spectrum) and y
// transforms, all in LDS.  Each workgroup looks at the high words of every atom's z
// position, 32 atoms per thread at a time; a wave lists the atoms whose stencil covers
// the plane and spreads 64 of them together, one per lane (16 points each) with LDS
// atomics, as int64 fixed point in the mixed form: the same terms and integer
// sums as the global-atomic and brick spreads, so the plane holds the same
// values, and the line transforms are those of the x and y passes, so the half
// spectrum is the same to the bit.  No grid accumulator is read or cleared.
// Inverse: y, then x (half spectrum to real) transforms of the plane into the
// potential grid, again the passes' arithmetic.
// LDS: plane_dyn_lds (the charge sum lives in the second buffer until it is read, the
// waves' lists in the first).
// What bounds it: the latency of the scan, of one gather of the listed atoms and of
// the transforms' passes: few workgroups, one per plane.  Eight atoms at a time, those
// on the plane found by ballot and spread four to a wave by shuffles, the forward
// kernel took 37 us at 19,000 atoms and 15.8 at 1,000; this 23.1 and 12.8.
// Workgroups of NT threads: 1,024 where a launch holds few planes (the atom
// scan of one workgroup per plane needs many waves to hide its load latency
// behind) or a plane takes most of a compute unit's LDS, 512 of them where planes are
// small (the passes have no work for more), 256 where it holds many (a batch of small
// systems: more workgroups per CU).  1,024 -> 512 threads, forward and inverse: 24 x 24
// points 12.7 -> 11.1 and 8.7 -> 7.0 us, 45 x 45 in FP64 20.0 -> 19.2 and 11.5 -> 10.2;
// 88 x 88 46 -> 61 forward.
constexpr int PLANE_SCAN = 32;  // atoms per thread looked at together

template <bool MIXED, int NT>
__global__ __launch_bounds__(NT) void k_pme_plane_fwd(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  using A = typename std::conditional<MIXED, unsigned long long, double>::type;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int z = blockIdx.x - block_base(pre, nsys, s_);
  const int K0 = d.K[0], K1 = d.K[1], K2 = d.K[2], Kxh = d.Kxh;
  const int KP = K0 * K1, pad = plane_pad(K0, K1, sizeof(C)), PB = plane_buf(K0, K1, pad, sizeof(C));
  C* b0 = (C*)smem;
  C* b1 = b0 + PB;
  C* twx = b1 + PB;
  C* twy = twx + K0;
  A* acc = (A*)b1;
  for (int e = threadIdx.x; e < KP; e += NT) acc[e] = A(0);
  for (int k = threadIdx.x; k < K0 + K1; k += NT) twx[k] = ((const C*)d.tw)[k];
  __syncthreads();
  const int na = d.n_atoms, lane = threadIdx.x & 63;
  int* list = (int*)b0 + (threadIdx.x >> 6) * PLANE_LIST;  // the wave's atoms of the plane; free until the transforms
  int n = 0;
  const FZ_GLOBAL unsigned* uz32 = (const FZ_GLOBAL unsigned*)d.uz;  // high words at odd indices
  for (int base = 0; base < na; base += NT * PLANE_SCAN) {
    unsigned hz[PLANE_SCAN];
#pragma unroll
    for (int k = 0; k < PLANE_SCAN; k++)
      if (base + k * NT < na) hz[k] = uz32[2 * min(base + k * NT + (int)threadIdx.x, na - 1) + 1];
    // the cell of the high word is the atom's, or the one below where the low word carries
    unsigned bits = 0u;
#pragma unroll
    for (int k = 0; k < PLANE_SCAN; k++)
      if (base + k * NT < na) {
        const unsigned long long p = (unsigned long long)hz[k] * (unsigned)K2;
        int c = z + 3 - (int)(p >> 32);
        c += c < 0 ? K2 : 0;
        c -= c >= K2 ? K2 : 0;
        const bool hit = (c < 4 || (c == 4 && (unsigned)p >= 0u - (unsigned)K2)) && base + k * NT + (int)threadIdx.x < na;
        bits |= hit ? 1u << k : 0u;
      }
    const bool end = base + NT * PLANE_SCAN >= na;
    while (true) {
      const unsigned long long m = __ballot(bits != 0u);
      if (bits) {
        const int at = n + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        list[at] = base + (__ffs((int)bits) - 1) * NT + (int)threadIdx.x;
        bits &= bits - 1u;
      }
      n += __builtin_popcountll(m);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (n >= 64 || (!m && end && n > 0)) {  // an atom per lane
        if (lane < n) {
          const int a = list[lane];
          R fx, fy, fz;
          const R q = (R)d.q[a];
          const int gx = spline_pos<R>(d.ux[a], K0, fx), gy = spline_pos<R>(d.uy[a], K1, fy);
          int c = z - spline_pos<R>(d.uz[a], K2, fz);
          c += c < 0 ? K2 : 0;
          if (c < 4 && q != R(0)) {
            const R wz = bspline4_k<R>(fz, c);
            R qx[4];
            int ix[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
              qx[i] = q * bspline4_k<R>(fx, i);
              ix[i] = gx + i - (gx + i >= K0 ? K0 : 0);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const R wy = bspline4_k<R>(fy, j);
              A* row = acc + (gy + j - (gy + j >= K1 ? K1 : 0)) * K0;
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const R v = qx[i] * wy * wz;
                if (MIXED) atomicAdd((unsigned long long*)&row[ix[i]], fixed_f32((float)v));
                else atomicAdd((double*)&row[ix[i]], (double)v);
              }
            }
          }
        }
        const int rest = n - 64;
        const int keep = lane < rest ? list[64 + lane] : 0;
        if (lane < rest) list[lane] = keep;
        n = max(rest, 0);
      }
      if (!m) break;
    }
  }
  __syncthreads();
  // x lines (one per y) out of the charge sum, kept kx as y lines, then those
  const int LX = fft_line(K0, pad, sizeof(C)), LY = fft_line(K1, pad, sizeof(C));
  C* r = fft_lines<C, R, false>(
      K1, K0, pad, twx, R(-1), b0, b1, LX,
      [&](int y, int x) {
        C v;
        v.x = MIXED ? (R)from_fixed_acc(((const unsigned long long*)acc)[y * K0 + x]) : (R)((const double*)acc)[y * K0 + x];
        v.y = R(0);
        return v;
      },
      [&](int y, int kx, C v, C* out) {
        if (kx < Kxh) out[kx * LY + y] = v;
      });
  __syncthreads();
  C* Qc = (C*)d.Qc + (size_t)z * K1 * Kxh;
  fft_lines<C, R, true>(
      Kxh, K1, pad, twy, R(-1), r == b0 ? b1 : b0, r, LY, [&](int kx, int y) { return r[kx * LY + y]; },
      [&](int kx, int y, C v, C*) { Qc[y * Kxh + kx] = v; });
}

template <bool MIXED, int NT>
__global__ __launch_bounds__(NT) void k_pme_plane_inv(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using C = typename C2<R>::t;
  extern __shared__ char smem[];
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int z = blockIdx.x - block_base(pre, nsys, s_);
  const int K0 = d.K[0], K1 = d.K[1], Kxh = d.Kxh;
  const int pad = plane_pad(K0, K1, sizeof(C)), PB = plane_buf(K0, K1, pad, sizeof(C));
  C* b0 = (C*)smem;
  C* b1 = b0 + PB;
  C* twx = b1 + PB;
  C* twy = twx + K0;
  for (int k = threadIdx.x; k < K0 + K1; k += NT) twx[k] = ((const C*)d.tw)[k];
  __syncthreads();
  const C* Qc = (const C*)d.Qc + (size_t)z * K1 * Kxh;
  const int LX = fft_line(K0, pad, sizeof(C)), LY = fft_line(K1, pad, sizeof(C));
  C* r = fft_lines<C, R, true>(
      Kxh, K1, pad, twy, R(1), b0, b1, LY, [&](int kx, int y) { return Qc[y * Kxh + kx]; },
      [&](int kx, int y, C v, C* out) { out[kx * LY + y] = v; });
  __syncthreads();
  R* phi = (R*)d.phi + (size_t)z * K0 * K1;
  fft_lines<C, R, false>(
      K1, K0, pad, twx, R(1), r == b0 ? b1 : b0, r, LX,
      [&](int y, int k) {
        const bool up = k >= Kxh;
        C v = r[(up ? K0 - k : k) * LY + y];
        v.y = up ? -v.y : v.y;
        return v;
      },
      [&](int y, int x, C v, C*) { phi[y * K0 + x] = v.x; });
}

// Force gather into the atom-ordered gather term (a store: each atom has one):
// it needs no slot layout, so it runs beside the neighbour build.  The sum over
// the 4x4x4 stencil is formed per stencil plane c (16 potential values each),
// and the planes' partial sums are added as (p0 + p1) + (p2 + p3), with no
// contraction into fused multiply-adds.  LPA lanes per atom: with 4 (launches
// over few atoms, latency bound) lane c forms plane c's sum and the quad adds
// them by lane exchange; with 1 (many atoms) one lane forms all four.  Both
// give the same bits, so a system's trajectory does not depend on the batch
// around it.
template <bool MIXED, int LPA>
__global__ __launch_bounds__(256) void k_pme_gather(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
#pragma clang fp contract(off)
  using R = typename std::conditional<MIXED, float, double>::type;
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int a = (blockIdx.x - block_base(pre, nsys, s_)) * (256 / LPA) + (int)(threadIdx.x / LPA);
  const int c0 = (int)(threadIdx.x % LPA);
  if (a >= d.n_atoms) return;  // the atom's lanes together
  const double qd = d.q[a];
  const int n = d.n_atoms;
  if (qd == 0.0) {
    if (c0 == 0) {
      if (MIXED) {
        unsigned long long* F = (unsigned long long*)d.Fg;
        F[a] = 0ull; F[n + a] = 0ull; F[2 * n + a] = 0ull;
      } else {
        double* F = (double*)d.Fg;
        F[a] = 0.0; F[n + a] = 0.0; F[2 * n + a] = 0.0;
      }
    }
    return;  // the atom's lanes together
  }
  const int K0 = d.K[0], K1 = d.K[1], K2 = d.K[2];
  R fx, fy, fz, tx[4], ty[4], tz[4], dx[4], dy[4], dz[4];
  const int gx = spline_pos<R>(d.ux[a], K0, fx);
  const int gy = spline_pos<R>(d.uy[a], K1, fy);
  const int gz = spline_pos<R>(d.uz[a], K2, fz);
  bspline4<R>(fx, tx, dx);
  bspline4<R>(fy, ty, dy);
  bspline4<R>(fz, tz, dz);
  const R* phi = (const R*)d.phi;
  int ix[4];
#pragma unroll
  for (int k = 0; k < 4; k++) ix[k] = gx + k >= K0 ? gx + k - K0 : gx + k;
  // per plane partial sums (this lane's planes)
  R p0[4 / LPA], p1[4 / LPA], p2[4 / LPA];
#pragma unroll
  for (int j = 0; j < 4 / LPA; j++) {
    const int c = j * LPA + c0;
    const R tzc = LPA == 1 ? tz[j] : (c == 0 ? tz[0] : c == 1 ? tz[1] : c == 2 ? tz[2] : tz[3]);
    const R dzc = LPA == 1 ? dz[j] : (c == 0 ? dz[0] : c == 1 ? dz[1] : c == 2 ? dz[2] : dz[3]);
    const int z = gz + c >= K2 ? gz + c - K2 : gz + c;
    R g0 = 0, g1 = 0, g2 = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int y = gy + b >= K1 ? gy + b - K1 : gy + b;
      const R* row = phi + ((size_t)z * K1 + y) * K0;
      R sx = 0, sdx = 0;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const R p = row[ix[k]];
        sx += tx[k] * p;
        sdx += dx[k] * p;
      }
      g0 += sdx * ty[b] * tzc;
      g1 += sx * dy[b] * tzc;
      g2 += sx * ty[b] * dzc;
    }
    p0[j] = g0; p1[j] = g1; p2[j] = g2;
  }
  R g0, g1, g2;
  if (LPA == 4) {
    g0 = p0[0]; g1 = p1[0]; g2 = p2[0];
    g0 += __shfl_xor(g0, 1, 64); g1 += __shfl_xor(g1, 1, 64); g2 += __shfl_xor(g2, 1, 64);
    g0 += __shfl_xor(g0, 2, 64); g1 += __shfl_xor(g1, 2, 64); g2 += __shfl_xor(g2, 2, 64);
    if (c0 != 0) return;
  } else {
    g0 = (p0[0] + p0[1 % (4 / LPA)]) + (p0[2 % (4 / LPA)] + p0[3 % (4 / LPA)]);
    g1 = (p1[0] + p1[1 % (4 / LPA)]) + (p1[2 % (4 / LPA)] + p1[3 % (4 / LPA)]);
    g2 = (p2[0] + p2[1 % (4 / LPA)]) + (p2[2 % (4 / LPA)] + p2[3 % (4 / LPA)]);
  }
  const double fxv = -qd * (double)g0 * K0 / d.L[0];
  const double fyv = -qd * (double)g1 * K1 / d.L[1];
  const double fzv = -qd * (double)g2 * K2 / d.L[2];
  if (MIXED) {
    unsigned long long* F = (unsigned long long*)d.Fg;
    F[a] = to_fixed_acc(fxv);
    F[n + a] = to_fixed_acc(fyv);
    F[2 * n + a] = to_fixed_acc(fzv);
  } else {
    double* F = (double*)d.Fg;
    F[a] = fxv;
    F[n + a] = fyv;
    F[2 * n + a] = fzv;
  }
}

template <bool MIXED>
static void launch_gather(const Launch& L) {
  // four lanes per atom up to GATHER_QUAD_BLOCKS blocks of 256 atoms per launch
  if (L.w_atoms.total <= GATHER_QUAD_BLOCKS)
    hipLaunchKernelGGL((k_pme_gather<MIXED, 4>), dim3(L.w_atoms64.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms64.pre);
  else
    hipLaunchKernelGGL((k_pme_gather<MIXED, 1>), dim3(L.w_atoms.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_atoms.pre);
}

template <bool MIXED>
static void launch_fft_passes(const Launch& L, bool ev, int mode, bool bricks) {
  const size_t lds = L.fft_lds;
  const int NL = L.fft_nl;
  if (bricks) hipLaunchKernelGGL((k_fft_x_r2c<MIXED, true>), dim3(L.w_fftx.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftx.pre, NL);
  else hipLaunchKernelGGL((k_fft_x_r2c<MIXED, false>), dim3(L.w_fftx.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftx.pre, NL);
  hipLaunchKernelGGL(k_fft_y<MIXED>, dim3(L.w_ffty.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_ffty.pre, NL, -1);
  if (ev) hipLaunchKernelGGL((k_fft_z_conv<MIXED, true>), dim3(L.w_fftz.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftz.pre, NL, mode);
  else hipLaunchKernelGGL((k_fft_z_conv<MIXED, false>), dim3(L.w_fftz.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftz.pre, NL, mode);
  hipLaunchKernelGGL(k_fft_y<MIXED>, dim3(L.w_ffty.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_ffty.pre, NL, 1);
  hipLaunchKernelGGL(k_fft_x_c2r<MIXED>, dim3(L.w_fftx.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftx.pre, NL);
}

template <bool MIXED, int NT>
static void launch_planes(const Launch& L, int part, bool ev) {
  if (part == 0) {
    hipLaunchKernelGGL((k_pme_plane_fwd<MIXED, NT>), dim3(L.w_planes.total), dim3(NT), L.plane_lds, L.stream, L.d_sys, L.nsys,
                       L.w_planes.pre);
    return;
  }
  const size_t lds = L.fft_lds;
  const int NL = L.fft_nl;
  if (ev) hipLaunchKernelGGL((k_fft_z_conv<MIXED, true>), dim3(L.w_fftz.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftz.pre, NL, 0);
  else hipLaunchKernelGGL((k_fft_z_conv<MIXED, false>), dim3(L.w_fftz.total), dim3(256), lds, L.stream, L.d_sys, L.nsys, L.w_fftz.pre, NL, 0);
  hipLaunchKernelGGL((k_pme_plane_inv<MIXED, NT>), dim3(L.w_planes.total), dim3(NT), L.plane_lds, L.stream, L.d_sys, L.nsys,
                     L.w_planes.pre);
}

void launch_pme_part(const Launch& L, int part, bool ev) {
  if (L.w_fftx.total == 0) return;
  if (part < 2 && L.pme_planes) {
    const bool wide = L.w_planes.total < PLANE_WIDE_BELOW || L.plane_lds > PLANE_SMALL_LDS;
    const bool mid = wide && L.plane_points <= PLANE_MID_POINTS;
    if (L.mixed) mid ? launch_planes<true, 512>(L, part, ev) : wide ? launch_planes<true, 1024>(L, part, ev) : launch_planes<true, 256>(L, part, ev);
    else mid ? launch_planes<false, 512>(L, part, ev) : wide ? launch_planes<false, 1024>(L, part, ev) : launch_planes<false, 256>(L, part, ev);
  } else if (part == 0) {
    launch_spread(L);
  } else if (part == 1) {
    if (L.mixed) launch_fft_passes<true>(L, ev, 0, L.spread_bricks);
    else launch_fft_passes<false>(L, ev, 0, L.spread_bricks);
  } else {
    if (L.mixed) launch_gather<true>(L);
    else launch_gather<false>(L);
  }
}

void launch_pme_fft_only(const Launch& L, int conv_mode) {
  if (L.mixed) launch_fft_passes<true>(L, true, conv_mode, false);
  else launch_fft_passes<false>(L, true, conv_mode, false);
}

}  // namespace fz
