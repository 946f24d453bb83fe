// fz_pair.hip -- real-space LJ + Ewald pair kernel over the cluster-pair list.
//
// Replaces the reference's nonbondforce (src/nonbonded_forces.cu:25-270): same
// functional forms (erfc Coulomb, CHARMM-switched LJ with the exact gradient
// of the switched energy, reference defect B1 not reproduced), Newton's third
// law instead of a full list.
//
// One wave64 evaluates one or two 8x8 tiles (an i cluster x eight j slots) per
// pair group: lane l holds i = l & 7, j = l >> 3.  j forces are summed over the 8
// lanes that share j (xor 1, 2, 4), tile by tile, and added once per group (in the
// mixed form the tiles' sums are added in fixed point: a sum of both in FP32 would
// round once more and saved nothing, 227,000 atoms 288 and 290 us); i forces stay in
// registers for the whole work item (a run of the groups of two clusters), then are
// reduced over lanes l, l+8, ... (xor 8, 16, 32).
//
// What bounds it: vector issue (every lane of a tile costs the same whether its
// pair is inside the cutoff or not), and the j-force atomics, which resolve beyond
// the per-XCD L2 at 21-23 G cache lines of 64 bytes a second whatever is in them.
// A tile of two whole clusters carries a pair inside the cutoff in 0.33 of its
// lanes (cutoff 12, list 13.5; 0.29 at 10 / 11.5): most j clusters of an entry
// reach the list distance with some of their atoms only.  The groups hold the j
// slots one by one, without those no atom of the i cluster is near: 0.46 and 0.41
// of the lanes, three tenths fewer tiles.  With a list per i cluster the atomics then
// bound the kernel (227,000 atoms: 400 us, 234 without them); two neighbouring
// clusters share their groups, which leaves 0.64 of the cache lines.  A j slot's
// record is one 32-byte sector, gathered with a per-lane byte offset that the list
// holds ready (no address arithmetic).
//
// Mixed form: int32 fixed-point displacements (the top 32 bits of the 64-bit
// fractions; int32 wrap-around is the minimum image), FP32 arithmetic, own
// FP32 erfc fit, int64 fixed-point force sums (order independent).
// FP64 form: int64 displacements, FP64 arithmetic, FP64 atomics.
#include "fz_device.h"
#include "fz_erfc_fit.h"
#include "fz_launch.h"

namespace fz {

// ---------------------------------------------------------------------------
// Slot-ordered copies of positions, charges and LJ parameters for the pair
// kernel (k_step_first and the list build keep them current in dynamics).
template <bool MIXED>
__global__ __launch_bounds__(256) void k_gather_sorted(const SysDev* __restrict__ S, int nsys, const int* __restrict__ pre) {
  const int s_ = block_sys(pre, nsys, blockIdx.x);
  const SysDev& d = S[s_];
  const int sl = (blockIdx.x - block_base(pre, nsys, s_)) * 256 + threadIdx.x;
  // (more clusters than the capacity: counted by a build that was then left out)
  if (sl >= min(*d.n_clusters * CLUSTER, d.n_slots_cap)) return;
  store_slot(d, sl, d.slot_atom[sl]);
}

// chunks of an entry list
__device__ __forceinline__ int entry_chunks(const SysDev& d) { return (int)((*d.n_pairs + PAIR_CHUNK - 1) / PAIR_CHUNK); }

// One block: the pair kernels' work items (none of a system after an overflow)
// as prefixes over the systems of a batch: those of pair groups, then those of
// entry lists (low and high word of one scan).
// Systems are taken 1024 at a time, one per thread, with a block scan and a
// running carry.  MODE 0: every system, and the rebuild decisions are spent;
// MODE 1: only the systems without a pending rebuild (their lists are valid
// before the build runs); MODE 2: only the systems with one (after the build),
// and the rebuild decisions are spent.
template <int MODE>
__global__ __launch_bounds__(1024) void k_chunk_prefix(const SysDev* __restrict__ S, int nsys, int* __restrict__ chunk_pre) {
  __shared__ unsigned long long part[1024];
  __shared__ unsigned long long carry;
  const int t = threadIdx.x;
  int* entry_pre = chunk_pre + nsys + 1;
  if (t == 0) { carry = 0ull; chunk_pre[0] = entry_pre[0] = 0; }
  for (int base = 0; base < nsys; base += 1024) {
    const int s = base + t;
    unsigned long long c = 0ull;
    if (s < nsys) {
      const bool pending = S[s].flags[F_REBUILD] != 0;
      const bool take = MODE == 0 || (MODE == 1 ? !pending : pending);
      if (take && !S[s].flags[F_OVERFLOW])
        c = S[s].entry_list ? (unsigned long long)(unsigned)entry_chunks(S[s]) << 32 : *S[s].pg_n >> 40;
      if (MODE != 1) S[s].flags[F_REBUILD] = 0;
    }
    part[t] = c;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {  // Hillis-Steele inclusive scan
      const unsigned long long v = t >= o ? part[t - o] : 0ull;
      __syncthreads();
      part[t] += v;
      __syncthreads();
    }
    if (s < nsys) {
      const unsigned long long v = carry + part[t];
      chunk_pre[s + 1] = (int)(unsigned)v;
      entry_pre[s + 1] = (int)(unsigned)(v >> 32);
    }
    __syncthreads();
    if (t == 1023) carry += part[1023];
    __syncthreads();
  }
}

void launch_chunk_prefix(const Launch& L) {
  hipLaunchKernelGGL(k_chunk_prefix<0>, dim3(1), dim3(1024), 0, L.stream, L.d_sys, L.nsys, L.chunk_pre);
}
void launch_chunk_split(const Launch& L, bool built) {
  if (built) hipLaunchKernelGGL(k_chunk_prefix<2>, dim3(1), dim3(1024), 0, L.stream, L.d_sys, L.nsys, L.chunk_pre);
  else hipLaunchKernelGGL(k_chunk_prefix<1>, dim3(1), dim3(1024), 0, L.stream, L.d_sys, L.nsys, L.chunk_pre_a);
}

void launch_gather_sorted(const Launch& L) {
  if (L.mixed)
    hipLaunchKernelGGL(k_gather_sorted<true>, dim3(L.w_slots.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_slots.pre);
  else
    hipLaunchKernelGGL(k_gather_sorted<false>, dim3(L.w_slots.total), dim3(256), 0, L.stream, L.d_sys, L.nsys, L.w_slots.pre);
  launch_chunk_prefix(L);
}

// ---------------------------------------------------------------------------
__device__ __forceinline__ int rfl(int v) { return __builtin_amdgcn_readfirstlane(v); }
// DPP lane moves within rows: quad_perm [1,0,3,2] (xor 1), quad_perm [2,3,0,1]
// (xor 2), row_half_mirror (i <-> 7 - i inside each group of 8)
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// sum over the 8 lanes sharing lane >> 3; every lane of the group gets the sum
template <class T>
__device__ __forceinline__ T red8(T v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  return v;
}

// j forces of one FP64 tile: group g = lane >> 3 holds the sums of j slot g; lanes
// 8 g + c (c < 3) of the lane mask m add component c at byte offset off
__device__ __forceinline__ void store_j(double* F, unsigned off, unsigned long long m, int lane, double jx, double jy,
                                        double jz) {
  const int c = lane & 7;
  const double v = c == 0 ? jx : (c == 1 ? jy : jz);
  if (__builtin_amdgcn_inverse_ballot_w64(m)) unsafeAtomicAdd((double*)((char*)F + off), v);
}
// Global-address-space views of the buffers: loads and atomics through them
// compile to global_* instructions (SGPR base + VGPR offset) instead of flat_*,
// which also keeps them out of the LDS counter the DPP/permute traffic waits on.
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef FZ_GLOBAL v2f GF2;
// work items and group masks are read through the scalar cache: the address is
// the wave's, and a scalar load leaves the vector memory counter to the j gathers
typedef const __attribute__((address_space(4))) v4i CI4;
typedef int v2i __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(4))) v2i CI2;
typedef const __attribute__((address_space(4))) unsigned long long CU64;
typedef FZ_GLOBAL unsigned long long GU64;

__device__ __forceinline__ void atomic_add_g(GU64* p, unsigned long long v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Raw buffer views of the slot arrays: a load is (SGPR descriptor, SGPR byte
// offset of the cluster, VGPR byte offset of the lane), with no 64-bit address
// arithmetic on the vector ALU.  gfx9 descriptor word 3 (raw, 32-bit format).
// On gfx9 the scalar offset is not part of the range check, so num_records
// only covers the lane offsets; the caller's indices are in range.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4i buf_ld4(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}
__device__ __forceinline__ unsigned buf_ld1(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0);
}
__device__ __forceinline__ v2f buf_ld2(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
}

// Lanes 8k + c (c < 3) of a 64-bit lane mask whose byte k is not zero.
__device__ __forceinline__ unsigned long long byte_any3(unsigned long long a) {
  a |= a >> 4;
  a |= a >> 2;
  a |= a >> 1;
  a &= 0x0101010101010101ull;
  return a | (a << 1) | (a << 2);
}

template <class T>
__device__ __forceinline__ T red_stride8(T v) {  // sum over lanes sharing lane & 7
  v += __shfl_xor(v, 8, 64);
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

// i forces of cluster I at the end of its run of entries: sums over the lanes
// sharing lane & 7; lane i + 8c (c < 3) adds component c of slot i
__device__ __forceinline__ void flush_i(FZ_GLOBAL char* Fb, int I, int lane, float fix, float fiy, float fiz) {
  const float rx = red_stride8(fix), ry = red_stride8(fiy), rz = red_stride8(fiz);
  const int c = lane >> 3;
  const float v = c == 0 ? rx : (c == 1 ? ry : rz);
  if (lane < 24)
    atomic_add_g((GU64*)(Fb + (size_t)I * (CLUSTER * SLOT_BYTES) + (unsigned)(lane & 7) * SLOT_BYTES + (unsigned)c * 8u),
                 fixed_f32(v));
}

// Sums of three values over the 8 lanes sharing lane >> 3, every lane of the
// group getting them: nine v_add_f32 with a DPP operand (xor 1, xor 2, mirror
// within 8).  Written out because the compiler fuses the first add with the
// product that feeds it (a mov_dpp + fma pair per value) and sinks the last
// stage into the store's branch (mov_dpp + add).  s_nop 1 gives the two wait
// states a DPP read needs after the VALU write of its operand; inside the block
// each read comes two instructions after the write.  Called with all lanes on.
__device__ __forceinline__ void red8x3(float& x, float& y, float& z) {
  float a, b, c;
  __asm__(
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %1, %4, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %2, %5, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_add_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1"
      : "=&v"(a), "=&v"(b), "=&v"(c)
      : "v"(x), "v"(y), "v"(z));
  x = a;
  y = b;
  z = c;
}

__device__ __forceinline__ float erfc_fit(float x, float ex) {
  // erfc(x) = exp(-x^2) * t * P(t), t = 1 / (1 + p x); coefficients fitted for
  // relative error (fz_erfc_fit.h, generated by gen_erfc_fit.py)
  float t = __builtin_amdgcn_rcpf(1.0f + FZ_ERFC_P * x);
  float p = FZ_ERFC_C6;
  p = p * t + FZ_ERFC_C5;
  p = p * t + FZ_ERFC_C4;
  p = p * t + FZ_ERFC_C3;
  p = p * t + FZ_ERFC_C2;
  p = p * t + FZ_ERFC_C1;
  p = p * t + FZ_ERFC_C0;
  return ex * t * p;
}

__device__ __forceinline__ void add3(double* F, int slot, double fx, double fy, double fz) {
  unsafeAtomicAdd(F + (size_t)slot * 4, fx);
  unsafeAtomicAdd(F + (size_t)slot * 4 + 1, fy);
  unsafeAtomicAdd(F + (size_t)slot * 4 + 2, fz);
}

// Energy / virial sums of an evaluation step.  Each lane sums one work item in
// FP64; eight lanes' sums are added and converted to fixed point (2^28) before
// they join the first one's running total, so the totals do not depend on which
// wave ran which item: results are the same for any persistent-grid size and any
// batch around the system.  (A conversion per lane rounds eight times as often:
// 1.9e-6 kcal/mol off in the LJ energy of 18,000 atoms with a 24 A cutoff.)
struct EvAcc {
  long long e[8];  // vdw, elec, virial xx yy zz xy xz yz
  int npr;
  long long ntl;  // list entries of the systems whose first item the wave ran (the same in every lane)
  __device__ void zero() {
#pragma unroll
    for (int k = 0; k < 8; k++) e[k] = 0;
    npr = 0;
    ntl = 0;
  }
  __device__ void add_item(const double (&c)[8], int lane) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const double v = red8(c[k]);
      if ((lane & 7) == 0) e[k] += __double2ll_rn(v * E_SCALE);
    }
  }
  // into this wave's copy of the system's spread sums (folded by k_ev_fold)
  __device__ void flush(const SysDev& d, int lane) {
    long long v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = wave_sum(e[k]);
    const int np = wave_sum(npr);
    if (lane == 0) {
      const unsigned wv = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (EV_SPREAD - 1);
      unsigned long long* c = d.acc_ev + (size_t)wv * EV_W;
#pragma unroll
      for (int k = 0; k < 8; k++) atomicAdd(c + k, (unsigned long long)v[k]);
      atomicAdd(c + 8, (unsigned long long)np);
      atomicAdd(c + 9, (unsigned long long)ntl);
    }
  }
};

// Adds each system's EV_SPREAD copies into its accumulators and clears the copies
// (a barostat step does so in its piston kernel).
__global__ __launch_bounds__(EV_SPREAD) void k_ev_fold(const SysDev* __restrict__ S) {
  long long v[EV_NV];
  ev_fold(S[blockIdx.x], v);
}

// ---------------------------------------------------------------------------
// Work items of a launch: a batch's are laid out as a prefix over its systems
// (chunk_pre); a single system's are all of its own (none after an overflow).
__device__ __forceinline__ int work_items(const SysDev* __restrict__ S, int nsys, const int* __restrict__ chunk_pre) {
  if (nsys > 1) return chunk_pre[nsys];
  return S[0].flags[F_OVERFLOW] ? 0 : (int)(*S[0].pg_n >> 40);
}

__device__ __forceinline__ int entry_items(const SysDev* __restrict__ S, int nsys, const int* __restrict__ entry_pre) {
  if (nsys > 1) return entry_pre[nsys];
  return S[0].flags[F_OVERFLOW] ? 0 : entry_chunks(S[0]);
}

// One i cluster of a work item in registers (mixed form).
struct ICluster {
  int x, y, z, t;      // position top words, LJ table row
  float q, q_raw;      // charge times the Coulomb constant, charge
  v2f p;               // LJ parameters
  __device__ __forceinline__ void set(const v4i& v, const v2f& lp, int n_types) {
    p = lp;
    x = v.x; y = v.y; z = v.z;
    q_raw = __int_as_float(v.w);
    q = q_raw * (float)CC;
    t = __float_as_int(lp.x) * n_types;
  }
};

// Horner's rule.  The coefficients are scalars of the launch; written out so that they
// are taken from scalar registers (left to itself the compiler forms v_fmac, whose
// addend is the destination, and copies every coefficient into a vector register pair
// first: three instructions for one).
template <int N>
__device__ __forceinline__ double horner_s(const double (&c)[N], double y) {
  double p = c[N - 1];
#pragma unroll
  for (int k = N - 2; k >= 0; k--) {
    double r;
    __asm__("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(y), "s"(c[k]));
    p = r;
  }
  return p;
}

// Factors of the real-space Ewald terms at distance r = r2 / sqrt(r2): ex = e^{-z^2},
// cx = e^{z^2} erfc z, z = beta r (fit_ewald)
__device__ __forceinline__ void ewald_factors(const SysDev& d, double r2, double r, double& ex, double& cx) {
  const double n = __builtin_rint(r2 * d.ew_c);
  ex = __builtin_amdgcn_ldexp(horner_s(d.ew_x, fma(r2, d.ew_c, -n)), (int)n);
  cx = horner_s(d.ew_g, fma(r, d.ew_a, -1.0));
}

// 1 / sqrt(x) in FP64: the hardware estimate (relative error e below 2^-23) and one
// third-order step, y (1 + e/2 + 3 e^2/8), e = 1 - x y^2.  Off by 1.3e-16 at most (rms
// 5.5e-17), as is the quotient 1 / sqrt(x) of two rounded operations.
__device__ __forceinline__ double rsqrt_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// (u_j - u_i) as a displacement: both halves converted and scaled by themselves
__device__ __forceinline__ double disp_f64(unsigned long long u, double sc) {
  return fma((double)(int)(u >> 32), 4294967296.0 * sc, (double)(unsigned)u * sc);
}

// System constants of the mixed tile arithmetic.  CHARMM switch
// S(r2) = (rc2 - r2)^2 (rc2 + 2 r2 - 3 ron2) / (rc2 - ron2)^3 in the form
// 6 S = c1^2 (sw_a r2 + sw_b), c1 = rc2 - r2, and -2 dS/dr2 = sw_a c1 (r2 - ron2);
// r2 is clamped to ron2 below the switching range, where 6 S = 6 and dS = 0.
struct PairConst {
  float sx, sy, sz, rc2, ron2, sw_a, sw_b, pb, ccb, nb2l2e;
  __device__ __forceinline__ explicit PairConst(const SysDev& d) {
    sx = d.sc32[0]; sy = d.sc32[1]; sz = d.sc32[2];
    rc2 = (float)d.rc2; ron2 = (float)d.ron2;
    sw_a = (float)(12.0 * d.sw_inv);
    sw_b = (float)(6.0 * d.sw_inv * (d.rc2 - 3.0 * d.ron2));
    pb = (float)(FZ_ERFC_P * d.beta);
    ccb = (float)(TWO_OVER_SQRT_PI * d.beta);
    nb2l2e = -(float)(d.beta * d.beta * 1.4426950408889634);
  }
};

// a sum rounded by itself, whatever product feeds it
__device__ __forceinline__ float add_rn(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
__device__ __forceinline__ void sub3_rn(float (&f)[3], float x, float y, float z) {
  f[0] = add_rn(f[0], -x);
  f[1] = add_rn(f[1], -y);
  f[2] = add_rn(f[2], -z);
}

// One tile: forces of the lane's pair on its j (fx, fy, fz), energies into cev;
// returns the lanes with a pair inside the cutoff.
template <int EV, bool SEP>
__device__ __forceinline__ unsigned long long tile_mixed(const SysDev& d, const PairConst& c, const GF2* lj,
                                                         unsigned long long mask, const ICluster& ic, const v4i& xj,
                                                         const v2f& pj, float& fx, float& fy, float& fz, double (&cev)[8],
                                                         int& npr) {
  const float dx = (float)(int)((unsigned)xj.x - (unsigned)ic.x) * c.sx;
  const float dy = (float)(int)((unsigned)xj.y - (unsigned)ic.y) * c.sy;
  const float dz = (float)(int)((unsigned)xj.z - (unsigned)ic.z) * c.sz;
  // sums of two products name the one that is fused: which one the compiler takes
  // differs between the kernel's variants, and a run would then depend on which of
  // its steps evaluates energies
  float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  // pairs inside the cutoff as a lane mask: lane l's bit of the group's mask is
  // tested in scalar registers, not shifted out per lane
  const unsigned long long actm = mask & __builtin_amdgcn_ballot_w64(r2 < c.rc2);
  const bool act = __builtin_amdgcn_inverse_ballot_w64(actm);
  r2 = act ? r2 : 1.0f;
  const float rinv = __builtin_amdgcn_rsqf(r2);
  const float rinv2 = rinv * rinv;
  const float r = r2 * rinv;
  // Lennard-Jones with CHARMM switch (energy switched, exact gradient):
  // e6 = E_LJ, f6 = r2 F_LJ / (6 r) unswitched
  v2f p;
  if (SEP || d.lj_sep) {
    const float h = ic.p.y + pj.y;
    p = v2f{ic.p.x * pj.x, h * h};
  } else {
    p = lj[ic.t + __float_as_int(pj.x)];
  }
  const float s2 = p.y * rinv2;
  const float s6 = s2 * s2 * s2;
  const float a6 = p.x * s6, a12 = a6 * s6;
  const float e6 = a12 - a6;
  const float f6 = 2.0f * a12 - a6;
  // max(r2, ron2) of two non-negative floats as an integer max of their bits
  const float r2c = __int_as_float(max(__float_as_int(r2), __float_as_int(c.ron2)));
  const float c1 = c.rc2 - r2c;
  const float sw6 = c1 * c1 * (c.sw_a * r2c + c.sw_b);  // 6 S
  const float dsw = c1 * (r2c - c.ron2) * c.sw_a;       // -2 dS/dr2
  // real-space Ewald: erfc(beta r) = exp(-beta^2 r2) t P(t), t = 1 / (1 + p beta r)
  const float t = __builtin_amdgcn_rcpf(c.pb * r + 1.0f);
  const float ex = __builtin_amdgcn_exp2f(c.nb2l2e * r2);
  float tp = FZ_ERFC_C6;
  tp = tp * t + FZ_ERFC_C5;
  tp = tp * t + FZ_ERFC_C4;
  tp = tp * t + FZ_ERFC_C3;
  tp = tp * t + FZ_ERFC_C2;
  tp = tp * t + FZ_ERFC_C1;
  tp = tp * t + FZ_ERFC_C0;
  tp *= t;
  const float qex = ic.q * __int_as_float(xj.w) * ex;
  const float fc2 = (tp * rinv + c.ccb) * qex;  // r2 F_C / r
  // F / r = (r2 F_C / r + 6 S f6) / r2 + E_LJ (-2 dS/dr2)
  const float fs = act ? fmaf(e6, dsw, fmaf(f6, sw6, fc2) * rinv2) : 0.0f;
  fx = fs * dx; fy = fs * dy; fz = fs * dz;
  if (EV && act) {
    if (EV == 1) {
      cev[0] += (double)(e6 * sw6 * (1.0f / 6.0f));
      cev[1] += (double)(qex * tp * rinv);
    } else {
#pragma clang fp contract(off)  // as in tile_f64
      // energies of an evaluation step in FP64 from the same FP32 distance, so
      // that no FP32 bias of the erfc/exp approximations sums over millions of pairs
      const double r2d = (double)r2, rid = rsqrt_f64(r2d), ri2d = rid * rid;
      const double s2d = (double)p.y * ri2d, s6d = s2d * s2d * s2d;
      const double a6d = (double)p.x * s6d;
      double eljd = fma(a6d, s6d, -a6d);
      if (r2d > (double)c.ron2) {
        const double c1d = (double)c.rc2 - r2d, c2d = (double)c.rc2 + 2.0 * r2d - 3.0 * (double)c.ron2;
        eljd *= c1d * c1d * c2d * d.sw_inv;
      }
      cev[0] += eljd;
      const double qq = CC * (double)ic.q_raw * (double)__int_as_float(xj.w);
      double ec;
      if (EV == 2 || d.ew_poly) {
        double ex, cx;
        ewald_factors(d, r2d, r2d * rid, ex, cx);
        ec = ex * cx;
      } else {
        ec = erfc(d.beta * (r2d * rid));
      }
      cev[1] += qq * ec * rid;
    }
    npr++;
    cev[2] += (double)(fx * dx); cev[3] += (double)(fy * dy); cev[4] += (double)(fz * dz);
    cev[5] += (double)(fx * dy); cev[6] += (double)(fx * dz); cev[7] += (double)(fy * dz);
  }
  return actm;
}

// EV: 0 forces only; 1 also energies and virial summed from the FP32 pair terms
// (the minimisers' accept/reject tests); 2 energies recomputed in FP64 from the
// FP32 distance (reported energies), 3 the same in a launch with a system that has
// no Ewald polynomials (that one: the library's erfc).  SEP: every system of the launch follows the
// combination rule (per-slot LJ parameters, no table lookup).
template <int EV, bool SEP>
__global__ __launch_bounds__(256) void k_pair_mixed(const SysDev* __restrict__ S, int nsys, const int* __restrict__ chunk_pre,
                                                    int spend) {
  // spend: a single system's rebuild decision of this step is spent here
  if (spend && blockIdx.x == 0 && threadIdx.x == 0) S[0].flags[F_REBUILD] = 0;
  const int lane = threadIdx.x & 63, il = lane & 7, jl = lane >> 3;
  const int total = rfl(work_items(S, nsys, chunk_pre));
  const int nw = gridDim.x * 4;
  // energy / virial totals stay in registers until the wave moves to another system
  int evs = -1;
  EvAcc ev;
  ev.zero();
  for (int w = rfl(blockIdx.x * 4 + (threadIdx.x >> 6)); w < total; w += nw) {
    const int s = nsys == 1 ? 0 : rfl(locate(chunk_pre, nsys, w));
    const int wk = nsys == 1 ? w : w - chunk_pre[s];
    const SysDev& d = S[s];
    if (EV && s != evs) {
      if (evs >= 0) ev.flush(S[evs], lane);
      ev.zero();
      evs = s;
    }
    double cev[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const v4i item = ((const CI4*)d.pg_item)[wk];
    const int g0 = rfl(item.x), ne = rfl(item.y), I0 = rfl(item.z), I1 = rfl(item.w);
    if (EV && wk == 0) ev.ntl += *d.n_pairs;
    // slot record of a slot at (uniform base) + 32-bit byte offset per lane
    const __amdgpu_buffer_rsrc_t xsr = raw_rsrc(d.xs, (unsigned)d.n_slots_cap * SLOT_BYTES);
    // the item's j offsets, eight to a group
    const __amdgpu_buffer_rsrc_t jr = raw_rsrc(d.pg_j + 8 * (size_t)(unsigned)g0, (unsigned)(ne + 2) * 32u);
    const CI4* msk = (const CI4*)(d.pg_mask + (unsigned)g0);
    const GF2* lj = (const GF2*)d.lj32;
    FZ_GLOBAL char* Fb = (FZ_GLOBAL char*)d.Fs;
    const PairConst pc(d);
    // force atomics: lane 8k + c (c < 3) adds component c of the k-th j slot
    const unsigned coff = (unsigned)(lane & 7) * 8u;
    // Three groups are in flight: the arithmetic of one, the slot records of the
    // next, the j offsets of the one after that.
    const unsigned jlo = (unsigned)jl * 4u;
    unsigned jon = buf_ld1(jr, jlo, 0u), jonn = buf_ld1(jr, jlo, 32u);
    ICluster ic[2];
    float fi[2][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};  // their force sums
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const unsigned so = (unsigned)(h ? I1 : I0) * (CLUSTER * SLOT_BYTES);
      const v4i v = buf_ld4(xsr, (unsigned)il * SLOT_BYTES, so);
      ic[h].set(v, buf_ld2(xsr, (unsigned)il * SLOT_BYTES + 16u, so), d.n_types);
    }
    v4i xjn = buf_ld4(xsr, jon, 0u);
    v2f pjn = buf_ld2(xsr, jon + 16u, 0u);
    v4i mn = msk[0];
    // The j-force atomic of a group is issued one group late, after the next
    // prefetch: the wait for prefetched data (vmcnt counts loads and atomics in
    // issue order) then covers only an atomic issued a whole group earlier.
    unsigned long long pend_m = 0ull, pend_v = 0ull;
    unsigned pend_o = 0u;
    for (int k = 0; k < ne; k++) {
      const unsigned long long m0 = ((unsigned long long)(unsigned)rfl(mn.y) << 32) | (unsigned)rfl(mn.x);
      const unsigned long long m1 = ((unsigned long long)(unsigned)rfl(mn.w) << 32) | (unsigned)rfl(mn.z);
      const v4i xj = xjn;
      const v2f pj = pjn;
      const unsigned jo = jon;
      mn = msk[k + 1];
      jon = jonn;
      xjn = buf_ld4(xsr, jon, 0u);
      pjn = buf_ld2(xsr, jon + 16u, 0u);
      jonn = buf_ld1(jr, jlo, (unsigned)(k + 2) * 32u);
      if (__builtin_amdgcn_inverse_ballot_w64(pend_m)) atomic_add_g((GU64*)(Fb + pend_o), pend_v);
      // j sums: every lane of group j = lane >> 3 holds slot j's; lane 8j + c adds
      // component c when a pair of slot j is inside the cutoff.  Each tile's sum is
      // converted by itself and the two are added in fixed point.
      unsigned long long actm = 0ull;
      pend_v = 0ull;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const unsigned long long m = h ? m1 : m0;
        if (m) {
          float fx, fy, fz;
          actm |= tile_mixed<EV, SEP>(d, pc, lj, m, ic[h], xj, pj, fx, fy, fz, cev, ev.npr);
          sub3_rn(fi[h], fx, fy, fz);
          red8x3(fx, fy, fz);
          const int c = lane & 7;
          pend_v += fixed_f32(c == 0 ? fx : (c == 1 ? fy : fz));
        }
      }
      pend_m = byte_any3(actm);
      pend_o = jo + coff;
    }
    if (__builtin_amdgcn_inverse_ballot_w64(pend_m)) atomic_add_g((GU64*)(Fb + pend_o), pend_v);
    flush_i(Fb, I0, lane, fi[0][0], fi[0][1], fi[0][2]);
    if (I1 != I0) flush_i(Fb, I1, lane, fi[1][0], fi[1][1], fi[1][2]);
    if (EV) ev.add_item(cev, lane);
  }
  if (EV && evs >= 0) ev.flush(S[evs], lane);
}

// Mixed form over entry lists (SysDev::entry_list): tiles of two whole clusters.
//
// Forces on i are FP32 sums over an i cluster's run of entries within a chunk of
// PAIR_CHUNK, in list order.  A small system's trajectory runs many steps between two
// looks at it and multiplies a rounding difference about eightfold in 40 steps of 2 fs,
// so the order of these sums is part of its results: it is the list's, whatever wave
// forms a tile.  One workgroup per chunk: its four waves form the tiles of eight
// entries each, all their records loaded before the first is used, and leave the i
// terms in LDS; then one wave per component adds them up entry by entry.
//
// What bounds it: latency (1,000 atoms: 274 chunks).  8 to 12 us at 1,000 atoms, back to
// back; a wave per chunk takes 18 (the step 66 us, 54 with this), pair groups 6.7, and
// eight or sixteen waves save 1.5 us, which no step shows (the PME kernels beside it take
// longer).
constexpr int ENTRY_WAVE = PAIR_CHUNK / 4;  // entries of a wave

template <int EV, bool SEP>
__global__ __launch_bounds__(256) void k_pair_entry(const SysDev* __restrict__ S, int nsys, const int* __restrict__ chunk_pre,
                                                    int spend) {
  if (spend && blockIdx.x == 0 && threadIdx.x == 0) S[0].flags[F_REBUILD] = 0;
  __shared__ float term[PAIR_CHUNK][3][64];
  const int lane = threadIdx.x & 63, il = lane & 7, jl = lane >> 3, wv = rfl(threadIdx.x >> 6);
  chunk_pre += nsys + 1;  // the entry lists' prefix
  const int total = rfl(entry_items(S, nsys, chunk_pre));
  int evs = -1;
  EvAcc ev;
  ev.zero();
  for (int w = blockIdx.x; w < total; w += gridDim.x) {
    const int s = nsys == 1 ? 0 : rfl(locate(chunk_pre, nsys, w));
    const int wk = nsys == 1 ? w : w - chunk_pre[s];
    const SysDev& d = S[s];
    if (EV && s != evs) {
      if (evs >= 0) ev.flush(S[evs], lane);
      ev.zero();
      evs = s;
    }
    double cev[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const long long np = *d.n_pairs, e0 = (long long)wk * PAIR_CHUNK;
    const int ne = rfl((int)(np - e0 < PAIR_CHUNK ? np - e0 : PAIR_CHUNK));
    if (EV && wk == 0 && wv == 0) ev.ntl += np;
    const __amdgpu_buffer_rsrc_t xsr = raw_rsrc(d.xs, (unsigned)d.n_slots_cap * SLOT_BYTES);
    const CI2* ent = (const CI2*)(d.pl_ij + e0);
    const CU64* msk = (const CU64*)(d.pl_mask + e0);
    const GF2* lj = (const GF2*)d.lj32;
    FZ_GLOBAL char* Fb = (FZ_GLOBAL char*)d.Fs;
    const PairConst pc(d);
    // the wave's entries (past the list's end: the last one, no lanes)
    unsigned Js[ENTRY_WAVE];
    unsigned long long m[ENTRY_WAVE];
    v4i xi[ENTRY_WAVE], xj[ENTRY_WAVE];
    v2f pi[ENTRY_WAVE], pj[ENTRY_WAVE];
#pragma unroll
    for (int k = 0; k < ENTRY_WAVE; k++) {
      const int e = wv * ENTRY_WAVE + k, at = e < ne ? e : ne - 1;
      const v2i ij = ent[at];
      m[k] = e < ne ? msk[at] : 0ull;
      const unsigned Is = (unsigned)ij.x * (CLUSTER * SLOT_BYTES);
      Js[k] = (unsigned)ij.y * (CLUSTER * SLOT_BYTES);
      xi[k] = buf_ld4(xsr, (unsigned)il * SLOT_BYTES, Is);
      pi[k] = buf_ld2(xsr, (unsigned)il * SLOT_BYTES + 16u, Is);
      xj[k] = buf_ld4(xsr, (unsigned)jl * SLOT_BYTES, Js[k]);
      pj[k] = buf_ld2(xsr, (unsigned)jl * SLOT_BYTES + 16u, Js[k]);
    }
#pragma unroll
    for (int k = 0; k < ENTRY_WAVE; k++) {
      float fx = 0.f, fy = 0.f, fz = 0.f;
      float* t = &term[wv * ENTRY_WAVE + k][0][lane];
      unsigned long long actm = 0ull;
      if (m[k]) {
        ICluster ic;
        ic.set(xi[k], pi[k], d.n_types);
        actm = tile_mixed<EV, SEP>(d, pc, lj, m[k], ic, xj[k], pj[k], fx, fy, fz, cev, ev.npr);
      }
      t[0] = fx; t[64] = fy; t[128] = fz;
      if (m[k]) {
        red8x3(fx, fy, fz);
        const int c = lane & 7;
        const unsigned long long v = fixed_f32(c == 0 ? fx : (c == 1 ? fy : fz));
        if (__builtin_amdgcn_inverse_ballot_w64(byte_any3(actm)))
          atomic_add_g((GU64*)(Fb + (size_t)Js[k] + (unsigned)jl * SLOT_BYTES + (unsigned)c * 8u), v);
      }
    }
    __syncthreads();
    if (wv < 3) {  // component wv of the i forces
      float f = 0.f;
      int I = ent[0].x;
      auto flush = [&]() {
        const float r = red_stride8(f);
        if (lane < 8)
          atomic_add_g((GU64*)(Fb + (size_t)I * (CLUSTER * SLOT_BYTES) + (unsigned)lane * SLOT_BYTES + (unsigned)wv * 8u), fixed_f32(r));
      };
      float t[PAIR_CHUNK];
#pragma unroll
      for (int k = 0; k < PAIR_CHUNK; k++) t[k] = term[k][wv][lane];
#pragma unroll
      for (int k = 0; k < PAIR_CHUNK; k++) {
        const int Ik = k < ne ? ent[k].x : I;
        if (Ik != I) {
          flush();
          f = 0.f;
          I = Ik;
        }
        f = add_rn(f, -t[k]);
      }
      flush();
    }
    __syncthreads();
    if (EV) ev.add_item(cev, lane);
  }
  if (EV && evs >= 0) ev.flush(S[evs], lane);
}

// The same sums with a wave per chunk, for launches of many chunks (ENTRY_WAVE_CHUNKS):
// no terms pass through LDS and no wave waits for another.
template <int EV, bool SEP>
__global__ __launch_bounds__(256) void k_pair_entry_wave(const SysDev* __restrict__ S, int nsys, const int* __restrict__ chunk_pre,
                                                         int spend) {
  if (spend && blockIdx.x == 0 && threadIdx.x == 0) S[0].flags[F_REBUILD] = 0;
  const int lane = threadIdx.x & 63, il = lane & 7, jl = lane >> 3;
  chunk_pre += nsys + 1;  // the entry lists' prefix
  const int total = rfl(entry_items(S, nsys, chunk_pre));
  const int nw = gridDim.x * 4;
  int evs = -1;
  EvAcc ev;
  ev.zero();
  for (int w = rfl(blockIdx.x * 4 + (threadIdx.x >> 6)); w < total; w += nw) {
    const int s = nsys == 1 ? 0 : rfl(locate(chunk_pre, nsys, w));
    const int wk = nsys == 1 ? w : w - chunk_pre[s];
    const SysDev& d = S[s];
    if (EV && s != evs) {
      if (evs >= 0) ev.flush(S[evs], lane);
      ev.zero();
      evs = s;
    }
    double cev[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const long long np = *d.n_pairs, e0 = (long long)wk * PAIR_CHUNK;
    const int ne = rfl((int)(np - e0 < PAIR_CHUNK ? np - e0 : PAIR_CHUNK));
    if (EV && wk == 0) ev.ntl += np;
    const __amdgpu_buffer_rsrc_t xsr = raw_rsrc(d.xs, (unsigned)d.n_slots_cap * SLOT_BYTES);
    const CI2* ent = (const CI2*)(d.pl_ij + e0);
    const CU64* msk = (const CU64*)(d.pl_mask + e0);
    const GF2* lj = (const GF2*)d.lj32;
    FZ_GLOBAL char* Fb = (FZ_GLOBAL char*)d.Fs;
    const PairConst pc(d);
    const unsigned ioff = (unsigned)il * SLOT_BYTES, joff = (unsigned)jl * SLOT_BYTES;
    const unsigned foff = joff + (unsigned)(lane & 7) * 8u;
    ICluster ic;
    float fi[3];
    int I = -1;
    v2i en = ent[0];
    unsigned Js = (unsigned)en.y * (CLUSTER * SLOT_BYTES);
    v4i xjn = buf_ld4(xsr, joff, Js);
    v2f pjn = buf_ld2(xsr, joff + 16u, Js);
    // j cluster one entry ahead, the j-force atomic one late (as in k_pair_mixed)
    unsigned long long pend_m = 0ull, pend_v = 0ull;
    unsigned pend_o = 0u;
    for (int k = 0; k < ne; k++) {
      const int Ik = rfl(en.x);
      const unsigned long long m = msk[k];
      const unsigned Jk = Js;
      const v4i xj = xjn;
      const v2f pj = pjn;
      en = ent[min(k + 1, ne - 1)];
      Js = (unsigned)en.y * (CLUSTER * SLOT_BYTES);
      xjn = buf_ld4(xsr, joff, Js);
      pjn = buf_ld2(xsr, joff + 16u, Js);
      if (__builtin_amdgcn_inverse_ballot_w64(pend_m)) atomic_add_g((GU64*)(Fb + pend_o), pend_v);
      if (Ik != I) {
        const unsigned Is = (unsigned)Ik * (CLUSTER * SLOT_BYTES);
        const v4i v = buf_ld4(xsr, ioff, Is);
        const v2f lp = buf_ld2(xsr, ioff + 16u, Is);
        if (I >= 0) flush_i(Fb, I, lane, fi[0], fi[1], fi[2]);
        I = Ik;
        ic.set(v, lp, d.n_types);
        // the i loads consumed here: one in flight where this branch rejoins the loop
        // would make every tile wait for all memory operations
        __asm__ volatile("" ::"v"(ic.q), "v"(ic.x), "v"(ic.y), "v"(ic.z), "v"(ic.p.x), "v"(ic.p.y));
        fi[0] = fi[1] = fi[2] = 0.f;
      }
      float fx, fy, fz;
      const unsigned long long actm = tile_mixed<EV, SEP>(d, pc, lj, m, ic, xj, pj, fx, fy, fz, cev, ev.npr);
      sub3_rn(fi, fx, fy, fz);
      red8x3(fx, fy, fz);
      const int c = lane & 7;
      pend_v = fixed_f32(c == 0 ? fx : (c == 1 ? fy : fz));
      pend_m = byte_any3(actm);
      pend_o = Jk + foff;
      if (EV && (k + 1) % ENTRY_WAVE == 0) {  // energies by the same eight entries as a workgroup's waves
        ev.add_item(cev, lane);
#pragma unroll
        for (int q = 0; q < 8; q++) cev[q] = 0.0;
      }
    }
    if (__builtin_amdgcn_inverse_ballot_w64(pend_m)) atomic_add_g((GU64*)(Fb + pend_o), pend_v);
    flush_i(Fb, I, lane, fi[0], fi[1], fi[2]);
    if (EV) ev.add_item(cev, lane);
  }
  if (EV && evs >= 0) ev.flush(S[evs], lane);
}

struct ICluster64 {
  unsigned long long x, y, z;
  int t;
  double q, fx, fy, fz;
};

// One FP64 tile.  Real-space Ewald terms from polynomials (fit_ewald: 41 fused
// multiply-adds); of a system without them (beta rc above EW_MAX_Z) with the library's
// erfc and exp, which took most of the kernel's 250 FP64 instructions a tile.
// Force-only launch over 131,000 atoms 652 us with the library, 395 with the polynomials.
// POLY: every system of the launch has them.
template <bool EV, bool POLY>
__device__ __forceinline__ void tile_f64(const SysDev& d, const double2* __restrict__ lj, unsigned long long mask,
                                         ICluster64& ic, const Slot64& xj, int tj, double& jx, double& jy, double& jz,
                                         double (&cev)[8], int& npr) {
#pragma clang fp contract(off)  // fused where written: the variants of the kernel then agree to the bit
  const double dx = disp_f64(xj.x - ic.x, d.sc[0]), dy = disp_f64(xj.y - ic.y, d.sc[1]), dz = disp_f64(xj.z - ic.z, d.sc[2]);
  double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
  const bool act = __builtin_amdgcn_inverse_ballot_w64(mask & __builtin_amdgcn_ballot_w64(r2 < d.rc2));
  r2 = act ? r2 : 1.0;
  const double rinv = rsqrt_f64(r2);
  const double rinv2 = rinv * rinv;
  const double2 p = lj[ic.t + tj];
  const double s2 = p.y * rinv2;
  const double s6 = s2 * s2 * s2;
  const double a6 = p.x * s6, a12 = a6 * s6;
  double e_lj = fma(a6, s6, -a6);
  // CHARMM switch; below ron 1 (slope 0) itself, not its formula at ron, whose last
  // factors cancel
  const bool sw_on = r2 > d.ron2;
  const double c1 = d.rc2 - r2, c2 = fma(2.0, r2, d.rc2 - 3.0 * d.ron2);
  const double sw = sw_on ? c1 * c1 * c2 * d.sw_inv : 1.0;
  const double dsw = sw_on ? 12.0 * c1 * (r2 - d.ron2) * d.sw_inv : 0.0;
  const double f_lj = fma(fma(12.0, a12, -6.0 * a6) * rinv2, sw, e_lj * dsw);
  e_lj *= sw;
  const double qq = ic.q * xj.q;
  double e_c = 0.0, f_c;
  if (POLY || d.ew_poly) {
    double ex, cx;
    const double r = r2 * rinv;
    ewald_factors(d, r2, r, ex, cx);
    f_c = qq * (ex * fma(r, d.ew_b, cx)) * (rinv * rinv2);
    if (EV) e_c = qq * rinv * (ex * cx);
  } else {
    const double x = d.beta * (r2 * rinv);
    e_c = qq * erfc(x) * rinv;
    f_c = fma(qq * (TWO_OVER_SQRT_PI * d.beta), exp(-x * x), e_c) * rinv2;
  }
  const double fs = act ? f_c + f_lj : 0.0;
  ic.fx = fma(-fs, dx, ic.fx); ic.fy = fma(-fs, dy, ic.fy); ic.fz = fma(-fs, dz, ic.fz);
  jx = fma(fs, dx, jx); jy = fma(fs, dy, jy); jz = fma(fs, dz, jz);
  if (EV && act) {
    const double fx = fs * dx, fy = fs * dy, fz = fs * dz;
    cev[0] += e_lj; cev[1] += e_c; npr++;
    cev[2] = fma(fx, dx, cev[2]); cev[3] = fma(fy, dy, cev[3]); cev[4] = fma(fz, dz, cev[4]);
    cev[5] = fma(fx, dy, cev[5]); cev[6] = fma(fx, dz, cev[6]); cev[7] = fma(fy, dz, cev[7]);
  }
}

template <bool EV, bool POLY>
__global__ __launch_bounds__(256) void k_pair_f64(const SysDev* __restrict__ S, int nsys, const int* __restrict__ chunk_pre,
                                                  int spend) {
  if (spend && blockIdx.x == 0 && threadIdx.x == 0) S[0].flags[F_REBUILD] = 0;
  const int lane = threadIdx.x & 63, il = lane & 7, jl = lane >> 3;
  const int total = rfl(work_items(S, nsys, chunk_pre));
  const int nw = gridDim.x * 4;
  int evs = -1;
  EvAcc ev;
  ev.zero();
  for (int w = rfl(blockIdx.x * 4 + (threadIdx.x >> 6)); w < total; w += nw) {
    const int s = nsys == 1 ? 0 : rfl(locate(chunk_pre, nsys, w));
    const int wk = nsys == 1 ? w : w - chunk_pre[s];
    const SysDev& d = S[s];
    if (EV && s != evs) {
      if (evs >= 0) ev.flush(S[evs], lane);
      ev.zero();
      evs = s;
    }
    double cev[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const v4i item = ((const CI4*)d.pg_item)[wk];
    const int g0 = rfl(item.x), ne = rfl(item.y), I0 = rfl(item.z), I1 = rfl(item.w);
    if (EV && wk == 0) ev.ntl += *d.n_pairs;
    const Slot64* __restrict__ xs = (const Slot64*)d.xs;
    const int* __restrict__ ts = d.ts;
    const double2* __restrict__ lj = d.lj64;
    const CI4* msk = (const CI4*)(d.pg_mask + (unsigned)g0);
    const unsigned* __restrict__ jof = d.pg_j + 8 * (size_t)(unsigned)g0 + jl;  // the lane's j of each group
    double* F = (double*)d.Fs;
    const unsigned coff = (unsigned)(lane & 7) * 8u;
    ICluster64 ic[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int sl = (h ? I1 : I0) * CLUSTER + il;
      const Slot64 v = xs[sl];
      ic[h].x = v.x; ic[h].y = v.y; ic[h].z = v.z;
      ic[h].q = v.q * CC;
      ic[h].t = ts[sl] * d.n_types;
      ic[h].fx = ic[h].fy = ic[h].fz = 0.0;
    }
    // as in the mixed kernel: slot records one group ahead, offsets two (an offset
    // past the item may be anything: it is not followed)
    unsigned jon = jof[0], jonn = jof[8];
    Slot64 xjn = *(const Slot64*)((const char*)xs + jon);
    int tjn = ts[jon / SLOT_BYTES];
    v4i mkn = msk[0];
    for (int k = 0; k < ne; k++) {
      const v4i mk = mkn;
      const unsigned long long m0 = ((unsigned long long)(unsigned)rfl(mk.y) << 32) | (unsigned)rfl(mk.x);
      const unsigned long long m1 = ((unsigned long long)(unsigned)rfl(mk.w) << 32) | (unsigned)rfl(mk.z);
      const unsigned jo = jon;
      const Slot64 xj = xjn;
      const int tj = tjn;
      mkn = msk[k + 1];
      jon = jonn;
      if (k + 1 < ne) {
        xjn = *(const Slot64*)((const char*)xs + jon);
        tjn = ts[jon / SLOT_BYTES];
        jonn = jof[8 * (k + 2)];
      }
      double jx = 0.0, jy = 0.0, jz = 0.0;
      if (m0) tile_f64<EV, POLY>(d, lj, m0, ic[0], xj, tj, jx, jy, jz, cev, ev.npr);
      if (m1) tile_f64<EV, POLY>(d, lj, m1, ic[1], xj, tj, jx, jy, jz, cev, ev.npr);
      store_j(F, jo + coff, byte_any3(m0 | m1), lane, red8(jx), red8(jy), red8(jz));
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const double rx = red_stride8(ic[h].fx), ry = red_stride8(ic[h].fy), rz = red_stride8(ic[h].fz);
      if (jl == 0 && (h == 0 || I1 != I0)) add3(F, (h ? I1 : I0) * CLUSTER + il, rx, ry, rz);
    }
    if (EV) ev.add_item(cev, lane);
  }
  if (EV && evs >= 0) ev.flush(S[evs], lane);
}

template <int EV, bool SEP>
static void launch_pair_mixed(const Launch& L, const int* cp, int sp) {
  if (L.n_entry < L.nsys)
    hipLaunchKernelGGL((k_pair_mixed<EV, SEP>), dim3(L.pair_grid), dim3(256), 0, L.stream, L.d_sys, L.nsys, cp, sp);
  if (L.n_entry > 0 && L.entry_waves)
    hipLaunchKernelGGL((k_pair_entry_wave<EV, SEP>), dim3(L.entry_grid), dim3(256), 0, L.stream, L.d_sys, L.nsys, cp, sp);
  else if (L.n_entry > 0)
    hipLaunchKernelGGL((k_pair_entry<EV, SEP>), dim3(L.entry_grid), dim3(256), 0, L.stream, L.d_sys, L.nsys, cp, sp);
}

template <bool EV, bool POLY>
static void launch_pair_f64(const Launch& L, const int* cp, int sp) {
  hipLaunchKernelGGL((k_pair_f64<EV, POLY>), dim3(L.pair_grid), dim3(256), 0, L.stream, L.d_sys, L.nsys, cp, sp);
}

void launch_pair(const Launch& L, int ev, const int* cp, bool fold, bool spend) {
  const int sp = spend ? 1 : 0;
  if (!cp) cp = L.chunk_pre;
  if (L.mixed) {
    if (ev == 2 && !L.ew_poly) ev = 3;
    if (L.lj_sep) {
      if (ev == 3) launch_pair_mixed<3, true>(L, cp, sp);
      else if (ev == 2) launch_pair_mixed<2, true>(L, cp, sp);
      else if (ev == 1) launch_pair_mixed<1, true>(L, cp, sp);
      else launch_pair_mixed<0, true>(L, cp, sp);
    } else {
      if (ev == 3) launch_pair_mixed<3, false>(L, cp, sp);
      else if (ev == 2) launch_pair_mixed<2, false>(L, cp, sp);
      else if (ev == 1) launch_pair_mixed<1, false>(L, cp, sp);
      else launch_pair_mixed<0, false>(L, cp, sp);
    }
  } else {
    // with a system that has no Ewald polynomials: chosen system by system, so that
    // the batch around a system does not change its sums
    if (L.ew_poly) {
      if (ev) launch_pair_f64<true, true>(L, cp, sp);
      else launch_pair_f64<false, true>(L, cp, sp);
    } else {
      if (ev) launch_pair_f64<true, false>(L, cp, sp);
      else launch_pair_f64<false, false>(L, cp, sp);
    }
  }
  if (ev && fold) launch_ev_fold(L);
}

void launch_ev_fold(const Launch& L) {
  hipLaunchKernelGGL(k_ev_fold, dim3(L.nsys), dim3(EV_SPREAD), 0, L.stream, L.d_sys);
}

}  // namespace fz
