// fz_launch.h -- host-side launch description shared by the kernel launchers.
#pragma once
#include <hip/hip_runtime.h>

#include "fz_fft.h"
#include "fz_sys.h"

namespace fz {

// A static work decomposition: pre[s] = first block of system s, total blocks.
struct Work {
  int* pre = nullptr;  // device, nsys + 1 entries
  int total = 0;
};

// pair-search waves per I cluster of a system: its buffer parts, at most the launch's cap
__host__ __device__ inline int search_split(int parts, int cap) { return parts < cap ? parts : cap; }

// Size of a PME grid plane in LDS: two buffers of K0 K1 complex values of csz bytes
// and the x and y twiddles.  The plane kernels are used up to this many atoms per
// system (each of a system's K2 workgroups reads every atom's z position) and
// planes of this size (all the LDS of a compute unit), over PLANE_SMALL_LDS only
// where there are enough planes.
inline int plane_lds_bytes(int K0, int K1, int csz) { return (2 * K0 * K1 + K0 + K1) * csz; }
constexpr int PLANE_MAX_ATOMS = 65536, PLANE_MAX_LDS = 163840, PLANE_SMALL_LDS = 65536;
constexpr int PLANE_LIST = 128;  // atoms a wave of the forward kernel collects before it spreads 64 of them
// elements of each buffer: the plane, its x lines and its kept y lines (padded: fft_line)
__host__ __device__ inline int plane_buf(int K0, int K1, int pad, int csz) {
  const int x = K1 * fft_line(K0, pad, csz), y = (K0 / 2 + 1) * fft_line(K1, pad, csz), p = K0 * K1;
  const int l = PLANE_LIST * 16 * 4 / csz;  // the waves' atom lists
  const int xy = x > y ? x : y, pl = p > l ? p : l;
  return xy > pl ? xy : pl;
}
// padded lines where they fit in PLANE_MAX_LDS too
__host__ __device__ inline int plane_pad(int K0, int K1, int csz) {
  return (2 * plane_buf(K0, K1, 1, csz) + K0 + K1) * csz <= PLANE_MAX_LDS;
}
// dynamic LDS of the plane kernels
inline int plane_dyn_lds(int K0, int K1, int csz) {
  return (2 * plane_buf(K0, K1, plane_pad(K0, K1, csz), csz) + K0 + K1) * csz;
}
// dynamic LDS of the grid passes, lines of up to kmax points
inline int fft_dyn_lds(int NL, const int (&K)[3], int csz) {
  int b = 0;
  for (int k : K) {
    const int n = (2 * NL * fft_line(k, 1, csz) + k) * csz;
    b = n > b ? n : b;
  }
  return b;
}
// launches of fewer planes than this use workgroups of 1,024 threads, others 256
// (planes over PLANE_SMALL_LDS, one to a compute unit, always 1,024)
constexpr int PLANE_WIDE_BELOW = 512;
constexpr int PLANE_MID_POINTS = 2304;  // 512 threads, not 1,024, over planes of up to this many points
// PME gather: four lanes per atom in launches of up to this many 256-atom blocks
constexpr int GATHER_QUAD_BLOCKS = 512;

struct Launch {
  hipStream_t stream = nullptr;
  const SysDev* d_sys = nullptr;  // device array of nsys descriptors
  int nsys = 0;
  int mixed = 0;                  // 0 = FP64 form, 1 = mixed form
  Work w_atoms;   // 256 atoms per block
  Work w_atoms64; // 64 atoms per block
  Work w_slots;   // 256 slots per block
  Work w_cols;    // one block per column
  Work w_clus;    // 4 clusters (waves) per block
  Work w_fill;    // 4 pairs of clusters (waves) per block
  Work w_search;  // 4 search waves per block, search_split(parts, search_cap) waves per cluster
  Work w_terms;   // 256 bonded terms per block
  Work w_ccl;     // 128 constraint clusters per block
  Work w_step;    // 128 per block: constraint clusters, then free atoms
  Work w_fftx;    // x-line groups
  Work w_ffty;    // y-line groups
  Work w_fftz;    // z-line groups
  Work w_bricks;  // one block per PME brick
  Work w_planes;  // one block per PME grid z plane
  int* chunk_pre = nullptr;  // device: pair-kernel work items per system (prefix; a single system's are in its pg_n), then those of entry lists
  int* chunk_pre_a = nullptr;  // device: the same for the systems without a pending rebuild
  int pair_grid = 0;         // persistent pair-kernel blocks
  int n_entry = 0;           // systems with an entry list (a kernel of their own)
  int entry_grid = 0;        // its blocks
  int entry_waves = 0;       // a wave per chunk (1) or a workgroup (0)
  int fft_lds = 0;           // dynamic LDS bytes for the FFT kernels
  int fft_nl = 16;           // lines per FFT workgroup
  int lj_sep = 0;            // every system follows the LJ combination rule
  int ew_poly = 0;           // every system has the FP64 Ewald polynomials
  int com_any = 0;           // some system has a COM restraint
  int spread_bricks = 1;     // PME spread by bricks (1) or by global atomics (0)
  int pme_planes = 0;        // PME spread and x, y transforms by the plane kernels
  int plane_lds = 0;         // their dynamic LDS bytes
  int plane_points = 0;      // the largest plane's grid points
  int search_cap = 1;  // cap on the pair-search waves per I cluster (1, 2 or 4)
  int npt = 0;         // every system has the Andersen barostat on
};

// check: run the displacement test first (the fused step kernel does it otherwise)
void launch_nblist(const Launch& L, bool check);
// list entries (I, J) and lane masks of a single system's last build, in list order
void launch_pair_entries(const Launch& L, int2* pairs, unsigned long long* masks);
void launch_gather_sorted(const Launch& L);
void launch_chunk_prefix(const Launch& L);  // pair-kernel work items of every system, rebuild flags cleared
// pair-kernel work items of the systems without (built = false, into
// chunk_pre_a) or with (built = true, into chunk_pre; flags cleared) a pending rebuild
void launch_chunk_split(const Launch& L, bool built);
// 0 forces, 1 + FP32 energies, 2 + FP64 energies; work items cp (null: chunk_pre);
// fold: the energy / virial copies are folded after it (else launch_ev_fold
// later); spend: the kernel clears a single system's rebuild decision
void launch_pair(const Launch& L, int ev, const int* cp = nullptr, bool fold = true, bool spend = false);
void launch_ev_fold(const Launch& L);
void launch_bonded(const Launch& L, bool ev);
void launch_pme_fft_only(const Launch& L, int conv_mode);
void launch_pme_gtable(const SysDev& d, hipStream_t st);  // d.pme_g from d's box tables (host descriptor)
void launch_pme_part(const Launch& L, int part, bool ev);  // 0 spread, 1 FFT + convolution, 2 gather
// kick, drift, SHAKE, rebuild test; finish: the previous step's kick + RATTLE first
void launch_step_first(const Launch& L, bool finish = false);
void launch_step_second(const Launch& L);  // kick, RATTLE
void launch_shake(const Launch& L);
void launch_rattle(const Launch& L);
void launch_kinetic(const Launch& L);
void launch_maxwell(const Launch& L, double T, unsigned long long seed, unsigned long long counter);
void launch_zero_acc(const Launch& L);
void launch_clear_shake_flag(const Launch& L);
// every member's positions, velocities, build positions and flags into its
// snapshot (clear_shake: the SHAKE-failure flag cleared first)
void launch_snapshot(const Launch& L, bool clear_shake);
void launch_zero_forces(const Launch& L);
void launch_restraint(const Launch& L);  // COM restraint forces (systems with com_on)
// Andersen barostat step phases (every system of the launch has the barostat on)
void launch_npt_a(const Launch& L);
void launch_npt_b(const Launch& L);
void launch_npt_c(const Launch& L);
void launch_npt_d(const Launch& L);
void launch_npt_intra(const Launch& L);  // the clusters' internal virial (after the forces)
void launch_npt_g(const Launch& L, bool next);  // the pair sums too; next: the following step's launch_npt_a
// box fields and PME tables from the state (after a restore); build_scale: at the
// box of the last list build
void launch_npt_apply(const Launch& L, bool build_scale);
void launch_npt_mark(const Launch& L);  // a list build since: build scale = current box
void launch_npt_wtr(const Launch& L);   // piston virial from a stand-alone evaluation
// host layout <-> device arrays (fz_state.hip); d: host copy of the descriptor, pointers to device memory, nullable
void launch_get_state(const SysDev& d, double* xyz, unsigned long long* u, double* v, hipStream_t st);
void launch_set_positions(const SysDev& d, const double* xyz, const unsigned long long* u, hipStream_t st);
void launch_set_velocities(const SysDev& d, const double* v, hipStream_t st);
void launch_get_forces(const SysDev& d, double* f, hipStream_t st);
void launch_status(const Launch& L, StatusRec* out);

}  // namespace fz
