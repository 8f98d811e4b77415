// ocfd_chem.hip -- MI355X kernels for OpenCFD-Comb's finite-rate chemistry:
// the per-cell 0-D integrators of chemical_timeAdv (CHEM_reactions.f90:374-602)
// over a batch of independent cells, FP64 throughout.
//
//   * k_chem_fixed<MODE>: the reference integrator, nsub equal substeps per
//     cell, one cell per thread (MODE = CHEM_TimeAdv: 1 Euler, 2 RK2, 3 RK3,
//     -1 point-implicit Euler).
//   * k_chem_adaptive: point-implicit Euler with the adaptive per-cell substep
//     controller, one cell per thread.
//   * k_chem_queue: the same integrator in a persistent kernel whose lanes
//     pull cells from a device work queue, so lanes that finish early take
//     new cells instead of idling while the slowest lane of the wavefront
//     works through hundreds of substeps.
//
// Layout: rho is species-major [ns][n] (coalesced per species), E and dt [n].
// The mechanism lives in constant memory, the arithmetic in ocfd_chem_core.h.
// Sums keep the reference's order; the exponentials are the core's own and the
// logarithms the device library's, so results agree with the CPU restatement
// to a few ulps per call.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>

#include "../../include/ocfd_hip.h"
#include "ocfd_mlp.h"
#include "ocfd_mlp_tile.h"

#include "ocfd_chem_core.h"

// threads per workgroup of the one-cell-per-lane kernels: one wavefront, so
// that no wavefront waits for another's LDS to be freed
constexpr int CH_BLOCK = 64;

// Integration state of a cell handed from the per-lane queue to the
// cooperative kernel (struct of arrays, capacity cap records).
struct HeavyBuf {
  double* di;  // [CH_NS][cap]
  double *E, *t, *h_cap;
  int *nsub, *nrej, *cell;
  long cap;
};

namespace {
struct ChemCtx {
  bool ready = false;
  bool h2 = false;         // the mechanism has the structure of ChemH2
  bool rev_ready = false;  // reverse-rate data present (always for ReReac = 0)
  ChemMech h{};
  hipStream_t stream = nullptr, own = nullptr;
  unsigned long long* counter = nullptr;  // [0] queue head, [1] unfinished, [2] surrogate fallbacks
  int* fb_list = nullptr;                  // cells handed to the fallback integrator
  unsigned char* surr_buf = nullptr;       // surrogate phases: X[cap][16] (bf16), O[9][cap] (float), ok[cap]
  tbf16* surr_wpack = nullptr;             // network weights in MFMA fragment order
  long surr_wpack_cap = 0;
  const tbf16* surr_wp[MLP_MAX_LAYERS] = {};  // per layer, into surr_wpack
  unsigned long long surr_wp_version = ~0ull;  // network weights version packed
  long fb_cap = 0;
  HeavyBuf heavy{};                        // cells handed to the cooperative kernel
  int fallback_scheduler = 2;              // scheduler of the surrogate's fallback
  int coop_direct_max = 16384;             // fallback lists up to this size go to the cooperative kernel
  int coop_budget = 128;                   // attempts on one lane before the cooperative kernel
  unsigned char* heavy_mem = nullptr;
  // longest-first order of a batch: cell indices sorted by decreasing dt
  int order = 1;                           // 0: index order, 1: longest dt first
  int *ord_in = nullptr, *ord_out = nullptr;
  unsigned int *ord_keys = nullptr, *ord_keys_in = nullptr;
  unsigned long long* ord_count = nullptr;
  void* ord_temp = nullptr;
  size_t ord_temp_bytes = 0;
  long ord_cap = 0;
  unsigned char* ord_mem = nullptr;
  bool surr_ready = false;
  int surr_variant = 0;                    // tile shape of k_surr_mlp (SurrTile)
  float surr_tune_ms[8] = {};
  std::string err;
};
ChemCtx CX;
int cfail(const std::string& m) {
  CX.err = m;
  return 1;
}
}  // namespace

template <int MODE, class ST>
__global__ __launch_bounds__(CH_BLOCK, MODE == 1 ? 3 : 2) void k_chem_fixed(long n, double* rho, double* Ecell,
                                                                         const double* dtcell, int nsub) {
  __shared__ LaneLds<CH_BLOCK, MODE == -1> L;
  // the waves that the launch bounds ask for, four SIMDs a CU, fit its LDS
  static_assert(4 * (MODE == 1 ? 3 : 2) * sizeof(L) <= 160 * 1024, "LDS of a CU");
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  lane_lds_init(L);
  if (c >= n) return;
  double di[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) di[i] = rho[(long)i * n + c];
  double E = Ecell[c];
  const double h = dtcell[c] / nsub;
  Mech m = (Mech)&cm;
  for (int s = 0; s < nsub; s++) {
    m = mech_opaque(m);
    chem_step<MODE, ST>(m, L, di, E, h);
  }
#pragma unroll
  for (int i = 0; i < CH_NS; i++) rho[(long)i * n + c] = di[i];
  Ecell[c] = E;
}

// queue[0]: next cell of the work queue; queue[1]: cells left unfinished
// (budget of max_sub accepted and max_sub rejected attempts spent before dt)
__device__ __forceinline__ void chem_finish(long c, long n, double* rho, double* Ecell, const double* di, double E,
                                            int nsub, bool finished, int* nsub_out, unsigned long long* queue) {
#pragma unroll
  for (int i = 0; i < CH_NS; i++) rho[(long)i * n + c] = di[i];
  Ecell[c] = E;
  if (nsub_out) nsub_out[c] = nsub;
  if (!finished) atomicAdd(queue + 1, 1ull);
}

template <class ST>
__global__ __launch_bounds__(CH_BLOCK, 2) void k_chem_adaptive(long n, double* rho, double* Ecell, const double* dtcell,
                                                        ChemCtl ctl, int* nsub_out, unsigned long long* queue) {
  __shared__ LaneLds<CH_BLOCK, true> L;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  lane_lds_init(L);
  if (c >= n) return;
  double di[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) di[i] = rho[(long)i * n + c];
  double E = Ecell[c];
  const double dt = dtcell[c];
  double t = 0.0, h_cap = dt, h = 0.0;
  int nsub = 0, nrej = 0;
  Mech m = (Mech)&cm;
  while (t < dt && nsub < ctl.max_sub && nrej < ctl.max_sub) {
    m = mech_opaque(m);
    if (!chem_adaptive_attempt<ST>(m, L, di, E, dt, t, h_cap, ctl, h)) {
      nrej++;
      continue;
    }
    t = t + h;
    nsub++;
    if (dt - t <= 1e-12 * dt) break;
  }
  chem_finish(c, n, rho, Ecell, di, E, nsub, t >= dt || dt - t <= 1e-12 * dt, nsub_out, queue);
}

// The rest of one cell's integration on a whole wavefront; every lane holds
// the state.  Ends after at most 2 max_sub attempts.
template <class ST>
__device__ __forceinline__ void coop_cell(Mech m, CoopLds& L, const double2* tab, int lane, long c, long n, double* rho,
                                          double* Ecell, double* di, double E, double dt, double t, double h_cap,
                                          int nsub, int nrej, const ChemCtl& ctl, int* nsub_out,
                                          unsigned long long* queue) {
  // readfirstlane states that the loop decisions are uniform, which keeps
  // the control flow scalar
  while (__builtin_amdgcn_readfirstlane((t < dt && nsub < ctl.max_sub && nrej < ctl.max_sub) ? 1 : 0)) {
    m = mech_opaque(m);
    double h = 0.0;
    if (!coop_attempt<ST>(m, L, tab, lane, di, E, dt, t, h_cap, ctl, h)) {
      nrej++;
      continue;
    }
    t = t + h;
    nsub++;
    if (__builtin_amdgcn_readfirstlane((dt - t <= 1e-12 * dt) ? 1 : 0)) break;
  }
  if (lane == 0) chem_finish(c, n, rho, Ecell, di, E, nsub, t >= dt || dt - t <= 1e-12 * dt, nsub_out, queue);
  __builtin_amdgcn_wave_barrier();  // the wavefront goes on together
}

// Persistent kernel with a lane-level work queue, one wavefront a workgroup.
// Each pass runs one attempt per busy lane, with the same per-cell loop as
// k_chem_adaptive.  With a list, the cells are list[0 .. *list_count) instead
// of 0 .. n (n stays the array stride).
//   - First cells: all resident wavefronts are launched and share the
//     cells, so that a batch of fewer cells than lanes spreads over them.
//     With a list (longest first), lane l of wavefront w takes entry w + l W:
//     every wavefront gets one cell of each stratum instead of 64 of the
//     longest; without one, consecutive cells (their loads coalesce).
//   - Refill: a lane whose cell is done takes the next one; the wavefront
//     asks the queue once for all its idle lanes.
//   - Tail: once the queue is empty and one lane (COOP_TAIL) of the wavefront
//     still runs, its cell goes on with the whole wavefront (coop_attempt: 7 us
//     an attempt against 10 us for any number of lanes, so two cells gain only
//     where one of them ends early; with a tail of 1 / 2 / 3 cells, ms over three
//     seeds: 50,021 cells 1.47-1.61 / 1.51-1.83 / 1.62-1.90, 2,097,152 cells
//     3.49-3.60 / 3.70-3.83 / 3.81-3.96).
//   - budget > 0: a cell still running after `budget` attempts is handed to
//     k_chem_coop with its full controller state.  A list of at most
//     direct_max cells (the surrogate's rejects: few, and mostly stiff) hands
//     every cell over after its first attempt.
// A cell ends after at most 2 max_sub attempts, and a lane leaves once the
// queue is empty and its cell is done, so every wave reaches the exit.
constexpr int COOP_TAIL = 1;
template <class ST>
__global__ __launch_bounds__(CH_BLOCK, 2) void k_chem_queue(long n, double* rho, double* Ecell, const double* dtcell,
                                                     ChemCtl ctl, int* nsub_out, unsigned long long* queue,
                                                     const int* list, const unsigned long long* list_count, int budget,
                                                     int direct_max, HeavyBuf hb) {
  // the lanes' columns, and in the tail the one-cell tables, whose space
  // they share
  __shared__ union Lds {
    LaneLds<CH_BLOCK, true> lane;
    struct {
      CoopLds L;
      double2 tab[CH_EXPN];
    } coop;
    __device__ Lds() {}
  } U;
  LaneLds<CH_BLOCK, true>& L = U.lane;
  lane_lds_init(L);
  const unsigned long long count =
      list ? (*list_count < (unsigned long long)n ? *list_count : (unsigned long long)n) : (unsigned long long)n;
  if (list && budget > 0 && count <= (unsigned long long)direct_max) budget = 1;
  const int lane = threadIdx.x & 63;
  const unsigned long long lt = (1ull << lane) - 1ull;
  const unsigned long long W = gridDim.x, per = (count + W - 1) / W;
  const unsigned long long quota = per < 64ull ? per : 64ull;  // first cells of a wavefront
  long cell = -1;  // -1: needs work, -2: queue exhausted
  double di[CH_NS];
  double E = 0.0, dt = 0.0, t = 0.0, h_cap = 0.0;
  int nsub = 0, nrej = 0;
  bool first = true;
  Mech m = (Mech)&cm;
  while (true) {
    m = mech_opaque(m);
    const bool need = (cell == -1);
    const unsigned long long mask = __ballot(need);
    if (mask) {
      unsigned long long my;
      if (first) {
        my = list ? blockIdx.x + (unsigned long long)lane * W : blockIdx.x * quota + lane;
        if ((unsigned long long)lane >= quota) my = count;
        first = false;
      } else {
        const int leader = __ffsll((long long)mask) - 1;
        unsigned long long base = 0;
        if (lane == leader) base = atomicAdd(queue, (unsigned long long)__popcll(mask));
        my = W * quota + __shfl(base, leader) + (unsigned long long)__popcll(mask & lt);
      }
      if (need) {
        if (my < count) {
          cell = list ? (long)list[my] : (long)my;
          if (cell < 0 || cell >= n) cell = -1;  // a list entry outside the batch is skipped
        } else {
          cell = -2;
        }
        if (cell >= 0) {
#pragma unroll
          for (int i = 0; i < CH_NS; i++) di[i] = rho[(long)i * n + cell];
          E = Ecell[cell];
          dt = dtcell[cell];
          t = 0.0;
          h_cap = dt;
          nsub = 0;
          nrej = 0;
        }
      }
    }
    const unsigned long long busy = __ballot(cell != -2);
    if (busy == 0) break;  // every lane has found the queue empty
    if (budget == 0 && __popcll(busy) <= COOP_TAIL && __ballot(cell == -1) == 0) break;  // the tail
    if (cell >= 0) {
      bool done = !(t < dt && nsub < ctl.max_sub && nrej < ctl.max_sub);
      double h = 0.0;
      if (!done) {
        if (chem_adaptive_attempt<ST>(m, L, di, E, dt, t, h_cap, ctl, h)) {
          t = t + h;
          nsub++;
          done = dt - t <= 1e-12 * dt;
        } else {
          nrej++;
        }
        done = done || !(t < dt && nsub < ctl.max_sub && nrej < ctl.max_sub);
      }
      if (done) {
        chem_finish(cell, n, rho, Ecell, di, E, nsub, t >= dt || dt - t <= 1e-12 * dt, nsub_out, queue);
        cell = -1;
      } else if (budget > 0 && nsub + nrej >= budget) {
        const unsigned long long r = atomicAdd(queue + 3, 1ull);
#pragma unroll
        for (int i = 0; i < CH_NS; i++) hb.di[(long)i * hb.cap + r] = di[i];
        hb.E[r] = E;
        hb.t[r] = t;
        hb.h_cap[r] = h_cap;
        hb.nsub[r] = nsub;
        hb.nrej[r] = nrej;
        hb.cell[r] = (int)cell;
        cell = -1;
      }
    }
  }
  unsigned long long left = __ballot(cell >= 0);
  if (left == 0) return;
  __syncthreads();
  U.coop.tab[lane] = make_double2(cm.exp2t[lane][0], cm.exp2t[lane][1]);
  coop_lds_init(m, U.coop.L, lane);
  while (left) {
    const int src = __ffsll((long long)left) - 1;
    left &= left - 1;
    double d1[CH_NS];
#pragma unroll
    for (int i = 0; i < CH_NS; i++) d1[i] = bcast(di[i], src);
    const long c = __double_as_longlong(bcast(__longlong_as_double(cell), src));
    coop_cell<ST>(m, U.coop.L, U.coop.tab, lane, c, n, rho, Ecell, d1, bcast(E, src), bcast(dt, src), bcast(t, src),
                  bcast(h_cap, src), __builtin_amdgcn_readlane(nsub, src), __builtin_amdgcn_readlane(nrej, src), ctl,
                  nsub_out, queue);
  }
}

// One wavefront per handed-off cell, taken from a queue over the records.
template <class ST>
__global__ __launch_bounds__(64, 2) void k_chem_coop(long n, double* rho, double* Ecell, const double* dtcell, ChemCtl ctl,
                                                  int* nsub_out, unsigned long long* queue, HeavyBuf hb) {
  __shared__ CoopLds L;
  __shared__ double2 tab[CH_EXPN];
  const int lane = threadIdx.x;
  Mech m = (Mech)&cm;
  const unsigned long long count = queue[3];
  tab[lane] = make_double2(cm.exp2t[lane][0], cm.exp2t[lane][1]);
  coop_lds_init(m, L, lane);
  while (true) {
    // No branch on the lane here: with `if (lane == 0)` at the end of one
    // pass (chem_finish) and at the start of the next, the compiler may join
    // the two and let the other lanes run ahead of lane 0, into a shuffle
    // that reads a lane which is not there.
    const unsigned long long rl = atomicAdd(queue + 4, lane == 0 ? 1ull : 0ull);
    const unsigned long long r = (unsigned long long)__double_as_longlong(bcast(__longlong_as_double((long long)rl), 0));
    if (r >= count) break;
    const long c = hb.cell[r];
    double di[CH_NS];
#pragma unroll
    for (int i = 0; i < CH_NS; i++) di[i] = hb.di[(long)i * hb.cap + r];
    coop_cell<ST>(m, L, tab, lane, c, n, rho, Ecell, di, hb.E[r], dtcell[c], hb.t[r], hb.h_cap[r], hb.nsub[r],
                  hb.nrej[r], ctl, nsub_out, queue);
  }
}

__global__ void k_chem_reset(unsigned long long* queue) {
  if (threadIdx.x < 8 && blockIdx.x == 0) queue[threadIdx.x] = 0;
}

// ===========================================================================
// Learned surrogate (no reference counterpart).  Per cell: T from E by the
// reference's Newton iteration, features
//   f = [T, ln p, cbrt(Y_0..Y_8), ln dt],   x = (f - in_shift) * in_scale,
// the MLP (BF16 MFMA, FP32 accumulation) gives z, and in FP64
//   dY = P (z * out_scale)          (P projects onto element conservation)
// is accepted when the cell lies in the training domain, the H/O/N balance of
// dY is within elem_tol of the cell's total element content (moles of H, O
// and N per kg), Y + dY >= -y_neg_tol, every
// |dY_k| <= dy_max (the increment size up to which the network's error was
// measured to stay within tolerance) and the temperature after the update
// (Newton on the new state, update_Et energy) is finite and within
// [T_out_lo, T_out_hi].  Accepted cells are written
// (rho_k += rho dY_k, E by update_Et); the others go to a list for the plain
// FP64 integrator.
struct SurrCfg {
  double in_shift[12], in_scale[12];
  double out_scale[CH_NS];
  double T_lo, T_hi, p_lo, p_hi, dt_lo, dt_hi;
  double y_neg_tol, elem_tol, T_out_lo, T_out_hi, dy_max;
  double P[CH_NS][CH_NS];
  double Cel[3][CH_NS];
};
__constant__ SurrCfg scfg;
__constant__ MlpDevice cnet;
// the network's weights in fragment order (mt_pack_src): layer 0 over K = 32,
// hidden layers over 256, the output layer's first 16 rows
struct SurrPacked {
  const tbf16* W[MLP_MAX_LAYERS];
};
__constant__ SurrPacked cwp;

__global__ void k_pack_frag(long count, int KS, int ldw, const tbf16* __restrict__ src, tbf16* __restrict__ dst) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < count) dst[e] = src[mt_pack_src(e, KS, ldw)];
}

// raw surrogate features of one cell: [T, ln p, cbrt(Y_0..Y_8), ln dt]
__device__ __forceinline__ void surr_raw_features(Mech m, const double* di, double r, double E, double dt, double* f,
                                                  double& T, double& p) {
  T = chem_T(m, di, E);
  p = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) p = p + di[i] * m->ri[i] * T;
  f[0] = T;
  f[1] = log(p);
#pragma unroll
  for (int i = 0; i < CH_NS; i++) f[2 + i] = cbrt(di[i] / r);
  f[11] = log(dt);
}

// mode 0: T [n]; 1: raw features [n][12] (f64); 2: normalised inputs [n][12]
// (f32, (f - in_shift) * in_scale)
__global__ __launch_bounds__(128) void k_cell_features(long n, const double* __restrict__ rho,
                                                        const double* __restrict__ Ecell, const double* __restrict__ dtcell,
                                                        int mode, void* out) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Mech m = (Mech)&cm;
  double di[CH_NS], r = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    di[i] = rho[(long)i * n + c];
    r = r + di[i];
  }
  if (mode == 0) {
    ((double*)out)[c] = chem_T(m, di, Ecell[c]);
    return;
  }
  double f[12], T, p;
  surr_raw_features(m, di, r, Ecell[c], dtcell[c], f, T, p);
#pragma unroll
  for (int j = 0; j < 12; j++) {
    if (mode == 1) ((double*)out)[c * 12 + j] = f[j];
    else ((float*)out)[c * 12 + j] = (float)((f[j] - scfg.in_shift[j]) * scfg.in_scale[j]);
  }
}

// normalised targets: y [n][9] = ((rho1_k - rho0_k) / rho0) / out_scale_k
__global__ void k_surr_targets(long n, const double* __restrict__ rho0, const double* __restrict__ rho1, float* y) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) r = r + rho0[(long)i * n + c];
#pragma unroll
  for (int i = 0; i < CH_NS; i++)
    y[c * CH_NS + i] = (float)((rho1[(long)i * n + c] - rho0[(long)i * n + c]) / r / scfg.out_scale[i]);
}

__global__ void k_fill_u64(unsigned long long* p, int count) {
  if ((int)threadIdx.x < count && blockIdx.x == 0) p[threadIdx.x] = 0;
}

// Tile shapes of the surrogate network kernel (cells per workgroup, waves,
// workgroups per CU the register budget aims at, row groups of waves: with
// NWR = 2 the waves form 2 x 2 blocks of ROWS/2 rows x 128 columns, which
// halves the LDS reads per MFMA and doubles the weight loads).  All give
// bit-identical results; ocfd_chem_surrogate_autotune picks the fastest.
template <int V> struct SurrTile;
template <> struct SurrTile<0> { static constexpr int ROWS = 128, NW = 4, OCC = 2, NWR = 1; };
template <> struct SurrTile<1> { static constexpr int ROWS = 128, NW = 4, OCC = 2, NWR = 2; };
template <> struct SurrTile<2> { static constexpr int ROWS = 64, NW = 4, OCC = 3, NWR = 1; };
template <> struct SurrTile<3> { static constexpr int ROWS = 96, NW = 4, OCC = 2, NWR = 1; };
#define SURR_VARIANTS 4

// The surrogate step runs as three launches, so that every phase keeps all
// of its threads busy: the per-cell FP64 work (features with the Newton
// temperature; projection, checks, update_Et and a second Newton
// temperature) takes one cell per thread, and the network takes whole
// workgroups of MFMA waves.  (Fused into one kernel, the per-cell phases ran
// on the ROWS threads of a workgroup of NW * 64 while the other waves waited
// at its barriers.)
//
// Phase 1: normalised inputs X[n][16] (bfloat16, rounded to nearest even;
// features 12..15 zero), the network's first-layer operand rows, and the
// domain check ok[n].
__global__ __launch_bounds__(256) void k_surr_features(long n, const double* __restrict__ rho,
                                                       const double* __restrict__ Ecell,
                                                       const double* __restrict__ dtcell, tbf16* __restrict__ X,
                                                       unsigned char* __restrict__ okv) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Mech m = (Mech)&cm;
  float x[12];
  double di[CH_NS];
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    di[i] = rho[(long)i * n + c];
    r = r + di[i];
  }
  const double E = Ecell[c], dt = dtcell[c];
  double f[12], T, p;
  surr_raw_features(m, di, r, E, dt, f, T, p);
  int ok = (T >= scfg.T_lo && T <= scfg.T_hi && p >= scfg.p_lo && p <= scfg.p_hi && dt >= scfg.dt_lo &&
            dt <= scfg.dt_hi && r > 0.0) ? 1 : 0;
#pragma unroll
  for (int j = 0; j < 12; j++) {
    x[j] = (float)((f[j] - scfg.in_shift[j]) * scfg.in_scale[j]);
    if (!(fabsf(x[j]) <= 1e6f)) ok = 0;  // also catches NaN
  }
  tbf16x8 lo, hi;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    lo[j] = (tbf16)(ok ? x[j] : 0.f);
    hi[j] = (tbf16)(ok && j < 4 ? x[8 + j] : 0.f);
  }
  *(tbf16x8*)&X[c * 16] = lo;
  *(tbf16x8*)&X[c * 16 + 8] = hi;
  okv[c] = (unsigned char)ok;
}

// Phase 2: the network on tiles of ROWS cells, O[9][n] (float) from X.  The
// input rows are staged into LDS columns 0..15 with columns 16..31 zeroed:
// the first layer runs over K = 32 (its weights beyond input 12 are zero).
template <int V>
__global__ __launch_bounds__(SurrTile<V>::NW * 64, SurrTile<V>::OCC) void k_surr_mlp(long n,
                                                                                       const tbf16* __restrict__ X,
                                                                                       float* __restrict__ Oout) {
  constexpr int ROWS = SurrTile<V>::ROWS, NW = SurrTile<V>::NW, NT = NW * 64;
  __shared__ __attribute__((aligned(16))) tbf16 H[ROWS * MT_LDH];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const long c0 = (long)blockIdx.x * ROWS;
  const tbf16x8 zero8 = {};
  for (int e = t; e < ROWS * 2; e += NT) {
    const int row = e >> 1, h = (e & 1) * 8;
    const long c = c0 + row;
    *(tbf16x8*)&H[row * MT_LDH + h] = c < n ? *(const tbf16x8*)&X[c * 16 + h] : zero8;
    *(tbf16x8*)&H[row * MT_LDH + 16 + h] = zero8;
  }
  __syncthreads();
  const int L = cnet.n_layers;
  constexpr int NWR = SurrTile<V>::NWR;
  mt_layer256<true, ROWS, NW, 32, NWR>(H, cwp.W[0], cnet.b[0], lane, w);
  for (int l = 1; l < L - 1; l++) mt_layer256<true, ROWS, NW, 256, NWR>(H, cwp.W[l], cnet.b[l], lane, w);
  mt_out_cols<ROWS, NW, 256, CH_NS>(H, cwp.W[L - 1], cnet.b[L - 1], Oout, n, c0, lane, w);
}

// Phase 3: in FP64, dY = P (O * out_scale) (P projects onto element
// conservation); the cell is accepted when it lies in the training domain,
// the H/O/N balance of dY is within elem_tol of the cell's total element
// content (moles of H, O and N per kg), Y + dY >= -y_neg_tol, every
// |dY_k| <= dy_max (the increment size up to which the network's error was
// measured to stay within tolerance) and the temperature after the update
// (Newton on the new state, update_Et energy) is finite and within
// [T_out_lo, T_out_hi].  Accepted cells are written (rho_k += rho dY_k, E by
// update_Et); the others go to a list for the plain FP64 integrator.
__global__ __launch_bounds__(256) void k_surr_finish(long n, double* rho, double* Ecell,
                                                     const float* __restrict__ Oin,
                                                     const unsigned char* __restrict__ okv, int* flag_out,
                                                     int* fb_list, unsigned long long* counters) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Mech m = (Mech)&cm;
  int why = okv[c] ? 0 : 1;
  double di[CH_NS], dY[CH_NS], dYp[CH_NS], dinew[CH_NS];
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    di[i] = rho[(long)i * n + c];
    r = r + di[i];
    dY[i] = (double)Oin[(long)i * n + c] * scfg.out_scale[i];
  }
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    double a = 0.0;
#pragma unroll
    for (int j = 0; j < CH_NS; j++) a = a + scfg.P[i][j] * dY[j];
    dYp[i] = a;
  }
  // each element's balance to elem_tol of the cell's total element content
  // (mol/kg): a cell without one element (pure air has no H) is held to the
  // same absolute bound as the others, not to zero
  double content = 0.0;
#pragma unroll
  for (int e = 0; e < 3; e++)
#pragma unroll
    for (int i = 0; i < CH_NS; i++) content = content + scfg.Cel[e][i] * fmax(di[i] / r, 0.0);
#pragma unroll
  for (int e = 0; e < 3; e++) {
    double res = 0.0;
#pragma unroll
    for (int i = 0; i < CH_NS; i++) res = res + scfg.Cel[e][i] * dYp[i];
    if (!(fabs(res) <= scfg.elem_tol * content + 1e-300)) why |= 2;
  }
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    if (!(di[i] / r + dYp[i] >= -scfg.y_neg_tol)) why |= 4;
    if (!(fabs(dYp[i]) <= scfg.dy_max)) why |= 16;  // also NaN
    dinew[i] = di[i] + r * dYp[i];
  }
  double E = Ecell[c];
  chem_update_et(m, di, dinew, E);
  const double Tn = chem_T(m, dinew, E);
  if (!(Tn >= scfg.T_out_lo && Tn <= scfg.T_out_hi)) why |= 8;  // also NaN
  if (why == 0) {
#pragma unroll
    for (int i = 0; i < CH_NS; i++) rho[(long)i * n + c] = dinew[i];
    Ecell[c] = E;
  } else {
    const unsigned long long k = atomicAdd(counters + 2, 1ull);
    fb_list[k] = (int)c;
  }
  if (flag_out) flag_out[c] = why;
}

// checks of the surrogate network, fallback list capacity, network view into
// the constant bank, counters cleared (on CX.stream)
int surr_prepare(long n, const char* who) {
  if (!CX.ready || !CX.surr_ready) return cfail(std::string(who) + ": mechanism or surrogate not set");
  if (!CX.rev_ready) return cfail(std::string(who) + ": ReReac 1/2 needs ocfd_chem_set_reverse_rates");
  const MlpDevice* net = ocfd_mlp_device_view();
  if (!net) return cfail(std::string(who) + ": no network (ocfd_mlp_create)");
  const int L = net->n_layers;
  bool shape_ok = L >= 2 && net->din[0] == 12 && net->dinp[0] == 64 && net->dout[L - 1] == CH_NS;
  for (int l = 0; l < L - 1; l++) shape_ok = shape_ok && net->dout[l] == 256;
  if (!shape_ok) return cfail(std::string(who) + ": the network must be 12 -> 256 x k -> 9");
  if (n > 0x7fffffffL) return cfail(std::string(who) + ": at most 2^31-1 cells");
  if (n > CX.fb_cap) {
    if (CX.fb_list) hipFree(CX.fb_list);
    if (CX.surr_buf) hipFree(CX.surr_buf);
    CX.fb_list = nullptr;
    CX.surr_buf = nullptr;
    CX.fb_cap = 0;
    // the phases' buffers: inputs X[n][16] (bf16), outputs O[9][n] (float), ok[n]
    if (hipMalloc(&CX.fb_list, (size_t)n * sizeof(int)) != hipSuccess ||
        hipMalloc(&CX.surr_buf, (size_t)n * (16 * sizeof(tbf16) + 9 * sizeof(float) + 1)) != hipSuccess)
      return cfail(std::string(who) + ": hipMalloc");
    CX.fb_cap = n;
  }
  // the weights in fragment order, repacked whenever the network's weights
  // changed: 16 output blocks x 1 chunk for layer 0, 16 x 8 for the hidden
  // layers, 1 x 8 for the output layer
  long off[MLP_MAX_LAYERS], need = 0;
  for (int l = 0; l < L; l++) {
    off[l] = need;
    need += (l == L - 1 ? 1 : 16) * (l == 0 ? 1 : 8) * 512L;
  }
  if (need > CX.surr_wpack_cap) {
    CX.surr_wp_version = ~0ull;
    if (CX.surr_wpack) hipFree(CX.surr_wpack);
    CX.surr_wpack = nullptr;
    CX.surr_wpack_cap = 0;
    if (hipMalloc(&CX.surr_wpack, need * sizeof(tbf16)) != hipSuccess)
      return cfail(std::string(who) + ": hipMalloc");
    CX.surr_wpack_cap = need;
  }
  if (CX.surr_wp_version != ocfd_mlp_weights_version()) {
    for (int l = 0; l < L; l++) {
      const long cnt = (l == L - 1 ? 1 : 16) * (l == 0 ? 1 : 8) * 512L;
      hipLaunchKernelGGL(k_pack_frag, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, CX.stream, cnt,
                         l == 0 ? 1 : 8, net->dinp[l], (const tbf16*)net->W[l], CX.surr_wpack + off[l]);
      CX.surr_wp[l] = CX.surr_wpack + off[l];
    }
    CX.surr_wp_version = ocfd_mlp_weights_version();
  }
  if (hipMemcpyToSymbolAsync(HIP_SYMBOL(cnet), net, sizeof(MlpDevice), 0, hipMemcpyHostToDevice, CX.stream) !=
          hipSuccess ||
      hipMemcpyToSymbolAsync(HIP_SYMBOL(cwp), CX.surr_wp, sizeof(SurrPacked), 0, hipMemcpyHostToDevice,
                             CX.stream) != hipSuccess)
    return cfail(std::string(who) + ": copy failed");
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, CX.stream, CX.counter, 8);
  return 0;
}

template <int V>
void launch_surrogate_v(long n, double* rho, double* E, const double* dt, int* flag_out) {
  constexpr int R = SurrTile<V>::ROWS, NW = SurrTile<V>::NW;
  tbf16* X = (tbf16*)CX.surr_buf;
  float* O = (float*)(X + 16 * (size_t)CX.fb_cap);
  unsigned char* ok = (unsigned char*)(O + 9 * (size_t)CX.fb_cap);
  const dim3 g1((unsigned)((n + 255) / 256));
  hipLaunchKernelGGL(k_surr_features, g1, dim3(256), 0, CX.stream, n, (const double*)rho, (const double*)E, dt, X, ok);
  hipLaunchKernelGGL(k_surr_mlp<V>, dim3((unsigned)((n + R - 1) / R)), dim3(NW * 64), 0, CX.stream, n,
                     (const tbf16*)X, O);
  hipLaunchKernelGGL(k_surr_finish, g1, dim3(256), 0, CX.stream, n, rho, E, (const float*)O,
                     (const unsigned char*)ok, flag_out, CX.fb_list, CX.counter);
}
void launch_surrogate(int v, long n, double* rho, double* E, const double* dt, int* flag_out) {
  switch (v) {
    case 1: launch_surrogate_v<1>(n, rho, E, dt, flag_out); break;
    case 2: launch_surrogate_v<2>(n, rho, E, dt, flag_out); break;
    case 3: launch_surrogate_v<3>(n, rho, E, dt, flag_out); break;
    default: launch_surrogate_v<0>(n, rho, E, dt, flag_out); break;
  }
}

int ensure_heavy(long n) {
  if (n <= CX.heavy.cap) return 0;
  if (CX.heavy_mem) hipFree(CX.heavy_mem);
  CX.heavy_mem = nullptr;
  CX.heavy = HeavyBuf{};
  const size_t bytes = (size_t)n * ((CH_NS + 3) * sizeof(double) + 3 * sizeof(int)) + 256;
  if (hipMalloc(&CX.heavy_mem, bytes) != hipSuccess) return cfail("chemistry: out of device memory (work records)");
  HeavyBuf& h = CX.heavy;
  double* d = (double*)CX.heavy_mem;
  h.di = d;
  h.E = d + (size_t)CH_NS * n;
  h.t = h.E + n;
  h.h_cap = h.t + n;
  int* q = (int*)(h.h_cap + n);
  h.nsub = q;
  h.nrej = q + n;
  h.cell = q + 2 * n;
  h.cap = n;
  return 0;
}

// Sort key of a cell, an estimate of its work: dt T^2 (T by comput_T_rgas).
// A 2^21-cell jet-flame batch laid out in this order takes 2.70 ms, by dt alone
// 2.74, by the true substep counts 2.22 and in index order 2.97; with the sort,
// 0.3 ms, 3.01 (50,000 cells: 1.27, 1.30, 1.16, 1.33; with the sort 1.52).  The
// key is the top 32 bits of the value (sign, exponent and 20 mantissa bits,
// which order like the values for a positive finite number: to within 1e-6); 0
// otherwise (such cells go last).
__device__ __forceinline__ unsigned int cell_key(Mech m, const double* __restrict__ rho,
                                                 const double* __restrict__ Ecell, const double* __restrict__ dtcell,
                                                 long n, long c) {
  double di[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) di[i] = rho[(long)i * n + c];
  const double T = chem_T(m, di, Ecell[c]);
  const double w = dtcell[c] * T * T;
  return (w > 0.0 && w <= 1.7976931348623157e308) ? (unsigned int)((unsigned long long)__double_as_longlong(w) >> 32)
                                                  : 0u;
}

// keys[c] = cell_key of cell c, idx[c] = c for c < n, and *count = n
__global__ void k_order_keys(long n, const double* __restrict__ rho, const double* __restrict__ Ecell,
                             const double* __restrict__ dt, unsigned int* __restrict__ keys, int* idx,
                             unsigned long long* count) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) {
    keys[c] = cell_key((Mech)&cm, rho, Ecell, dt, n, c);
    idx[c] = (int)c;
  }
  if (c == 0) *count = (unsigned long long)n;
}

int ensure_order(long n) {
  if (n <= CX.ord_cap) return 0;
  if (CX.ord_mem) hipFree(CX.ord_mem);
  CX.ord_mem = nullptr;
  CX.ord_cap = 0;
  size_t temp = 0;
  if (hipcub::DeviceRadixSort::SortPairsDescending(nullptr, temp, (const unsigned int*)nullptr, (unsigned int*)nullptr,
                                                   (const int*)nullptr, (int*)nullptr, (int)n) != hipSuccess)
    return cfail("chemistry: radix sort query failed");
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t b_keys = up(sizeof(unsigned int) * (size_t)n), b_idx = up(sizeof(int) * (size_t)n), b_cnt = 256;
  if (hipMalloc(&CX.ord_mem, 2 * b_keys + 2 * b_idx + b_cnt + up(temp)) != hipSuccess)
    return cfail("chemistry: out of device memory (cell order)");
  unsigned char* p = CX.ord_mem;
  CX.ord_keys = (unsigned int*)p;
  CX.ord_keys_in = (unsigned int*)(p + b_keys);
  p += 2 * b_keys;
  CX.ord_in = (int*)p;
  CX.ord_out = (int*)(p + b_idx);
  CX.ord_count = (unsigned long long*)(p + 2 * b_idx);
  CX.ord_temp = p + 2 * b_idx + b_cnt;
  CX.ord_temp_bytes = temp;
  CX.ord_cap = n;
  return 0;
}

// Cell indices in order of decreasing cell_key, ties in index order (a
// stable radix sort): the cells with the longest integrations start first,
// so the batch does not end waiting on a stiff cell that a lane took up
// late.  The result is CX.ord_out[0 .. n) with *CX.ord_count = n.
int order_longest_first(long n, const double* rho, const double* E, const double* dt) {
  if (n > 0x7fffffffL) return cfail("chemistry: the cell order needs n < 2^31");
  if (ensure_order(n)) return 1;
  hipLaunchKernelGGL(k_order_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, CX.stream, n, rho, E, dt,
                     CX.ord_keys_in, CX.ord_in, CX.ord_count);
  size_t temp = CX.ord_temp_bytes;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairsDescending(CX.ord_temp, temp, CX.ord_keys_in, CX.ord_keys,
                                                                    CX.ord_in, CX.ord_out, (int)n, 0, 32, CX.stream);
  if (e != hipSuccess) return cfail(std::string("chemistry: radix sort failed: ") + hipGetErrorString(e));
  return 0;
}

// Sort keys of a cell list whose length is on the device: cell_key of each
// listed cell, 0 past the end.  A stable descending sort keeps every listed
// cell ahead of the slots past the end (their keys are the smallest, and
// among equal keys the listed cells come first in index order).
__global__ void k_list_keys(long n, long cap, const int* __restrict__ list, const unsigned long long* __restrict__ count,
                            const double* __restrict__ rho, const double* __restrict__ Ecell,
                            const double* __restrict__ dt, unsigned int* __restrict__ keys) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cap) return;
  unsigned int k = 0u;
  if ((unsigned long long)i < *count) {
    const long c = list[i];
    if (c >= 0 && c < n) k = cell_key((Mech)&cm, rho, Ecell, dt, n, c);
  }
  keys[i] = k;
}

// The cells of list[0 .. *count) (count <= cap <= n) in order of decreasing
// cell_key, into CX.ord_out[0 .. *count).
int order_list_longest_first(long n, long cap, const int* list, const unsigned long long* count, const double* rho,
                             const double* E, const double* dt) {
  if (n > 0x7fffffffL || cap > n) return cfail("chemistry: the cell order needs cap <= n < 2^31");
  if (ensure_order(n)) return 1;
  hipLaunchKernelGGL(k_list_keys, dim3((unsigned)((cap + 255) / 256)), dim3(256), 0, CX.stream, n, cap, list, count,
                     rho, E, dt, CX.ord_keys_in);
  size_t temp = CX.ord_temp_bytes;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairsDescending(CX.ord_temp, temp, CX.ord_keys_in, CX.ord_keys,
                                                                    list, CX.ord_out, (int)cap, 0, 32, CX.stream);
  if (e != hipSuccess) return cfail(std::string("chemistry: radix sort failed: ") + hipGetErrorString(e));
  return 0;
}

// the kernels for the mechanism's structure
template <class F>
auto chem_kernel(F f) {
  return CX.h2 ? f(ChemH2{}) : CX.h.rereac != 0 ? f(ChemRev{}) : f(ChemAny{});
}

// the adaptive integrator over cells 0..n-1, or over list[0 .. *list_count)
// when list is given; counters [0,1,3,4] must be zero.  scheduler 0: one
// cell per thread; 1: per-lane work queue; 2: work queue with the cooperative
// kernel taking the cells that outlast CX.coop_budget attempts.  direct: a
// list of at most CX.coop_direct_max cells goes to the cooperative kernel
// after one attempt per cell (the surrogate's rejects).
int launch_adaptive(long n, double* rho, double* E, const double* dt, const ChemCtl& ctl, int* nsub_out, int scheduler,
                    const int* list, const unsigned long long* list_count, bool direct = true,
                    unsigned long long* counter = nullptr) {
  if (!counter) counter = CX.counter;
  if (scheduler == 0 && !list) {
    const auto kern = chem_kernel([](auto st) { return &k_chem_adaptive<decltype(st)>; });
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + CH_BLOCK - 1) / CH_BLOCK)), dim3(CH_BLOCK), 0, CX.stream, n, rho, E, dt,
                       ctl, nsub_out, counter);
    return hipGetLastError() == hipSuccess ? 0 : cfail("chemistry: launch failed");
  }
  const auto queue = chem_kernel([](auto st) { return &k_chem_queue<decltype(st)>; });
  int dev = 0, ncu = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, queue, CH_BLOCK, 0) != hipSuccess)
    return cfail("chemistry: device query failed");
  if (per < 1) per = 1;
  long blocks = (long)ncu * per;
  if (blocks > n) blocks = n;
  const bool coop = scheduler == 2;
  if (coop && ensure_heavy(n)) return 1;
  hipLaunchKernelGGL(queue, dim3((unsigned)blocks), dim3(CH_BLOCK), 0, CX.stream, n, rho, E, dt, ctl, nsub_out,
                     counter, list, list_count, coop ? CX.coop_budget : 0, direct ? CX.coop_direct_max : 0,
                     coop ? CX.heavy : HeavyBuf{});
  if (coop) {
    const auto coopk = chem_kernel([](auto st) { return &k_chem_coop<decltype(st)>; });
    int per2 = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per2, coopk, 64, 0) != hipSuccess)
      return cfail("chemistry: device query failed");
    long b2 = (long)ncu * (per2 < 1 ? 1 : per2);
    if (b2 > n) b2 = n;
    hipLaunchKernelGGL(coopk, dim3((unsigned)b2), dim3(64), 0, CX.stream, n, rho, E, dt, ctl, nsub_out,
                       counter, CX.heavy);
  }
  return hipGetLastError() == hipSuccess ? 0 : cfail("chemistry: launch failed");
}

// ===========================================================================
// The batch entry behind ocfd_chem_adaptive_batch; the flow solver calls it
// with order = false (its cells share one dt, so the order is the index order).
int chem_adaptive_batch(long n, double* rho, double* E, const double* dt, double rtol_y, double y_floor, double rtol_t,
                        int max_sub, int* nsub_out, int scheduler, bool order) {
  if (!CX.ready) return cfail("ocfd_chem_adaptive_batch: call ocfd_chem_set_mechanism first");
  if (!CX.rev_ready) return cfail("ocfd_chem_adaptive_batch: ReReac 1/2 needs ocfd_chem_set_reverse_rates");
  if (max_sub < 1 || !(rtol_y > 0.0) || !(y_floor >= 0.0) || !(rtol_t > 0.0))
    return cfail("ocfd_chem_adaptive_batch: bad controller parameters");
  if (scheduler < 0 || scheduler > 2) return cfail("ocfd_chem_adaptive_batch: scheduler 0, 1 or 2");
  // the cooperative hand-off records a cell index as int
  if (scheduler == 2 && n > 0x7fffffffL) return cfail("ocfd_chem_adaptive_batch: scheduler 2 takes at most 2^31-1 cells");
  const ChemCtl ctl{rtol_y, y_floor, rtol_t, max_sub};
  hipLaunchKernelGGL(k_chem_reset, dim3(1), dim3(64), 0, CX.stream, CX.counter);
  if (n <= 0) return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_adaptive_batch: launch failed");
  // the order lists cells as int: a batch of 2^31 cells or more runs in index order
  if (order && scheduler != 0 && n > 1 && n <= 0x7fffffffL) {
    if (order_longest_first(n, rho, E, dt)) return 1;
    return launch_adaptive(n, rho, E, dt, ctl, nsub_out, scheduler, CX.ord_out, CX.ord_count, false);
  }
  return launch_adaptive(n, rho, E, dt, ctl, nsub_out, scheduler, nullptr, nullptr);
}

// The batch entry behind ocfd_chem_surrogate_batch; with order, the fallback
// list is taken by decreasing dt (the flow solver passes false: one dt).
int chem_surrogate_batch(long n, double* rho, double* E, const double* dt, bool fallback, double rtol_y, double y_floor,
                         double rtol_t, int max_sub, int* flag_out, bool order) {
  if (fallback && (max_sub < 1 || !(rtol_y > 0.0) || !(y_floor >= 0.0) || !(rtol_t > 0.0)))
    return cfail("ocfd_chem_surrogate_batch: bad controller parameters");
  if (surr_prepare(n, "ocfd_chem_surrogate_batch")) return 1;
  if (n <= 0) return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_surrogate_batch: launch failed");
  launch_surrogate(CX.surr_variant, n, rho, E, dt, flag_out);
  if (fallback) {
    const ChemCtl ctl{rtol_y, y_floor, rtol_t, max_sub};
    const int* list = CX.fb_list;
    if (order && CX.fallback_scheduler != 0 && n > 1) {
      // the list's length decides the work: none (no launch), or a sort of
      // that many keys only (sorting all n slots cost 0.3 ms on 2^21 cells)
      unsigned long long cnt = 0;
      if (hipMemcpyAsync(&cnt, CX.counter + 2, sizeof(cnt), hipMemcpyDeviceToHost, CX.stream) != hipSuccess ||
          hipStreamSynchronize(CX.stream) != hipSuccess)
        return cfail("ocfd_chem_surrogate_batch: reading the fallback count failed");
      if (cnt == 0) return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_surrogate_batch: launch failed");
      const long cap = (long)std::min<unsigned long long>(cnt, (unsigned long long)n);
      if (cap > 1) {
        if (order_list_longest_first(n, cap, CX.fb_list, CX.counter + 2, rho, E, dt)) return 1;
        list = CX.ord_out;
      }
    }
    if (launch_adaptive(n, rho, E, dt, ctl, nullptr, CX.fallback_scheduler, list, CX.counter + 2)) return 1;
  }
  if (hipGetLastError() != hipSuccess) return cfail("ocfd_chem_surrogate_batch: launch failed");
  return 0;
}

// ===========================================================================
// Workspace of ocfd_chem_adaptive_batch_noalloc (no reference counterpart):
// the work counters, the cell-order keys and index lists and the radix-sort
// workspace of one batch of at most NA_MAX_CELLS cells, in one file-scope
// device array.  Each GPU holds its own copy (about 32.5 MiB) from module
// load until the process ends; host code reaches it only through the
// per-device address from hipGetSymbolAddress, never through the symbol.
constexpr long NA_MAX_CELLS = 1L << 20;
constexpr size_t NA_COUNTERS = 256;  // 8 u64 work counters (k_chem_reset), then padding
constexpr size_t NA_COUNT = 256;     // length of the ordered list (u64)
constexpr size_t NA_KEYS = sizeof(unsigned int) * NA_MAX_CELLS;
constexpr size_t NA_LIST = sizeof(int) * NA_MAX_CELLS;
constexpr size_t NA_TEMP = size_t(16) << 20;  // radix-sort workspace
constexpr size_t NA_BYTES = NA_COUNTERS + NA_COUNT + 2 * NA_KEYS + 2 * NA_LIST + NA_TEMP;
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

constexpr int NA_MAX_DEVICES = 64;
unsigned char* na_base[NA_MAX_DEVICES] = {};

// The current device's copy of scratch, resolved once per device (with that
// device current) on the first call there.
int na_workspace(unsigned char** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NA_MAX_DEVICES)
    return cfail("ocfd_chem_adaptive_batch_noalloc: no usable current device");
  if (!na_base[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return cfail(std::string("ocfd_chem_adaptive_batch_noalloc: hipGetSymbolAddress failed: ") + hipGetErrorString(e));
    na_base[dev] = (unsigned char*)p;
  }
  *out = na_base[dev];
  return 0;
}

extern "C" {

const char* ocfd_chem_last_error(void) { return CX.err.c_str(); }

int32_t ocfd_chem_set_mechanism(int32_t ns, int32_t nr, int32_t rereac, const int32_t* af_type,
                                const int32_t* third_body, const double* fc_troe, const double* arrhenius,
                                const int32_t* vf, const int32_t* vr, const double* eff, int32_t n_tct,
                                const double* tct, double tct_max, const double* mi, const double* coef) {
  if (ns != CH_NS) return cfail("ocfd_chem_set_mechanism: this build is compiled for 9 species");
  if (nr > CH_NR_MAX || n_tct > CH_NT_MAX || n_tct < 1) return cfail("ocfd_chem_set_mechanism: too many reactions or ranges");
  if (rereac < 0 || rereac > 2) return cfail("ocfd_chem_set_mechanism: ReReac must be 0, 1 or 2");
  ChemMech& h = CX.h;
  h = ChemMech{};
  h.ns = ns;
  h.rereac = rereac;
  CX.rev_ready = rereac == 0;
  h.nr = nr;
  h.n_tct = n_tct;
  for (int j = 0; j < nr; j++) {
    ChemRx& R = h.rx[j];
    R.af_type = af_type[j];
    R.tb = third_body[j];
    const double* a = arrhenius + j * 6;
    R.a0 = a[0]; R.b0 = a[1]; R.e0 = a[2];
    R.a1 = a[3]; R.b1 = a[4]; R.e1 = a[5];
    if (af_type[j] != 0 && af_type[j] != 2) {
      R.lfc = std::log10(fc_troe[j]);
      R.ac = -0.4 - (double)0.67f * R.lfc;  // REAL(4) literals of the reference
      R.an = 0.75 - (double)1.27f * R.lfc;
    }
    for (int i = 0; i < ns; i++) {
      const int f = vf[j * ns + i], r = vr[j * ns + i];
      R.vf[i] = f;
      R.vr[i] = r;
      R.nu[i] = r - f;
      R.eff[i] = eff[j * ns + i];
      R.sgm += r - f;
      if (f != 0 || r != 0) R.part |= 1 << i;
    }
    // the mass-action products as species slots, where they fit (else ipow)
    auto slots = [&](const int32_t* v, unsigned long long& s) {
      s = 0;
      int c = 0;
      for (int i = 0; i < ns; i++) {
        if (v[i] < 0 || c + v[i] > 8) return -1;
        for (int q = 0; q < v[i]; q++) s |= (unsigned long long)i << (8 * c++);
      }
      for (int q = c; q < CH_SLOTS; q++) s |= (unsigned long long)CH_NS << (8 * q);
      return c;
    };
    R.nsf = slots(vf + j * ns, R.sf);
    R.nsr = slots(vr + j * ns, R.sr);
  }
  for (int j = 0; j < n_tct - 1; j++) h.tct[j] = tct[j];
  h.tct_max = tct_max;
  auto P2 = [](double x) { return x * x; };
  auto P3 = [](double x) { double x2 = x * x; return x2 * x; };
  auto P4 = [](double x) { double x2 = x * x; return x2 * x2; };
  auto P5 = [](double x) { double x2 = x * x; return (x2 * x2) * x; };
  for (int k = 0; k < ns; k++) {
    h.mi[k] = mi[k];
    h.ri[k] = CH_R0 / mi[k];
    h.ci6[k] = 1.0e-6 / mi[k];
    h.rcv[k] = 2.5 * h.ri[k];
    for (int j = 0; j < n_tct; j++)
      for (int c = 0; c < 7; c++) h.coef[k][j][c] = coef[(k * n_tct + j) * 7 + c];
    h.rf[k] = h.ri[k] * h.coef[k][0][5];
    double ect = 0.0;  // read_Spec, CHEM_thermdyn.f90:43-47
    for (int j = 0; j < n_tct; j++) {
      const double* c = h.coef[k][j];
      if (j > 0) {
        const double t = h.tct[j - 1];
        const double* p = h.coef[k][j - 1];
        ect = -((c[0] - p[0]) * t + (c[1] - p[1]) * P2(t) / 2.0 + (c[2] - p[2]) * P3(t) / 3.0 +
                (c[3] - p[3]) * P4(t) / 4.0 + (c[4] - p[4]) * P5(t) / 5.0) +
              ect;
      }
      h.ev[j][0][k] = (c[0] - 1.0) * h.ri[k];
      for (int a = 1; a < 5; a++) h.ev[j][a][k] = c[a] * h.ri[k];
      h.ev[j][5][k] = ect * h.ri[k];
      const double gb[7] = {c[0], c[1] / 2.0, c[2] / 6.0, c[3] / 12.0, c[4] / 20.0, c[5], c[6]};
      for (int a = 0; a < 7; a++) h.gb[k][j][a] = gb[a];
    }
  }
  chem_exp_table(h.exp2t);
  CX.h2 = rereac == 0 && nr == ChemH2::NR && n_tct == ChemH2::NT;
  for (int j = 0; CX.h2 && j < nr; j++) {
    const ChemRx& R = h.rx[j];
    const int ar = (R.b0 != 0.0) | (R.e0 != 0.0) << 1 | (R.b1 != 0.0) << 2 | (R.e1 != 0.0) << 3;
    CX.h2 = R.af_type == ChemH2::af[j] && (R.tb == 1) == (ChemH2::tb[j] == 1) && ar == ChemH2::ar[j];
    for (int i = 0; i < ns; i++) CX.h2 = CX.h2 && R.vf[i] == ChemH2::vf[j][i] && R.vr[i] == ChemH2::vr[j][i];
  }
  if (!CX.own) {
    if (hipStreamCreateWithFlags(&CX.own, hipStreamNonBlocking) != hipSuccess) return cfail("no HIP device/stream");
    if (hipMalloc(&CX.counter, 8 * sizeof(unsigned long long)) != hipSuccess) return cfail("hipMalloc failed");
  }
  CX.stream = CX.own;
  // kernels still in flight read the constant bank being replaced
  if (hipDeviceSynchronize() != hipSuccess) return cfail("ocfd_chem_set_mechanism: device error");
  if (hipMemcpyToSymbol(HIP_SYMBOL(cm), &h, sizeof(ChemMech)) != hipSuccess) return cfail("hipMemcpyToSymbol failed");
  CX.ready = true;
  return 0;
}

// Reverse-rate data of ReReac = 1 or 2, rev[j*5 .. j*5+4] per reaction (the
// line read_Reac reads after the Arrhenius lines, CHEM_reactions.f90:46-47).
int32_t ocfd_chem_set_reverse_rates(const double* rev) {
  if (!CX.ready) return cfail("ocfd_chem_set_reverse_rates: call ocfd_chem_set_mechanism first");
  if (!rev) return cfail("ocfd_chem_set_reverse_rates: null data");
  ChemMech& h = CX.h;
  for (int j = 0; j < h.nr; j++)
    for (int a = 0; a < 5; a++) h.rx[j].r[a] = rev[j * 5 + a];
  if (hipDeviceSynchronize() != hipSuccess) return cfail("ocfd_chem_set_reverse_rates: device error");
  if (hipMemcpyToSymbol(HIP_SYMBOL(cm), &h, sizeof(ChemMech)) != hipSuccess) return cfail("hipMemcpyToSymbol failed");
  CX.rev_ready = true;
  return 0;
}

// Chemical_time_advance over a batch of independent cells (OCFD_Time_Adv.f90:169-196
// calls chemical_timeAdv per cell); device pointers; nsub substeps of dt/nsub.
int32_t ocfd_chem_timeadv_batch(int64_t n, double* rho, double* E, const double* dt, int32_t mode, int32_t nsub) {
  if (!CX.ready) return cfail("ocfd_chem_timeadv_batch: call ocfd_chem_set_mechanism first");
  if (!CX.rev_ready) return cfail("ocfd_chem_timeadv_batch: ReReac 1/2 needs ocfd_chem_set_reverse_rates");
  if (n <= 0) return 0;
  if (nsub < 1) return cfail("ocfd_chem_timeadv_batch: nsub must be >= 1");
  dim3 g((unsigned)((n + CH_BLOCK - 1) / CH_BLOCK)), b(CH_BLOCK);
  switch (mode) {
    case 1: hipLaunchKernelGGL(chem_kernel([](auto st) { return &k_chem_fixed<1, decltype(st)>; }), g, b, 0, CX.stream, (long)n, rho, E, dt, nsub); break;
    case 2: hipLaunchKernelGGL(chem_kernel([](auto st) { return &k_chem_fixed<2, decltype(st)>; }), g, b, 0, CX.stream, (long)n, rho, E, dt, nsub); break;
    case 3: hipLaunchKernelGGL(chem_kernel([](auto st) { return &k_chem_fixed<3, decltype(st)>; }), g, b, 0, CX.stream, (long)n, rho, E, dt, nsub); break;
    case -1: hipLaunchKernelGGL(chem_kernel([](auto st) { return &k_chem_fixed<-1, decltype(st)>; }), g, b, 0, CX.stream, (long)n, rho, E, dt, nsub); break;
    default: return cfail("ocfd_chem_timeadv_batch: CHEM_TimeAdv must be 1, 2, 3 or -1");
  }
  if (hipGetLastError() != hipSuccess) return cfail("ocfd_chem_timeadv_batch: launch failed");
  return 0;
}

int32_t ocfd_chem_adaptive_batch(int64_t n, double* rho, double* E, const double* dt, double rtol_y, double y_floor,
                                 double rtol_t, int32_t max_sub, int32_t* nsub_out, int32_t scheduler) {
  return chem_adaptive_batch((long)n, rho, E, dt, rtol_y, y_floor, rtol_t, (int)max_sub, (int*)nsub_out,
                             (int)scheduler, CX.order != 0);
}

int32_t ocfd_chem_adaptive_batch_noalloc(int64_t n, double* rho, double* E, const double* dt, double rtol_y,
                                         double y_floor, double rtol_t, int32_t max_sub, int32_t* nsub_out) {
  const char* who = "ocfd_chem_adaptive_batch_noalloc";
  if (!CX.ready) return cfail(std::string(who) + ": call ocfd_chem_set_mechanism first");
  if (!CX.rev_ready) return cfail(std::string(who) + ": ReReac 1/2 needs ocfd_chem_set_reverse_rates");
  if (max_sub < 1 || !(rtol_y > 0.0) || !(y_floor >= 0.0) || !(rtol_t > 0.0))
    return cfail(std::string(who) + ": bad controller parameters");
  if (n < 0 || n > NA_MAX_CELLS)
    return cfail(std::string(who) + ": n must be 0 .. 2^20 (" + std::to_string(NA_MAX_CELLS) +
                 ", the capacity of its static workspace), got " + std::to_string((long long)n));
  unsigned char* base = nullptr;
  if (na_workspace(&base)) return 1;
  unsigned long long* counter = (unsigned long long*)base;
  unsigned long long* count = (unsigned long long*)(base + NA_COUNTERS);
  unsigned char* p = base + NA_COUNTERS + NA_COUNT;
  unsigned int* keys_in = (unsigned int*)p;
  unsigned int* keys_out = (unsigned int*)(p + NA_KEYS);
  int* idx_in = (int*)(p + 2 * NA_KEYS);
  int* idx_out = (int*)(p + 2 * NA_KEYS + NA_LIST);
  void* temp = p + 2 * NA_KEYS + 2 * NA_LIST;
  const ChemCtl ctl{rtol_y, y_floor, rtol_t, max_sub};
  // the previous call's counters are still there: clear them (a kernel)
  hipLaunchKernelGGL(k_chem_reset, dim3(1), dim3(64), 0, CX.stream, counter);
  if (n == 0) return hipGetLastError() == hipSuccess ? 0 : cfail(std::string(who) + ": launch failed");
  const int* list = nullptr;
  const unsigned long long* list_count = nullptr;
  if (n > 1) {
    // the longest-first order of ocfd_chem_adaptive_batch, on the workspace
    size_t need = 0;
    if (hipcub::DeviceRadixSort::SortPairsDescending(nullptr, need, (const unsigned int*)nullptr, (unsigned int*)nullptr,
                                                     (const int*)nullptr, (int*)nullptr, (int)n) != hipSuccess)
      return cfail(std::string(who) + ": radix sort query failed");
    if (need > NA_TEMP)
      return cfail(std::string(who) + ": the radix sort needs " + std::to_string(need) + " bytes of workspace, more than " +
                   std::to_string(NA_TEMP));
    hipLaunchKernelGGL(k_order_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, CX.stream, (long)n, rho, E, dt,
                       keys_in, idx_in, count);
    size_t tb = need;
    const hipError_t e = hipcub::DeviceRadixSort::SortPairsDescending(temp, tb, keys_in, keys_out, idx_in, idx_out,
                                                                      (int)n, 0, 32, CX.stream);
    if (e != hipSuccess) return cfail(std::string(who) + ": radix sort failed: " + hipGetErrorString(e));
    list = idx_out;
    list_count = count;
  }
  return launch_adaptive((long)n, rho, E, dt, ctl, (int*)nsub_out, 1, list, list_count, false, counter);
}

int32_t ocfd_chem_surrogate_set(const double* cfg, int32_t count) {
  if (!CX.ready) return cfail("ocfd_chem_surrogate_set: call ocfd_chem_set_mechanism first");
  if (count != (int32_t)(sizeof(SurrCfg) / sizeof(double)))
    return cfail("ocfd_chem_surrogate_set: expected " + std::to_string(sizeof(SurrCfg) / sizeof(double)) + " values");
  SurrCfg h;
  std::memcpy(&h, cfg, sizeof(SurrCfg));
  if (hipStreamSynchronize(CX.stream) != hipSuccess ||
      hipMemcpyToSymbol(HIP_SYMBOL(scfg), &h, sizeof(SurrCfg)) != hipSuccess)
    return cfail("ocfd_chem_surrogate_set: copy failed");
  CX.surr_ready = true;
  return 0;
}

int32_t ocfd_chem_surrogate_batch(int64_t n, double* rho, double* E, const double* dt, int32_t fallback,
                                  double rtol_y, double y_floor, double rtol_t, int32_t max_sub, int32_t* flag_out) {
  return chem_surrogate_batch((long)n, rho, E, dt, fallback != 0, rtol_y, y_floor, rtol_t, (int)max_sub,
                              (int*)flag_out, CX.order != 0);
}

// Autotuner of the surrogate network kernel: every tile shape runs `reps`
// times on scratch copies of the batch (the inputs are not modified), timed
// with HIP events on the chemistry stream; the fastest is kept.  Results are
// bit-identical for every shape.  ms_out (may be NULL) receives the mean ms
// per launch of each shape (SURR_VARIANTS floats).  Synchronises.
int32_t ocfd_chem_surrogate_autotune(int64_t n, const double* rho, const double* E, const double* dt, int32_t reps,
                                     float* ms_out) {
  if (reps < 1 || n <= 0) return cfail("ocfd_chem_surrogate_autotune: need reps >= 1 and cells");
  if (surr_prepare((long)n, "ocfd_chem_surrogate_autotune")) return 1;
  double *r2 = nullptr, *e2 = nullptr;
  if (hipMalloc(&r2, sizeof(double) * (size_t)n * CH_NS) != hipSuccess ||
      hipMalloc(&e2, sizeof(double) * (size_t)n) != hipSuccess) {
    if (r2) hipFree(r2);
    return cfail("ocfd_chem_surrogate_autotune: out of device memory");
  }
  hipEvent_t a, b;
  hipEventCreate(&a);
  hipEventCreate(&b);
  int best = 0;
  for (int v = 0; v < SURR_VARIANTS; v++) {
    float tot = 0.f;
    for (int r = 0; r <= reps; r++) {  // the first run warms up and is not counted
      hipMemcpyAsync(r2, rho, sizeof(double) * (size_t)n * CH_NS, hipMemcpyDeviceToDevice, CX.stream);
      hipMemcpyAsync(e2, E, sizeof(double) * (size_t)n, hipMemcpyDeviceToDevice, CX.stream);
      hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, CX.stream, CX.counter, 8);
      hipEventRecord(a, CX.stream);
      launch_surrogate(v, (long)n, r2, e2, dt, nullptr);
      hipEventRecord(b, CX.stream);
      hipEventSynchronize(b);
      float ms = 0.f;
      hipEventElapsedTime(&ms, a, b);
      if (r > 0) tot += ms;
    }
    CX.surr_tune_ms[v] = tot / reps;
    if (CX.surr_tune_ms[v] < CX.surr_tune_ms[best]) best = v;
  }
  hipEventDestroy(a);
  hipEventDestroy(b);
  hipFree(r2);
  hipFree(e2);
  CX.surr_variant = best;
  if (ms_out)
    for (int v = 0; v < SURR_VARIANTS; v++) ms_out[v] = CX.surr_tune_ms[v];
  return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_surrogate_autotune: launch failed");
}

// the tile shape in use (and force one with variant >= 0)
int32_t ocfd_chem_surrogate_tile(int32_t variant, int32_t* rows, int32_t* waves) {
  if (variant >= SURR_VARIANTS) return cfail("ocfd_chem_surrogate_tile: unknown variant");
  if (variant >= 0) CX.surr_variant = variant;
  const int v = CX.surr_variant;
  const int R[SURR_VARIANTS] = {SurrTile<0>::ROWS, SurrTile<1>::ROWS, SurrTile<2>::ROWS, SurrTile<3>::ROWS};
  const int W[SURR_VARIANTS] = {SurrTile<0>::NW, SurrTile<1>::NW, SurrTile<2>::NW, SurrTile<3>::NW};
  if (rows) *rows = R[v];
  if (waves) *waves = W[v];
  return v;
}

// T [n] (mode 0), raw features [n][12] f64 (mode 1) or normalised surrogate
// inputs [n][12] f32 (mode 2) of a batch; device pointers
int32_t ocfd_chem_cell_features(int64_t n, const double* rho, const double* E, const double* dt, int32_t mode,
                                void* out) {
  if (!CX.ready) return cfail("ocfd_chem_cell_features: call ocfd_chem_set_mechanism first");
  if (mode < 0 || mode > 2) return cfail("ocfd_chem_cell_features: mode 0, 1 or 2");
  if (mode == 2 && !CX.surr_ready) return cfail("ocfd_chem_cell_features: surrogate normalisation not set");
  if (mode > 0 && !dt) return cfail("ocfd_chem_cell_features: dt required");
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_cell_features, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, CX.stream, (long)n, rho, E, dt,
                     (int)mode, out);
  return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_cell_features: launch failed");
}

int32_t ocfd_chem_surrogate_targets(int64_t n, const double* rho0, const double* rho1, float* y) {
  if (!CX.ready || !CX.surr_ready) return cfail("ocfd_chem_surrogate_targets: surrogate normalisation not set");
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_surr_targets, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, CX.stream, (long)n, rho0, rho1, y);
  return hipGetLastError() == hipSuccess ? 0 : cfail("ocfd_chem_surrogate_targets: launch failed");
}

int64_t ocfd_chem_surrogate_fallbacks(void) {
  if (!CX.ready) {
    cfail("ocfd_chem_surrogate_fallbacks: call ocfd_chem_set_mechanism first");
    return -1;
  }
  unsigned long long v = 0;
  if (hipMemcpyAsync(&v, CX.counter + 2, sizeof(v), hipMemcpyDeviceToHost, CX.stream) != hipSuccess ||
      hipStreamSynchronize(CX.stream) != hipSuccess) {
    cfail("ocfd_chem_surrogate_fallbacks: copy failed");
    return -1;
  }
  return (int64_t)v;
}

int32_t ocfd_chem_synchronize(void) {
  if (!CX.stream) return 0;
  if (hipStreamSynchronize(CX.stream) != hipSuccess) return cfail("ocfd_chem_synchronize: stream error");
  return 0;
}

void* ocfd_chem_stream(void) { return (void*)CX.stream; }

int32_t ocfd_chem_set_option(int32_t key, int32_t value) {
  switch (key) {
    case 1:
      if (value < 1) return cfail("ocfd_chem_set_option: the attempt budget must be >= 1");
      CX.coop_budget = value;
      return 0;
    case 2:
      if (value < 1 || value > 2) return cfail("ocfd_chem_set_option: fallback scheduler 1 or 2");
      CX.fallback_scheduler = value;
      return 0;
    case 3:
      if (value < 0) return cfail("ocfd_chem_set_option: the direct cooperative list size must be >= 0");
      CX.coop_direct_max = value;
      return 0;
    case 4:
      if (value < 0 || value > 1) return cfail("ocfd_chem_set_option: cell order 0 or 1");
      CX.order = value;
      return 0;
  }
  return cfail("ocfd_chem_set_option: unknown option");
}

int32_t ocfd_chem_counters(int64_t* out, int32_t count) {
  if (!CX.ready) return cfail("ocfd_chem_counters: call ocfd_chem_set_mechanism first");
  if (count < 0 || count > 8) return cfail("ocfd_chem_counters: at most 8 counters");
  unsigned long long v[8] = {};
  if (hipMemcpyAsync(v, CX.counter, sizeof(v), hipMemcpyDeviceToHost, CX.stream) != hipSuccess ||
      hipStreamSynchronize(CX.stream) != hipSuccess)
    return cfail("ocfd_chem_counters: copy failed");
  for (int i = 0; i < count; i++) out[i] = (int64_t)v[i];
  return 0;
}

int64_t ocfd_chem_unfinished(void) {
  if (!CX.ready) {
    cfail("ocfd_chem_unfinished: call ocfd_chem_set_mechanism first");
    return -1;
  }
  unsigned long long v = 0;
  if (hipMemcpyAsync(&v, CX.counter + 1, sizeof(v), hipMemcpyDeviceToHost, CX.stream) != hipSuccess ||
      hipStreamSynchronize(CX.stream) != hipSuccess) {
    cfail("ocfd_chem_unfinished: copy failed");
    return -1;
  }
  return (int64_t)v;
}

int32_t ocfd_chem_set_stream(void* stream) {
  if (!CX.ready) return cfail("ocfd_chem_set_stream: call ocfd_chem_set_mechanism first");
  CX.stream = (hipStream_t)stream;
  return 0;
}

}  // extern "C"
