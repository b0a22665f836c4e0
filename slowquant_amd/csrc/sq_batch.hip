// Batched energy + adjoint gradient for many independent UPS instances of
// uneven active spaces in ONE persistent launch (the reference's batching
// primitive is the _SA family, operator_state_algebra.py:282-410,633-781,
// which needs equal dimensions; here every instance has its own space,
// Hamiltonian, gate list and theta).
//
// One workgroup owns a list of instances (longest-processing-time order,
// assigned on the host, no atomics).  Per instance, inside the workgroup:
//   psi = HF;  forward rotations;  D build;  G = A.D with FP64 MFMA;
//   sigma gather + energy;  reverse sweep with fused <lambda|T_i psi> dots.
// psi and lambda live in LDS where all of the launch's instances fit beside A,
// else, like G, in a per-workgroup slot of global scratch (L2-resident for the
// small spaces), so instances never interact.
// The launch can be captured in a hipGraph and replayed.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <numeric>
#include <string>

#include "sq_internal.h"

namespace sq {

constexpr int kBT = 512;    // threads per batch workgroup (8 waves)
constexpr int kBW = kBT / 64;
constexpr int kBRot = 128;  // rotations whose records and angles are staged in LDS at a time
constexpr size_t kBatchLds = 160 * 1024 - kBRot * 64 - 1024;  // dynamic LDS of a workgroup
constexpr int kBatchMT = 5;  // row tiles of the sigma GEMM (kpad <= 80: up to 12 orbitals)

// k -> whether packed pair k = p(p+1)/2 + q is diagonal (p == q), k < 91
__constant__ uint8_t c_bdiag[91];

struct BatchSpace {
  int n, nsa, nsb, npair, K4, kpad;
  const uint32_t* astr;
  const uint32_t* bstr;
  const int32_t* arank;
  const int32_t* brank;
  const int32_t* aexc;  // packed, k-major
  const int32_t* bexc;
};

struct BatchInstance {
  int space;        // index into spaces
  int gate0, ngate; // rotation records [gate0, gate0 + ngate)
  int theta0;       // offset into theta array (one theta per layout gate)
  int nparam;
  int A_off;        // offset into A storage (K4 * kpad doubles)
  double e_core;
  int out0;         // offset of the gradient in the output array
};

// One rotation half: string G = sgn * Ga * Gb with distinct indices; the
// layout gate's theta index and angle scale.
// A rotation string touches exactly the (alpha, beta) pairs where both spin
// parts apply: precomputed lists of (string, image | parity << 31) per spin
// (shared between rotations with the same spin part on the same space); a
// spin part without operators acts on every string (list offset -1).
struct BatchRot {
  double sgn, scale;
  int theta_idx;    // index relative to the instance's theta0
  int grad_idx;     // same, for the gradient accumulation
  int aoff, na;     // alpha list [aoff, aoff + na), or aoff = -1: every alpha string
  int boff, nb;     // beta list, likewise
};

struct BatchDev {
  const BatchSpace* spaces;
  const BatchInstance* inst;
  const BatchRot* rots;
  const int2* lists;       // (string, image | parity << 31) entries of the spin-part lists
  const double* theta;
  const double* A;
  const int32_t* wg_list;  // concatenated instance lists per workgroup
  const int32_t* wg_off;   // [nwg + 1]
  double* scratch;         // per-workgroup slots
  int64_t slot_doubles;
  int64_t dmax;
  int64_t vec0;            // psi | lambda in the dynamic LDS from here (in doubles)
  double* energy;          // [ninst]
  double* grad;            // concatenated gradients
  const double* const* psi0;  // [ninst] start states (engine convention), nullptr: HF determinant
};

// Visit every (alpha row, beta column) of a space with 32-bit index math:
// a block-wide 2-D walk, rows_per_step rows of min(nsb, blockDim) columns.
template <class F>
__device__ __forceinline__ void for_each_det(int nsa, int nsb, F&& f) {
  const int cols = nsb < (int)blockDim.x ? nsb : (int)blockDim.x;
  const int rps = (int)blockDim.x / cols;
  const int r0 = (int)threadIdx.x / cols, c0 = (int)threadIdx.x - r0 * cols;
  if (r0 >= rps) return;
  for (int ia = r0; ia < nsa; ia += rps)
    for (int ib = c0; ib < nsb; ib += cols) f(ia, ib, ia * nsb + ib);
}

__device__ __forceinline__ int2 list_entry(const int2* lists, int off, int i) {
  return off < 0 ? int2{i, i} : lists[off + i];
}

// One rotation half of the forward (REV = false) or reverse sweep over its
// spin-part lists, U pairs of determinants per thread in flight: the loads of
// all U pairs are issued before any of them is updated (the pairs of one
// rotation are disjoint).  Returns this thread's part of
// scale * <lam|T psi> (reverse sweep).
template <int U, bool REV>
__device__ __forceinline__ double rotate_lists(const int2* __restrict__ lists, const BatchRot& R, int nsb, double c,
                                               double s, bool apply, double* psi, double* lam) {
  const int na = R.na, nb = R.nb;
  const int cols = nb < (int)blockDim.x ? (nb > 0 ? nb : 1) : (int)blockDim.x;
  const int rps = (int)blockDim.x / cols;
  const int r0 = (int)threadIdx.x / cols, c0 = (int)threadIdx.x - r0 * cols;
  double dot = 0.0;
  if (r0 >= rps) return 0.0;
  for (int bi = c0; bi < nb; bi += cols) {
    const int2 Bq = list_entry(lists, R.boff, bi);
    for (int a0 = r0; a0 < na; a0 += rps * U) {
      int x[U], J[U];
      double sg[U], pd[U], pj[U], ld[U], lj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int ai = a0 + u * rps;
        x[u] = -1;
        if (ai < na) {
          const int2 A = list_entry(lists, R.aoff, ai);
          x[u] = A.x * nsb + Bq.x;
          J[u] = (A.y & 0x7fffffff) * nsb + (Bq.y & 0x7fffffff);
          sg[u] = (((uint32_t)(A.y ^ Bq.y) >> 31) ? -1.0 : 1.0) * R.sgn;
          pd[u] = psi[x[u]];
          pj[u] = psi[J[u]];
          if (REV) {
            ld[u] = lam[x[u]];
            lj[u] = lam[J[u]];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (x[u] < 0) continue;
        if (REV) dot += R.scale * sg[u] * (lj[u] * pd[u] - ld[u] * pj[u]);
        if (apply) {
          psi[x[u]] = c * pd[u] - sg[u] * s * pj[u];
          psi[J[u]] = sg[u] * s * pd[u] + c * pj[u];
          if (REV) {
            lam[x[u]] = c * ld[u] - sg[u] * s * lj[u];
            lam[J[u]] = sg[u] * s * ld[u] + c * lj[u];
          }
        }
      }
    }
  }
  return dot;
}

// U: rotation pairs per thread in flight; CT: 16-column tiles per wave in the
// sigma GEMM (sharing each LDS read of A).  Both are picked by the autotuner.
// LDS: psi and lambda at vec0 of the dynamic LDS.  The sweeps are a chain of one
// rotation after the other; what it waits for is kept short: records and angles
// of a chunk of rotations are staged at once (a thread-wide sincos per rotation
// before), one barrier per rotation (four in the reverse sweep before), psi and
// lambda in LDS.  One 3-layer evaluation of (7: 4,3) 419 -> 238 us, of (8e,8o)
// 994 -> 608; 38 instances of 4 to 7 orbitals 449 -> 270.
template <int U, int CT, bool LDS>
__global__ __launch_bounds__(kBT) void k_batch(BatchDev B) {
  __shared__ double red[2][kBW];
  __shared__ BatchRot recs[kBRot];
  __shared__ double2 cs[kBRot];
  extern __shared__ double sA[];
  double* slot = B.scratch + (size_t)blockIdx.x * B.slot_doubles;
  double* psi = LDS ? sA + B.vec0 : slot;
  double* lam = psi + B.dmax;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int li = B.wg_off[blockIdx.x]; li < B.wg_off[blockIdx.x + 1]; ++li) {
    const BatchInstance I = B.inst[B.wg_list[li]];
    const BatchSpace S = B.spaces[I.space];
    const int nsb = S.nsb;
    const int dim = S.nsa * nsb;  // < 2^30, checked at creation
    double* G = LDS ? slot : slot + 2 * B.dmax;
    const double* th = B.theta + I.theta0;
    const double* start = B.psi0[B.wg_list[li]];
    if (start) {
      for (int64_t x = threadIdx.x; x < dim; x += blockDim.x) psi[x] = start[x];
    } else {
      // psi = HF determinant (alpha string 0, beta string 0) in the engine's
      // sign convention: (-1)^{sum_{p in alpha} #{q in beta : q < p}}.
      for (int64_t x = threadIdx.x; x < dim; x += blockDim.x) psi[x] = 0.0;
      __syncthreads();
      if (threadIdx.x == 0) {
        uint32_t a = S.astr[0], b = S.bstr[0];
        int par = 0;
        for (uint32_t aa = a; aa; aa &= aa - 1) par += __popc(b & ((1u << (__ffs(aa) - 1)) - 1u));
        psi[0] = (par & 1) ? -1.0 : 1.0;
      }
    }
    __syncthreads();
    // records and angles of rotations [r0, r0 + n); c = 1, s = 0 where theta
    // vanishes
    auto stage = [&](int r0, int n, bool rev) {
      __syncthreads();
      for (int i = threadIdx.x; i < n; i += kBT) {
        const BatchRot R = B.rots[I.gate0 + r0 + i];
        const double t0 = th[R.theta_idx];
        double s = 0.0, c = 1.0;
        if (rev ? !(fabs(t0) < 1e-28) : fabs(t0) >= 1e-28) sincos(R.scale * t0, &s, &c);
        recs[i] = R;
        cs[i] = double2{c, rev ? -s : s};
      }
      __syncthreads();
    };
    // forward sweep
    for (int r0 = 0; r0 < I.ngate; r0 += kBRot) {
      const int n = min(kBRot, I.ngate - r0);
      stage(r0, n, false);
      for (int r = 0; r < n; ++r) {
        const double2 x = cs[r];
        if (x.x != 1.0 || x.y != 0.0)
          (void)rotate_lists<U, false>(B.lists, recs[r], nsb, x.x, x.y, true, psi, nullptr);
        __syncthreads();
      }
    }
    // stage A (K4 x kpad, transposed coefficient matrix) in LDS
    const double* Ag = B.A + I.A_off;
    for (int i = threadIdx.x; i < S.K4 * S.kpad; i += blockDim.x) sA[i] = Ag[i];
    __syncthreads();
    // G = A . D with v_mfma_f64_16x16x4f64, the B operand D[k][c] = (E+_k psi)[c]
    // (row npair: psi) generated in registers: each wave walks 16-column tiles
    // and keeps all kpad/16 row tiles in flight, so D is never stored.
    {
      typedef double double4_t __attribute__((ext_vector_type(4)));
      const int kq = lane >> 4, li = lane & 15;
      const int nwaves = blockDim.x >> 6;
      const int MT = S.kpad / 16;
      for (int c0 = wave * 16 * CT; c0 < dim; c0 += nwaves * 16 * CT) {
        int ccol[CT], ia[CT], ib[CT];
        bool ok[CT];
        double pc[CT];
#pragma unroll
        for (int u = 0; u < CT; ++u) {
          ccol[u] = c0 + u * 16 + li;
          ok[u] = ccol[u] < dim;
          ia[u] = ok[u] ? ccol[u] / nsb : 0;
          ib[u] = ok[u] ? ccol[u] - ia[u] * nsb : 0;
          pc[u] = ok[u] ? psi[ccol[u]] : 0.0;
        }
        auto dval = [&](int u, int k) -> double {
          if (!ok[u] || k > S.npair) return 0.0;
          if (k == S.npair) return pc[u];
          const int32_t ea = S.aexc[k * S.nsa + ia[u]];
          const int32_t eb = S.bexc[k * nsb + ib[u]];
          if (c_bdiag[k]) return (double)(ea + eb) * pc[u];
          double v = 0.0;
          if (ea) v += (ea > 0 ? 1.0 : -1.0) * psi[(abs(ea) - 1) * nsb + ib[u]];
          if (eb) v += (eb > 0 ? 1.0 : -1.0) * psi[ia[u] * nsb + abs(eb) - 1];
          return v;
        };
        double4_t acc[CT][kBatchMT];
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int t = 0; t < kBatchMT; ++t) acc[u][t] = double4_t{0.0, 0.0, 0.0, 0.0};
        double bnext[CT];
#pragma unroll
        for (int u = 0; u < CT; ++u) bnext[u] = dval(u, kq);
        for (int k4 = 0; k4 < S.K4; k4 += 4) {
          double bv[CT];
#pragma unroll
          for (int u = 0; u < CT; ++u) {
            bv[u] = bnext[u];
            if (k4 + 4 < S.K4) bnext[u] = dval(u, k4 + 4 + kq);
          }
          const double* arow = sA + (k4 + kq) * S.kpad + li;
#pragma unroll
          for (int t = 0; t < kBatchMT; ++t) {
            if (t < MT) {
              const double a = arow[t * 16];
#pragma unroll
              for (int u = 0; u < CT; ++u) acc[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bv[u], acc[u][t], 0, 0, 0);
            }
          }
        }
#pragma unroll
        for (int u = 0; u < CT; ++u) {
          if (!ok[u]) continue;
#pragma unroll
          for (int t = 0; t < kBatchMT; ++t) {
            if (t >= MT) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int m = t * 16 + kq + 4 * r;
              if (m < S.npair) G[(size_t)m * dim + ccol[u]] = acc[u][t][r];
            }
          }
        }
      }
    }
    __syncthreads();
    // sigma gather into lam, energy
    double e = 0.0;
    for_each_det(S.nsa, nsb, [&](int ia, int ib, int x) {
      double v = I.e_core * psi[x];
      int k = 0;
      for (int p = 0; p < S.n; ++p) {
        for (int q = 0; q <= p; ++q, ++k) {
          const double* Gk = G + (size_t)k * dim;
          const int32_t ea = S.aexc[(size_t)k * S.nsa + ia];
          const int32_t eb = S.bexc[(size_t)k * nsb + ib];
          if (p == q) {
            v += (double)(ea + eb) * Gk[x];
          } else {
            if (ea) v += (ea > 0 ? 1.0 : -1.0) * Gk[(size_t)(abs(ea) - 1) * nsb + ib];
            if (eb) v += (eb > 0 ? 1.0 : -1.0) * Gk[(size_t)ia * nsb + abs(eb) - 1];
          }
        }
      }
      lam[x] = v;
      e += v * psi[x];
    });
    e = wave_sum63(e);
    if (lane == 63) red[0][wave] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
      e = 0.0;
      for (int w = 0; w < kBW; ++w) e += red[0][w];
      B.energy[B.wg_list[li]] = e;
    }
    // reverse sweep with gradient dots; the last wave adds the wave sums of one
    // rotation to its gate's gradient during the next
    for (int p = threadIdx.x; p < I.nparam; p += blockDim.x) B.grad[I.out0 + p] = 0.0;
    int par = 0, done = -1;  // grad index of the previous rotation
    double sum = 0.0;
    auto finish = [&](int now) {
      if (wave != kBW - 1 || done < 0) return;
      sum += row16_sum(lane < kBW ? red[par ^ 1][lane] : 0.0);
      if (now != done) {
        if (lane == 15) B.grad[I.out0 + done] = 2.0 * sum;
        sum = 0.0;
      }
    };
    for (int r1 = I.ngate; r1 > 0; r1 -= kBRot) {
      const int r0 = max(0, r1 - kBRot);
      stage(r0, r1 - r0, true);
      for (int r = r1 - r0 - 1; r >= 0; --r) {
        const double2 x = cs[r];
        const double dot = wave_sum63(
            rotate_lists<U, true>(B.lists, recs[r], nsb, x.x, x.y, x.x != 1.0 || x.y != 0.0, psi, lam));
        const int now = recs[r].grad_idx;
        finish(now);
        if (lane == 63) red[par][wave] = dot;
        done = now;
        par ^= 1;
        __syncthreads();
      }
    }
    finish(-1);
    __syncthreads();
  }
}

// Large instances of one (space, gate layout) run together through the
// single-instance kernels with an instance grid dimension (window stages, row
// sigma, gradient): one persistent workgroup per instance would leave them
// bound by one CU each.  Per-instance buffers are contiguous at fixed
// strides.
struct BatchGroup {
  const Space* space = nullptr;
  const Program* prog = nullptr;
  std::shared_ptr<const TilePlan> tiles;  // the program's plan and the space's shape when the batch was made
  SigmaShape sigma;
  int n = 0, ng = 0;
  int64_t dim = 0, A_stride = 0, Ma_stride = 0, Mb_stride = 0, mats_stride = 0, tpart_stride = 0, spart_stride = 0;
  double hf = 1.0;  // the HF determinant's amplitude in the engine's sign convention
  int plan_gen = 0;  // the program's tile-plan generation (check_group)
  int32_t *d_inst = nullptr, *d_theta0 = nullptr, *d_out0 = nullptr;  // per member
  double *theta = nullptr, *A = nullptr, *Ma = nullptr, *Mb = nullptr, *psi = nullptr, *lam = nullptr, *mats = nullptr,
         *tpart = nullptr, *spart = nullptr, *grad = nullptr;
};

// theta_g[m][i] = theta_all[theta0[m] + i] (member m = blockIdx.y)
__global__ void k_group_theta(const double* __restrict__ theta_all, const int32_t* __restrict__ theta0, int ng,
                              double* __restrict__ theta_g) {
  const int m = blockIdx.y;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ng; i += gridDim.x * blockDim.x)
    theta_g[(size_t)m * ng + i] = theta_all[theta0[m] + i];
}

// psi_g[m] = the member's start state, or the HF determinant (amplitude hf at 0)
__global__ void k_group_init(const double* const* __restrict__ psi0, const int32_t* __restrict__ inst, int64_t dim,
                             double hf, double* __restrict__ psi) {
  const int m = blockIdx.y;
  const double* src = psi0[inst[m]];
  double* dst = psi + (size_t)m * dim;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < dim; i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src ? src[i] : (i == 0 ? hf : 0.0);
}

// energy[inst[m]] = sum of member m's sigma energy partials (fixed order);
// grad[out0[m] + g] = grad_g[m][g]
__global__ void k_group_out(const double* __restrict__ spart, int64_t nblk, const double* __restrict__ grad_g, int ng,
                            const int32_t* __restrict__ inst, const int32_t* __restrict__ out0,
                            double* __restrict__ energy, double* __restrict__ grad) {
  __shared__ double red[4];
  const int m = blockIdx.x;
  const double* p = spart + (size_t)m * nblk;
  double v = 0.0;
  for (int64_t i = threadIdx.x; i < nblk; i += blockDim.x) v += p[i];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) energy[inst[m]] = red[0] + red[1] + red[2] + red[3];
  for (int g = threadIdx.x; g < ng; g += blockDim.x) grad[out0[m] + g] = grad_g[(size_t)m * ng + g];
}

// Instances this large go to groups (the persistent launch keeps the rest):
// one workgroup runs a 3-layer (8e,8o) evaluation in 590 us, the large kernels
// in 92, but a 2-layer (6e,6o) one takes 100, less than the launches of another
// group.  Groups from 16384, 4096 and 1200 determinants: 256 instances of 4 to
// 10 orbitals 1158, 1136, 1145 us; 100 of 5 to 8 orbitals 801, 365, 424; 12 of 6
// to 9 orbitals 3030, 375, 377; 38 of 4 to 7 orbitals 272, 271, 244.
constexpr int64_t kGroupMinDim = 4096;

// From here on instances are always grouped (one workgroup needs 3 ms and more
// for an evaluation), and the batch's user keeps their programs (check_group).
constexpr int64_t kKeepMinDim = 16384;

// Streams the groups run on: one group's short kernels and the ends of its long
// ones leave CUs idle that another group's fill (256 instances as above on 1,
// 3 and 4: 1549, 1329, 1206 us; there are four hardware queues).
constexpr int kGroupLanes = 4;
constexpr int kBatchShapes = 6;  // of the persistent launch: 1, 2 or 4 rotation pairs, 1 or 2 column tiles

struct Batch {
  std::vector<BatchInstance> inst;
  int nwg = 0;
  int64_t dmax = 0, slot = 0, ngrad = 0;
  double bytes = 0.0, flops = 0.0;  // algorithmic totals of one launch
  size_t lds = 0;
  bool vec_lds = false;  // psi and lambda of the persistent launch in LDS
  std::vector<void*> allocs;
  BatchDev dev{};
  double* d_theta = nullptr;
  const double** d_psi0 = nullptr;  // start-state pointer table [inst]
  std::vector<BatchGroup> groups;   // instances run through the tile and row-sigma kernels
  std::vector<std::pair<int, int>> group_members;  // (group, instance), in instance order
  // a captured launch per kernel shape (kernel_shape), kept until the batch goes
  hipGraph_t graph[kBatchShapes] = {};
  hipGraphExec_t exec[kBatchShapes] = {};
  std::vector<int32_t> grad_off;
  double* host_out = nullptr;  // pinned: energies | gradients on their way to the caller
  mutable std::mutex host_mu;
  hipStream_t side = nullptr;  // the persistent launch beside the groups (default priority, as the lanes)
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  hipStream_t lane[kGroupLanes] = {};  // [0] unused: the caller's stream
  hipEvent_t ev_lane[kGroupLanes] = {};
  int rot_pairs = 2;    // rotation pairs per thread in flight (1, 2, 4)
  int gemm_tiles = 1;   // sigma GEMM column tiles per wave (1, 2)
  // 0 to kBatchShapes - 1; one when the persistent launch holds no instance
  int kernel_shape() const {
    return nwg == 0 ? 0 : (rot_pairs == 1 ? 0 : rot_pairs == 2 ? 1 : 2) * 2 + gemm_tiles - 1;
  }
  ~Batch() {
    for (hipGraphExec_t e : exec)
      if (e) (void)hipGraphExecDestroy(e);
    for (hipGraph_t g : graph)
      if (g) (void)hipGraphDestroy(g);
    if (host_out) (void)hipHostFree(host_out);
    if (side) (void)hipStreamDestroy(side);
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    if (ev_join) (void)hipEventDestroy(ev_join);
    for (hipStream_t l : lane)
      if (l) (void)hipStreamDestroy(l);
    for (hipEvent_t e : ev_lane)
      if (e) (void)hipEventDestroy(e);
    for (void* p : allocs) (void)hipFree(p);
  }
};

template <class T>
static T* bupload(Batch& B, const std::vector<T>& v) {
  T* d = nullptr;
  SQ_HIP(hipMalloc(&d, sizeof(T) * std::max<size_t>(v.size(), 1)));
  if (!v.empty()) SQ_HIP(hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
  B.allocs.push_back(d);
  return d;
}

// Bytes of a program's gate layout (kinds, pairs, scales and generator
// terms): equal keys on one space give identical tile plans.
static std::string layout_key(const Program& p) {
  std::string k;
  auto put = [&](const void* x, size_t n) { k.append(reinterpret_cast<const char*>(x), n); };
  for (size_t g = 0; g < p.gates.size(); ++g) {
    const GateDev& gd = p.gates[g];
    put(&gd.kind, sizeof gd.kind);
    put(&gd.scale, sizeof gd.scale);
    const int32_t pp = g < p.pair_p.size() ? p.pair_p[g] : -1;
    put(&pp, sizeof pp);
    const int32_t nt = gd.term_end - gd.term_begin;
    put(&nt, sizeof nt);
    for (int t = gd.term_begin; t < gd.term_end; ++t) {
      const Term& T = p.terms[t];
      put(&T.coef, sizeof T.coef);
      for (const SpinOps* o : {&T.a, &T.b}) {
        put(&o->n, sizeof o->n);
        put(o->orb, (size_t)o->n);
        put(o->cre, (size_t)o->n);
      }
    }
  }
  return k;
}

// About how long a group takes on its stream (us): its chain of launches and its
// work (29 instances of (10e,10o) with three layers: 800).
static double group_us(int n, const Space& s, int ng) {
  return 100.0 + 1.3e-6 * (double)n * (double)s.dim * (ng + 4.0 * s.npair);
}

static size_t a_bytes(const Space& s) {
  return sizeof(double) * (size_t)((s.npair + 1 + 3) / 4 * 4) * (size_t)((s.npair + 1 + 15) / 16 * 16);
}

// Work of an instance of the persistent launch, in amplitudes touched.
static int64_t persistent_cost(const Space& s, int rotations) {
  const int K4 = (s.npair + 1 + 3) / 4 * 4;
  return s.dim * (int64_t)(2 * rotations + 4 + 2 * s.npair + (s.npair * K4) / 8);
}

// About how long one workgroup takes for it (us, vectors in LDS or not): (7: 4,3)
// with three layers 238, (8e,8o) 608, (9: 5,4) in scratch 3030.
static double persistent_us(const Space& s, const Program& p, bool vec_lds) {
  int rotations = 0;
  for (const GateDev& g : p.gates) rotations += g.kind == GC_SA_SINGLE ? 2 : 1;
  return (vec_lds ? 1.0 : 1.6) * (1.4 * rotations + 2e-4 * (double)persistent_cost(s, rotations));
}

// Instances of one space and gate layout that can run as a group.
struct GroupCand {
  std::shared_ptr<const TilePlan> tiles;
  std::vector<int> mem;
  bool keep = true;
};

// Many groups of few instances below kKeepMinDim are chains of launches that
// wait for the four streams, while one persistent launch holds 256 of them: the
// ones with the fewest members go there (to 12 orbitals) as far as that takes
// less by a fifth (by the times above).  Sixty instances of (8e,8o) with as many layouts: groups
// 2550 us, persistent launch 765; 256 instances of 4 to 10 orbitals keep their
// groups.
static void drop_small_groups(std::vector<GroupCand>& cands, const std::vector<int>& rest,
                              const sq_space* const* spaces, const sq_program* const* programs, int n_workgroups) {
  auto space = [&](int i) -> const Space& { return spaces[i]->s; };
  auto program = [&](int i) -> const Program& { return programs[i]->p; };
  double tg = 0.0;
  std::vector<int> order;
  auto time = [&](const GroupCand& c) {  // many chains in a graph: 50 us more each
    return (50.0 + group_us((int)c.mem.size(), space(c.mem[0]), (int)program(c.mem[0]).gates.size())) / kGroupLanes;
  };
  for (size_t i = 0; i < cands.size(); ++i) {
    tg += time(cands[i]);
    if (space(cands[i].mem[0]).dim < kKeepMinDim && space(cands[i].mem[0]).n <= 12) order.push_back((int)i);
  }
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return cands[a].mem.size() < cands[b].mem.size(); });
  // the persistent launch with the rest and the first k candidates of the order
  size_t lds = 0, count = 0;
  int64_t dmax = 0;
  double longest[2] = {0.0, 0.0}, total[2] = {0.0, 0.0};  // scratch, LDS
  auto add = [&](int i) {
    lds = std::max(lds, a_bytes(space(i)));
    dmax = std::max(dmax, space(i).dim);
    ++count;
    for (int l = 0; l < 2; ++l) {
      const double us = persistent_us(space(i), program(i), l == 1);
      longest[l] = std::max(longest[l], us);
      total[l] += us;
    }
  };
  auto persistent = [&] {
    if (count == 0) return 0.0;
    const int l = lds + 2 * sizeof(double) * (size_t)dmax <= kBatchLds ? 1 : 0;
    return std::max(longest[l], total[l] / (double)std::min<size_t>(n_workgroups > 0 ? n_workgroups : 256, count));
  };
  for (int i : rest) add(i);
  auto both = [&] {  // side by side, in each other's way
    const double tp = persistent();
    return std::max(tg, tp) + 0.5 * std::min(tg, tp);
  };
  double best = 0.8 * both();
  size_t drop = 0;
  for (size_t k = 0; k < order.size(); ++k) {
    const GroupCand& c = cands[order[k]];
    tg -= time(c);
    for (int i : c.mem) add(i);
    const double t = both();
    if (t < best) best = t, drop = k + 1;
  }
  for (size_t k = 0; k < drop; ++k) cands[order[k]].keep = false;
}

template <class T>
static T* balloc(Batch& B, size_t n) {
  T* d = nullptr;
  SQ_HIP(hipMalloc(&d, sizeof(T) * std::max<size_t>(n, 1)));
  B.allocs.push_back(d);
  return d;
}

// Buffers of every group: members' theta offsets, output offsets, their
// Hamiltonians copied into contiguous A and Ma arrays, and the work vectors.
static void build_groups(Batch& B, const sq_hamiltonian* const* hams, const sq_space* const* spaces) {
  (void)spaces;
  std::vector<std::vector<int>> members(B.groups.size());
  for (const auto& gm : B.group_members) members[gm.first].push_back(gm.second);
  for (size_t gi = 0; gi < B.groups.size(); ++gi) {
    BatchGroup& G = B.groups[gi];
    const Space& s = *G.space;
    const std::vector<int>& mem = members[gi];
    G.n = (int)mem.size();
    SQ_CHECK(G.n <= 65535, SQ_ERR_ARG, "too many instances in one batched group");
    G.dim = s.dim;
    const Hamiltonian& H0 = hams[mem[0]]->h;
    const int K4 = (s.npair + 1 + 3) / 4 * 4;
    G.A_stride = (int64_t)K4 * H0.kpad;
    G.Ma_stride = (int64_t)s.nsa * s.nsa;
    G.plan_gen = G.prog->plan_gen;
    G.sigma = s.sig;
    G.mats_stride = tiles_mats_doubles(*G.tiles);
    G.tpart_stride = tiles_partial_doubles(*G.tiles);
    G.spart_stride = row_sigma_group_partials(s, G.sigma, G.n);
    SQ_CHECK(G.mats_stride > 0 && G.tpart_stride > 0 && G.spart_stride > 0, SQ_ERR_ARG, "group path unavailable");
    {
      const uint32_t a = s.h_astr[0], b = s.h_bstr[0];
      int par = 0;
      for (uint32_t aa = a; aa; aa &= aa - 1) par += __builtin_popcount(b & ((1u << __builtin_ctz(aa)) - 1u));
      G.hf = (par & 1) ? -1.0 : 1.0;
    }
    std::vector<int32_t> inst(mem.begin(), mem.end()), th0, out0;
    for (int i : mem) {
      th0.push_back(B.inst[i].theta0);
      out0.push_back(B.inst[i].out0);
    }
    G.d_inst = bupload(B, inst);
    G.d_theta0 = bupload(B, th0);
    G.d_out0 = bupload(B, out0);
    const size_t n = (size_t)G.n;
    G.theta = balloc<double>(B, n * G.ng);
    G.A = balloc<double>(B, n * G.A_stride);
    G.Ma = balloc<double>(B, n * G.Ma_stride);
    G.Mb_stride = H0.d_Mb ? (int64_t)s.nsb * s.nsb : G.Ma_stride;
    G.Mb = H0.d_Mb ? balloc<double>(B, n * G.Mb_stride) : G.Ma;
    G.psi = balloc<double>(B, n * G.dim);
    G.lam = balloc<double>(B, n * G.dim);
    G.mats = balloc<double>(B, n * G.mats_stride);
    G.tpart = balloc<double>(B, n * G.tpart_stride);
    G.spart = balloc<double>(B, n * G.spart_stride);
    G.grad = balloc<double>(B, n * G.ng);
    for (size_t m = 0; m < n; ++m) {
      const Hamiltonian& H = hams[mem[m]]->h;
      SQ_CHECK(H.kpad == H0.kpad && H.d_Ma && !H.d_Mb == !H0.d_Mb, SQ_ERR_ARG, "group Hamiltonians differ in shape");
      SQ_HIP(hipMemcpy(G.A + m * G.A_stride, H.d_A, sizeof(double) * G.A_stride, hipMemcpyDeviceToDevice));
      SQ_HIP(hipMemcpy(G.Ma + m * G.Ma_stride, H.d_Ma, sizeof(double) * G.Ma_stride, hipMemcpyDeviceToDevice));
      if (H.d_Mb)
        SQ_HIP(hipMemcpy(G.Mb + m * G.Mb_stride, H.d_Mb, sizeof(double) * G.Mb_stride, hipMemcpyDeviceToDevice));
    }
  }
}

// A group keeps the tile plan and the sigma shape that its buffers and graph
// are made for.  Of instances of kKeepMinDim or more determinants the program
// must outlive the batch, and a later change of its tile shape or of its
// space's sigma shape is refused, as such groups always did; smaller instances,
// which the persistent launch also serves, are free of both.
static void check_group(const BatchGroup& G) {
  if (G.dim < kKeepMinDim) return;
  SQ_CHECK(G.prog->plan_gen == G.plan_gen, SQ_ERR_ARG,
           "a batched program's tile shape changed after the batch was created; create the batch again");
  SQ_CHECK(row_sigma_group_partials(*G.space, G.space->sig, G.n) == G.spart_stride, SQ_ERR_ARG,
           "a batched space's sigma shape changed after the batch was created; create the batch again");
}

static void check_groups(const Batch& B) {
  for (const BatchGroup& G : B.groups) check_group(G);
}

// One group's evaluation on st: thetas and start states in, forward sweep,
// sigma and energies, reverse sweep with gradients, results out.
static void group_launch(const Batch& B, const BatchGroup& G, hipStream_t st) {
  const Space& s = *G.space;
  check_group(G);
  Multi M;
  M.n = G.n;
  M.theta = G.ng;
  M.mats = G.mats_stride;
  M.vec = G.dim;
  M.part = G.tpart_stride;
  M.grad = G.ng;
  k_group_theta<<<dim3((unsigned)((G.ng + 255) / 256), (unsigned)G.n), 256, 0, st>>>(B.dev.theta, G.d_theta0, G.ng,
                                                                                     G.theta);
  const unsigned ib = (unsigned)std::min<int64_t>((G.dim + 255) / 256, 64);
  k_group_init<<<dim3(ib, (unsigned)G.n), 256, 0, st>>>(B.dev.psi0, G.d_inst, G.dim, G.hf, G.psi);
  SQ_HIP(hipGetLastError());
  tiles_forward_group(s, *G.tiles, G.theta, G.psi, G.mats, M, G.lam, st);
  row_sigma_group(s, G.sigma, G.A, G.A_stride, G.Ma, G.Ma_stride, G.Mb, G.Mb_stride, G.psi, G.lam, G.spart, G.n, true, st);
  tiles_reverse_group(s, *G.tiles, G.theta, G.psi, G.lam, G.mats, G.tpart, G.grad, M, st);
  k_group_out<<<(unsigned)G.n, 256, 0, st>>>(G.spart, G.spart_stride, G.grad, G.ng, G.d_inst, G.d_out0,
                                             B.dev.energy, B.dev.grad);
  SQ_HIP(hipGetLastError());
}

}  // namespace sq

using namespace sq;

struct sq_batch {
  Batch b;
};

extern "C" {

int sq_batch_create(int n_inst, const sq_space* const* spaces, const sq_program* const* programs,
                    const sq_hamiltonian* const* hams, int n_workgroups, sq_batch** out) {
  return guarded([&] {
    SQ_CHECK(n_inst > 0 && spaces && programs && hams && out, SQ_ERR_ARG, "invalid arguments");
    {
      uint8_t diag[91] = {0};
      for (int p = 0; p < 13; ++p) diag[p * (p + 1) / 2 + p] = 1;
      SQ_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_bdiag), diag, sizeof(diag)));
    }
    auto* bo = new sq_batch();
    Batch& B = bo->b;
    try {
      std::map<const sq_space*, int> sp_index;
      std::vector<int2> lists;
      std::map<std::pair<const void*, std::vector<int>>, std::pair<int, int>> list_cache;
      // (string, image | parity << 31) of every string a spin part applies to
      auto spin_list = [&](const std::vector<uint32_t>& strs, const SpinOps& o, int& off, int& len) {
        spin_part_list(strs, o, lists, list_cache, off, len);
      };
      std::vector<BatchSpace> bsp;
      std::vector<BatchRot> rots;
      std::vector<double> Astore;
      std::vector<int64_t> cost(n_inst, 0);
      std::vector<char> grouped(n_inst, 0);
      std::vector<GroupCand> cands;
      std::vector<int> cand_of(n_inst, -1), cand_group;
      {
        const char* genv = getenv("SQ_BATCH_GROUPS");
        const bool groups_on = !(genv && genv[0] == '0');
        std::map<std::pair<const Space*, std::string>, int> index;  // (space, gate layout) -> candidate
        std::vector<int> rest;
        for (int i = 0; i < n_inst; ++i) {
          const Space& s = spaces[i]->s;
          const Program& p = programs[i]->p;
          SQ_CHECK(p.space == &s && hams[i]->h.space == &s, SQ_ERR_ARG,
                   "program / Hamiltonian built for another space");
          std::shared_ptr<const TilePlan> tiles;
          if (groups_on && s.dim >= kGroupMinDim && hams[i]->h.d_Ma && row_sigma_group_ok(s))
            tiles = group_tiles_for(s, p);
          if (!tiles) {
            rest.push_back(i);
            continue;
          }
          const auto key = std::make_pair(&s, layout_key(p));
          auto it = index.find(key);
          if (it == index.end()) {
            it = index.emplace(key, (int)cands.size()).first;
            cands.push_back(GroupCand{tiles, {}, true});
          }
          cand_of[i] = it->second;
          cands[it->second].mem.push_back(i);
        }
        drop_small_groups(cands, rest, spaces, programs, n_workgroups);
        cand_group.assign(cands.size(), -1);
      }
      int theta_off = 0, grad_off = 0;
      int64_t gmax = 0;  // G of the persistent launch's instances, at most
      for (int i = 0; i < n_inst; ++i) {
        const Space& s = spaces[i]->s;
        const Program& p = programs[i]->p;
        const Hamiltonian& H = hams[i]->h;
        SQ_CHECK(s.dim < (int64_t)1 << 30, SQ_ERR_ARG, "batched spaces must have fewer than 2^30 determinants");
        if (cand_of[i] >= 0 && cands[cand_of[i]].keep) {
          // grouped with the instances of the same space and gate layout
          int& group = cand_group[cand_of[i]];
          if (group < 0) {
            group = (int)B.groups.size();
            BatchGroup G;
            G.space = &s;
            G.prog = &p;
            G.tiles = cands[cand_of[i]].tiles;
            G.ng = (int)p.gates.size();
            B.groups.push_back(G);
          }
          grouped[i] = 1;
          BatchInstance I{};
          I.theta0 = theta_off;
          I.nparam = (int)p.gates.size();
          theta_off += I.nparam;
          I.out0 = grad_off;
          B.grad_off.push_back(grad_off);
          grad_off += I.nparam;
          B.inst.push_back(I);
          B.group_members.push_back({group, i});
          continue;
        }
        if (!sp_index.count(spaces[i])) {
          sp_index[spaces[i]] = (int)bsp.size();
          BatchSpace b{};
          b.n = s.n;
          b.nsa = s.nsa;
          b.nsb = s.nsb;
          b.npair = s.npair;
          b.K4 = (s.npair + 1 + 3) / 4 * 4;
          b.kpad = (s.npair + 1 + 15) / 16 * 16;
          b.astr = s.d_astr;
          b.bstr = s.d_bstr;
          b.arank = s.d_arank;
          b.brank = s.d_brank;
          b.aexc = s.d_aexc;
          b.bexc = s.d_bexc;
          bsp.push_back(b);
        }
        const BatchSpace& bs = bsp[sp_index[spaces[i]]];
        BatchInstance I{};
        I.space = sp_index[spaces[i]];
        I.gate0 = (int)rots.size();
        for (int g = 0; g < (int)p.gates.size(); ++g) {
          const GateDev& gd = p.gates[g];
          SQ_CHECK(gd.kind == GC_ROT || gd.kind == GC_SA_SINGLE, SQ_ERR_ARG,
                   "batched launches support rotation gates (single, double, sa_single, pair doubles) only");
          const int halves = gd.kind == GC_SA_SINGLE ? 2 : 1;
          for (int h = 0; h < halves; ++h) {
            const Term& T = p.terms[gd.term_begin + 2 * h];
            BatchRot R{};
            spin_list(s.h_astr, T.a, R.aoff, R.na);
            spin_list(s.h_bstr, T.b, R.boff, R.nb);
            R.sgn = T.coef < 0 ? -1.0 : 1.0;
            R.scale = halves == 2 ? 1.0 : gd.scale;
            R.theta_idx = g;
            R.grad_idx = g;
            rots.push_back(R);
          }
        }
        I.ngate = (int)rots.size() - I.gate0;
        I.theta0 = theta_off;
        I.nparam = (int)p.gates.size();
        theta_off += I.nparam;
        I.out0 = grad_off;
        B.grad_off.push_back(grad_off);
        grad_off += I.nparam;
        // A copied from the device Hamiltonian (K4 x kpad, same packing)
        I.A_off = (int)Astore.size();
        std::vector<double> A((size_t)bs.K4 * bs.kpad);
        SQ_HIP(hipMemcpy(A.data(), H.d_A, sizeof(double) * A.size(), hipMemcpyDeviceToHost));
        Astore.insert(Astore.end(), A.begin(), A.end());
        I.e_core = H.e_core;
        B.inst.push_back(I);
        B.lds = std::max(B.lds, a_bytes(s));
        B.dmax = std::max<int64_t>(B.dmax, s.dim);
        gmax = std::max<int64_t>(gmax, bs.npair * s.dim);
        cost[i] = persistent_cost(s, I.ngate);
      }
      SQ_CHECK(B.lds <= 65536, SQ_ERR_ARG, "batched spaces limited to 12 orbitals (LDS)");
      for (const auto& bs : bsp)
        SQ_CHECK(bs.kpad <= 16 * kBatchMT && bs.npair < 91, SQ_ERR_ARG, "batched spaces limited to 12 orbitals");
      B.ngrad = grad_off;
      // longest processing time first, each to the least-loaded workgroup
      // (the instances of the persistent launch: those not in a group)
      int n_small = 0;
      for (int i = 0; i < n_inst; ++i) n_small += grouped[i] ? 0 : 1;
      int nwg = n_workgroups > 0 ? n_workgroups : 256;
      nwg = std::min(nwg, n_small);
      std::vector<int> order;
      for (int i = 0; i < n_inst; ++i)
        if (!grouped[i]) order.push_back(i);
      std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost[a] > cost[b]; });
      std::vector<std::vector<int32_t>> wg_inst(nwg);
      std::vector<int64_t> load(nwg, 0);
      for (int i : order) {
        int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        wg_inst[w].push_back(i);
        load[w] += cost[i];
      }
      std::vector<int32_t> wl, wo{0};
      for (auto& l : wg_inst) {
        wl.insert(wl.end(), l.begin(), l.end());
        wo.push_back((int32_t)wl.size());
      }
      B.nwg = nwg;
      B.dev.vec0 = (int64_t)(B.lds / sizeof(double));
      const size_t with_vec = B.lds + 2 * sizeof(double) * (size_t)B.dmax;
      B.vec_lds = with_vec <= kBatchLds;
      if (B.vec_lds) B.lds = with_vec;
      B.slot = gmax + (B.vec_lds ? 0 : 2 * B.dmax);
      B.dev.spaces = bupload(B, bsp);
      B.dev.inst = bupload(B, B.inst);
      B.dev.rots = bupload(B, rots);
      B.dev.lists = bupload(B, lists);
      B.dev.A = bupload(B, Astore);
      B.dev.wg_list = bupload(B, wl);
      B.dev.wg_off = bupload(B, wo);
      B.dev.slot_doubles = B.slot;
      B.dev.dmax = B.dmax;
      double* scratch = nullptr;
      SQ_HIP(hipMalloc(&scratch, sizeof(double) * std::max<size_t>((size_t)B.slot * nwg, 1)));
      B.allocs.push_back(scratch);
      B.dev.scratch = scratch;
      // energies | gradients, one copy to the host
      double* en = nullptr;
      SQ_HIP(hipMalloc(&en, sizeof(double) * ((size_t)n_inst + grad_off)));
      B.allocs.push_back(en);
      B.dev.energy = en;
      B.dev.grad = en + n_inst;
      SQ_HIP(hipHostMalloc(reinterpret_cast<void**>(&B.host_out), sizeof(double) * ((size_t)n_inst + grad_off),
                           hipHostMallocDefault));
      SQ_HIP(hipMalloc(&B.d_theta, sizeof(double) * std::max(theta_off, 1)));
      B.allocs.push_back(B.d_theta);
      B.dev.theta = B.d_theta;
      B.d_psi0 = bupload(B, std::vector<const double*>(n_inst, nullptr));
      B.dev.psi0 = B.d_psi0;
      build_groups(B, hams, spaces);
      const int nl = std::min<int>(kGroupLanes, (int)B.groups.size());
      if (nl > 1 || (nl > 0 && nwg > 0)) SQ_HIP(hipEventCreateWithFlags(&B.ev_fork, hipEventDisableTiming));
      if (nl > 0 && nwg > 0) {
        SQ_HIP(hipStreamCreateWithFlags(&B.side, hipStreamNonBlocking));
        SQ_HIP(hipEventCreateWithFlags(&B.ev_join, hipEventDisableTiming));
      }
      for (int l = 1; l < nl; ++l) {
        SQ_HIP(hipStreamCreateWithFlags(&B.lane[l], hipStreamNonBlocking));
        SQ_HIP(hipEventCreateWithFlags(&B.ev_lane[l], hipEventDisableTiming));
      }
    } catch (...) {
      delete bo;
      throw;
    }
    *out = bo;
  });
}

int sq_batch_destroy(sq_batch* b) {
  return guarded([&] { delete b; });
}

int64_t sq_batch_num_params(const sq_batch* b) { return b ? b->b.ngrad : -1; }

/* theta: host array of all instances' parameters (concatenated in instance
 * order); copied into the batch's device buffer. */
int sq_batch_set_theta(sq_batch* bo, const double* theta, void* stream) {
  return guarded([&] {
    SQ_CHECK(bo && theta, SQ_ERR_ARG, "NULL argument");
    SQ_HIP(hipMemcpyAsync(bo->b.d_theta, theta, sizeof(double) * bo->b.ngrad, hipMemcpyHostToDevice,
                          as_stream(stream)));
  });
}

/* psi0: host array of n_inst device pointers, each to its instance's start
 * state (engine convention, space dim doubles) or NULL for the HF
 * determinant.  The pointers are read at every launch (graph replays
 * included): the states must stay allocated while the batch runs. */
int sq_batch_set_start_states(sq_batch* bo, const double* const* psi0, void* stream) {
  return guarded([&] {
    SQ_CHECK(bo && psi0, SQ_ERR_ARG, "NULL argument");
    Batch& B = bo->b;
    hipStream_t st = as_stream(stream);
    SQ_HIP(hipMemcpyAsync(B.d_psi0, psi0, sizeof(double*) * B.inst.size(), hipMemcpyHostToDevice, st));
    SQ_HIP(hipStreamSynchronize(st));
  });
}

using BatchKernel = void (*)(BatchDev);

static BatchKernel batch_kernel(const Batch& B) {
  static const BatchKernel table[2][3][2] = {{{k_batch<1, 1, false>, k_batch<1, 2, false>},
                                              {k_batch<2, 1, false>, k_batch<2, 2, false>},
                                              {k_batch<4, 1, false>, k_batch<4, 2, false>}},
                                             {{k_batch<1, 1, true>, k_batch<1, 2, true>},
                                              {k_batch<2, 1, true>, k_batch<2, 2, true>},
                                              {k_batch<4, 1, true>, k_batch<4, 2, true>}}};
  const int u = B.rot_pairs == 1 ? 0 : (B.rot_pairs == 2 ? 1 : 2);
  const BatchKernel k = table[B.vec_lds ? 1 : 0][u][B.gemm_tiles - 1];
  // with the static part above 64 KB the launch needs the permission too
  allow_lds(k, B.lds + kBRot * 64 + 1024 > 65536 ? std::max<size_t>(B.lds, 65536 + 8) : B.lds);
  return k;
}

// The persistent launch and the groups write disjoint outputs: between a fork
// and join events the persistent launch runs on the batch's side stream, first
// (last, or in a lane of the groups: 955 -> 980 to 1100 us), and the groups on
// the lanes (the first is st), the longest first, each on the lane with the
// least work.
static void batch_launch(Batch& B, hipStream_t st) {
  const int nl = std::min<int>(kGroupLanes, (int)B.groups.size());
  if (nl == 0) {
    if (B.nwg > 0) SQ_PROF(PC_BATCH, st, B.bytes, B.flops, batch_kernel(B)<<<B.nwg, kBT, B.lds, st>>>(B.dev));
    return;
  }
  if (B.ev_fork) SQ_HIP(hipEventRecord(B.ev_fork, st));
  if (B.nwg > 0) {
    SQ_HIP(hipStreamWaitEvent(B.side, B.ev_fork, 0));
    SQ_PROF(PC_BATCH, B.side, B.bytes, B.flops, batch_kernel(B)<<<B.nwg, kBT, B.lds, B.side>>>(B.dev));
  }
  for (int l = 1; l < nl; ++l) SQ_HIP(hipStreamWaitEvent(B.lane[l], B.ev_fork, 0));
  auto us = [&](int i) { return group_us(B.groups[i].n, *B.groups[i].space, B.groups[i].ng); };
  std::vector<int> order(B.groups.size());
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return us(a) > us(b); });
  double load[kGroupLanes] = {};
  for (int i : order) {
    const int l = (int)(std::min_element(load, load + nl) - load);
    load[l] += us(i);
    group_launch(B, B.groups[i], l == 0 ? st : B.lane[l]);
  }
  for (int l = 1; l < nl; ++l) {
    SQ_HIP(hipEventRecord(B.ev_lane[l], B.lane[l]));
    SQ_HIP(hipStreamWaitEvent(st, B.ev_lane[l], 0));
  }
  if (B.nwg > 0) {
    SQ_HIP(hipEventRecord(B.ev_join, B.side));
    SQ_HIP(hipStreamWaitEvent(st, B.ev_join, 0));
  }
}

/* Kernel shape: rotation pairs per thread in flight (1, 2 or 4) and sigma
 * GEMM column tiles per wave (1 or 2).  Every shape keeps its captured graph. */
int sq_batch_configure(sq_batch* bo, int rot_pairs, int gemm_tiles) {
  return guarded([&] {
    SQ_CHECK(bo, SQ_ERR_ARG, "NULL argument");
    SQ_CHECK(rot_pairs == 1 || rot_pairs == 2 || rot_pairs == 4, SQ_ERR_ARG, "rot_pairs must be 1, 2 or 4");
    SQ_CHECK(gemm_tiles == 1 || gemm_tiles == 2, SQ_ERR_ARG, "gemm_tiles must be 1 or 2");
    Batch& B = bo->b;
    B.rot_pairs = rot_pairs;
    B.gemm_tiles = gemm_tiles;
  });
}

int sq_batch_run(sq_batch* bo, void* stream) {
  return guarded([&] {
    check_groups(bo->b);
    batch_launch(bo->b, as_stream(stream));
  });
}

/* Capture the launch in a hipGraph (once per kernel shape) and replay it. */
int sq_batch_run_graph(sq_batch* bo, void* stream) {
  return guarded([&] {
    Batch& B = bo->b;
    hipStream_t st = as_stream(stream);
    check_groups(B);
    const int shape = B.kernel_shape();
    if (!B.exec[shape]) {
      // the groups' kernels take their shared-memory attributes on an eager
      // launch first (not a stream operation, so kept out of the capture)
      if (!B.groups.empty()) {
        batch_launch(B, st);
        SQ_HIP(hipStreamSynchronize(st));
      }
      hipStream_t cap;
      SQ_HIP(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
      const bool prof_was = prof_pause();  // event records would become graph nodes
      SQ_HIP(hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal));
      hipError_t e = hipSuccess;
      try {
        batch_launch(B, cap);
        e = hipGetLastError();
      } catch (...) {
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(cap, &g);
        if (g) (void)hipGraphDestroy(g);
        (void)hipStreamDestroy(cap);
        prof_resume(prof_was);
        throw;
      }
      hipGraph_t g = nullptr;
      hipError_t e2 = hipStreamEndCapture(cap, &g);
      (void)hipStreamDestroy(cap);
      prof_resume(prof_was);
      SQ_CHECK(e == hipSuccess && e2 == hipSuccess, SQ_ERR_HIP, "graph capture failed");
      if (B.graph[shape]) (void)hipGraphDestroy(B.graph[shape]);  // of a failed instantiation
      B.graph[shape] = g;
      SQ_HIP(hipGraphInstantiate(&B.exec[shape], g, nullptr, nullptr, 0));
    }
    SQ_HIP(hipGraphLaunch(B.exec[shape], st));
  });
}

int sq_batch_results(const sq_batch* bo, double* energies, double* grads, void* stream) {
  return guarded([&] {
    SQ_CHECK(bo && energies && grads, SQ_ERR_ARG, "NULL argument");
    const Batch& B = bo->b;
    hipStream_t st = as_stream(stream);
    const size_t n = B.inst.size();
    std::lock_guard<std::mutex> lock(B.host_mu);
    SQ_HIP(hipMemcpyAsync(B.host_out, B.dev.energy, sizeof(double) * (n + (size_t)B.ngrad), hipMemcpyDeviceToHost, st));
    SQ_HIP(hipStreamSynchronize(st));
    std::memcpy(energies, B.host_out, sizeof(double) * n);
    std::memcpy(grads, B.host_out + n, sizeof(double) * (size_t)B.ngrad);
  });
}

}  // extern "C"
