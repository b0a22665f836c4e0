// 1- and 2-RDMs by spin parts (replaces the rdm1 and rdm2 properties,
// ups_wavefunction.py:409-476, with the conventions of density_matrix.py:5-136).
//
// With E_x = Ea_x + Eb_x (x = (p, q), n^2 of them) and C the state as an
// [alpha string][beta string] matrix,
//     G(x,y) = <E_x psi|E_y psi> = Ta(x,y) + Tb(x,y) + AB(x,y) + AB(y,x),
//     Ta(x,y) = sum_S s_x(S) s_y(S) (C C^T)[P_x(S)][P_y(S)]   (Tb: C^T C),
//     AB(x,y) = <Ea_x psi|Eb_y psi>,
//     rdm1_pq = <psi|E_pq psi>,   rdm2_pqrs = G((q,p),(r,s)) - d_qr rdm1_ps,
// (E_x psi)[S] = s_x(S) psi[P_x(S)] per spin.  The same-spin parts are two
// Gram products over strings and a sum over strings with two table lookups per
// pair (k_rdm_same).  The opposite-spin part is the work (k_rdm_ab): on an
// alpha string only Na (n - Na) + Na of the n^2 Ea_x do not vanish, and
// AB(x^T, y^T) = AB(x, y) for real psi, so it needs those rows against the
// n (n + 1) / 2 pairs y = (c <= d): 6.6 GFLOP at (12e,12o) (and 1.6 for the
// Gram products) where the Gram matrix of all E_x psi takes 15.7 with its
// symmetries, and its operands need no vector instruction beside their loads
// (the rows E_x psi, generated element by element, took thirty per product).
// Every sum has a fixed order.
// RDMs of a state, the Gram matrix of all E_x psi -> this: (4e,4o) 37 -> 34 us,
// (6e,6o) 63 -> 37, (8e,8o) 653 -> 54, (10e,10o) 387 -> 80, (12e,12o) 733 -> 253
// (k_rdm_ab 139: 47 TFLOP/s of the products it executes; Gram products 60),
// (14e,14o) 9850 -> 4390, (14,7,0) 808 -> 500.

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "sq_internal.h"

namespace sq {

typedef double double4_t __attribute__((ext_vector_type(4)));

// Two doubles of an 8-byte aligned address in one load.
struct __attribute__((packed, aligned(8))) Pair {
  double a, b;
};

static inline int rup(int x, int m) { return (x + m - 1) / m * m; }

namespace {

// alist[s][w] (w a multiple of 16): the Ea_x that do not vanish on alpha
// string s, {partner row * nsb, x | negative << 31}; the rest {own row, n^2}.
__global__ void k_rdm_alist(int n, int nsa, int nsb, int w, const int32_t* __restrict__ full,
                            int2* __restrict__ alist) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsa) return;
  int2* out = alist + (size_t)s * w;
  int m = 0;
  for (int p = 0; p < n; ++p)
    for (int q = 0; q < n; ++q) {
      const int32_t v = full[(size_t)(q * n + p) * nsa + s];
      if (v == 0) continue;
      const int P = p == q ? s : abs(v) - 1;
      out[m++] = make_int2(P * nsb, (p * n + q) | (v < 0 ? (int)0x80000000 : 0));
    }
  for (; m < w; ++m) out[m] = make_int2(s * nsb, n * n);
}

// btab[k][s] (k = (c <= d) packed, padded rows; s < nsp): the byte offset of the
// partner of beta string s under Eb_cd in the LDS rows {row | 0 | -row}; where
// there is none, of the zero.
__global__ void k_rdm_btab(int n, int npair, int nsb, int nsp, const int32_t* __restrict__ full,
                           int32_t* __restrict__ btab) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
  if (s >= nsp) return;
  int32_t v = nsb;
  if (k < npair && s < nsb) {
    int d = 0;
    while ((d + 1) * (d + 2) / 2 <= k) ++d;
    const int c = k - d * (d + 1) / 2;
    const int32_t t = full[(size_t)(d * n + c) * nsb + s];
    if (t != 0) v = c == d ? s : abs(t) - 1 + (t < 0 ? nsb + 1 : 0);
  }
  btab[(size_t)k * nsp + s] = 8 * v;
}

struct AbArgs {
  const double* psi;  // followed by 16 readable doubles
  const int2* alist;
  const int32_t* btab;
  double* partial;
  int n2, nsa, nsb, nsp, nkb, nblk;
  int full, ks, kper, nunits;  // units: full whole rows, then each other row in ks ranges of kper 16-column blocks
};

constexpr int kAbThreads = 256, kAbWaves = 4;
constexpr int kRowPer = 14;  // amplitudes of a row per thread: at most 3432 beta strings

// Opposite-spin part.  A block owns M = AB[x][its YT 16-column tiles of y] in
// LDS and walks alpha rows.  Per row the product A (listed x) . B over the
// beta strings runs on FP64 MFMA, the waves splitting the contraction: lane
// (li, kq) holds A[x = li][4 kq .. 4 kq + 3] of a 16-column block (two 16-byte
// loads of the partner row) and gathers B[the same][y = li] from the row and
// its negative in LDS by the partner table: no vector instruction beside the
// loads (columns past the row read the next one; B is zero there).  One wave
// per SIMD: XT x YT accumulator tiles, and the next block's operands loaded
// during the products of the current one.
// At the end of a row the waves add their tiles to M in turn (rows of M by the
// list, a spare one for its padding), so the order of every sum is fixed; the
// first operands of the next row are loaded meanwhile.
template <int XT, int YT>
__global__ __launch_bounds__(kAbThreads, 1) void k_rdm_ab(AbArgs P) {
  constexpr int W = YT * 16;
  extern __shared__ double smem[];
  double* row = smem;  // row | 0 | -row
  int32_t* xl = reinterpret_cast<int32_t*>(row + 2 * P.nsb + 2);
  double* M = reinterpret_cast<double*>(xl + XT * 16);
  const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, li = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nsb = P.nsb;
  for (int i = tid; i < P.n2 * W; i += kAbThreads) M[i] = 0.0;
  if (tid == 0) row[nsb] = 0.0;
  const char* __restrict__ psib = reinterpret_cast<const char*>(P.psi);
  const int32_t* __restrict__ tab = P.btab;
  auto unit_row = [&](int u) { return u < P.full ? u : P.full + (u - P.full) / P.ks; };
  // block b of an XCD's share walks rows next to those of its neighbours there
  int b0 = blockIdx.x;
  if ((P.nblk & 7) == 0) b0 = (b0 & 7) * (P.nblk >> 3) + (b0 >> 3);
  uint32_t tofs[YT];
#pragma unroll
  for (int v = 0; v < YT; ++v) tofs[v] = (uint32_t)((v * 16 + li) * P.nsp + kq * 4) * 4u;
  double nr[kRowPer];
  int32_t noff[XT];
  int32_t nx = 0;
  uint32_t off[XT];
  double A[2][XT][4], B[2][YT][4];
  int4 T[2][YT];
  int k0 = 0, k1 = 0;
  auto load_t = [&](int kb, int e) {
    const char* __restrict__ p = reinterpret_cast<const char*>(tab + min(kb, k1 - 1) * 16);
#pragma unroll
    for (int v = 0; v < YT; ++v) T[e][v] = *reinterpret_cast<const int4*>(p + tofs[v]);
  };
  auto load_a = [&](int kb, int e) {
    const char* __restrict__ p = psib + (size_t)min(kb, k1 - 1) * 128;
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const Pair x = *reinterpret_cast<const Pair*>(p + off[t] + h * 16);
        A[e][t][2 * h] = x.a;
        A[e][t][2 * h + 1] = x.b;
      }
  };
  auto gather = [&](int e) {
    const char* rb = reinterpret_cast<const char*>(row);
#pragma unroll
    for (int v = 0; v < YT; ++v) {
      B[e][v][0] = *reinterpret_cast<const double*>(rb + T[e][v].x);
      B[e][v][1] = *reinterpret_cast<const double*>(rb + T[e][v].y);
      B[e][v][2] = *reinterpret_cast<const double*>(rb + T[e][v].z);
      B[e][v][3] = *reinterpret_cast<const double*>(rb + T[e][v].w);
    }
  };
  // unit u's row, list and contraction range, for the loads that follow
  auto fetch = [&](int u) {
    const int r = unit_row(u);
#pragma unroll
    for (int i = 0; i < kRowPer; ++i)
      if (i * kAbThreads < nsb) nr[i] = P.psi[(size_t)r * nsb + min(i * kAbThreads + tid, nsb - 1)];
    const int2* __restrict__ al = P.alist + (size_t)r * (XT * 16);
    if (tid < XT * 16) nx = al[tid].y;
#pragma unroll
    for (int t = 0; t < XT; ++t) noff[t] = al[t * 16 + li].x;
  };
  // the first operands of unit u (A of one block, the table of two)
  auto prime = [&](int u) {
    k0 = 0;
    k1 = P.nkb;
    if (u >= P.full) {
      k0 = ((u - P.full) % P.ks) * P.kper;
      k1 = min(P.nkb, k0 + P.kper);
    }
#pragma unroll
    for (int t = 0; t < XT; ++t) off[t] = (uint32_t)noff[t] * 8u + (uint32_t)kq * 32u;
    load_t(k0 + wave, 0);
    load_a(k0 + wave, 0);
    load_t(k0 + wave + kAbWaves, 1);
  };
  if (b0 < P.nunits) {
    fetch(b0);
    prime(b0);
  }
  for (int u = b0; u < P.nunits; u += P.nblk) {
    lds_barrier();  // everyone has left the previous row
#pragma unroll
    for (int i = 0; i < kRowPer; ++i)
      if (i * kAbThreads + tid < nsb) {
        row[i * kAbThreads + tid] = nr[i];
        row[nsb + 1 + i * kAbThreads + tid] = -nr[i];
      }
    if (tid < XT * 16) xl[tid] = nx;
    lds_barrier();
    if (u + P.nblk < P.nunits) fetch(u + P.nblk);
    double4_t acc[XT][YT];
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
      for (int v = 0; v < YT; ++v) acc[t][v] = double4_t{0.0, 0.0, 0.0, 0.0};
    auto step = [&](int kb, int e) {  // block kb, its operands in buffers e
      load_t(kb + 2 * kAbWaves, e);
      load_a(kb + kAbWaves, e ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      gather(e ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < XT; ++t)
#pragma unroll
          for (int v = 0; v < YT; ++v)
            acc[t][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[e][t][s], B[e][v][s], acc[t][v], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    int kb = k0 + wave;
    if (kb < k1) {
      gather(0);
      for (; kb < k1; kb += 2 * kAbWaves) {
        step(kb, 0);
        if (kb + kAbWaves < k1) step(kb + kAbWaves, 1);
      }
    }
    if (u + P.nblk < P.nunits) prime(u + P.nblk);
    double* mr[XT][4];
#pragma unroll
    for (int t = 0; t < XT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = xl[t * 16 + kq + 4 * r];
        mr[t][r] = M + (size_t)(e & 0xffff) * W + li;
#pragma unroll
        for (int v = 0; v < YT; ++v) {
          double x = flip(acc[t][v][r], e);
          __asm__ volatile("" : "+v"(x));  // before the turn
          acc[t][v][r] = x;
        }
      }
    for (int w = 0; w < kAbWaves; ++w) {
      if (w == wave) {
#pragma unroll
        for (int t = 0; t < XT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int v = 0; v < YT; ++v) atomicAdd(mr[t][r] + v * 16, acc[t][v][r]);
      }
      lds_barrier();
    }
  }
  double* __restrict__ out = P.partial + (size_t)blockIdx.x * P.n2 * W;
  for (int i = tid; i < P.n2 * W; i += kAbThreads) out[i] = M[i];
}

// Ta, Tb (blockIdx.y: spin) for x <= y, x and y up to n^2 (the identity): one
// wave per pair, lanes over strings.  rho holds its upper 64 x 64 tiles.
__global__ __launch_bounds__(256) void k_rdm_same(int n, int nsa, int nsb, const int32_t* __restrict__ afull,
                                                  const int32_t* __restrict__ bfull, const double* __restrict__ rho_a,
                                                  const double* __restrict__ rho_b, double* __restrict__ T) {
  const int n2 = n * n, m = n2 + 1, lane = threadIdx.x & 63;
  const int pair = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pair >= m * (m + 1) / 2) return;
  int y = (int)((sqrtf(8.0f * (float)pair + 1.0f) - 1.0f) * 0.5f);
  while (y * (y + 1) / 2 > pair) --y;
  while ((y + 1) * (y + 2) / 2 <= pair) ++y;
  const int x = pair - y * (y + 1) / 2;
  const bool beta = blockIdx.y != 0;
  const int ns = beta ? nsb : nsa;
  const int32_t* __restrict__ full = beta ? bfull : afull;
  const double* __restrict__ rho = beta ? rho_b : rho_a;
  auto entry = [&](int e) { return (size_t)((e % n) * n + e / n) * ns; };  // E_pq psi: the image under E_qp
  const int32_t* __restrict__ tx = full + (x < n2 ? entry(x) : 0);
  const int32_t* __restrict__ ty = full + (y < n2 ? entry(y) : 0);
  const bool dx = x == n2 || x / n == x % n, dy = y == n2 || y / n == y % n;
  double v = 0.0;
  constexpr int U = 4;  // strings in flight per lane
  for (int s0 = lane; s0 < ns; s0 += 64 * U) {
    int px[U], py[U];
    double r[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int s = s0 + 64 * i;
      px[i] = s < ns ? (x == n2 ? 1 : tx[s]) : 0;
      py[i] = s < ns ? (y == n2 ? 1 : ty[s]) : 0;
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int s = s0 + 64 * i;
      r[i] = 0.0;
      if (px[i] != 0 && py[i] != 0) {
        const int a = dx ? s : abs(px[i]) - 1, b = dy ? s : abs(py[i]) - 1;
        r[i] = rho[(size_t)min(a, b) * ns + max(a, b)];
      }
    }
#pragma unroll
    for (int i = 0; i < U; ++i) v += (px[i] ^ py[i]) < 0 ? -r[i] : r[i];
  }
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if (lane == 0) T[((size_t)blockIdx.y * m + x) * m + y] = v;
}

constexpr int kSumParts = 8;  // partial sums over the blocks of k_rdm_ab

// sums[z][x][y] (wtot columns): the blocks of part z (blockIdx.z), in order, of
// the columns [y0, y0 + w) that are in the partials.
__global__ void k_rdm_sum(const double* __restrict__ partial, int nblk, int n2, int w, int y0, int wtot,
                          double* __restrict__ sums) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, len = n2 * w, z = blockIdx.z;
  if (i >= len) return;
  const int b0 = nblk * z / kSumParts, b1 = nblk * (z + 1) / kSumParts;
  const double* __restrict__ p = partial + i;
  double v = 0.0;
#pragma unroll 8
  for (int b = b0; b < b1; ++b) v += p[(size_t)b * len];
  sums[((size_t)z * n2 + i / w) * wtot + y0 + i % w] = v;
}

// out: rdm1 [n^2] | rdm2 [n^4].
__global__ void k_rdm_assemble(int n, int w, const double* __restrict__ sums, const double* __restrict__ T,
                               double* __restrict__ out) {
  const int n2 = n * n, m = n2 + 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  auto g1 = [&](int p, int q) {
    const int x = min(p, q) * n + max(p, q);
    return T[(size_t)x * m + n2] + T[((size_t)m + x) * m + n2];
  };
  if (i < n2) out[i] = g1(i / n, i % n);
  if (i >= n2 * n2) return;
  auto ab = [&](int a, int b, int c, int d) {
    const bool t = c > d;
    const int x = t ? b * n + a : a * n + b, lo = min(c, d), hi = max(c, d);
    const int k = hi * (hi + 1) / 2 + lo;
    double v = 0.0;
#pragma unroll
    for (int z = 0; z < kSumParts; ++z) v += sums[((size_t)z * n2 + x) * w + k];
    return v;
  };
  const int p = i / (n2 * n), q = i / n2 % n, r = i / n % n, s = i % n;
  const int x = q * n + p, y = r * n + s, lo = min(x, y), hi = max(x, y);
  double v = T[(size_t)lo * m + hi] + T[((size_t)m + lo) * m + hi];
  v += ab(q, p, r, s) + ab(r, s, q, p);
  if (q == r) v -= g1(p, s);
  out[n2 + i] = v;
}

// Ct = C^T (nsa x nsb): 32 x 32 tiles through LDS; Cp = C followed by 16 zeros.
__global__ __launch_bounds__(256) void k_transpose(const double* __restrict__ C, double* __restrict__ Ct,
                                                   double* __restrict__ Cp, int nsa, int nsb) {
  __shared__ double t[32][33];
  const int a0 = blockIdx.y * 32, b0 = blockIdx.x * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (int j = y; j < 32; j += 8)
    if (a0 + j < nsa && b0 + x < nsb) {
      const size_t i = (size_t)(a0 + j) * nsb + b0 + x;
      Cp[i] = t[j][x] = C[i];
    }
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 16) Cp[(size_t)nsa * nsb + threadIdx.x] = 0.0;
  __syncthreads();
  for (int j = y; j < 32; j += 8)
    if (b0 + j < nsb && a0 + x < nsa) Ct[(size_t)(b0 + j) * nsa + a0 + x] = t[x][j];
}

struct RdmPlan {
  int xt, ytot, npass, nblk, nsp, nkb, full, ks, kper, nunits;
  int yt(int pass) const { return ytot * (pass + 1) / npass - ytot * pass / npass; }
  int y0(int pass) const { return ytot * pass / npass; }
};

size_t ab_lds(const Space& s, int xt, int yt) {
  return 8 * (((size_t)s.n * s.n + 1) * yt * 16 + 2 * (size_t)s.nsb + 2) + 4 * (size_t)xt * 16;
}

// Shape of k_rdm_ab: the y tiles in the fewest even groups (a launch each) of
// at most 20 tiles with the x tiles (registers) whose M fits in LDS; one block per CU; the rows that do
// not fill a round of blocks are cut into the ranges that balance best
// ((12e,12o): 924 rows on 256 blocks, 3 rounds and 156 rows in thirds, 3.67 row
// times instead of 4).  The limits hold for every space of up to 14 orbitals.
bool rdm_plan(const Space& s, RdmPlan* out) {
  out->xt = std::max(1, (s.na * (s.n - s.na) + s.na + 15) / 16);
  out->ytot = (s.npair + 15) / 16;
  if (out->xt > 4 || s.nsb > kRowPer * kAbThreads || s.dim >= ((int64_t)1 << 29) || s.dim == 0) return false;
  out->npass = 0;
  for (int np = 1; np <= out->ytot; ++np) {
    const int yt = (out->ytot + np - 1) / np;
    if (yt <= 6 && out->xt * yt <= 20 && ab_lds(s, out->xt, yt) <= 160 * 1024 - 256) {
      out->npass = np;
      break;
    }
  }
  if (out->npass == 0) return false;
  out->nblk = std::min(s.nsa, 256);
  out->nsp = rup(s.nsb, 16);
  out->nkb = out->nsp / 16;
  out->full = s.nsa / out->nblk * out->nblk;
  const int rest = s.nsa - out->full;
  out->ks = 1;
  if (rest > 0) {
    double best = 1e9;
    for (int ks = 1; ks <= 4 && out->nkb >= 4 * ks; ++ks) {
      const double t = (double)((rest * ks + out->nblk - 1) / out->nblk) / ks;
      if (t < best - 1e-9) best = t, out->ks = ks;
    }
  }
  out->kper = (out->nkb + out->ks - 1) / out->ks;
  out->nunits = out->full + rest * out->ks;
  return true;
}

struct RdmWork {
  int64_t ct, cp, rho_a, rho_b, T, partial, sums, out, total;  // offsets in doubles
};

RdmWork rdm_work(const Space& s, const RdmPlan& p) {
  const int64_t n2 = (int64_t)s.n * s.n;
  int yt = 0;
  for (int i = 0; i < p.npass; ++i) yt = std::max(yt, p.yt(i));
  RdmWork w;
  w.ct = 0;
  w.cp = w.ct + s.dim;
  w.rho_a = w.cp + s.dim + 16;
  w.rho_b = w.rho_a + (int64_t)s.nsa * s.nsa;
  w.T = w.rho_b + (int64_t)s.nsb * s.nsb;
  w.partial = w.T + 2 * (n2 + 1) * (n2 + 1);
  w.sums = w.partial + p.nblk * n2 * yt * 16;
  w.out = w.sums + kSumParts * n2 * p.ytot * 16;
  w.total = w.out + n2 + n2 * n2;
  return w;
}

}  // namespace

int64_t rdm_work_bytes(const Space& s) {
  RdmPlan p;
  return rdm_plan(s, &p) ? 8 * rdm_work(s, p).total : 8;
}

// The space's tables, on first use; freed with the space.
static void rdm_tables(const Space& s, const RdmPlan& p) {
  std::lock_guard<std::mutex> lock(s.rdm_mu);
  if (s.d_rdm_btab) return;
  int2* al = nullptr;
  int32_t* bt = nullptr;
  try {
    const int w = p.xt * 16, rows = p.ytot * 16;
    SQ_HIP(hipMalloc(&al, sizeof(int2) * (size_t)w * s.nsa));
    SQ_HIP(hipMalloc(&bt, sizeof(int32_t) * (size_t)rows * p.nsp));
    k_rdm_alist<<<(s.nsa + 63) / 64, 64>>>(s.n, s.nsa, s.nsb, w, s.d_aexc_full, al);
    SQ_HIP(hipGetLastError());
    k_rdm_btab<<<dim3((p.nsp + 255) / 256, rows), 256>>>(s.n, s.npair, s.nsb, p.nsp, s.d_bexc_full, bt);
    SQ_HIP(hipGetLastError());
    SQ_HIP(hipDeviceSynchronize());
  } catch (...) {
    if (al) (void)hipFree(al);
    if (bt) (void)hipFree(bt);
    throw;
  }
  s.d_rdm_alist = al;
  s.d_rdm_btab = bt;
}

void rdm_tables_free(Space& s) {
  if (s.d_rdm_alist) (void)hipFree(s.d_rdm_alist);
  if (s.d_rdm_btab) (void)hipFree(s.d_rdm_btab);
  s.d_rdm_alist = nullptr;
  s.d_rdm_btab = nullptr;
}

void rdm_impl(const Space& s, const double* psi, double* rdm1, double* rdm2, double* work, hipStream_t st) {
  RdmPlan p;
  SQ_CHECK(rdm_plan(s, &p), SQ_ERR_ARG, "RDMs support at most 14 orbitals and need a determinant");
  rdm_tables(s, p);
  const RdmWork w = rdm_work(s, p);
  const int n2 = s.n * s.n, m = n2 + 1;
  double *ct = work + w.ct, *cp = work + w.cp, *ra = work + w.rho_a, *rb = work + w.rho_b, *T = work + w.T, *partial = work + w.partial,
         *sums = work + w.sums;
  k_transpose<<<dim3((s.nsb + 31) / 32, (s.nsa + 31) / 32), 256, 0, st>>>(psi, ct, cp, s.nsa, s.nsb);
  SQ_HIP(hipGetLastError());
  string_grams(psi, ct, ra, rb, s.nsa, s.nsb, st);
  k_rdm_same<<<dim3((m * (m + 1) / 2 + 3) / 4, 2), 256, 0, st>>>(s.n, s.nsa, s.nsb, s.d_aexc_full, s.d_bexc_full, ra,
                                                               rb, T);
  SQ_HIP(hipGetLastError());
  for (int i = 0; i < p.npass; ++i) {
    const int yt = p.yt(i), wy = yt * 16;
    const AbArgs A{cp,   s.d_rdm_alist, s.d_rdm_btab + (size_t)p.y0(i) * 16 * p.nsp,
                   partial, n2, s.nsa, s.nsb, p.nsp, p.nkb, p.nblk, p.full, p.ks, p.kper, p.nunits};
    const size_t lds = ab_lds(s, p.xt, yt);
    auto go = [&](auto kernel) {
      allow_lds(kernel, lds);
      const double flops = 2.0 * 256.0 * p.xt * yt * (double)s.nsa * p.nsp;
      const double bytes = 8.0 * (double)s.dim + 8.0 * (double)n2 * wy * p.nblk;
      SQ_PROF(PC_RDM_GRAM, st, bytes, flops, kernel<<<p.nblk, kAbThreads, lds, st>>>(A));
    };
    switch (p.xt * 8 + yt) {
#define SQ_AB(X, Y)     \
  case X * 8 + Y:       \
    go(k_rdm_ab<X, Y>); \
    break;
#define SQ_ABX(X) SQ_AB(X, 1) SQ_AB(X, 2) SQ_AB(X, 3) SQ_AB(X, 4) SQ_AB(X, 5)
      SQ_ABX(1) SQ_AB(1, 6) SQ_ABX(2) SQ_AB(2, 6) SQ_ABX(3) SQ_AB(3, 6) SQ_ABX(4)
#undef SQ_ABX
#undef SQ_AB
      default:
        throw Error{SQ_ERR_ARG, "unsupported orbital count for the RDM kernel"};
    }
    k_rdm_sum<<<dim3((n2 * wy + 255) / 256, 1, kSumParts), 256, 0, st>>>(partial, p.nblk, n2, wy, p.y0(i) * 16,
                                                                       p.ytot * 16, sums);
    SQ_HIP(hipGetLastError());
  }
  k_rdm_assemble<<<(n2 * n2 + 255) / 256, 256, 0, st>>>(s.n, p.ytot * 16, sums, T, work + w.out);
  SQ_HIP(hipGetLastError());
  std::vector<double> h((size_t)n2 + (size_t)n2 * n2);
  copy_to_host_pinned(h.data(), work + w.out, h.size(), st);
  std::memcpy(rdm1, h.data(), sizeof(double) * n2);
  std::memcpy(rdm2, h.data() + n2, sizeof(double) * (size_t)n2 * n2);
}

}  // namespace sq
