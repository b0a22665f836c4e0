// sigma = H psi by alpha rows, with no intermediate in HBM (replaces the
// H application of propagate_state([H]) / expectation_value,
// operator_state_algebra.py:472-824, for H = hamiltonian_0i_0a,
// operators.py:476-529).
//
// Spin split.  With E+_k = E+a_k + E+b_k over packed pairs k = (p >= q),
// A(k,k') = 1/2 g(k,k') and h'_k = h_pq - 1/2 sum_r g_prrq (the alpha and
// beta parts commute):
//     H = Ha + Hb + sum_{k,k'} g(k,k') E+b_k E+a_k',
//     Ha = sum_k h'_k E+a_k + sum_{k,k'} A(k,k') E+a_k E+a_k'   (Hb alike),
// With C the state as an [alpha string][beta string] matrix and Ma, Mb the
// matrices of Ha and Hb over strings (built once per Hamiltonian, k_string_ham,
// half of e_core on each diagonal; one matrix where both spins have the same
// strings), the list form:
//     sigma = Ma C + C Mb + sum_k E+b_k G_k,   G_k = sum_k' g(k,k') E+a_k' psi.
//   1. The string products are dense FP64-MFMA GEMMs: tiles in the launch of
//      step 2 where two of its blocks share a CU (to 12 orbitals at half
//      filling), else a launch of their own (k_string_gemm).
//   2. k_sigma_rows_list: one block per group of R alpha rows.  On an alpha
//      string only Na (n - Na) + Na of the npair E+a_k' do not vanish, and the
//      row of G is A . B over those, B[k'][I_b] = +- psi[Pa_k'(I_a), I_b] (the
//      partner row is uniform over the row of G: a list per string).  B is
//      loaded straight into the MFMA operand registers, A comes from LDS by
//      the listed k'.  Every G_k[I_a, J_b] goes to the sigma row at Pb_k(J_b)
//      (E+b_k is symmetric) by an LDS atomic add; G never leaves the CU.
// The full form contracts all npair + 1 rows with the beta part of H in the
// operand (no Mb):
//     sigma = Ma C + e_core / 2 C + sum_k E+b_k G_k,
//     G_k   = h'_k psi + sum_k' A(k,k') (2 E+a_k' + E+b_k') psi.
// It takes 1.4 ((12e,12o)) to 1.03 ((15e,15o)) times the products of the list
// form and more vector instructions per product: (12e,12o) 271 -> 200 us a
// sigma, (14e,14o) 7.07 -> 5.40 ms (rows 5.89 -> 2.76, string products 1.18 ->
// 2.64), (15: 7,7) 43.9 -> 28.9, (16: 6,6) 165 -> 55 (one 16-row tile of A at a
// time beside two rows of 8008 in LDS), 10 orbitals in groups 325 -> 245 us.  It
// serves deterministic runs, with a fixed order of every sum (k_sigma_rows: each
// wave's tile of G is staged in LDS and every target adds the staged values of
// its beta neighbours in list order).

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>

#include <rocblas/rocblas.h>

#include "sq_internal.h"

namespace sq {

void reduce_impl(const double* partial, int64_t n, double* out_dev, int slot, bool accumulate, double factor,
                 hipStream_t st);

namespace {

constexpr int kRowThreads = 512;
constexpr int kRowWaves = kRowThreads / 64;
constexpr int kMaxMt = 9;       // 16-row tiles of G per wave
constexpr int kMaxFusedMt = 6;  // where two blocks share a CU (its LDS holds no two A slices of 7)
constexpr int kMaxTargets = 8;  // targets (alpha row, beta string) per thread
constexpr size_t kLdsMax = 160 * 1024 - 256;  // dynamic LDS per block (the static part stays below 256 bytes)
constexpr int kMaxSplit = 4;     // string product partials (workspace is sized for this many)

int env_int(const char* name, int dflt) {
  const char* e = getenv(name);
  return (e && e[0]) ? atoi(e) : dflt;
}

__host__ __device__ inline int rup(int x, int m) { return (x + m - 1) / m * m; }

__global__ void k_zero(double* __restrict__ x, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] = 0.0;
}

// ---------------------------------------------------------------------------
// Space tables.
// rta[k][s] (k < K8 + 16): {partner row * nsb, 2 * coefficient} of E+a_k on
// alpha string s (diagonal: 2 * occupation; absent / k >= npair: {own, 0}).
// rtb[k][s] (k < K8 + 32): {partner column, coefficient} of E+b_k on beta
// string s (diagonal: occupation; k == npair: {own, 1}; absent: {own, 0}).
__global__ void k_row_tables(int npair, int nstr, int nsb, int alpha, const int32_t* __restrict__ exc,
                             int2* __restrict__ tab) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  if (s >= nstr) return;
  const int own = alpha ? s * nsb : s;
  const int f = alpha ? 2 : 1;
  int2 e = make_int2(own, 0);
  if (k < npair) {
    int p = 0;
    while ((p + 1) * (p + 2) / 2 <= k) ++p;
    const int q = k - p * (p + 1) / 2;
    const int32_t x = exc[(size_t)k * nstr + s];
    if (p == q) e = make_int2(own, f * x);
    else if (x != 0) e = make_int2(alpha ? (abs(x) - 1) * nsb : abs(x) - 1, x > 0 ? f : -f);
  } else if (k == npair && !alpha) {
    e = make_int2(own, 1);
  }
  tab[(size_t)k * nstr + s] = e;
}

// Beta neighbour lists: for target string s, the entries (J, k, sign) with
// (E+b_k)[s][J] != 0 (J = partner, or s itself with occupation 1 on the
// diagonal), packed J | k << 14 | negative << 31 and sorted by J; tile[s][c]
// (c = 0..tpr) counts the entries with J < 16 c.
__global__ void k_nbr_count(int npair, int nsb, const int32_t* __restrict__ bexc, int32_t* __restrict__ cnt) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsb) return;
  int c = 0;
  for (int k = 0; k < npair; ++k) c += bexc[(size_t)k * nsb + s] != 0;
  cnt[s] = c;
}

__global__ void k_nbr_fill(int npair, int nsb, int tpr, const int32_t* __restrict__ bexc,
                           const int32_t* __restrict__ off, uint32_t* __restrict__ nbr, uint8_t* __restrict__ tile) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsb) return;
  uint32_t* out = nbr + off[s];
  int m = 0, k = 0;
  for (int p = 0; p < 32 && k < npair; ++p) {
    for (int q = 0; q <= p; ++q, ++k) {
      const int32_t x = bexc[(size_t)k * nsb + s];
      if (x == 0) continue;
      uint32_t e;
      if (p == q) e = (uint32_t)s | ((uint32_t)k << 14);
      else e = (uint32_t)(abs(x) - 1) | ((uint32_t)k << 14) | (x < 0 ? 0x80000000u : 0u);
      // insertion by partner column (stable: equal columns keep k order)
      int j = m++;
      while (j > 0 && (out[j - 1] & 0x3FFFu) > (e & 0x3FFFu)) {
        out[j] = out[j - 1];
        --j;
      }
      out[j] = e;
    }
  }
  int e = 0;
  for (int c = 0; c <= tpr; ++c) {
    while (e < m && (int)(out[e] & 0x3FFFu) < 16 * c) ++e;
    tile[(size_t)s * (tpr + 1) + c] = (uint8_t)e;
  }
}

// ---------------------------------------------------------------------------
// M[J][I] = <I|Hx|J> + e0 delta_IJ (symmetric) for the part Hx = Ha or Hb of
// one spin, one block per column J:
//   Hx|J> = sum_k E+x_k u_k,  u_k = h'_k |J> + sum_k' A(k,k') E+x_k' |J>,
// where E+x_k'|J> is J itself (diagonal k', coefficient = occupation) or one
// single excitation of J (distinct for distinct off-diagonal k'): u_k lives
// on at most 1 + N (n - N) strings ("slots"), every slot but the first with
// one k', and
//   <I|Hx|J> = sum_k c_k(I) u_k[slot(P_k(I))].
__global__ void k_string_ham(int nstr, int npair, int kpad, const int32_t* __restrict__ exc,
                             const double* __restrict__ At, double e0, double* __restrict__ M) {
  extern __shared__ unsigned char smem_raw[];
  const int J = blockIdx.x;
  // LDS: slot of every string (-1: none) | slot -> k' | k' coefficient | u[npair][nslot_max]
  int16_t* slotmap = reinterpret_cast<int16_t*>(smem_raw);
  int16_t* slotk = slotmap + rup(nstr, 8);
  int32_t* kcoef = reinterpret_cast<int32_t*>(slotk + rup(npair + 1, 8));
  double* u = reinterpret_cast<double*>(kcoef + rup(npair, 2));
  __shared__ int nslot;
  for (int i = threadIdx.x; i < nstr; i += blockDim.x) slotmap[i] = -1;
  __syncthreads();
  if (threadIdx.x == 0) {
    slotmap[J] = 0;
    int ns = 1;
    int k = 0;
    for (int p = 0; k < npair; ++p)
      for (int q = 0; q <= p; ++q, ++k) {
        const int32_t x = exc[(size_t)k * nstr + J];
        if (p == q || x == 0) {
          kcoef[k] = p == q ? x : 0;
        } else {
          const int P = abs(x) - 1;
          slotmap[P] = (int16_t)ns;
          slotk[ns++] = (int16_t)k;
          kcoef[k] = x > 0 ? 1 : -1;
        }
      }
    nslot = ns;
  }
  __syncthreads();
  const int ns = nslot;
  // u[k][slot] in a fixed k' order
  for (int i = threadIdx.x; i < npair * ns; i += blockDim.x) {
    const int k = i / ns, sl = i - k * ns;
    double v;
    if (sl == 0) {
      v = At[(size_t)npair * kpad + k];
      for (int p = 0, kp = 0; kp < npair; ++p, kp += p + 1)  // the diagonal k'
        v += At[(size_t)kp * kpad + k] * (double)kcoef[kp];
    } else {
      const int kp = slotk[sl];
      v = At[(size_t)kp * kpad + k] * (double)kcoef[kp];
    }
    u[i] = v;
  }
  __syncthreads();
  for (int I = threadIdx.x; I < nstr; I += blockDim.x) {
    double v = I == J ? e0 : 0.0;
    int k = 0;
    for (int p = 0; k < npair; ++p)
      for (int q = 0; q <= p; ++q, ++k) {
        const int32_t x = exc[(size_t)k * nstr + I];
        if (x == 0) continue;
        const int K = p == q ? I : abs(x) - 1;
        const int sl = slotmap[K];
        if (sl < 0) continue;
        const double c = p == q ? (double)x : (x > 0 ? 1.0 : -1.0);
        v += c * u[k * ns + sl];
      }
    M[(size_t)J * nstr + I] = v;
  }
}

// ---------------------------------------------------------------------------
// out[z] = the part of L0 R0 + L1 R1 in split z of the joined contraction range
// [0, k0n + k1n) (L m x k, R k x n, row-major; k1n may be 0).  256 threads,
// T x T tile, a wave owns a quarter of it as 16 x 16 MFMA tiles; 16-deep slices
// in two LDS buffers, the next slice loaded into registers during the MFMAs of
// the current one (one barrier per slice, which leaves those loads in flight).
// Row k of a slice holds its columns at c ^ swz(k), swz(k) = 16 (k & 1) +
// 4 ((k >> 1) & 3): the sixteen k of a store go to eight bank groups, the two
// k of a half-wave's read to separate halves.
// Blocks take tiles in strips of 8 tile rows, contiguous per XCD.
typedef double double4_t __attribute__((ext_vector_type(4)));

struct GemmArgs {
  const double *L0, *R0, *L1, *R1;
  double* out;
  int m, n, k0n, k1n, kchunk;
};

template <int T>
__device__ __forceinline__ void string_gemm_block(const GemmArgs& P, int i0, int j0, int z) {
  constexpr int F = T / 32;  // MFMA tiles per wave and side
  constexpr int LJ = T / 16;
  __shared__ double sL[2][16][T];
  __shared__ double sR[2][16][T];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, kq = lane >> 4, li = lane & 15;
  const int wi = (wave >> 1) * (T / 2), wj = (wave & 1) * (T / 2);
  double4_t acc[F][F];
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b) acc[a][b] = double4_t{0.0, 0.0, 0.0, 0.0};
  // c ^ swz(k) for c = 16 x + low: 16 (x & ~1) + at(k, low, x & 1)
  auto at = [](int k, int low, int odd) {
    const int b4 = (odd ^ k) & 1;
    return 16 * b4 + (low ^ (4 * ((k >> 1) & 3)));
  };
  // loaders: L column t % 16 of rows t / 16 + 16 j, R row t / 16, columns t % 16 + 16 j
  const int tk = t & 15, tr = t >> 4;
  const int wl[2] = {at(tk, tr, 0), at(tk, tr, 1)}, wr[2] = {at(tr, tk, 0), at(tr, tk, 1)};
  const int rd[2][2] = {{at(kq, li, 0), at(kq, li, 1)}, {at(4 + kq, li, 0), at(4 + kq, li, 1)}};
  // (rows past m and columns past n read the last one), as byte offsets from
  // the slice's uniform base
  uint32_t lofs[LJ], rofs[LJ];
  double pl[LJ], pr[LJ];
  const int zb = z * P.kchunk, ze = min(P.k0n + P.k1n, zb + P.kchunk);
  for (int phase = 0; phase < 2; ++phase) {
    const double* __restrict__ L = phase ? P.L1 : P.L0;
    const double* __restrict__ R = phase ? P.R1 : P.R0;
    const int off = phase ? P.k0n : 0, kn = phase ? P.k1n : P.k0n;
    const int kb = max(zb - off, 0), ke = min(ze - off, kn);
    if (kb >= ke) continue;
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
      lofs[j] = ((uint32_t)min(tr + 16 * j, P.m - 1 - i0) * (uint32_t)kn + tk) * 8u;
      rofs[j] = ((uint32_t)tr * (uint32_t)P.n + (uint32_t)min(tk + 16 * j, P.n - 1 - j0)) * 8u;
    }
    // slice at k; bl, br: bytes back to the last column / row for lanes past it
    auto load = [&](int k, uint32_t bl, uint32_t br) {
      const char* __restrict__ Lk = reinterpret_cast<const char*>(L + (size_t)i0 * kn + k);
      const char* __restrict__ Rk = reinterpret_cast<const char*>(R + (size_t)k * P.n + j0);
#pragma unroll
      for (int j = 0; j < LJ; ++j) {
        pl[j] = *reinterpret_cast<const double*>(Lk + (lofs[j] - bl));
        pr[j] = *reinterpret_cast<const double*>(Rk + (rofs[j] - br));
      }
    };
    auto store = [&](int buf) {
#pragma unroll
      for (int j = 0; j < LJ; ++j) {
        sL[buf][tk][16 * (j & ~1) + wl[j & 1]] = pl[j];
        sR[buf][tr][16 * (j & ~1) + wr[j & 1]] = pr[j];
      }
    };
    auto products = [&](int buf) {
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4) {
        double a[F], b[F];
#pragma unroll
        for (int x = 0; x < F; ++x) {
          a[x] = sL[buf][kk + kq][wi + 16 * (x & ~1) + rd[(kk >> 2) & 1][x & 1]];
          b[x] = sR[buf][kk + kq][wj + 16 * (x & ~1) + rd[(kk >> 2) & 1][x & 1]];
        }
#pragma unroll
        for (int x = 0; x < F; ++x)
#pragma unroll
          for (int y = 0; y < F; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], b[y], acc[x][y], 0, 0, 0);
      }
    };
    const int kf = kb + ((ke - kb) & ~15);  // end of the whole slices
    int buf = 0;
    if (kb < kf) {
      load(kb, 0, 0);
      store(0);  // the previous phase ended with a barrier
      lds_barrier();
      for (int k = kb; k < kf; k += 16, buf ^= 1) {
        if (k + 16 < kf) load(k + 16, 0, 0);
        products(buf);
        if (k + 16 < kf) store(buf ^ 1);
        lds_barrier();
      }
    }
    if (kf < ke) {
      const int pl_over = kf + tk - (ke - 1), pr_over = kf + tr - (ke - 1);
      load(kf, 8u * (uint32_t)max(0, pl_over), 8u * (uint32_t)max(0, pr_over) * (uint32_t)P.n);
#pragma unroll
      for (int j = 0; j < LJ; ++j) {
        if (pl_over > 0) pl[j] = 0.0;
        if (pr_over > 0) pr[j] = 0.0;
      }
      store(0);
      lds_barrier();
      products(0);
      lds_barrier();
    }
  }
  double* o = P.out + (size_t)z * P.m * P.n;
#pragma unroll
  for (int x = 0; x < F; ++x)
#pragma unroll
    for (int y = 0; y < F; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int I = i0 + wi + x * 16 + kq + 4 * r, J = j0 + wj + y * 16 + li;
        if (I < P.m && J < P.n) o[(size_t)I * P.n + J] = acc[x][y][r];
      }
}

template <int T>
__global__ __launch_bounds__(256, 2) void k_string_gemm(GemmArgs P) {
  const int tn = (P.n + T - 1) / T, tm = (P.m + T - 1) / T, nt = tm * tn;
  int id = blockIdx.x;
  if (id < (nt & ~7)) id = (id & 7) * (nt >> 3) + (id >> 3);
  const int strip = id / (8 * tn), sr = min(8, tm - strip * 8), rem = id - strip * 8 * tn;
  const int i0 = (strip * 8 + rem % sr) * T, j0 = (rem / sr) * T;
  string_gemm_block<T>(P, i0, j0, blockIdx.y);
}

// L0 R0 of two symmetric products (blockIdx.y: which), their tiles i <= j only.
template <int T>
__global__ __launch_bounds__(256, 2) void k_string_grams(GemmArgs A, GemmArgs B) {
  const GemmArgs& P = blockIdx.y ? B : A;
  const int tn = (P.n + T - 1) / T;
  int i = 0, id = blockIdx.x;
  while (i < tn && id >= tn - i) id -= tn - i++;
  if (i >= tn) return;
  string_gemm_block<T>(P, i * T, (i + id) * T, 0);
}

// ---------------------------------------------------------------------------
// One 16-column tile of G for the alpha row whose psi row is ps (LDS) and
// whose alpha operand entries are ra (LDS): acc[t] holds the 16 x 16 block
// of rows m0 + 16 t (the A slice sA [K8][W] is in LDS); column ib = c*16 + li
// (columns past nsb compute garbage that is never used).  The k-steps are
// unrolled by two with ping-pong registers: step s issues the alpha
// amplitude and beta table loads of later steps before its MFMAs.

template <int MT>
__device__ __forceinline__ void row_tile(double4_t (&acc)[MT], const double* __restrict__ sA,
                                         const double* __restrict__ ps, const int2* __restrict__ ra,
                                         const double* __restrict__ psi, const int2* __restrict__ rtb, int nsb,
                                         int ib, int kq, int li, int nsteps) {
  constexpr int W = MT * 16;
  const uint32_t ibc = (uint32_t)(ib < nsb ? ib : nsb - 1);
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = double4_t{0.0, 0.0, 0.0, 0.0};
  const uint32_t sb = 4u * (uint32_t)nsb;
  const uint32_t tb_i = (uint32_t)kq * (uint32_t)nsb + ibc;
  // slot 0: even steps, slot 1: odd steps
  int2 tb0 = rtb[tb_i], tb1 = rtb[tb_i + sb];
  int2 a = ra[kq];
  double xa0 = psi[(uint32_t)a.x + ibc];
  int ca0 = a.y;
  double xb0 = ps[tb0.x];
  int cb0 = tb0.y;
  tb0 = rtb[tb_i + 2 * sb];
  double xa1, xb1;
  int ca1, cb1;
  const double* arow = sA + (size_t)kq * W + li;
#pragma unroll
  for (int s = 0; s < nsteps; s += 2) {
    a = ra[(s + 1) * 4 + kq];
    xa1 = psi[(uint32_t)a.x + ibc];
    ca1 = a.y;
    xb1 = ps[tb1.x];
    cb1 = tb1.y;
    tb1 = rtb[tb_i + (uint32_t)(s + 3) * sb];
    __asm__ volatile("" ::: "memory");
    {
      const double b = (double)ca0 * xa0 + (double)cb0 * xb0;
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(arow[t * 16], b, acc[t], 0, 0, 0);
    }
    arow += 4 * W;
    a = ra[(s + 2) * 4 + kq];
    xa0 = psi[(uint32_t)a.x + ibc];
    ca0 = a.y;
    xb0 = ps[tb0.x];
    cb0 = tb0.y;
    tb0 = rtb[tb_i + (uint32_t)(s + 4) * sb];
    __asm__ volatile("" ::: "memory");
    {
      const double b = (double)ca1 * xa1 + (double)cb1 * xb1;
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(arow[t * 16], b, acc[t], 0, 0, 0);
    }
    arow += 4 * W;
  }
}

// Row kernel, staged form (deterministic): LDS = A slice [K8][W] | staged G
// tiles [waves][W][16] | psi rows [R][nsb] | alpha operand rows [R][K8 + 16].
// Per round every wave computes one tile; after a barrier each target adds
// its beta neighbours' staged values in neighbour-list order.
template <int MT>
__global__ __launch_bounds__(kRowThreads) void k_sigma_rows(
    const double* __restrict__ At, int kpad, int K4, int K8, int mgroups, const double* __restrict__ psi,
    const double* __restrict__ sin, int nsplit, double* __restrict__ sigma, double* __restrict__ partial,
    const int2* __restrict__ rta, const int2* __restrict__ rtb, const uint32_t* __restrict__ nbr,
    const int32_t* __restrict__ nbr_off, const uint8_t* __restrict__ nbr_tile, int nsa, int nsb, int R,
    double e0) {
  constexpr int W = MT * 16;
  extern __shared__ double smem[];
  __shared__ double red[kRowWaves];
  const int tpr = (nsb + 15) >> 4;
  const int RA = K8 + 16;
  double* sA = smem;
  double* sG = sA + (size_t)K8 * W;
  double* sPsi = sG + (size_t)kRowWaves * W * 16;
  int2* sRA = reinterpret_cast<int2*>(sPsi + (size_t)R * nsb);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, kq = lane >> 4, li = lane & 15;
  const int row0 = blockIdx.x * R;
  const int nr = min(R, nsa - row0);
  const int ntg = nr * nsb;
  const size_t base = (size_t)row0 * nsb;
  for (int i = tid; i < ntg; i += kRowThreads) sPsi[i] = psi[base + i];
  for (int i = tid; i < nr * RA; i += kRowThreads) {
    const int r = i / RA, k = i - r * RA;
    sRA[i] = rta[(size_t)k * nsa + row0 + r];
  }
  double tacc[kMaxTargets];
#pragma unroll
  for (int i = 0; i < kMaxTargets; ++i) tacc[i] = 0.0;
  const int ntiles = nr * tpr;
  const int nsteps = K8 / 4;
  for (int mg = 0; mg < mgroups; ++mg) {
    const int m0 = mg * W;
    __syncthreads();  // the previous m-group's reads of sA are done
    for (int i = tid; i < K8 * W; i += kRowThreads) {
      const int k = i / W, m = m0 + (i - k * W);
      sA[i] = (k < K4 && m < kpad) ? At[(size_t)k * kpad + m] : 0.0;
    }
    __syncthreads();
    for (int f0 = 0; f0 < ntiles; f0 += kRowWaves) {
      const int f = f0 + wave;
      if (f < ntiles) {
        const int r = f / tpr, c = f - r * tpr;
        double4_t acc[MT];
        row_tile<MT>(acc, sA, sPsi + (size_t)r * nsb, sRA + (size_t)r * RA, psi, rtb, nsb, c * 16 + li, kq, li,
                     nsteps);
        double* g = sG + (size_t)wave * W * 16 + li;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) g[(t * 16 + kq + 4 * q) * 16] = acc[t][q];
      }
      __syncthreads();
      // every target adds its beta neighbours' staged G_k values, by partner column
#pragma unroll
      for (int i = 0; i < kMaxTargets; ++i) {
        const int tau = tid + i * kRowThreads;
        if (tau >= ntg) break;
        const int r = tau / nsb, ib = tau - r * nsb;
        const int lo = max(f0, r * tpr), hi = min(f0 + kRowWaves, (r + 1) * tpr);
        if (lo >= hi) continue;
        const uint8_t* tl = nbr_tile + (size_t)ib * (tpr + 1);
        const int eb = nbr_off[ib];
        const int e0 = eb + tl[lo - r * tpr], e1 = eb + tl[hi - r * tpr];
        const int fb = r * tpr - f0;
        double v = tacc[i];
        for (int e = e0; e < e1; ++e) {
          const uint32_t x = nbr[e];
          const int jb = (int)(x & 0x3FFFu), k = (int)((x >> 14) & 0xFFu) - m0;
          if (k < 0 || k >= W) continue;
          const double gv = sG[((size_t)(fb + (jb >> 4)) * W + k) * 16 + (jb & 15)];
          v += (x >> 31) ? -gv : gv;
        }
        tacc[i] = v;
      }
      __syncthreads();
    }
  }
  const size_t dim = (size_t)nsa * nsb;
  double e = 0.0;
#pragma unroll
  for (int i = 0; i < kMaxTargets; ++i) {
    const int tau = tid + i * kRowThreads;
    if (tau >= ntg) break;
    double v = tacc[i] + e0 * sPsi[tau];
    for (int z = 0; z < nsplit; ++z) v += sin[(size_t)z * dim + base + tau];
    sigma[base + tau] = v;
    e += v * sPsi[tau];
  }
  for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
  if (lane == 0) red[wave] = e;
  __syncthreads();
  if (tid == 0) {
    double tsum = 0.0;
    for (int w = 0; w < kRowWaves; ++w) tsum += red[w];
    partial[blockIdx.x] = tsum;
  }
}

// One 128 x 64 tile of the string product L R (nsa x nk, nk x nsb) over the
// contraction range [kb, ke) for the fused sigma launch (512 threads: wave w
// owns rows 32 (w >> 1) and columns 32 (w & 1) as 2 x 2 MFMA tiles); the tile
// is added to sigma by global atomics and its <psi|.> partial returned
// (thread 0's value is the block's).  C: psi.
constexpr int kGemmRows = 128, kGemmCols = 64;

__device__ __forceinline__ double string_gemm_tile(int i0, int j0, int kb, int ke, const double* __restrict__ L,
                                                   int nk, const double* __restrict__ R,
                                                   const double* __restrict__ C, double* __restrict__ sigma, int nsa,
                                                   int nsb, double* smem, double* red) {
  // two buffers of L [16][128] | R [16][64], columns swizzled as in k_string_gemm
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, kq = lane >> 4, li = lane & 15;
  const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
  const bool idle = i0 + wi >= nsa || j0 + wj >= nsb;  // nothing of the wave's quarter is in the matrix
  double4_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = double4_t{0.0, 0.0, 0.0, 0.0};
  const int lk = t & 15, lr = t >> 4;  // L: column lk of rows lr + 32 j
  const int rk = t >> 5, rc = t & 31;  // R: row rk, columns rc + 32 j
  auto swz = [](int k) { return 16 * (k & 1) + 4 * ((k >> 1) & 3); };
  const int wl = lk * kGemmRows + (lr ^ swz(lk)), wr = 16 * kGemmRows + rk * kGemmCols + (rc ^ swz(rk));
  const int rd0 = li ^ swz(kq), rd1 = li ^ swz(4 + kq);
  uint32_t lofs[4], rofs[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) lofs[j] = ((uint32_t)min(lr + 32 * j, nsa - 1 - i0) * (uint32_t)nk + lk) * 8u;
#pragma unroll
  for (int j = 0; j < 2; ++j)
    rofs[j] = ((uint32_t)rk * (uint32_t)nsb + (uint32_t)min(rc + 32 * j, nsb - 1 - j0)) * 8u;
  double pl[4], pr[2];
  // slice at k; bl, br: bytes back to the last column / row for lanes past it
  auto load = [&](int k, uint32_t bl, uint32_t br) {
    const char* __restrict__ Lk = reinterpret_cast<const char*>(L + (size_t)i0 * nk + k);
    const char* __restrict__ Rk = reinterpret_cast<const char*>(R + (size_t)k * nsb + j0);
#pragma unroll
    for (int j = 0; j < 4; ++j) pl[j] = *reinterpret_cast<const double*>(Lk + (lofs[j] - bl));
#pragma unroll
    for (int j = 0; j < 2; ++j) pr[j] = *reinterpret_cast<const double*>(Rk + (rofs[j] - br));
  };
  constexpr int kBuf = 16 * (kGemmRows + kGemmCols);
  auto store = [&](int buf) {
    double* sb = smem + buf * kBuf;
#pragma unroll
    for (int j = 0; j < 4; ++j) sb[wl + 32 * j] = pl[j];
#pragma unroll
    for (int j = 0; j < 2; ++j) sb[wr + 32 * j] = pr[j];
  };
  auto products = [&](int buf) {
    const double* sb = smem + buf * kBuf;
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
      const int c = (kk & 4) ? rd1 : rd0;  // 16 columns from wi (wj); c ^ 16: the next 16
      const double* l = sb + (kk + kq) * kGemmRows + wi;
      const double* r = sb + 16 * kGemmRows + (kk + kq) * kGemmCols + wj;
      const double a0 = l[c], a1 = l[c ^ 16], b0 = r[c], b1 = r[c ^ 16];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
  };
  const int kf = kb + ((ke - kb) & ~15);  // end of the whole slices
  if (kb < kf) {
    load(kb, 0, 0);
    store(0);
    lds_barrier();
    int buf = 0;
    for (int k = kb; k < kf; k += 16, buf ^= 1) {
      if (k + 16 < kf) load(k + 16, 0, 0);
      if (!idle) products(buf);
      if (k + 16 < kf) store(buf ^ 1);
      lds_barrier();
    }
  }
  if (kf < ke) {
    const int pl_over = kf + lk - (ke - 1), pr_over = kf + rk - (ke - 1);
    load(kf, 8u * (uint32_t)max(0, pl_over), 8u * (uint32_t)max(0, pr_over) * (uint32_t)nsb);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (pl_over > 0) pl[j] = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (pr_over > 0) pr[j] = 0.0;
    store(0);
    lds_barrier();
    if (!idle) products(0);
  }
  double e = 0.0;
  if (!idle) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      double pc[2][4];  // psi of the tile, all loads first
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int I = i0 + wi + a * 16 + kq + 4 * r, c = j0 + wj + b * 16 + li;
          pc[b][r] = C[(size_t)min(I, nsa - 1) * nsb + min(c, nsb - 1)];
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int I = i0 + wi + a * 16 + kq + 4 * r, c = j0 + wj + b * 16 + li;
          if (I < nsa && c < nsb) {
            unsafeAtomicAdd(sigma + (size_t)I * nsb + c, acc[a][b][r]);
            e += acc[a][b][r] * pc[b][r];
          }
        }
    }
  }
  for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
  if (lane == 0) red[wave] = e;
  __syncthreads();
  double tsum = 0.0;
  if (t == 0)
    for (int w = 0; w < kRowWaves; ++w) tsum += red[w];
  return tsum;
}

// Row kernel over the alpha excitations that do not vanish: LDS = A slice
// [npair + 1][W] (doubled, the operand's factor 2; row npair is zero) | sigma
// rows [R][nsb] | lists [R][KA] of the row's nonzero E+a_k' (k_alpha_list).
// Waves take 16-column tiles independently.  The amplitudes of a step are
// loaded kAhead steps before its products, those of a tile's first steps before
// the LDS adds of the previous tile.  Each output G_k[I_a, J_b] goes to the sigma
// row at P_k(J_b) (E+b_k is symmetric) by an LDS atomic add.  The order of those
// adds varies between runs, so results agree to rounding, not bit for bit.
// FUSED: the launch also holds the tiles of Ma C and C Mb as extra blocks after
// the row blocks (they fill the CUs the last row blocks leave idle); every
// block adds its part to sigma (zeroed beforehand) by global atomics.  Else the
// nsplit partial products at sin are added and sigma written.  blockIdx.y: the
// instance of a group (zero strides: one instance).
constexpr int kAhead = 4;
constexpr int kTrash = 64;  // doubles past each sigma row in LDS: targets of outputs that vanish

struct RowArgs {
  const double *At, *psi, *sin, *Ma, *Mb;
  double *sigma, *partial;
  const int2* list;
  const int32_t* rtc;
  int kpad, mgroups, npair, nsteps, KA, nsplit, nsa, nsb, nsp, R, xcd, nrowblk, ngemm_a, kchunk, kchunk_b;
  int64_t A_stride, Ma_stride, Mb_stride, vec_stride, part_stride;
};

// Threads of a block: with two blocks on a CU four waves per SIMD; alone on it
// three (its registers allow no more): (14e,14o) 2.84 -> 2.76 ms against two.
template <bool FUSED>
constexpr int kListThreads = FUSED ? 512 : 768;

template <int MT, bool FUSED>
__global__ __launch_bounds__(kListThreads<FUSED>) __attribute__((amdgpu_waves_per_eu(FUSED ? 4 : 3, 8))) void
k_sigma_rows_list(RowArgs P) {
  constexpr int kThreads = kListThreads<FUSED>, kWaves = kThreads / 64;
  constexpr int W = MT * 16;
  extern __shared__ double smem[];
  __shared__ double red[kWaves];
  const double* __restrict__ At = P.At + blockIdx.y * P.A_stride;
  const double* __restrict__ psi = P.psi + blockIdx.y * P.vec_stride;
  double* __restrict__ sigma = P.sigma + blockIdx.y * P.vec_stride;
  double* __restrict__ partial = P.partial + blockIdx.y * P.part_stride;
  const int nsa = P.nsa, nsb = P.nsb, npair = P.npair, KA = P.KA;
  if (FUSED && (int)blockIdx.x >= P.nrowblk) {
    int g = (int)blockIdx.x - P.nrowblk;
    const bool beta = g >= P.ngemm_a;
    if (beta) g -= P.ngemm_a;
    const int tn = (nsb + kGemmCols - 1) / kGemmCols, tm = (nsa + kGemmRows - 1) / kGemmRows;
    const int z = g / (tm * tn), rem = g - z * (tm * tn);
    const int nk = beta ? nsb : nsa, kc = beta ? P.kchunk_b : P.kchunk, kb = z * kc;
    const double* L = beta ? psi : P.Ma + blockIdx.y * P.Ma_stride;
    const double* R = beta ? P.Mb + blockIdx.y * P.Mb_stride : psi;
    const double e = string_gemm_tile((rem / tn) * kGemmRows, (rem % tn) * kGemmCols, kb, min(nk, kb + kc), L, nk, R,
                                      psi, sigma, nsa, nsb, smem, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = e;
    return;
  }
  double* sA = smem;
  double* sAcc = sA + (size_t)(npair + 1) * W;
  const int SR = nsb + kTrash;
  int2* sL = reinterpret_cast<int2*>(sAcc + (size_t)P.R * SR);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kq = lane >> 4, li = lane & 15;
  // with xcd, XCD x (workgroups go to the eight XCDs round robin) takes a
  // contiguous range of row groups, whose alpha partner rows overlap in its L2
  int blk = blockIdx.x;
  const int nrb = FUSED ? P.nrowblk : (int)gridDim.x;
  if (P.xcd && blk < (nrb & ~7)) {  // the remainder past a multiple of 8 keeps its order
    const int q = nrb >> 3, x = blk & 7;
    blk = x * q + (blk >> 3);
  }
  const int row0 = blk * P.R;
  const int nr = min(P.R, nsa - row0);
  const int ntg = nr * nsb;
  const size_t base = (size_t)row0 * nsb;
  for (int i = tid; i < nr * SR; i += kThreads) sAcc[i] = 0.0;
  for (int i = tid; i < nr * KA; i += kThreads) {
    const int2 e = P.list[(size_t)row0 * KA + i];
    // byte offset of the partner row; half the byte offset of the row of A
    sL[i] = make_int2(e.x * 8, (e.y & 0xffff) * (W * 4) | (e.y & (int)0x80000000));
  }
  const int tpr = (nsb + 15) >> 4;
  const int ntiles = nr * tpr;
  for (int mg = 0; mg < P.mgroups; ++mg) {
    const int m0 = mg * W;
    __syncthreads();  // the previous m-group's reads of sA are done
    constexpr int kB = 4;  // A elements in flight per thread
    for (int i0 = tid; i0 < (npair + 1) * W; i0 += kB * kThreads) {
      double v[kB];
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int i = i0 + b * kThreads, k = min(i / W, npair), m = m0 + i % W;
        v[b] = At[(size_t)k * P.kpad + min(m, npair)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int i = i0 + b * kThreads, k = i / W, m = m0 + i % W;
        if (k <= npair) sA[i] = m < npair && k < npair ? 2.0 * v[b] : 0.0;
      }
    }
    __syncthreads();
    const int2* __restrict__ ls = nullptr;
    uint32_t col = 0;  // byte offset of the lane's column
    const char* __restrict__ psib = reinterpret_cast<const char*>(psi);
    const char* sAl = reinterpret_cast<const char*>(sA + li);
    auto amp = [&](int2 e) { return *reinterpret_cast<const double*>(psib + ((uint32_t)e.x + col)); };
    double x[kAhead];
    int ky[kAhead];
    int2 en[kAhead];  // the entries of the loads after those in flight
    // the first kAhead steps' amplitudes of tile f
    auto head = [&](int f) {
      const int r = f / tpr, c = f - r * tpr;
      ls = sL + (size_t)r * KA + kq;
      col = 8u * (uint32_t)min(c * 16 + li, nsb - 1);
#pragma unroll
      for (int d = 0; d < kAhead; ++d) {
        const int2 e = ls[4 * d];
        en[d] = ls[4 * (d + kAhead)];
        ky[d] = e.y;
        x[d] = amp(e);
      }
    };
    if (wave < ntiles) head(wave);
    for (int f = wave; f < ntiles; f += kWaves) {
      const int r = f / tpr;
      char* acc_row = reinterpret_cast<char*>(sAcc + (size_t)r * SR);
      double4_t acc[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = double4_t{0.0, 0.0, 0.0, 0.0};
      // step: the A fragments of the next step are read before the products
      double a[2][MT];
      auto frag = [&](int k, int e) {
        const double* arow = reinterpret_cast<const double*>(sAl + ((uint32_t)k << 1));
#pragma unroll
        for (int t = 0; t < MT; ++t) a[e][t] = arow[t * 16];
      };
      auto mul = [&](int d, int e) {
        const double b = flip(x[d], ky[d]);
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e][t], b, acc[t], 0, 0, 0);
      };
      frag(ky[0], 0);
      int st = 0;
      for (; st + kAhead < P.nsteps; st += kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
          frag(d + 1 < kAhead ? ky[d + 1] : ky[0], (d + 1) & 1);
          __builtin_amdgcn_sched_barrier(0);
          mul(d, d & 1);
          ky[d] = en[d].y;
          x[d] = amp(en[d]);
          en[d] = ls[4 * (2 * kAhead + d)];
        }
        ls += 4 * kAhead;
      }
      // LDS targets of the tile's 4 MT outputs
      int32_t tb[MT][4];
      const int32_t* __restrict__ tbase = P.rtc + (size_t)m0 * P.nsp + (f - r * tpr) * 16;
      const uint32_t tbo = (uint32_t)(kq * P.nsp + li) * 4u;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          tb[t][q] = *reinterpret_cast<const int32_t*>(
              reinterpret_cast<const char*>(tbase + (t * 16 + 4 * q) * P.nsp) + tbo);
      // the last 1 to kAhead steps
#pragma unroll
      for (int d = 0; d < kAhead; ++d) {
        if (st + d >= P.nsteps) break;
        if (d + 1 < kAhead) frag(ky[d + 1], (d + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        mul(d, d & 1);
      }
      // the next tile's first amplitudes are in flight during the LDS adds
      if (f + kWaves < ntiles) head(f + kWaves);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          atomicAdd(reinterpret_cast<double*>(acc_row + ((uint32_t)tb[t][q] << 1)), flip(acc[t][q], tb[t][q]));
    }
  }
  __syncthreads();
  const size_t dim = (size_t)nsa * nsb;
  double e = 0.0;
  constexpr int kB = 4;  // amplitudes in flight per thread
  for (int r = 0; r < nr; ++r)
    for (int c0 = tid; c0 < nsb; c0 += kB * kThreads) {
      const size_t at = base + (size_t)r * nsb;
      double x[kB], v[kB];
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int c = min(c0 + b * kThreads, nsb - 1);
        x[b] = psi[at + c];
        v[b] = sAcc[r * SR + c];
      }
      if (!FUSED)
        for (int z = 0; z < P.nsplit; ++z) {
#pragma unroll
          for (int b = 0; b < kB; ++b) v[b] += P.sin[(size_t)z * dim + at + min(c0 + b * kThreads, nsb - 1)];
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int c = c0 + b * kThreads;
        if (c < nsb) {
          if (FUSED) unsafeAtomicAdd(sigma + at + c, v[b]);
          else sigma[at + c] = v[b];
          e += v[b] * x[b];
        }
      }
    }
  for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
  if (lane == 0) red[wave] = e;
  __syncthreads();
  if (tid == 0) {
    double tsum = 0.0;
    for (int w = 0; w < kWaves; ++w) tsum += red[w];
    partial[blockIdx.x] = tsum;
  }
}

struct RowPlan {
  int mt, mgroups, R, ngroups, nsplit, kchunk;
  bool fused;
  bool list;  // k_sigma_rows_list, else k_sigma_rows
  int ngemm_a, ngemm_b, kchunk_b;  // fused: tile blocks of Ma C and C Mb after the row blocks
  size_t lds;
};

// Nonvanishing E+a_k' per alpha string, in 4-deep k-steps, and the entries of
// the list: whole groups of kAhead steps are read up to two groups ahead.
int list_steps(const Space& s) { return (s.na * (s.n - s.na) + s.na + 3) / 4; }
int list_entries(const Space& s) { return 4 * (rup(list_steps(s), kAhead) + 2 * kAhead); }

// LDS of one k_string_ham block (bytes).
size_t string_ham_lds(const Space& s, int nstr, int nel) {
  return 2 * (size_t)rup(nstr, 8) + 2 * (size_t)rup(s.npair + 1, 8) + 4 * (size_t)rup(s.npair, 2) +
         8 * (size_t)s.npair * (1 + nel * (s.n - nel));
}

// Whether the list form can run: 32-bit byte offsets into psi, and the matrix of
// Hb built in LDS.
bool list_form(const Space& s) {
  return s.dim < ((int64_t)1 << 29) && string_ham_lds(s, s.nsb, s.nb) <= kLdsMax;
}

int row_k8(const Space& s) { return rup(s.npair + 1, 8); }  // contraction rows: two 4-deep k-steps per iteration

// Dynamic LDS of one block (bytes): list form A slice | sigma rows | lists;
// staged form A slice | G tiles | psi rows | alpha operand rows.
size_t row_lds(const Space& s, int mt, int R, bool list) {
  if (list)
    return 8 * ((size_t)(s.npair + 1) * mt * 16 + (size_t)R * (s.nsb + kTrash) + (size_t)R * list_entries(s));
  const int K8 = row_k8(s);
  const size_t W = (size_t)mt * 16;
  return 8 * ((size_t)K8 * W + (size_t)kRowWaves * W * 16 + (size_t)R * s.nsb + (size_t)R * (K8 + 16));
}

// Spaces the list form takes: a row of psi and one of sigma fit a block's LDS
// beside a 16-row tile of A (to 15 orbitals, and 16 with up to 6 or from 10 beta
// electrons; the rest runs the two-kernel path).
bool list_fits(const Space& s) {
  const int K8 = row_k8(s);
  return list_form(s) && 8 * ((size_t)K8 * 16 + 2 * (size_t)s.nsb + K8 + 16) <= kLdsMax;
}

// The space's kernel shape choices (sq_sigma_configure) override these
// defaults: rows per block, string product split, and the deterministic (staged)
// form instead of the list form (default: SQ_SIGMA_DETERMINISTIC, else 0).
bool row_deterministic(const SigmaShape& shape) {
  if (shape.det >= 0) return shape.det != 0;
  static int v = -1;
  if (v < 0) v = env_int("SQ_SIGMA_DETERMINISTIC", 0) != 0 ? 1 : 0;
  return v == 1;
}

// The contraction split of the separate string products
// whose 128 x 128 tiles take the fewest block rounds (two blocks on each of 256
// CUs) per split: (14e,14o), 729 tiles: 2 rounds whole, 3 rounds of halves,
// 3.40 -> 2.64 ms.  More than one partial product only where they stay within
// the scratch memory of the no-allocation entry point.
int string_gemm_split(const Space& s) {
  const int64_t tiles = (int64_t)((s.nsa + 127) / 128) * ((s.nsb + 127) / 128);
  int best = 1;
  int64_t rounds = (tiles + 511) / 512;
  for (int z = 2; z <= 4; ++z) {
    const int64_t r = (tiles * z + 511) / 512;
    if (r * best < rounds * z) best = z, rounds = r;
  }
  const int64_t limit = ((int64_t)8 << 20) - s.nsa;
  return s.dim <= limit && best * s.dim > limit ? 1 : best;
}

// Kernel shape: the m-tile group (largest that fits, then balanced) and the
// rows per block R.  Staged form: R with the fewest block-rounds on 256 CUs
// (one block per CU).  List form: the smallest R that gives every wave a tile
// (more, smaller blocks), but two rows at least, which halves the staging of A
// per row: 10 orbitals in groups 1600 -> 1506 us, (11e,11o) 205 ->
// 186, (12e,12o) 437 -> 424 (energy and gradient); more rows gain no more.  A
// launch of many instances has blocks enough: four rows and the string products
// unsplit (a quarter of the atomic adds), 256 instances 1283 -> 1206 us.  But no
// more rows than leave two blocks on a CU where the single instance has two
// ((12e,12o): three), so that the fused form, which groups need, does not depend
// on n.
constexpr int kManyInst = 8;

bool row_plan(const Space& s, const SigmaShape& shape, RowPlan* out, int n) {
  if (s.dim == 0 || s.nsb > 16384 || s.npair + 1 > 255 || s.dim >= ((int64_t)1 << 31)) return false;
  const bool list = !row_deterministic(shape);
  if (!(list ? list_fits(s) : row_lds(s, 1, 1, false) <= kLdsMax)) return false;
  const int mt_total = rup(list ? s.npair : s.npair + 1, 16) / 16;
  int mt = std::min(mt_total, kMaxMt);
  while (mt > 1 && row_lds(s, mt, 1, list) > kLdsMax) --mt;
  const int mgroups = (mt_total + mt - 1) / mt;
  mt = (mt_total + mgroups - 1) / mgroups;
  const int tpr = (s.nsb + 15) / 16;
  int bestR = 0;
  if (list) {
    auto rows = [&](int least) {
      int R = std::max(1, std::min(s.nsa, std::max(least, (kRowWaves + tpr - 1) / tpr)));
      while (R > 1 && row_lds(s, mt, R, true) > kLdsMax) --R;
      return R;
    };
    bestR = rows(2);
    if (n >= kManyInst) {
      const int one = bestR;
      bestR = rows(4);
      while (bestR > one && 2 * row_lds(s, mt, bestR, true) > kLdsMax) --bestR;
    }
  } else {
    int64_t best = -1;
    for (int R = 1; R <= 64 && R <= s.nsa; ++R) {
      if (row_lds(s, mt, R, false) > kLdsMax) break;
      if ((int64_t)R * s.nsb > (int64_t)kMaxTargets * kRowThreads) break;
      const int64_t groups = (s.nsa + R - 1) / R;
      const int64_t cost = ((groups + 255) / 256) * (((int64_t)R * tpr + kRowWaves - 1) / kRowWaves);
      if (best < 0 || cost < best) {
        best = cost;
        bestR = R;
      }
    }
  }
  if (bestR == 0) return false;
  if (shape.R > 0) {
    const int R = shape.R;
    if (R <= s.nsa && row_lds(s, mt, R, list) <= kLdsMax &&
        (list || (int64_t)R * s.nsb <= (int64_t)kMaxTargets * kRowThreads))
      bestR = R;
  }
  out->mt = mt;
  out->mgroups = mgroups;
  out->R = bestR;
  out->list = list;
  out->ngroups = (s.nsa + bestR - 1) / bestR;
  // contraction split of the string products (Ma C and, in the list form, C Mb
  // in one joined range) that run as a launch of their own
  const int joined = s.nsa + (list ? s.nsb : 0);
  auto chunk = [](int len, int nsplit) {
    nsplit = std::max(1, std::min({nsplit, kMaxSplit, (len + 15) / 16}));
    return rup((len + nsplit - 1) / nsplit, 16);
  };
  int nsplit = shape.nsplit;
  if (nsplit <= 0) nsplit = list ? string_gemm_split(s) : (s.nsa >= 2048 ? 1 : 2);
  out->kchunk = chunk(joined, nsplit);
  out->nsplit = (joined + out->kchunk - 1) / out->kchunk;
  out->lds = row_lds(s, mt, bestR, list);
  // fused form: the tiles of the string products (128 x 64, each contraction
  // split in four: (12e,12o) 481, 441, 432, 424 us an energy and gradient for
  // 1 to 4, 450 for 8) as extra blocks of the row launch, where two row blocks
  // share a CU (the tile blocks then fill the slots the last row blocks
  // leave); with one row block per CU (14 orbitals) the tile blocks would run
  // at that block's LDS footprint, so the products stay separate
  static const int fuse_env = env_int("SQ_SIGMA_FUSED_GEMM", 1);
  out->fused = list && fuse_env != 0 && 2 * out->lds <= kLdsMax && mt <= kMaxFusedMt;
  out->ngemm_a = out->ngemm_b = out->kchunk_b = 0;
  if (out->fused) {
    const int split = shape.nsplit > 0 ? shape.nsplit : n >= kManyInst ? 1 : 4;
    out->kchunk = chunk(s.nsa, split);
    out->kchunk_b = chunk(s.nsb, split);
    const int tiles = ((s.nsa + kGemmRows - 1) / kGemmRows) * ((s.nsb + kGemmCols - 1) / kGemmCols);
    out->nsplit = (s.nsa + out->kchunk - 1) / out->kchunk;
    out->ngemm_a = tiles * out->nsplit;
    out->ngemm_b = tiles * ((s.nsb + out->kchunk_b - 1) / out->kchunk_b);
    const size_t glds = 8 * (size_t)2 * 16 * (kGemmRows + kGemmCols);
    out->lds = std::max(out->lds, glds);
  }
  return true;
}

bool row_plan(const Space& s, RowPlan* out) { return row_plan(s, s.sig, out, 1); }

bool rows_enabled() {
  static int v = -1;
  if (v < 0) v = env_int("SQ_SIGMA_ROWS", 1) != 0 ? 1 : 0;
  return v == 1;
}

}  // namespace

bool sigma_deterministic(const Space& s) { return row_deterministic(s.sig); }

void string_grams(const double* C, const double* Ct, double* rho_a, double* rho_b, int nsa, int nsb, hipStream_t st) {
  const GemmArgs A{C, Ct, nullptr, nullptr, rho_a, nsa, nsa, nsb, 0, nsb};
  const GemmArgs B{Ct, C, nullptr, nullptr, rho_b, nsb, nsb, nsa, 0, nsa};
  const double flops = (double)nsa * nsb * (nsa + nsb);
  const double bytes = 8.0 * ((double)nsa * nsb + (double)nsa * nsa + (double)nsb * nsb);
  const int t = (std::max(nsa, nsb) + 63) / 64;
  SQ_PROF(PC_ALPHA_GEMM, st, bytes, flops,
          (k_string_grams<64><<<dim3(t * (t + 1) / 2, 2), 256, 0, st>>>(A, B)));
}

bool row_sigma_applies(const Space& s) {
  RowPlan pl;
  return rows_enabled() && s.d_rtb != nullptr && row_plan(s, &pl);
}

// doubles of workspace: string product partials [nsplit][dim] | block energy
// partials [ngroups], sized for the largest shape (nsplit = kMaxSplit,
// ngroups = nsa) | scalars [64] at the end.
int64_t row_sigma_work_doubles(const Space& s) {
  return (int64_t)kMaxSplit * s.dim + s.nsa + 64;
}

namespace {

// list[s]: the E+a_k' that do not vanish on alpha string s (k' ascending) as
// {partner row * nsb, k' | negative << 31}; the rest {own row, npair}, whose
// row of A is zero.
__global__ void k_alpha_list(int npair, int nsa, int nsb, int KA, const int32_t* __restrict__ aexc,
                             int2* __restrict__ list) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsa) return;
  int2* out = list + (size_t)s * KA;
  int m = 0, k = 0;
  for (int p = 0; k < npair; ++p)
    for (int q = 0; q <= p; ++q, ++k) {
      const int32_t x = aexc[(size_t)k * nsa + s];
      if (x == 0) continue;
      out[m++] = p == q ? make_int2(s * nsb, k) : make_int2((abs(x) - 1) * nsb, k | (x < 0 ? (int)0x80000000 : 0));
    }
  for (; m < KA; ++m) out[m] = make_int2(s * nsb, npair);
}

// rtc[k][s] (k < a multiple of 16, s < nsp, a multiple of 16): half the byte
// offset in the LDS sigma row of the partner of beta string s under E+b_k |
// negative << 31; where there is none, of one of the kTrash doubles past it.
__global__ void k_beta_partners(int npair, int nsb, int nsp, const int2* __restrict__ rtb, int32_t* __restrict__ rtc) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
  if (s >= nsp) return;
  int32_t v = 4 * (nsb + 16 * (k & 3) + (s & 15));
  if (k < npair && s < nsb) {
    const int2 e = rtb[(size_t)k * nsb + s];
    if (e.y != 0) v = 4 * e.x | (e.y < 0 ? (int)0x80000000 : 0);
  }
  rtc[(size_t)k * nsp + s] = v;
}

}  // namespace

void build_row_tables(Space& s) {
  RowPlan pl;
  if (!row_plan(s, &pl)) return;
  const int K8 = row_k8(s);
  const int tpr = (s.nsb + 15) / 16;
  SQ_HIP(hipMalloc(&s.d_rta, sizeof(int2) * (size_t)(K8 + 16) * s.nsa));
  SQ_HIP(hipMalloc(&s.d_rtb, sizeof(int2) * (size_t)(K8 + 32) * s.nsb));
  k_row_tables<<<dim3((s.nsa + 255) / 256, K8 + 16), 256>>>(s.npair, s.nsa, s.nsb, 1, s.d_aexc, s.d_rta);
  SQ_HIP(hipGetLastError());
  k_row_tables<<<dim3((s.nsb + 255) / 256, K8 + 32), 256>>>(s.npair, s.nsb, s.nsb, 0, s.d_bexc, s.d_rtb);
  SQ_HIP(hipGetLastError());
  if (list_form(s)) {
    const int KA = list_entries(s);
    SQ_HIP(hipMalloc(&s.d_alist, sizeof(int2) * (size_t)KA * s.nsa));
    k_alpha_list<<<(s.nsa + 255) / 256, 256>>>(s.npair, s.nsa, s.nsb, KA, s.d_aexc, s.d_alist);
    SQ_HIP(hipGetLastError());
    // rows for every m-group (mt of them cover rup(npair, 16) rows, rounded up)
    const int rows = rup(s.npair, 16) + 16 * kMaxMt, nsp = rup(s.nsb, 16);
    SQ_HIP(hipMalloc(&s.d_rtc, sizeof(int32_t) * (size_t)rows * nsp));
    k_beta_partners<<<dim3((nsp + 255) / 256, rows), 256>>>(s.npair, s.nsb, nsp, s.d_rtb, s.d_rtc);
    SQ_HIP(hipGetLastError());
  }
  int32_t* cnt = nullptr;
  SQ_HIP(hipMalloc(&cnt, sizeof(int32_t) * s.nsb));
  k_nbr_count<<<(s.nsb + 255) / 256, 256>>>(s.npair, s.nsb, s.d_bexc, cnt);
  SQ_HIP(hipGetLastError());
  std::vector<int32_t> h(s.nsb), off(s.nsb + 1, 0);
  SQ_HIP(hipMemcpy(h.data(), cnt, sizeof(int32_t) * s.nsb, hipMemcpyDeviceToHost));
  for (int i = 0; i < s.nsb; ++i) off[i + 1] = off[i] + h[i];
  (void)hipFree(cnt);
  SQ_HIP(hipMalloc(&s.d_nbr_off, sizeof(int32_t) * (s.nsb + 1)));
  SQ_HIP(hipMemcpy(s.d_nbr_off, off.data(), sizeof(int32_t) * (s.nsb + 1), hipMemcpyHostToDevice));
  SQ_HIP(hipMalloc(&s.d_nbr, sizeof(uint32_t) * std::max(off[s.nsb], 1)));
  SQ_HIP(hipMalloc(&s.d_nbr_tile, (size_t)s.nsb * (tpr + 1)));
  k_nbr_fill<<<(s.nsb + 255) / 256, 256>>>(s.npair, s.nsb, tpr, s.d_bexc, s.d_nbr_off, s.d_nbr, s.d_nbr_tile);
  SQ_HIP(hipGetLastError());
  SQ_HIP(hipDeviceSynchronize());
}

void free_row_tables(Space& s) {
  for (void* p : {(void*)s.d_rta, (void*)s.d_rtb, (void*)s.d_alist, (void*)s.d_rtc, (void*)s.d_nbr, (void*)s.d_nbr_off, (void*)s.d_nbr_tile})
    if (p) (void)hipFree(p);
  s.d_rta = s.d_rtb = s.d_alist = nullptr;
  s.d_rtc = nullptr;
  s.d_nbr = nullptr;
  s.d_nbr_off = nullptr;
  s.d_nbr_tile = nullptr;
}

// Ma and (where the list form applies) Mb, the matrices of Ha and Hb over
// strings with half of e_core on each diagonal, for a Hamiltonian whose
// coefficient matrix is already on the device; one matrix where both spins
// have the same strings.
void build_string_hams(const Space& s, Hamiltonian& H) {
  if (s.d_rtb == nullptr || s.nsa == 0) return;
  auto build = [&](int nstr, int nel, const int32_t* exc, double** out) {
    SQ_HIP(hipMalloc(out, sizeof(double) * (size_t)nstr * nstr));
    const size_t lds = string_ham_lds(s, nstr, nel);
    SQ_CHECK(lds <= kLdsMax, SQ_ERR_ARG, "string Hamiltonian block does not fit in LDS");
    allow_lds(k_string_ham, lds);
    k_string_ham<<<nstr, 256, lds>>>(nstr, s.npair, H.kpad, exc, H.d_A, 0.5 * H.e_core, *out);
    SQ_HIP(hipGetLastError());
  };
  build(s.nsa, s.na, s.d_aexc, &H.d_Ma);
  if (list_form(s) && s.na != s.nb) build(s.nsb, s.nb, s.d_bexc, &H.d_Mb);
  SQ_HIP(hipDeviceSynchronize());
}

void free_string_hams(Hamiltonian& H) {
  if (H.d_Ma) (void)hipFree(H.d_Ma);
  if (H.d_Mb) (void)hipFree(H.d_Mb);
  H.d_Ma = H.d_Mb = nullptr;
}

namespace {

// rocBLAS handle of the current device, created on first use and kept until
// the process ends (creation allocates the library's workspace).
rocblas_handle blas_handle() {
  static std::mutex mu;
  static std::map<int, rocblas_handle> handles;
  int dev = 0;
  SQ_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  auto it = handles.find(dev);
  if (it != handles.end()) return it->second;
  rocblas_handle h = nullptr;
  SQ_CHECK(rocblas_create_handle(&h) == rocblas_status_success, SQ_ERR_HIP, "rocblas_create_handle failed");
  handles[dev] = h;
  return h;
}

// k_sigma_rows_list for n instances at the given strides (fused: sigma zeroed
// here unless it is already, and the string products' tiles in the launch; else the nsplit products
// at sin added).
void rows_list_launch(const Space& s, const RowPlan& pl, const double* A, int64_t A_stride, int kpad, const double* Ma,
                      int64_t Ma_stride, const double* Mb, int64_t Mb_stride, const double* psi, const double* sin,
                      int nsplit, double* sigma, double* partial, int n, bool zeroed, hipStream_t st) {
  static const int xcd = env_int("SQ_ROWS_XCD", 1) != 0 ? 1 : 0;
  RowArgs P{};
  P.At = A, P.psi = psi, P.sin = sin, P.Ma = Ma, P.Mb = Mb, P.sigma = sigma, P.partial = partial;
  P.list = s.d_alist, P.rtc = s.d_rtc;
  P.kpad = kpad, P.mgroups = pl.mgroups, P.npair = s.npair, P.nsteps = list_steps(s), P.KA = list_entries(s);
  P.nsplit = nsplit, P.nsa = s.nsa, P.nsb = s.nsb, P.nsp = rup(s.nsb, 16), P.R = pl.R, P.xcd = xcd, P.nrowblk = pl.ngroups;
  P.ngemm_a = pl.ngemm_a, P.kchunk = pl.kchunk, P.kchunk_b = pl.kchunk_b;
  const int nblk = pl.ngroups + pl.ngemm_a + pl.ngemm_b;
  P.A_stride = A_stride, P.Ma_stride = Ma_stride, P.Mb_stride = Mb_stride, P.vec_stride = s.dim, P.part_stride = nblk;
  const double rows = 2.0 * (double)s.npair * 4.0 * list_steps(s) * (double)s.dim;
  const double flops = n * (rows + (pl.fused ? 2.0 * (double)s.dim * (s.nsa + s.nsb) : 0.0));
  const double bytes = 8.0 * (double)s.dim * n * (pl.fused ? 3 : 2 + nsplit);
  if (pl.fused && !zeroed) {
    const int64_t total = (int64_t)n * s.dim;
    k_zero<<<(unsigned)std::min<int64_t>((total + 255) / 256, 16384), 256, 0, st>>>(sigma, total);
    SQ_HIP(hipGetLastError());
  }
  auto go = [&](auto kernel) {
    allow_lds(kernel, pl.lds);
    SQ_PROF(PC_SIGMA_ROWS, st, bytes, flops, kernel<<<dim3(nblk, n), pl.fused ? kListThreads<true> : kListThreads<false>, pl.lds, st>>>(P));
  };
  switch (pl.mt) {
#define SQ_RL(MT)                                                                       \
  case MT:                                                                              \
    if (!pl.fused) go(k_sigma_rows_list<MT, false>);                                    \
    else if constexpr (MT <= kMaxFusedMt) go(k_sigma_rows_list<MT, true>);              \
    break;
    SQ_RL(1) SQ_RL(2) SQ_RL(3) SQ_RL(4) SQ_RL(5) SQ_RL(6) SQ_RL(7) SQ_RL(8) SQ_RL(9)
#undef SQ_RL
    default:
      throw Error{SQ_ERR_ARG, "unsupported orbital count for the row sigma"};
  }
}

}  // namespace

// sigma = H psi and the block partials of <psi|sigma> (*partial_out, the
// count is returned).  The full form's Ma C is a plain dense GEMM and goes to
// rocBLAS unless allow_library is false (the no-allocation entry point) or
// SQ_ALPHA_GEMM_LIB=0: 66.5 TFLOP/s on 3432^3 against 62 for k_string_gemm.
int64_t row_sigma(const Space& s, const Hamiltonian& H, const double* psi, double* sigma, double* work,
                  double** partial_out, hipStream_t st, bool allow_library, bool zeroed) {
  RowPlan pl;
  SQ_CHECK(row_plan(s, &pl) && H.d_Ma, SQ_ERR_ARG, "row sigma does not apply to this space");
  SQ_CHECK(pl.nsplit <= kMaxSplit && pl.ngroups <= s.nsa, SQ_ERR_ARG, "row sigma shape exceeds its workspace");
  SQ_CHECK(!pl.fused || pl.ngroups + pl.ngemm_a + pl.ngemm_b <= row_sigma_work_doubles(s) - 64, SQ_ERR_ARG,
           "row sigma shape exceeds its workspace");
  const double* Mb = H.d_Mb ? H.d_Mb : H.d_Ma;
  if (pl.fused) {
    *partial_out = work;
    rows_list_launch(s, pl, H.d_A, 0, H.kpad, H.d_Ma, 0, Mb, 0, psi, nullptr, 0, sigma, work, 1, zeroed, st);
    return (int64_t)pl.ngroups + pl.ngemm_a + pl.ngemm_b;
  }
  double* sinp = work;
  double* partial = work + (size_t)pl.nsplit * s.dim;
  *partial_out = partial;
  int nsplit = pl.nsplit;  // partial products the row kernels add
  {
    static const int lib_env = env_int("SQ_ALPHA_GEMM_LIB", 1);
    const double flops = 2.0 * (double)s.dim * s.nsa, flops_b = pl.list ? 2.0 * (double)s.dim * s.nsb : 0.0;
    GemmArgs G{H.d_Ma, psi, psi, Mb, sinp, s.nsa, s.nsb, s.nsa, pl.list ? s.nsb : 0, pl.kchunk};
    const bool lib = allow_library && lib_env != 0;
    if (lib && !pl.list) {
      // row-major S = Ma C is the column-major product C' Ma' of the same
      // buffers (C' the nsb x nsa view of psi, Ma' that of Ma)
      rocblas_handle h = blas_handle();
      SQ_CHECK(rocblas_set_stream(h, st) == rocblas_status_success, SQ_ERR_HIP, "rocblas_set_stream failed");
      const double one = 1.0, zero = 0.0;
      rocblas_status rs = rocblas_status_success;
      const double bytes = 8.0 * ((double)s.nsa * s.nsa + 2.0 * (double)s.dim);
      SQ_PROF(PC_ALPHA_GEMM, st, bytes, flops,
              rs = rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, s.nsb, s.nsa, s.nsa, &one, psi,
                                 s.nsb, H.d_Ma, s.nsa, &zero, sinp, s.nsb));
      SQ_CHECK(rs == rocblas_status_success, SQ_ERR_HIP, "rocblas_dgemm failed");
      nsplit = 1;
    } else {
      const double bytes =
          8.0 * ((double)s.nsa * s.nsa + (pl.list ? (double)s.nsb * s.nsb : 0.0) + (double)s.dim * (1 + pl.nsplit));
      const int t128 = ((s.nsa + 127) / 128) * ((s.nsb + 127) / 128);
      if (t128 * pl.nsplit >= 256) {
        SQ_PROF(PC_ALPHA_GEMM, st, bytes, flops + flops_b,
                (k_string_gemm<128><<<dim3(t128, pl.nsplit), 256, 0, st>>>(G)));
      } else {
        const int t64 = ((s.nsa + 63) / 64) * ((s.nsb + 63) / 64);
        SQ_PROF(PC_ALPHA_GEMM, st, bytes, flops + flops_b,
                (k_string_gemm<64><<<dim3(t64, pl.nsplit), 256, 0, st>>>(G)));
      }
    }
  }
  if (pl.list) {
    rows_list_launch(s, pl, H.d_A, 0, H.kpad, H.d_Ma, 0, Mb, 0, psi, sinp, nsplit, sigma, partial, 1, false, st);
    return pl.ngroups;
  }
  const int K8 = row_k8(s);
  const int K4 = rup(s.npair + 1, 4);
  const double flops = 2.0 * (double)s.npair * (s.npair + 1) * (double)s.dim;
  const double e0 = 0.5 * H.e_core;  // the other half is on Ma's diagonal
  // algorithmic traffic: psi read (rows and alpha partners through the cache), the alpha partials read, sigma written
  const double bytes = 8.0 * (double)s.dim * (2 + nsplit);
  switch (pl.mt) {
#define SQ_RS(MT)                                                                                               \
  case MT:                                                                                                      \
    allow_lds(k_sigma_rows<MT>, pl.lds);                                                                        \
    SQ_PROF(PC_SIGMA_ROWS, st, bytes, flops,                                                                    \
            k_sigma_rows<MT><<<pl.ngroups, kRowThreads, pl.lds, st>>>(                                          \
                H.d_A, H.kpad, K4, K8, pl.mgroups, psi, sinp, nsplit, sigma, partial, s.d_rta, s.d_rtb,         \
                s.d_nbr, s.d_nbr_off, s.d_nbr_tile, s.nsa, s.nsb, pl.R, e0));                                   \
    break;
    SQ_RS(1) SQ_RS(2) SQ_RS(3) SQ_RS(4) SQ_RS(5) SQ_RS(6) SQ_RS(7) SQ_RS(8) SQ_RS(9)
#undef SQ_RS
    default:
      throw Error{SQ_ERR_ARG, "unsupported orbital count for the row sigma"};
  }
  return pl.ngroups;
}

// Doubles of workspace the row sigma uses at its chosen shape (string product
// partials and block partials), or -1 when it does not apply.
int64_t row_sigma_used_doubles(const Space& s) {
  RowPlan pl;
  if (!row_plan(s, &pl)) return -1;
  if (pl.fused) return (int64_t)pl.ngroups + pl.ngemm_a + pl.ngemm_b;
  // at least two partial products are asked for below 2048 alpha strings, so
  // that the spaces the no-allocation entry point takes do not depend on the form
  const int least = s.sig.nsplit > 0 ? pl.nsplit : s.nsa >= 2048 ? 1 : 2;
  return (int64_t)std::max(pl.nsplit, least) * s.dim + pl.ngroups;
}

bool row_sigma_wants_zero(const Space& s) {
  RowPlan pl;
  return row_plan(s, &pl) && pl.fused;
}

bool row_sigma_group_ok(const Space& s) {
  RowPlan pl;
  return rows_enabled() && s.d_rtb != nullptr && row_plan(s, &pl) && pl.fused;
}

int64_t row_sigma_group_partials(const Space& s, const SigmaShape& shape, int n) {
  RowPlan pl;
  if (!row_plan(s, shape, &pl, n) || !pl.fused) return 0;
  return (int64_t)pl.ngroups + pl.ngemm_a + pl.ngemm_b;
}

void row_sigma_group(const Space& s, const SigmaShape& shape, const double* A, int64_t A_stride, const double* Ma, int64_t Ma_stride,
                     const double* Mb, int64_t Mb_stride, const double* psi, double* sigma, double* partial, int n,
                     bool zeroed, hipStream_t st) {
  RowPlan pl;
  SQ_CHECK(row_plan(s, shape, &pl, n) && pl.fused && n > 0 && n <= 65535, SQ_ERR_ARG,
           "the grouped row sigma does not apply to this space");
  rows_list_launch(s, pl, A, A_stride, rup(s.npair + 1, 16), Ma, Ma_stride, Mb, Mb_stride, psi, nullptr, 0, sigma,
                   partial, n, zeroed, st);
}

}  // namespace sq

extern "C" int sq_sigma_configure(sq_space* sp, int rows_per_block, int nsplit, int deterministic) {
  return sq::guarded([&] {
    SQ_CHECK(sp, SQ_ERR_ARG, "NULL space");
    SQ_CHECK(rows_per_block >= 0 && rows_per_block <= 64 && nsplit >= 0 && nsplit <= 4, SQ_ERR_ARG,
             "rows_per_block must be in [0, 64] and nsplit in [0, 4] (0: automatic)");
    sq::Space& s = sp->s;
    sq::RowPlan pl;
    const bool before = sq::row_plan(s, &pl);
    const sq::SigmaShape old = s.sig;
    s.sig.R = rows_per_block;
    s.sig.nsplit = nsplit;
    s.sig.det = deterministic < 0 ? -1 : (deterministic != 0);
    if (before && !sq::row_plan(s, &pl)) {  // the workspace sizes assume the row path
      s.sig = old;
      throw sq::Error{SQ_ERR_ARG, "this sigma form does not fit the space"};
    }
  });
}
