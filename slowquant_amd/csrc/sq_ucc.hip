// Unfactorised UCC on the device (replaces construct_ucc_state /
// get_ucc_T / build_operator_matrix + scipy expm_multiply,
// operator_state_algebra.py:413-469,870-960, and the finite-difference theta
// gradient of ucc_wavefunction.py:1025-1098).
//
// T(theta) = sum_k theta_k T_k with every gate generator T_k taken from the
// program's raw terms.  T's sparsity pattern does not depend on theta: it is
// built once per program on the device (k_csr_count / k_csr_fill, rows of
// (source determinant, term, sign)), the entries of a row are sorted by
// source, and those that share one are merged (k_row_sort, k_row_merge):
// spin-adapted doubles give about five entries per matrix element.  An
// evaluation then assembles the numbers of T(theta) once (k_assemble) and
// every product is a plain sparse matrix-vector product over merged elements
// (k_spmv, 12 bytes each).
//
// exp(t T) v is a combination of K basis vectors, kept so that one series
// gives the state at every t in [0, 1] (k_combine).  The first kNormSteps
// products run at once on v and on a fixed pseudo-random vector (k_spmv's two
// columns); the latter's growth estimates ||T||_2 as a power iteration does,
// nu = 1.5 x the estimate + 0.05, at most the largest row sum of |T(theta)|
// (a rigorous bound the assembly yields).  Up to |t| nu = 2 the first column
// is the head of the Taylor series (the largest term is 2: one bit), which
// goes on to K terms with (|t| nu)^K / K! < 2^-60.  Above, the Chebyshev
// series of the exponential takes over: T = i A with A Hermitian, so
//   exp(t T) = sum_k (2 - delta_k0) J_k(t nu) phi_k,   phi_0 = 1,
//   phi_1 = T / nu,  phi_{k+1} = (2 T / nu) phi_k + phi_{k-1},
// where |phi_k v| <= |v|: no term exceeds the result and about nu / 2 times
// fewer products are needed than in Taylor steps of radius 2.
// Energy and gradient of UCCSD, one product per unmerged entry (8 bytes each)
// in Taylor steps -> this: (8e,8o) 663 -> 310 us (44 products of 4-5 us: launch
// latency), (10e,10o) 13.5 -> 2.1 ms (9.1 M merged elements of 44 M entries;
// a product takes 25 us, 105 us before).
// The first evaluation of a program, which builds the pattern: (10e,10o) 202
// -> 8.9 ms.
// The analytic gradient integrates <e^{-sT} lam | T_i | e^{-sT} psi> over
// s in [0, 1] by Gauss-Legendre (lam = H psi): the nodes of psi come from the
// forward series, those of lam from one more series, and one pass over the
// pattern forms the weighted sum over nodes of V_q[I] U_q[J] per merged
// element and adds it to the gates of its entries (k_gate_dots_rows).
//
// Patterns above 2^29 entries, and SQ_UCC_CSR=0, keep a scaled Taylor series
// whose products rescan the terms per determinant (tapply).

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "sq_internal.h"

namespace sq {

constexpr int kUB = 256;

// A fixed pseudo-random vector in [-1, 1) (integer hash of the index).
__device__ __forceinline__ double pattern_at(int64_t i) {
  uint64_t h = (uint64_t)i * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
  h ^= h >> 31;
  h *= 0xBF58476D1CE4E5B9ull;
  h ^= h >> 29;
  return (double)(h >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

struct SV {
  int nsa, nsb;
  const uint32_t* astr;
  const uint32_t* bstr;
  const int32_t* arank;
  const int32_t* brank;
};

__device__ __forceinline__ bool ops_adjoint(const SpinOps& o, uint32_t& m, int& par) {
  for (int j = 0; j < o.n; ++j) {
    uint32_t bit = 1u << o.orb[j];
    par += __popc(m & (bit - 1u));
    if (!o.cre[j]) {
      if (m & bit) return false;
      m |= bit;
    } else {
      if (!(m & bit)) return false;
      m &= ~bit;
    }
  }
  return true;
}

// Adjoint of term t on strings (a0, b0): images (a, b) and sign parity;
// false if it does not apply.
__device__ __forceinline__ bool term_adjoint(const TermFast& F, const Term* __restrict__ terms, int t, uint32_t a0,
                                             uint32_t b0, uint32_t& a, uint32_t& b, int& par) {
  if (F.flags & 1u) {
    if ((a0 & F.sa) != F.sa || (a0 & F.ca) || (b0 & F.sb) != F.sb || (b0 & F.cb)) return false;
    a = a0 ^ F.sa ^ F.ca;
    b = b0 ^ F.sb ^ F.cb;
    par = __popc(a0 & F.xa) + __popc(b0 & F.xb) + (int)(F.flags >> 1);
    return true;
  }
  const Term& T = terms[t];
  a = a0;
  b = b0;
  par = 0;
  return ops_adjoint(T.a, a, par) && ops_adjoint(T.b, b, par);
}

// part[y][I] = sum over the terms t = g, g + G, ... of w[t] <I|O_t|J> cur[J]
// summed over the groups g = y*nw + wave of one block (w = nullptr: unit
// weights).  A block is nw = min(G, kTG) waves over the same 64 determinants
// (lane = determinant, flattened across rows), one term group per wave; the
// waves' sums are added in LDS in wave order.  Splitting the terms over G groups
// keeps small spaces' grids full; k_tapply_sum adds the part rows in order.
constexpr int kTG = 8;

__global__ __launch_bounds__(64 * kTG) void k_tapply_part(SV v, const Term* __restrict__ terms,
                                                         const TermFast* __restrict__ fast,
                                                         const double* __restrict__ w, int nt, int G,
                                                         const double* __restrict__ cur, double* __restrict__ part) {
  __shared__ double red[kTG][64];
  const size_t dim = (size_t)v.nsa * v.nsb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  const size_t I = (size_t)blockIdx.x * 64 + lane;
  const int g = blockIdx.y * nw + wave;
  double val = 0.0;
  if (I < dim && g < G) {
    const int ia = (int)(I / (uint32_t)v.nsb), ib = (int)(I - (size_t)ia * v.nsb);
    const uint32_t a0 = v.astr[ia], b0 = v.bstr[ib];
    for (int t = g; t < nt; t += G) {
      const TermFast F = fast[t];
      uint32_t a, b;
      int par;
      if (!term_adjoint(F, terms, t, a0, b0, a, b, par)) continue;
      const int ra = v.arank[a], rb = v.brank[b];
      if (ra < 0 || rb < 0) continue;
      const double c = (w ? w[t] : 1.0) * F.coef;
      val += ((par & 1) ? -c : c) * cur[(size_t)ra * v.nsb + rb];
    }
  }
  red[wave][lane] = val;
  __syncthreads();
  if (wave == 0 && I < dim) {
    double s = 0.0;
    for (int q = 0; q < nw; ++q) s += red[q][lane];
    part[(size_t)blockIdx.y * dim + I] = s;
  }
}

// part[g][I] for one term group g = blockIdx.y per block (all waves of a
// block on the same term stream, so they share its scalar-cache lines); used
// when there are too few groups to fold (large spaces).
__global__ __launch_bounds__(kUB) void k_tapply_group(SV v, const Term* __restrict__ terms,
                                                     const TermFast* __restrict__ fast,
                                                     const double* __restrict__ w, int nt, int G,
                                                     const double* __restrict__ cur, double* __restrict__ part) {
  const size_t dim = (size_t)v.nsa * v.nsb;
  const size_t I = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= dim) return;
  const int ia = (int)(I / (uint32_t)v.nsb), ib = (int)(I - (size_t)ia * v.nsb);
  const uint32_t a0 = v.astr[ia], b0 = v.bstr[ib];
  const int g = blockIdx.y;
  double val = 0.0;
  for (int t = g; t < nt; t += G) {
    const TermFast F = fast[t];
    uint32_t a, b;
    int par;
    if (!term_adjoint(F, terms, t, a0, b0, a, b, par)) continue;
    const int ra = v.arank[a], rb = v.brank[b];
    if (ra < 0 || rb < 0) continue;
    const double c = (w ? w[t] : 1.0) * F.coef;
    val += ((par & 1) ? -c : c) * cur[(size_t)ra * v.nsb + rb];
  }
  part[(size_t)g * dim + I] = val;
}

// T's sparsity pattern, row I = the terms whose adjoint maps I to a
// determinant J of the space, in term order: count, then fill the entries
// (J, t | parity << 31) between rowp[I] and rowp[I + 1].
__device__ __forceinline__ bool term_entry(const SV& v, const Term* __restrict__ terms,
                                           const TermFast* __restrict__ fast, int t, uint32_t a0, uint32_t b0,
                                           uint32_t& J, int& par) {
  uint32_t a, b;
  if (!term_adjoint(fast[t], terms, t, a0, b0, a, b, par)) return false;
  const int ra = v.arank[a], rb = v.brank[b];
  if (ra < 0 || rb < 0) return false;
  J = (uint32_t)ra * (uint32_t)v.nsb + (uint32_t)rb;
  return true;
}

__global__ void k_csr_count(SV v, const Term* __restrict__ terms, const TermFast* __restrict__ fast, int nt,
                            int32_t* __restrict__ cnt) {
  const size_t dim = (size_t)v.nsa * v.nsb;
  const size_t I = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= dim) return;
  const int ia = (int)(I / (uint32_t)v.nsb), ib = (int)(I - (size_t)ia * v.nsb);
  const uint32_t a0 = v.astr[ia], b0 = v.bstr[ib];
  int c = 0;
  for (int t = 0; t < nt; ++t) {
    uint32_t J;
    int par;
    if (term_entry(v, terms, fast, t, a0, b0, J, par)) ++c;
  }
  cnt[I] = c;
}

__global__ void k_csr_fill(SV v, const Term* __restrict__ terms, const TermFast* __restrict__ fast, int nt,
                           const int64_t* __restrict__ rowp, uint2* __restrict__ ent) {
  const size_t dim = (size_t)v.nsa * v.nsb;
  const size_t I = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= dim) return;
  const int ia = (int)(I / (uint32_t)v.nsb), ib = (int)(I - (size_t)ia * v.nsb);
  const uint32_t a0 = v.astr[ia], b0 = v.bstr[ib];
  int64_t k = rowp[I];
  const int64_t e = rowp[I + 1];
  for (int t = 0; t < nt && k < e; ++t) {
    uint32_t J;
    int par;
    if (term_entry(v, terms, fast, t, a0, b0, J, par)) ent[k++] = make_uint2(J, (uint32_t)t | ((uint32_t)(par & 1) << 31));
  }
}

// out[I] = sum over the entries (J, t, sign) of row I of sign coef[t] in[J], one
// wave per row: lane l takes entries l, l + 64, ... and the wave sums in a
// fixed shuffle order.
constexpr int kCsrRows = 4;  // rows (waves) per block

__global__ __launch_bounds__(64 * kCsrRows) void k_tapply_csr(int64_t dim, const int64_t* __restrict__ rowp,
                                                              const uint2* __restrict__ ent,
                                                              const double* __restrict__ coef,
                                                              const double* __restrict__ in,
                                                              double* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t I = (int64_t)blockIdx.x * kCsrRows + (threadIdx.x >> 6);
  if (I >= dim) return;  // uniform per wave; no block barrier below
  const int64_t b = rowp[I], e = rowp[I + 1];
  double val = 0.0;
  for (int64_t k = b + lane; k < e; k += 64) {
    const uint2 x = ent[k];
    const uint32_t t = x.y & 0x7fffffffu;
    const double c = coef[t] * in[x.x];
    val += (x.y >> 31) ? -c : c;
  }
  for (int off = 32; off > 0; off >>= 1) val += __shfl_down(val, off, 64);
  if (lane == 0) out[I] = val;
}

// ---- merged pattern -------------------------------------------------------

// One contribution to a merged element: gate | index of |coefficient| << 24 |
// negative << 31.
constexpr int kGateBits = 24, kCoefBits = 7;
constexpr int kSortRow = 8192;  // longest row sorted in LDS (64 KB of keys); longer rows merge neighbours only

// Sorts a row's entries by (source, term) in place (bitonic, keys
// source << 32 | term << 1 | sign) and counts the distinct sources.  A block
// per row, on two grid dimensions: 256 threads per row would pass the limit of
// 2^32 in one from 2^24 rows.
constexpr int64_t kSortGrid = (int64_t)1 << 20;
__global__ __launch_bounds__(kUB) void k_row_sort(int64_t dim, const int64_t* __restrict__ rowp,
                                                  uint2* __restrict__ ent, int32_t* __restrict__ ucnt) {
  extern __shared__ uint64_t key[];
  __shared__ int red[kUB / 64];
  const int64_t row = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  if (row >= dim) return;
  const int64_t b = rowp[row];
  const int n = (int)(rowp[row + 1] - b);
  const int tid = threadIdx.x;
  int c = 0;
  if (n <= kSortRow) {
    int P = 1;
    while (P < n) P <<= 1;
    for (int i = tid; i < P; i += kUB) {
      uint64_t k = ~0ull;
      if (i < n) {
        const uint2 e = ent[b + i];
        k = (uint64_t)e.x << 32 | (uint64_t)(e.y & 0x7fffffffu) << 1 | (e.y >> 31);
      }
      key[i] = k;
    }
    for (int k = 2; k <= P; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        __syncthreads();
        for (int i = tid; i < P; i += kUB) {
          const int o = i ^ j;
          if (o <= i) continue;
          const uint64_t x = key[i], y = key[o];
          if ((x > y) == ((i & k) == 0)) {
            key[i] = y;
            key[o] = x;
          }
        }
      }
    __syncthreads();
    for (int i = tid; i < n; i += kUB) {
      const uint64_t x = key[i];
      ent[b + i] = make_uint2((uint32_t)(x >> 32), (uint32_t)(x >> 1 & 0x7fffffffu) | (uint32_t)(x & 1) << 31);
      c += i == 0 || (uint32_t)(key[i - 1] >> 32) != (uint32_t)(x >> 32);
    }
  } else {
    for (int i = tid; i < n; i += kUB) c += i == 0 || ent[b + i - 1].x != ent[b + i].x;
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
  if ((tid & 63) == 0) red[tid >> 6] = c;
  __syncthreads();
  if (tid == 0) {
    int tot = 0;
    for (int w = 0; w < kUB / 64; ++w) tot += red[w];
    ucnt[row] = tot;
  }
}

// Merged elements of row I at [urow[I], urow[I + 1]): source and first
// contribution; every entry's contribution word.  One wave per row.
constexpr int kRows = 4;  // rows (waves) per block
__global__ __launch_bounds__(64 * kRows) void k_row_merge(int64_t dim, const int64_t* __restrict__ rowp,
                                                          const uint2* __restrict__ ent,
                                                          const uint32_t* __restrict__ tword,
                                                          const int64_t* __restrict__ urow, uint32_t* __restrict__ col,
                                                          uint32_t* __restrict__ first, uint32_t* __restrict__ con) {
  const int lane = threadIdx.x & 63;
  const int64_t I = (int64_t)blockIdx.x * kRows + (threadIdx.x >> 6);
  if (I >= dim) return;
  const int64_t b = rowp[I], e = rowp[I + 1];
  int64_t u = urow[I];
  for (int64_t k0 = b; k0 < e; k0 += 64) {
    const int64_t k = k0 + lane;
    uint2 x = make_uint2(0, 0);
    bool head = false;
    if (k < e) {
      x = ent[k];
      head = k == b || ent[k - 1].x != x.x;
      con[k] = tword[x.y & 0x7fffffffu] ^ (x.y & 0x80000000u);
    }
    const uint64_t m = __ballot(head);
    if (head) {
      const int64_t at = u + __popcll(m & ((1ull << lane) - 1ull));
      col[at] = x.x;
      first[at] = (uint32_t)k;
    }
    u += __popcll(m);
  }
}

// val[u] = sum over the contributions of merged element u of sign theta[gate]
// |coef|; rmax[block]: largest sum of |val| over the block's rows.  One wave per
// row.  theta and the coefficients are read from LDS when theta fits (ng <=
// kLdsGates).  Also v = v0 and x = the pseudo-random vector, for the products
// that follow.
constexpr int kLdsGates = 4096;
__global__ __launch_bounds__(64 * kRows) void k_assemble(int64_t dim, const int64_t* __restrict__ urow,
                                                         const uint32_t* __restrict__ first,
                                                         const uint32_t* __restrict__ con,
                                                         const double* __restrict__ coefs, int ncoef,
                                                         const double* __restrict__ theta, int ng,
                                                         double* __restrict__ val, double* __restrict__ rmax,
                                                         const double* __restrict__ v0, double* __restrict__ v,
                                                         double* __restrict__ x) {
  extern __shared__ double sth[];
  __shared__ double sc[1 << kCoefBits];
  __shared__ double red[kRows];
  for (int64_t i = blockIdx.x * (int64_t)(64 * kRows) + threadIdx.x; i < dim; i += (int64_t)gridDim.x * 64 * kRows) {
    v[i] = v0[i];
    x[i] = pattern_at(i);
  }
  const bool lds = ng <= kLdsGates;
  if (lds)
    for (int i = threadIdx.x; i < ng; i += 64 * kRows) sth[i] = theta[i];
  for (int i = threadIdx.x; i < ncoef; i += 64 * kRows) sc[i] = coefs[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double most = 0.0;
  for (int64_t I = (int64_t)blockIdx.x * kRows + wave; I < dim; I += (int64_t)gridDim.x * kRows) {
    const int64_t b = urow[I], e = urow[I + 1];
    double sum = 0.0;
    for (int64_t u = b + lane; u < e; u += 64) {
      const uint32_t c0 = first[u], c1 = first[u + 1];
      double v = 0.0;
      for (uint32_t c = c0; c < c1; ++c) {
        const uint32_t w = con[c];
        const uint32_t g = w & ((1u << kGateBits) - 1u);
        const double x = (lds ? sth[g] : theta[g]) * sc[(w >> kGateBits) & ((1u << kCoefBits) - 1u)];
        v += (w >> 31) ? -x : x;
      }
      val[u] = v;
      sum += fabs(v);
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    most = sum > most || sum != sum ? sum : most;
  }
  if (lane == 0) red[wave] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kRows; ++w) most = red[w] > most || red[w] != red[w] ? red[w] : most;
    rmax[blockIdx.x] = most;
  }
}

// out = max of n values (NaN if one is).
__global__ __launch_bounds__(kUB) void k_max(const double* __restrict__ x, int n, double* __restrict__ out) {
  __shared__ double red[kUB / 64];
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += kUB) m = x[i] > m || x[i] != x[i] ? x[i] : m;
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(m, off, 64);
    m = o > m || o != o ? o : m;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kUB / 64; ++w) m = red[w] > m || red[w] != red[w] ? red[w] : m;
    out[0] = m;
  }
}

// out[0..2] = bound[0], |y|^2, |x|^2 (out in pinned host memory), summed in a
// fixed order by the last block.
// The blocks' sums pass between them by agent-scope stores and loads; a fence
// would write back the caches' other lines first (9 us against 5).
__global__ __launch_bounds__(kUB) void k_norms(const double* __restrict__ y, const double* __restrict__ x, int64_t n,
                                               const double* __restrict__ bound, double* __restrict__ part,
                                               int* __restrict__ count, double* __restrict__ out) {
  __shared__ double red[2][kUB / 64];
  __shared__ int last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto sums = [&](double a, double b) {
    for (int off = 32; off > 0; off >>= 1) {
      a += __shfl_down(a, off, 64);
      b += __shfl_down(b, off, 64);
    }
    if (lane == 0) {
      red[0][wave] = a;
      red[1][wave] = b;
    }
    __syncthreads();
  };
  double a = 0.0, b = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kUB + threadIdx.x; i < n; i += (int64_t)gridDim.x * kUB) {
    a += y[i] * y[i];
    b += x[i] * x[i];
  }
  sums(a, b);
  if (threadIdx.x == 0) {
    for (int w = 1; w < kUB / 64; ++w) {
      red[0][0] += red[0][w];
      red[1][0] += red[1][w];
    }
    __hip_atomic_store(part + 2 * blockIdx.x, red[0][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(part + 2 * blockIdx.x + 1, red[1][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the sums have arrived before the count says so
    last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  a = b = 0.0;
  for (int i = threadIdx.x; i < (int)gridDim.x; i += kUB) {
    a += __hip_atomic_load(part + 2 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    b += __hip_atomic_load(part + 2 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  sums(a, b);
  if (threadIdx.x == 0) {
    for (int w = 1; w < kUB / 64; ++w) {
      red[0][0] += red[0][w];
      red[1][0] += red[1][w];
    }
    out[0] = bound[0];
    out[1] = red[0][0];
    out[2] = red[1][0];
    *count = 0;
  }
}

// A row sum of |T| below this is zero to the exponential, and its reciprocal
// may overflow.
constexpr double kTinyBound = 1e-300;

// nxt[I] = f (T cur)[I] + prev[I] (prev: nullptr for none), LPR lanes per row;
// TWO: nxt2 = f T cur2 in the same pass.  With bound, f is divided by
// bound[0] (0 where that vanishes).  U rounds of a row's elements are loaded before
// any is used, the next U during the gathers of those.
// Bound by the chain row pointer -> elements -> gathers -> sum of a row, some
// 3 us that the waves of a SIMD overlap, not by bytes ((10e,10o): 9.1 M
// elements of 12 bytes; without the gathers' misses or the 8-byte numbers it
// takes as long), and by launch latency below about 10^5 elements.  So a row
// gets half a wave: 64, 32 and 16 lanes 2464, 2140 and 2200 us an energy and
// gradient of (10e,10o) UCCSD (U = 6); U = 1, 2, 4, 6: 2448, 2236, 2180, 2140.
template <int LPR, bool TWO>
__global__ __launch_bounds__(kUB) void k_spmv(int64_t dim, const int64_t* __restrict__ urow,
                                              const uint32_t* __restrict__ col, const double* __restrict__ val,
                                              const double* __restrict__ cur, const double* __restrict__ cur2,
                                              const double* __restrict__ prev, double f,
                                              const double* __restrict__ bound, double* __restrict__ nxt,
                                              double* __restrict__ nxt2) {
  constexpr int U = 6;
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t I = (int64_t)blockIdx.x * (kUB / LPR) + threadIdx.x / LPR;
  if (I >= dim) return;
  if (bound) f = bound[0] > kTinyBound ? f / bound[0] : 0.0;
  const int64_t e = urow[I + 1];
  int64_t u0 = urow[I] + lane;
  double a[U], v = 0.0, v2 = 0.0;
  uint32_t c[U];
  auto load = [&] {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int64_t u = u0 + j * LPR;
      a[j] = u < e ? val[u] : 0.0;
      c[j] = u < e ? col[u] : 0u;
    }
  };
  load();
  for (bool more = true; more;) {
    double m[U], x[U], x2[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      m[j] = a[j];
      x[j] = cur[c[j]];
      if (TWO) x2[j] = cur2[c[j]];
    }
    u0 += U * LPR;
    more = u0 - lane < e;
    if (more) load();
#pragma unroll
    for (int j = 0; j < U; ++j) {
      v += m[j] * x[j];
      if (TWO) v2 += m[j] * x2[j];
    }
  }
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) {
    v += __shfl_down(v, off, LPR);
    if (TWO) v2 += __shfl_down(v2, off, LPR);
  }
  if (lane == 0) {
    nxt[I] = f * v + (prev ? prev[I] : 0.0);
    if (TWO) nxt2[I] = f * v2;
  }
}

// Linear combinations of the basis vectors phi_k (k <= K, at basis + k dim):
// node q (q < nq) to nodes[I * stride + q], the last output (if fin) to fin[I];
// zero (if given; it may be a basis vector) is cleared.
constexpr int kMaxOut = 9, kMaxBasis = 44, kCB = 64;
struct Combine {
  double c[kMaxOut][kMaxBasis];
};

__global__ __launch_bounds__(kCB) void k_combine(int64_t dim, int K, Combine C, int nq, const double* basis,
                                                 double* __restrict__ nodes, int stride, double* __restrict__ fin,
                                                 double* zero) {
  const int64_t I = blockIdx.x * (int64_t)kCB + threadIdx.x;
  if (I >= dim) return;
  double o[kMaxOut];
#pragma unroll
  for (int q = 0; q < kMaxOut; ++q) o[q] = 0.0;
#pragma unroll 4
  for (int k = K; k >= 0; --k) {  // small terms first
    const double x = basis[(size_t)k * dim + I];
#pragma unroll
    for (int q = 0; q < kMaxOut; ++q) o[q] += C.c[q][k] * x;
  }
#pragma unroll
  for (int q = 0; q < kMaxOut - 1; ++q)
    if (q < nq) nodes[(size_t)I * stride + q] = o[q];
  if (fin) fin[I] = o[kMaxOut - 1];
  if (zero) zero[I] = 0.0;
}

// Gate dots: per merged element (I, J) r = sum_q V[I][q] U[J][q] over NQ
// nodes (V carries the weights), added with sign |coef| to every
// contribution's gate g in [g0, g0 + ng).  Gate sums in LDS, copies of them per
// block, then to dpart[block][ng]; with more gates than LDS holds (copies = 0)
// to dpart[0][ng] by global atomics (zeroed before).  One wave per row; a node
// row is 64 to 128 contiguous bytes.
// A copy per wave gives every sum a fixed order (a wave's LDS adds run in
// program order, and those of one instruction by lane), so that the gradient is
// the same bit for bit where lambda is.
template <int NQ>
__global__ __launch_bounds__(64 * kRows) void k_gate_dots_rows(
    int64_t dim, const int64_t* __restrict__ urow, const uint32_t* __restrict__ col,
    const uint32_t* __restrict__ first, const uint32_t* __restrict__ con, const double* __restrict__ coefs, int ncoef,
    const double* __restrict__ U, const double* __restrict__ V, int g0, int ng, int copies,
    double* __restrict__ dpart) {
  extern __shared__ double sg[];
  __shared__ double sc[1 << kCoefBits];
  for (int i = threadIdx.x; i < copies * ng; i += 64 * kRows) sg[i] = 0.0;
  for (int i = threadIdx.x; i < ncoef; i += 64 * kRows) sc[i] = coefs[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* own = sg + (copies > 1 ? wave * ng : 0);
  for (int64_t I = (int64_t)blockIdx.x * kRows + wave; I < dim; I += (int64_t)gridDim.x * kRows) {
    const int64_t e = urow[I + 1];
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = V[(size_t)I * NQ + q];
    for (int64_t u = urow[I] + lane; u < e; u += 64) {
      const double* x = U + (size_t)col[u] * NQ;
      double r = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) r += v[q] * x[q];
      const uint32_t c1 = first[u + 1];
      for (uint32_t c = first[u]; c < c1; ++c) {
        const uint32_t w = con[c];
        const double d = r * sc[(w >> kGateBits) & ((1u << kCoefBits) - 1u)];
        const uint32_t g = (w & ((1u << kGateBits) - 1u)) - (uint32_t)g0;
        if (g >= (uint32_t)ng) continue;
        if (copies) atomicAdd(own + g, (w >> 31) ? -d : d);
        else unsafeAtomicAdd(dpart + g, (w >> 31) ? -d : d);
      }
    }
  }
  if (!copies) return;
  __syncthreads();
  for (int i = threadIdx.x; i < ng; i += 64 * kRows) {
    double sum = sg[i];
    for (int c = 1; c < copies; ++c) sum += sg[c * ng + i];
    dpart[(size_t)blockIdx.x * ng + i] = sum;
  }
}

// nxt[I] = f * sum_g part[g][I]; acc[I] += nxt[I] when acc != nullptr.
__global__ void k_tapply_sum(const double* __restrict__ part, int G, int64_t dim, double f, double* __restrict__ nxt,
                             double* __restrict__ acc) {
  const int64_t I = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (I >= dim) return;
  double v = 0.0;
  for (int g = 0; g < G; ++g) v += part[(size_t)g * dim + I];
  v *= f;
  nxt[I] = v;
  if (acc) acc[I] += v;
}

// Per gate i, per block b of amplitudes: dpart[b*ng + i] = sum over the
// block's I of v[I] (T_i u)[I] with T_i the gate's generator (unit weight).
// Block (b, y) covers determinants [256 b, 256 b + 256) and takes the gates
// i = y, y + gridDim.y, ...; every (b, i) is written by exactly one block and
// summed over b in a fixed order later.
__global__ void k_gate_dots(SV sv, const Term* __restrict__ terms, const TermFast* __restrict__ fast,
                            const GateDev* __restrict__ gates, int ng, const double* __restrict__ u,
                            const double* __restrict__ v, double* __restrict__ dpart) {
  __shared__ double red[kUB / 64];
  const size_t dim = (size_t)sv.nsa * sv.nsb;
  const size_t I = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // determinants flattened
  const bool ok = I < dim;
  const int ia = ok ? (int)(I / (uint32_t)sv.nsb) : 0;
  const int ib = ok ? (int)(I - (size_t)ia * sv.nsb) : 0;
  const int b = blockIdx.x;
  const uint32_t a0 = sv.astr[ia], b0 = sv.bstr[ib];
  const double vI = ok ? v[I] : 0.0;
  for (int i = blockIdx.y; i < ng; i += gridDim.y) {
    double val = 0.0;
    if (ok && vI != 0.0) {
      for (int t = gates[i].term_begin; t < gates[i].term_end; ++t) {
        const TermFast F = fast[t];
        uint32_t a, bb;
        int par;
        if (!term_adjoint(F, terms, t, a0, b0, a, bb, par)) continue;
        const int ra = sv.arank[a], rb = sv.brank[bb];
        if (ra < 0 || rb < 0) continue;
        val += ((par & 1) ? -F.coef : F.coef) * u[(size_t)ra * sv.nsb + rb];
      }
    }
    double c = vI * val;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
      double tot = 0.0;
      for (int w = 0; w < (int)(blockDim.x >> 6); ++w) tot += red[w];
      dpart[(size_t)b * ng + i] = tot;
    }
    __syncthreads();  // red is reused by the next gate
  }
}

// gsum[i] = f * sum_b dpart[b*ng + i] (+ gsum[i] with add), one wave per gate;
// also to host (if given).
__global__ __launch_bounds__(64 * kRows) void k_gate_accum(const double* __restrict__ dpart, int nb, int ng, double f,
                                                           int add, double* __restrict__ gsum,
                                                           double* __restrict__ host) {
  const int lane = threadIdx.x & 63, i = blockIdx.x * kRows + (threadIdx.x >> 6);
  if (i >= ng) return;
  double s = 0.0;
  for (int b = lane; b < nb; b += 64) s += dpart[(size_t)b * ng + i];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane != 0) return;
  s = f * s + (add ? gsum[i] : 0.0);
  gsum[i] = s;
  if (host) host[i] = s;
}

// w[t] = theta[gate of term t]
__global__ void k_term_weights(const GateDev* __restrict__ gates, int ngates, const double* __restrict__ theta,
                               double* __restrict__ w) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ngates) return;
  for (int t = gates[g].term_begin; t < gates[g].term_end; ++t) w[t] = theta[g];
}

__global__ void k_zero(double* __restrict__ x, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

__global__ void k_fill_pattern(double* __restrict__ x, int64_t n) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = pattern_at(i);
}

__global__ void k_scale(double* __restrict__ x, int64_t n, const double* __restrict__ s, int slot) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] *= s[slot];
}

__global__ void k_inv_sqrt_slot(double* __restrict__ s, int from, int to) {
  if (threadIdx.x == 0 && blockIdx.x == 0) s[to] = s[from] > 0.0 ? 1.0 / sqrt(s[from]) : 0.0;
}

static SV sv(const Space& s) { return SV{s.nsa, s.nsb, s.d_astr, s.d_bstr, s.d_arank, s.d_brank}; }

// Mask form of one spin part's adjoint (ops applied in order as in
// ops_adjoint: a creator needs its orbital occupied and clears it, an
// annihilator needs it empty and sets it).  Op j adds popc(m_j & below_j)
// with m_j = m ^ (bits of the ops before j); mod 2 that is popc(m & below_j)
// + popc(flipped_before_j & below_j), so the parity is popc(m & x) + c0 with
// x = XOR of the below_j masks and c0 a constant.  False if an orbital
// repeats.
static bool part_fast(const SpinOps& o, uint32_t& set, uint32_t& clear, uint32_t& x, int& c0) {
  set = clear = x = 0;
  c0 = 0;
  uint32_t flipped = 0;
  for (int j = 0; j < o.n; ++j) {
    const uint32_t bit = 1u << o.orb[j];
    if (flipped & bit) return false;
    x ^= bit - 1u;
    c0 += __builtin_popcount(flipped & (bit - 1u));
    flipped |= bit;
    (o.cre[j] ? set : clear) |= bit;
  }
  return true;
}

// Terms in mask form where their spin parts allow it (uploaded).
static TermFast* upload_term_fast(const std::vector<Term>& terms) {
  std::vector<TermFast> f(std::max<size_t>(terms.size(), 1), TermFast{0, 0, 0, 0, 0, 0, 0u, 0u, 0.0});
  for (size_t t = 0; t < terms.size(); ++t) {
    TermFast& F = f[t];
    F.coef = terms[t].coef;
    int ca0 = 0, cb0 = 0;
    if (part_fast(terms[t].a, F.sa, F.ca, F.xa, ca0) && part_fast(terms[t].b, F.sb, F.cb, F.xb, cb0))
      F.flags = 1u | ((uint32_t)((ca0 + cb0) & 1) << 1);
    else
      F = TermFast{0, 0, 0, 0, 0, 0, 0u, 0u, terms[t].coef};
  }
  TermFast* d = nullptr;
  SQ_HIP(hipMalloc(&d, sizeof(TermFast) * f.size()));
  const hipError_t e = hipMemcpy(d, f.data(), sizeof(TermFast) * f.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(d);
    SQ_HIP(e);
  }
  return d;
}

static const TermFast* term_fast(const Program& p) {
  if (!p.d_term_fast) p.d_term_fast = upload_term_fast(p.terms);
  return p.d_term_fast;
}

struct UccCsr {
  int64_t nnz = 0;
  int64_t* rowp = nullptr;  // [dim + 1]
  uint2* ent = nullptr;     // [nnz]
  double* coef = nullptr;   // [terms]
};

void ucc_csr_free(UccCsr* c) {
  if (!c) return;
  if (c->rowp) (void)hipFree(c->rowp);
  if (c->ent) (void)hipFree(c->ent);
  if (c->coef) (void)hipFree(c->coef);
  delete c;
}

// T's merged pattern.  val holds the numbers of the evaluation under way: an
// evaluation locks mu while it enqueues its work, waits on the device for the
// last one (busy) and records busy at its end, so that evaluations on other
// streams and threads keep to their own theta.
struct UccT {
  int64_t nu = 0;             // merged elements
  int ncoef = 0;
  int lpr = 32;               // lanes per row of k_spmv
  int64_t* urow = nullptr;    // [dim + 1]
  uint32_t* col = nullptr;    // [nu]
  uint32_t* first = nullptr;  // [nu + 1]
  uint32_t* con = nullptr;    // [entries]
  double* coefs = nullptr;    // [ncoef]
  double* val = nullptr;      // [nu]
  int* count = nullptr;       // blocks done of k_norms, zero between launches
  double* host = nullptr;     // pinned: norms [3] | energy | gradient
  std::mutex mu;
  hipEvent_t busy = nullptr;
  ~UccT() {
    if (host) (void)hipHostFree(host);
    for (void* p : {(void*)count, (void*)urow, (void*)col, (void*)first, (void*)con, (void*)coefs, (void*)val})
      if (p) (void)hipFree(p);
    if (busy) (void)hipEventDestroy(busy);
  }
};

void ucc_t_free(UccT* t) { delete t; }

// Largest pattern kept (entries of 8 bytes); above it, and with SQ_UCC_CSR=0,
// T is applied by the term-scan kernels below.
constexpr int64_t kCsrMaxEntries = (int64_t)1 << 29;
// Largest pattern kept for a compiled operator (256 MB); larger operators
// (a Hamiltonian over a big space) keep the term scan.
constexpr int64_t kOpMaxEntries = (int64_t)1 << 25;

// Sparsity pattern of sum_t coef_t O_t (terms on the device, with their mask
// forms) on space s: per determinant I, the entries (J, t | parity << 31) of
// the terms whose adjoint maps I into the space (synchronous); nullptr when
// it is empty, above max_nnz entries, or the one-wave-per-row product would
// not fit one grid dimension.
static UccCsr* build_pattern(const Space& s, const std::vector<Term>& terms, const Term* d_terms,
                             const TermFast* fast, int64_t max_nnz, hipStream_t st, int64_t* longest = nullptr) {
  const int nt = (int)terms.size();
  // k_tapply_csr runs one 64-lane wave per determinant: 64 * dim work-items
  // must stay below the 2^32 limit of one grid dimension
  if (s.dim == 0 || nt == 0 || 64 * s.dim >= ((int64_t)1 << 32)) return nullptr;
  const unsigned nb = (unsigned)((s.dim + kUB - 1) / kUB);
  int32_t* cnt = nullptr;
  SQ_HIP(hipMalloc(&cnt, sizeof(int32_t) * (size_t)s.dim));
  std::vector<int32_t> hc((size_t)s.dim);
  k_csr_count<<<nb, kUB, 0, st>>>(sv(s), d_terms, fast, nt, cnt);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(hc.data(), cnt, sizeof(int32_t) * hc.size(), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(cnt);
  SQ_HIP(e);
  std::vector<int64_t> rowp((size_t)s.dim + 1, 0);
  for (size_t i = 0; i < hc.size(); ++i) rowp[i + 1] = rowp[i] + hc[i];
  const int64_t nnz = rowp.back();
  if (nnz == 0 || nnz > max_nnz) return nullptr;
  if (longest) *longest = *std::max_element(hc.begin(), hc.end());
  UccCsr* c = new UccCsr;
  c->nnz = nnz;
  std::vector<double> coef((size_t)nt);
  for (int t = 0; t < nt; ++t) coef[t] = terms[t].coef;
  e = hipMalloc(&c->rowp, sizeof(int64_t) * rowp.size());
  if (e == hipSuccess) e = hipMalloc(&c->ent, sizeof(uint2) * (size_t)nnz);
  if (e == hipSuccess) e = hipMalloc(&c->coef, sizeof(double) * coef.size());
  if (e == hipSuccess) e = hipMemcpy(c->rowp, rowp.data(), sizeof(int64_t) * rowp.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(c->coef, coef.data(), sizeof(double) * coef.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    k_csr_fill<<<nb, kUB, 0, st>>>(sv(s), d_terms, fast, nt, c->rowp, c->ent);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) {
    ucc_csr_free(c);
    SQ_HIP(e);
  }
  return c;
}

static bool csr_enabled() {
  const char* env = getenv("SQ_UCC_CSR");
  return !(env && env[0] == '0');
}

// The program's merged pattern of T on space s, built on first use
// (synchronous); nullptr where it is not used.
static UccT* ucc_t(const Space& s, const Program& p, hipStream_t st) {
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  if (p.ucc_t_tried) return p.ucc_t;
  p.ucc_t_tried = true;
  const int ng = (int)p.gates.size();
  if (!csr_enabled() || ng >= (1 << kGateBits)) return nullptr;
  // the distinct |coefficients| and every term's word
  std::vector<double> coefs;
  std::vector<uint32_t> word(std::max<size_t>(p.terms.size(), 1), 0u);
  for (int g = 0; g < ng; ++g)
    for (int t = p.gates[g].term_begin; t < p.gates[g].term_end; ++t) {
      const double c = std::fabs(p.terms[t].coef);
      size_t k = std::find(coefs.begin(), coefs.end(), c) - coefs.begin();
      if (k == coefs.size()) coefs.push_back(c);
      if (k >= (1u << kCoefBits)) return nullptr;
      word[t] = (uint32_t)g | (uint32_t)k << kGateBits | (p.terms[t].coef < 0 ? 0x80000000u : 0u);
    }
  int64_t longest = 0;
  std::unique_ptr<UccCsr, void (*)(UccCsr*)> c(
      build_pattern(s, p.terms, p.d_terms, term_fast(p), kCsrMaxEntries, st, &longest), ucc_csr_free);
  if (!c) return nullptr;
  std::unique_ptr<UccT> T(new UccT);
  struct Tmp {
    void* p = nullptr;
    ~Tmp() { if (p) (void)hipFree(p); }
  } ucnt, tword;
  SQ_HIP(hipMalloc(&ucnt.p, sizeof(int32_t) * (size_t)s.dim));
  SQ_HIP(hipMalloc(&tword.p, sizeof(uint32_t) * word.size()));
  SQ_HIP(hipMemcpyAsync(tword.p, word.data(), sizeof(uint32_t) * word.size(), hipMemcpyHostToDevice, st));
  int P = 1;
  while (P < std::min<int64_t>(longest, kSortRow)) P <<= 1;
  allow_lds(k_row_sort, (size_t)P * 8 + 1024);
  const dim3 sort_grid((unsigned)std::min(s.dim, kSortGrid), (unsigned)((s.dim + kSortGrid - 1) / kSortGrid));
  k_row_sort<<<sort_grid, kUB, (size_t)P * 8, st>>>(s.dim, c->rowp, c->ent, (int32_t*)ucnt.p);
  SQ_HIP(hipGetLastError());
  std::vector<int32_t> hc((size_t)s.dim);
  SQ_HIP(hipMemcpyAsync(hc.data(), ucnt.p, sizeof(int32_t) * hc.size(), hipMemcpyDeviceToHost, st));
  SQ_HIP(hipStreamSynchronize(st));
  std::vector<int64_t> urow((size_t)s.dim + 1, 0);
  for (size_t i = 0; i < hc.size(); ++i) urow[i + 1] = urow[i] + hc[i];
  T->nu = urow.back();
  T->ncoef = (int)coefs.size();
  T->lpr = T->nu <= 32 * s.dim ? 16 : 32;
  SQ_HIP(hipMalloc(&T->urow, sizeof(int64_t) * urow.size()));
  SQ_HIP(hipMalloc(&T->col, sizeof(uint32_t) * (size_t)T->nu));
  SQ_HIP(hipMalloc(&T->first, sizeof(uint32_t) * ((size_t)T->nu + 1)));
  SQ_HIP(hipMalloc(&T->con, sizeof(uint32_t) * (size_t)c->nnz));
  SQ_HIP(hipMalloc(&T->coefs, sizeof(double) * coefs.size()));
  SQ_HIP(hipMalloc(&T->val, sizeof(double) * (size_t)T->nu));
  SQ_HIP(hipMalloc(&T->count, sizeof(double)));
  k_zero<<<1, 1, 0, st>>>(reinterpret_cast<double*>(T->count), 1);
  SQ_HIP(hipGetLastError());
  SQ_HIP(hipHostMalloc(reinterpret_cast<void**>(&T->host), sizeof(double) * (4 + (size_t)ng),
                       hipHostMallocPortable | hipHostMallocCoherent));
  SQ_HIP(hipEventCreateWithFlags(&T->busy, hipEventDisableTiming));
  SQ_HIP(hipMemcpyAsync(T->urow, urow.data(), sizeof(int64_t) * urow.size(), hipMemcpyHostToDevice, st));
  SQ_HIP(hipMemcpyAsync(T->coefs, coefs.data(), sizeof(double) * coefs.size(), hipMemcpyHostToDevice, st));
  const uint32_t end = (uint32_t)c->nnz;
  SQ_HIP(hipMemcpyAsync(T->first + T->nu, &end, sizeof(end), hipMemcpyHostToDevice, st));
  k_row_merge<<<(unsigned)((s.dim + kRows - 1) / kRows), 64 * kRows, 0, st>>>(
      s.dim, c->rowp, c->ent, (const uint32_t*)tword.p, T->urow, T->col, T->first, T->con);
  SQ_HIP(hipGetLastError());
  SQ_HIP(hipStreamSynchronize(st));
  p.ucc_t = T.release();
  return p.ucc_t;
}

bool operator_apply_pattern(const Space& s, sq_operator& op, const double* in, double* out, hipStream_t st) {
  if (!op.csr_tried) {
    op.csr_tried = true;
    if (!csr_enabled()) return false;
    op.d_fast = upload_term_fast(op.terms);
    op.csr = build_pattern(s, op.terms, op.d_terms, op.d_fast, kOpMaxEntries, st);
  }
  const UccCsr* c = op.csr;
  if (!c) return false;
  SQ_PROF(PC_TAPPLY, st, 16.0 * (double)s.dim + 8.0 * (double)c->nnz, 0.0,
          k_tapply_csr<<<(unsigned)((s.dim + kCsrRows - 1) / kCsrRows), 64 * kCsrRows, 0, st>>>(
              s.dim, c->rowp, c->ent, c->coef, in, out));
  return true;
}

void operator_pattern_free(sq_operator& op) {
  if (op.csr) ucc_csr_free(op.csr);
  op.csr = nullptr;
  if (op.d_fast) (void)hipFree(op.d_fast);
  op.d_fast = nullptr;
}

// Term groups of the split T application: enough (determinant, group)
// threads to fill the GPU for small spaces, at most 64 groups.
static int term_groups(const Space& s) {
  const int64_t G = 262144 / std::max<int64_t>(s.dim, 1);
  return (int)std::max<int64_t>(1, std::min<int64_t>(64, G));
}

// Work of the term-scan routines (doubles), carved in this order.
struct UccWork {
  double *A, *B, *C, *D, *w, *part, *dpart, *partial, *scal;
};

static int64_t dot_blocks(const Space& s) { return (s.dim + kUB - 1) / kUB; }

static int gate_groups(const Space& s, int ng) {
  const int64_t nb = dot_blocks(s);
  return (int)std::max<int64_t>(1, std::min<int64_t>(ng, std::max<int64_t>(1, 512 / nb)));
}

static int64_t scan_work_doubles(const Space& s, const Program& p) {
  const int64_t ng = (int64_t)std::max<size_t>(p.gates.size(), 1);
  return 4 * s.dim + (int64_t)p.terms.size() + 64 + (int64_t)term_groups(s) * s.dim + dot_blocks(s) * ng + 1024 + 64;
}

static UccWork carve_ucc(const Space& s, const Program& p, double* work) {
  UccWork u;
  const int64_t ng = (int64_t)std::max<size_t>(p.gates.size(), 1);
  u.A = work;
  u.B = u.A + s.dim;
  u.C = u.B + s.dim;
  u.D = u.C + s.dim;
  u.w = u.D + s.dim;
  u.part = u.w + p.terms.size() + 64;
  u.dpart = u.part + (size_t)term_groups(s) * s.dim;
  u.partial = u.dpart + (size_t)dot_blocks(s) * ng;
  u.scal = u.partial + 1024;
  return u;
}

// Largest nu t of one series and the nodes it needs: the n-point
// Gauss-Legendre rule on an interval of length h integrates frequencies up to
// omega = 2 nu with an error below h (n!)^4 / ((2n+1) (2n)!^3) (h omega)^2n
// max|f|: 1e-13 at h nu = 2, 5.5 and 9.7 for n = 8, 12 and 16.  Spaces above
// 2^22 determinants take h nu <= 2 (24 basis vectors and 8 nodes of
// workspace instead of 44 and 16).
constexpr int kNormSteps = 16;  // products of the norm estimate (and head of the Taylor series)
static double nu_limit(const Space& s) { return s.dim > ((int64_t)1 << 22) ? 2.0 : 9.7; }
static int max_nodes(const Space& s) { return s.dim > ((int64_t)1 << 22) ? 8 : 16; }
static int max_basis(const Space& s) { return s.dim > ((int64_t)1 << 22) ? 24 : kMaxBasis; }

// Work of the merged-pattern routines (doubles): U nodes | scal | rmax |
// basis | V nodes | C | D | dpart; from basis on it also serves sigma.
struct ChebWork {
  double *U, *scal, *rmax, *basis, *V, *C, *D, *dpart;
};

constexpr int kAsmBlocks = 2048;
static int64_t row_blocks(const Space& s, int64_t cap) { return std::min<int64_t>((s.dim + kRows - 1) / kRows, cap); }

static int64_t cheb_head(const Space& s) { return (int64_t)max_nodes(s) * s.dim + 64 + kAsmBlocks; }
static int64_t cheb_tail(const Space& s, int64_t ng) {
  return (int64_t)(max_basis(s) + max_nodes(s) + 2) * s.dim + std::max(ng, row_blocks(s, 1024) * std::min<int64_t>(ng, kLdsGates));
}

static ChebWork carve_cheb(const Space& s, double* work) {
  ChebWork u;
  u.U = work;
  u.scal = u.U + (size_t)max_nodes(s) * s.dim;
  u.rmax = u.scal + 64;
  u.basis = u.rmax + kAsmBlocks;
  u.V = u.basis + (size_t)max_basis(s) * s.dim;
  u.C = u.V + (size_t)max_nodes(s) * s.dim;
  u.D = u.C + s.dim;
  u.dpart = u.D + s.dim;
  return u;
}

static int64_t ucc_work_doubles(const Space& s, const Program& p) {
  const int64_t ng = (int64_t)std::max<size_t>(p.gates.size(), 1);
  int64_t n = std::max<int64_t>(scan_work_doubles(s, p), sigma_work_bytes(s) / 8);
  if (64 * s.dim < ((int64_t)1 << 32))  // spaces the merged pattern can serve
    n = std::max<int64_t>(n, cheb_head(s) + std::max<int64_t>(cheb_tail(s, ng), sigma_work_bytes(s) / 8));
  return n;
}

// nxt = f T cur (w: term weights, nullptr for unit weights); acc += nxt.
static void tapply(const Space& s, const Program& p, const double* w, const double* cur, double f, double* nxt,
                   double* acc, double* part, hipStream_t st) {
  const int G = term_groups(s);
  int rows = G;  // part rows
  if (G >= kTG) {  // small space: fold kTG groups per block in LDS
    rows = (G + kTG - 1) / kTG;
    const dim3 grid((unsigned)((s.dim + 63) / 64), rows);
    SQ_PROF(PC_TAPPLY, st, 24.0 * (double)s.dim, 0.0,
            k_tapply_part<<<grid, 64 * kTG, 0, st>>>(sv(s), p.d_terms, term_fast(p), w, (int)p.terms.size(), G,
                                                      cur, part));
  } else {
    const dim3 grid((unsigned)((s.dim + kUB - 1) / kUB), G);
    SQ_PROF(PC_TAPPLY, st, 24.0 * (double)s.dim, 0.0,
            k_tapply_group<<<grid, kUB, 0, st>>>(sv(s), p.d_terms, term_fast(p), w, (int)p.terms.size(), G, cur,
                                                 part));
  }
  k_tapply_sum<<<(unsigned)((s.dim + kUB - 1) / kUB), kUB, 0, st>>>(part, rows, s.dim, f, nxt, acc);
  SQ_HIP(hipGetLastError());
}

static double read_slot(const double* scal, int slot, hipStream_t st) {
  double h = 0.0;
  SQ_HIP(hipMemcpyAsync(&h, scal + slot, sizeof(double), hipMemcpyDeviceToHost, st));
  SQ_HIP(hipStreamSynchronize(st));
  return h;
}

// Terms of a Taylor series of exp(t T) with |t| ||T||_2 <= r: the smallest K
// with r^K / K! < 2^-60 (at most 60).
static int taylor_terms(double r) {
  int K = 1;
  double term = r;
  while (term > std::ldexp(1.0, -60) && K < 60) {
    ++K;
    term *= r / K;
  }
  return K;
}

// Taylor plan for exp(t T) with ||T||_2 <= nu: s steps of exp(t T / s) with
// |t| nu / s <= 2 and taylor_terms(|t| nu / s) terms per step (a radius of 2
// costs one bit to cancellation: the largest term is 2).
struct TaylorPlan {
  int steps, K;
  double a;  // t / steps
};

static TaylorPlan taylor_plan(double nu, double t) {
  const double b = std::fabs(t) * nu;
  TaylorPlan P;
  P.steps = std::max(1, (int)std::ceil(b / 2.0));
  P.K = taylor_terms(b / P.steps);
  P.a = t / P.steps;
  return P;
}

// ||T||_2 for the weights w: T is real antisymmetric (normal), so its
// 2-norm is its spectral radius.  Power iteration (16 steps from a fixed
// pseudo-random vector, in A and B) estimates it from below as
// ||T x_15|| / ||x_15||; the returned value is 1.5 x the estimate + 0.05,
// capped by the triangle-inequality bound b = sum_t |w_t coef_t| (each raw
// string has at most one unit entry per column).  The iterates are taken of
// T / b (norm <= 1), so they need no renormalisation between steps and the
// 16 products run back to back; two dots and one read-back finish it.  If
// they underflow (||T|| below 2^-60 b), the steps are rerun with a
// renormalisation each.
static double t_norm(const Space& s, const Program& p, const std::vector<double>& th, const UccWork& u,
                     hipStream_t st) {
  double bound = 0.0;
  for (size_t g = 0; g < p.gates.size(); ++g)
    for (int k = p.gates[g].term_begin; k < p.gates[g].term_end; ++k) bound += std::fabs(th[g] * p.terms[k].coef);
  if (bound == 0.0 || s.dim == 0) return 0.0;
  const unsigned nb = (unsigned)((s.dim + kUB - 1) / kUB);
  double* x = u.A;
  double* y = u.B;
  k_fill_pattern<<<nb, kUB, 0, st>>>(x, s.dim);
  SQ_HIP(hipGetLastError());
  for (int it = 0; it < 15; ++it) {
    tapply(s, p, u.w, x, 1.0 / bound, y, nullptr, u.part, st);  // y = (T / b) x
    std::swap(x, y);
  }
  tapply(s, p, u.w, x, 1.0 / bound, y, nullptr, u.part, st);
  dot_dev(x, x, s.dim, u.scal, 0, 1.0, u.partial, st);
  dot_dev(y, y, s.dim, u.scal, 1, 1.0, u.partial, st);
  double d[2];
  SQ_HIP(hipMemcpyAsync(d, u.scal, 2 * sizeof(double), hipMemcpyDeviceToHost, st));
  SQ_HIP(hipStreamSynchronize(st));
  double est;
  if (d[0] > 1e-200 && std::isfinite(d[1])) {
    est = bound * std::sqrt(std::max(0.0, d[1] / d[0]));
  } else {
    k_fill_pattern<<<nb, kUB, 0, st>>>(x, s.dim);
    SQ_HIP(hipGetLastError());
    for (int it = 0; it < 16; ++it) {
      dot_dev(x, x, s.dim, u.scal, 0, 1.0, u.partial, st);
      k_inv_sqrt_slot<<<1, 64, 0, st>>>(u.scal, 0, 1);
      k_scale<<<nb, kUB, 0, st>>>(x, s.dim, u.scal, 1);  // |x| = 1
      tapply(s, p, u.w, x, 1.0, y, nullptr, u.part, st);  // y = T x
      std::swap(x, y);
    }
    dot_dev(x, x, s.dim, u.scal, 0, 1.0, u.partial, st);
    est = std::sqrt(std::max(0.0, read_slot(u.scal, 0, st)));
  }
  return std::min(bound, 1.5 * est + 0.05);
}

// out = exp(t T) in over the plan for norm nu (A, B: Taylor terms).
static void expm_apply(const Space& s, const Program& p, const UccWork& u, double nu, double t, const double* in,
                       double* out, hipStream_t st) {
  const TaylorPlan P = taylor_plan(nu, t);
  if (in != out) copy_vec(in, out, s.dim, st);
  if (nu == 0.0) return;
  for (int step = 0; step < P.steps; ++step) {
    copy_vec(out, u.A, s.dim, st);
    double* cur = u.A;
    double* nxt = u.B;
    for (int k = 1; k <= P.K; ++k) {
      tapply(s, p, u.w, cur, P.a / k, nxt, out, u.part, st);
      std::swap(cur, nxt);
    }
  }
}

static std::vector<double> theta_host(const Program& p, const double* theta_dev, hipStream_t st) {
  const int ng = (int)p.gates.size();
  std::vector<double> th(ng);
  if (ng) SQ_HIP(hipMemcpyAsync(th.data(), theta_dev, sizeof(double) * ng, hipMemcpyDeviceToHost, st));
  SQ_HIP(hipStreamSynchronize(st));
  return th;
}

static void term_weights(const Program& p, const double* theta_dev, double* w, hipStream_t st) {
  const int ng = (int)p.gates.size();
  if (ng) k_term_weights<<<(ng + 255) / 256, 256, 0, st>>>(p.d_gates, ng, theta_dev, w);
  SQ_HIP(hipGetLastError());
}

// ---- Chebyshev series over the merged pattern ------------------------------

// n-point Gauss-Legendre nodes and weights on [0, 1] (Newton on P_n).
struct GaussRule {
  double x[16], w[16];
};

static const GaussRule& gauss_rule(int n) {
  auto make = [](int m) {
    GaussRule R{};
    for (int i = 0; i < m; ++i) {
      long double z = std::cos(3.14159265358979323846L * (i + 0.75L) / (m + 0.5L)), d = 1.0L;
      for (int it = 0; it < 100; ++it) {
        long double p0 = 1.0L, p1 = z;
        for (int k = 2; k <= m; ++k) {
          const long double p2 = ((2 * k - 1) * z * p1 - (k - 1) * p0) / k;
          p0 = p1;
          p1 = p2;
        }
        d = m * (z * p1 - p0) / (z * z - 1.0L);
        const long double dz = p1 / d;
        z -= dz;
        if (std::fabs(dz) < 1e-18L) break;
      }
      R.x[i] = (double)(0.5L * (1.0L - z));
      R.w[i] = (double)(1.0L / ((1.0L - z * z) * d * d));
    }
    return R;
  };
  static const GaussRule r8 = make(8), r12 = make(12), r16 = make(16);
  return n == 8 ? r8 : n == 12 ? r12 : r16;
}

// out[k] = (2 - delta_k0) J_k(x), k <= K: Miller's downward recurrence in
// long double, normalised by J_0 + 2 sum J_2k = 1.
static void cheb_coefs(double x, int K, double f, double* out) {
  const long double a = std::fabs((long double)x);
  if (!(a > 1e-300L)) {
    for (int k = 0; k <= K; ++k) out[k] = k == 0 ? f : 0.0;
    return;
  }
  const int M = K + 30 + (int)a;
  std::vector<long double> j(M + 2, 0.0L);
  j[M] = 1e-300L;
  for (int k = M; k > 0; --k) {
    j[k - 1] = 2.0L * k / a * j[k] - j[k + 1];
    if (std::fabs(j[k - 1]) > 1e250L)  // small arguments: rescale what is there
      for (int i = k - 1; i <= M; ++i) j[i] *= 1e-300L;
  }
  long double norm = j[0];
  for (int k = 2; k <= M; k += 2) norm += 2.0L * j[k];
  for (int k = 0; k <= K; ++k) {
    long double v = j[k] / norm * (k == 0 ? 1.0L : 2.0L);
    if (x < 0 && (k & 1)) v = -v;
    out[k] = (double)(v * f);
  }
}

static int cheb_terms(double r, int cap) {
  int K = 1;
  double term = r / 2;
  while (term > std::ldexp(1.0, -61) && K < cap) {
    ++K;
    term *= r / (2 * K);
  }
  return K;
}

// Guards a program's assembled T for one evaluation on st.
struct UccUse {
  UccT& T;
  std::unique_lock<std::mutex> lock;
  hipStream_t st;
  UccUse(UccT& t, hipStream_t stream) : T(t), lock(t.mu), st(stream) { SQ_HIP(hipStreamWaitEvent(st, T.busy, 0)); }
  ~UccUse() { (void)hipEventRecord(T.busy, st); }
};

static void spmv(const Space& s, const UccT& T, const double* cur, const double* prev, double f, const double* bound,
                 double* nxt, hipStream_t st, const double* cur2 = nullptr, double* nxt2 = nullptr) {
  auto* kernel = cur2 ? (T.lpr == 16 ? k_spmv<16, true> : k_spmv<32, true>)
                      : (T.lpr == 16 ? k_spmv<16, false> : k_spmv<32, false>);
  const int64_t rows = kUB / T.lpr;
  SQ_PROF(PC_TAPPLY, st, (cur2 ? 32.0 : 16.0) * (double)s.dim + 12.0 * (double)T.nu, 0.0,
          kernel<<<(unsigned)((s.dim + rows - 1) / rows), kUB, 0, st>>>(s.dim, T.urow, T.col, T.val, cur, cur2, prev, f,
                                                                      bound, nxt, nxt2));
}

// A series of exp(t T): basis[k] = (T / scale)^k in (taylor) or
// phi_k(T / scale) in, k <= K.
struct Series {
  bool taylor;
  double nu;     // >= ||T||_2
  double bound;  // largest row sum of |T|
  int K;
  double scale() const { return taylor ? bound : nu; }
  void coefs(double t, double f, double* out) const {
    if (!taylor) return cheb_coefs(nu * t, K, f, out);
    long double c = f;
    for (int k = 0; k <= K; ++k) {
      out[k] = (double)c;
      c *= (long double)t * bound / (k + 1);
    }
  }
};

// Basis vectors from + 1 .. K (basis[from] and, for from > 0, those before are there).
static void series_basis(const Space& s, const UccT& T, const Series& S, int from, const ChebWork& u,
                         hipStream_t st) {
  for (int k = from + 1; k <= S.K; ++k) {
    double* n = u.basis + (size_t)k * s.dim;
    const bool three = !S.taylor && k > 1;
    spmv(s, T, n - s.dim, three ? n - 2 * s.dim : nullptr, (three ? 2.0 : 1.0) / S.scale(), nullptr, n, st);
  }
}

// nodes[I][q] = f_q exp(t_q T) in (q < n) and fin = exp(tfin T) in; the last
// launch clears zero.
static void series_combine(const Space& s, const Series& S, int n, const double* t, const double* f, double* nodes,
                           double tfin, double* fin, const ChebWork& u, hipStream_t st, double* zero = nullptr) {
  for (int q0 = 0; q0 == 0 || q0 < n; q0 += kMaxOut - 1) {
    Combine C{};
    const int nq = std::min(kMaxOut - 1, n - q0);
    for (int q = 0; q < nq; ++q) S.coefs(t[q0 + q], f ? f[q0 + q] : 1.0, C.c[q]);
    double* out = q0 == 0 ? fin : nullptr;
    if (out) S.coefs(tfin, 1.0, C.c[kMaxOut - 1]);
    SQ_PROF(PC_OTHER, st, 8.0 * (double)s.dim * (S.K + 1 + nq + 1), 0.0,
            k_combine<<<(unsigned)((s.dim + kCB - 1) / kCB), kCB, 0, st>>>(s.dim, S.K, C, nq, u.basis, nodes + q0, n, out,
                                                                       q0 + kMaxOut - 1 >= n ? zero : nullptr));
  }
}

// Assembles T(theta), puts v into basis[0] and runs the first products on it
// and on the pseudo-random vector.  Returns the series for |t| <= 1 on an
// interval of length 1 / m; *done: basis vectors that are there.
static Series series_start(const Space& s, const Program& p, const UccT& T, const double* theta, const double* v,
                           double tmax, const ChebWork& u, int* m, int* done, hipStream_t st) {
  const int ng = (int)p.gates.size();
  const unsigned nb = (unsigned)row_blocks(s, kAsmBlocks);
  SQ_PROF(PC_OTHER, st, 12.0 * (double)T.nu, 0.0,
          k_assemble<<<nb, 64 * kRows, ng <= kLdsGates ? 8 * (size_t)ng : 0, st>>>(
              s.dim, T.urow, T.first, T.con, T.coefs, T.ncoef, theta, ng, T.val, u.rmax, v, u.basis, u.C));
  k_max<<<1, kUB, 0, st>>>(u.rmax, (int)nb, u.scal);
  SQ_HIP(hipGetLastError());
  double* x = u.C;
  double* y = u.D;
  for (int k = 1; k <= kNormSteps; ++k) {
    double* n = u.basis + (size_t)k * s.dim;
    spmv(s, T, n - s.dim, nullptr, 1.0, u.scal, n, st, x, y);
    std::swap(x, y);
  }
  k_norms<<<(unsigned)std::min<int64_t>((s.dim + kUB - 1) / kUB, 256), kUB, 0, st>>>(y, x, s.dim, u.scal, u.rmax,
                                                                                  T.count, T.host);
  SQ_HIP(hipGetLastError());
  SQ_HIP(hipStreamSynchronize(st));
  const double* d = T.host;
  Series S{};
  S.bound = S.nu = d[0];
  if (!std::isfinite(d[0])) S.bound = S.nu = 1.0;  // the result is NaN whatever the series
  else if (d[1] > 1e-200 && std::isfinite(d[2])) S.nu = std::min(d[0], 1.5 * d[0] * std::sqrt(d[2] / d[1]) + 0.05);
  const double r = S.nu * tmax;
  *m = std::max(1, (int)std::ceil(std::min(r / nu_limit(s), 1e9)));
  *done = 0;
  if (r == 0.0 || S.bound <= kTinyBound) {  // K = 0: the identity
    S.taylor = true;
  } else if (r <= 2.0 && S.bound < 1e6) {
    S.taylor = true;
    S.K = std::min(taylor_terms(r), max_basis(s) - 1);
    *done = std::min(S.K, kNormSteps);
  } else {
    S.K = cheb_terms(r / *m, max_basis(s) - 1);
  }
  return S;
}

// out = exp(t T) in, in m steps; the first step's basis is there up to done.
static void series_expm(const Space& s, const UccT& T, const Series& S, int m, int done, double t, double* out,
                        const ChebWork& u, hipStream_t st) {
  for (int k = 0; k < m; ++k) {
    if (k > 0) copy_vec(out, u.basis, s.dim, st);
    series_basis(s, T, S, k == 0 ? done : 0, u, st);
    series_combine(s, S, 0, nullptr, nullptr, u.U, t / m, out, u, st);
  }
}

static void gate_dots(const Space& s, const UccT& T, int n, int ng, const ChebWork& u, bool add, double* grad_dev,
                      double* grad_host, hipStream_t st) {
  // a copy of the sums per wave where two blocks fit a CU, or where a fixed order
  // is asked for, then at most kLdsGates gates per launch
  const bool det = sigma_deterministic(s);
  const int copies = det || ng <= kLdsGates / 2 ? kRows : ng <= kLdsGates ? 1 : 0;
  const unsigned nb = (unsigned)row_blocks(s, 1024);
  auto* kernel = n == 8 ? k_gate_dots_rows<8> : n == 12 ? k_gate_dots_rows<12> : k_gate_dots_rows<16>;
  const int per = copies ? std::min(ng, kLdsGates) : ng;
  const size_t lds = 8 * (size_t)copies * per;
  allow_lds(kernel, lds + 2048);
  if (!copies) k_zero<<<(unsigned)((ng + kUB - 1) / kUB), kUB, 0, st>>>(u.dpart, ng);
  for (int g0 = 0; g0 < ng; g0 += per) {
    const int m = std::min(per, ng - g0);
    SQ_PROF(PC_OTHER, st, 12.0 * (double)T.nu, 0.0,
            kernel<<<nb, 64 * kRows, lds, st>>>(s.dim, T.urow, T.col, T.first, T.con, T.coefs, T.ncoef, u.U, u.V, g0, m,
                                               copies, u.dpart));
    k_gate_accum<<<(unsigned)((m + kRows - 1) / kRows), 64 * kRows, 0, st>>>(
        u.dpart, copies ? (int)nb : 1, m, 1.0, add ? 1 : 0, grad_dev + g0, grad_host ? grad_host + g0 : nullptr);
  }
  SQ_HIP(hipGetLastError());
}

// Energy and gradient (grad may be nullptr; gdev: ng doubles) through the merged
// pattern.  grad_i = 2 int_0^1 <e^{-sT} lam | T_i | e^{-sT} psi> ds, and
// e^{-sT} psi = e^{(1-s)T} psi0: one interval while nu <= the limit, with psi's
// nodes from the forward series; else m intervals, both states propagated
// back through them.  With one interval and a sigma that adds into a zeroed
// vector, the last launch of the forward series clears basis[0] and sigma
// writes lam there.
static void cheb_energy_grad(const Space& s, const Program& p, UccT& T, const Hamiltonian& H, const double* theta,
                             const double* psi0, double* psi, double* lam, double* gdev, double* energy, double* grad,
                             double* work, hipStream_t st) {
  UccUse use(T, st);
  const ChebWork u = carve_cheb(s, work);
  const int ng = (int)p.gates.size();
  double *e_host = T.host + 3, *g_host = T.host + 4;
  int m, done;
  const Series S = series_start(s, p, T, theta, psi0, 1.0, u, &m, &done, st);
  const double r = S.nu / m;
  const int n = r <= 2.0 ? 8 : r <= 5.5 ? 12 : 16;
  const GaussRule& R = gauss_rule(n);
  double t[16], f[16];
  const bool direct = m == 1 && sigma_wants_zero(s, H);
  if (m == 1) {
    series_basis(s, T, S, done, u, st);
    for (int q = 0; q < n; ++q) t[q] = 1.0 - R.x[q];
    series_combine(s, S, grad ? n : 0, t, nullptr, u.U, 1.0, psi, u, st, direct ? u.basis : nullptr);
  } else {
    series_expm(s, T, S, m, done, 1.0, psi, u, st);
  }
  if (direct) lam = u.basis;
  double* epart = nullptr;
  // sigma's work: from the nodes of lam on where lam is basis[0]
  const int64_t ne = sigma_partials_dev(s, H, psi, lam, direct ? u.V : u.basis, &epart, direct, st);
  reduce_impl(epart, ne, e_host, 0, false, 1.0, st);
  if (grad) {
    for (int q = 0; q < n; ++q) {
      t[q] = -R.x[q] / m;
      f[q] = 2.0 * R.w[q] / m;
    }
    const double* c = psi;
    const double* d = lam;
    for (int j = 0; j < m; ++j) {
      if (m > 1) {
        copy_vec(c, u.basis, s.dim, st);
        series_basis(s, T, S, 0, u, st);
        series_combine(s, S, n, t, nullptr, u.U, -1.0 / m, u.C, u, st);
        c = u.C;
      }
      copy_vec(d, u.basis, s.dim, st);
      series_basis(s, T, S, 0, u, st);
      series_combine(s, S, n, t, f, u.V, -1.0 / m, j + 1 < m ? u.D : nullptr, u, st);
      d = u.D;
      gate_dots(s, T, n, ng, u, j > 0, gdev, j + 1 == m ? g_host : nullptr, st);
    }
  }
  SQ_HIP(hipStreamSynchronize(st));
  *energy = *e_host;
  if (grad) std::memcpy(grad, g_host, sizeof(double) * ng);
}

// out = exp(t T(theta)) in.  work: ucc_work_doubles.
void ucc_expm_impl(const Space& s, const Program& p, const double* theta_dev, double t, const double* in,
                   double* out, double* work, hipStream_t st) {
  if (UccT* T = ucc_t(s, p, st)) {
    UccUse use(*T, st);
    const ChebWork u = carve_cheb(s, work);
    int m, done;
    const Series S = series_start(s, p, *T, theta_dev, in, std::fabs(t), u, &m, &done, st);
    series_expm(s, *T, S, m, done, t, out, u, st);
    return;
  }
  const UccWork u = carve_ucc(s, p, work);
  const std::vector<double> th = theta_host(p, theta_dev, st);
  term_weights(p, theta_dev, u.w, st);
  const double nu = t_norm(s, p, th, u, st);
  expm_apply(s, p, u, nu, t, in, out, st);
}

// The gradient without a pattern: composite 8-point Gauss-Legendre over m
// subintervals of length h with h * 2 nu <= 4, psi and lam propagated from
// node to node (C, D), every node adding all gates' dots in one pass.
static void ucc_grad_impl(const Space& s, const Program& p, const UccWork& u, double nu, const double* psi,
                          const double* lam, double* grad_dev, hipStream_t st) {
  const int ng = (int)p.gates.size();
  const int m = std::max(1, (int)std::ceil(0.5 * nu));
  const GaussRule& R = gauss_rule(8);
  copy_vec(psi, u.C, s.dim, st);
  copy_vec(lam, u.D, s.dim, st);
  k_zero<<<(unsigned)((ng + kUB - 1) / kUB), kUB, 0, st>>>(grad_dev, ng);
  SQ_HIP(hipGetLastError());
  const int nb = (int)dot_blocks(s);
  const dim3 dgrid(nb, gate_groups(s, ng));
  double prev = 0.0;
  for (int j = 0; j < m; ++j) {
    for (int q = 0; q < 8; ++q) {
      const double node = (j + R.x[q]) / m;
      const double ds = node - prev;
      expm_apply(s, p, u, nu, -ds, u.C, u.C, st);
      expm_apply(s, p, u, nu, -ds, u.D, u.D, st);
      prev = node;
      k_gate_dots<<<dgrid, kUB, 0, st>>>(sv(s), p.d_terms, term_fast(p), p.d_gates, ng, u.C, u.D, u.dpart);
      k_gate_accum<<<(unsigned)((ng + kRows - 1) / kRows), 64 * kRows, 0, st>>>(u.dpart, nb, ng, 2.0 * R.w[q] / m, 1,
                                                                             grad_dev, nullptr);
      SQ_HIP(hipGetLastError());
    }
  }
}

}  // namespace sq

using namespace sq;

extern "C" {

int sq_ucc_expm(const sq_space* sp, const sq_program* pr, const double* theta, double t, const double* in,
                double* out, void* work_v, void* stream) {
  double* work = static_cast<double*>(work_v);
  return guarded([&] {
    SQ_CHECK(sp && pr && in && out && work && (theta || pr->p.gates.empty()), SQ_ERR_ARG, "NULL argument");
    SQ_CHECK(in != out, SQ_ERR_ARG, "in and out must differ");
    SQ_CHECK(pr->p.space == &sp->s, SQ_ERR_ARG, "program built for another space");
    ucc_expm_impl(sp->s, pr->p, theta, t, in, out, work, as_stream(stream));
  });
}

int sq_ucc_energy_grad(const sq_space* sp, const sq_program* pr, const sq_hamiltonian* H, const double* theta,
                       const double* psi0, double* energy, double* grad, void* work_v, void* stream) {
  double* work = static_cast<double*>(work_v);
  return guarded([&] {
    SQ_CHECK(sp && pr && H && psi0 && energy && work && (theta || pr->p.gates.empty()), SQ_ERR_ARG, "NULL argument");
    SQ_CHECK(pr->p.space == &sp->s && H->h.space == &sp->s, SQ_ERR_ARG,
             "program / Hamiltonian built for another space");
    const Space& s = sp->s;
    const Program& p = pr->p;
    const int ng = (int)p.gates.size();
    hipStream_t st = as_stream(stream);
    double* psi = work;
    double* lam = psi + s.dim;
    double* scal = lam + s.dim;            // 64
    double* gdev = scal + 64;              // ng
    double* rest = gdev + std::max(ng, 1) + 64;
    if (UccT* T = ucc_t(s, p, st)) {
      cheb_energy_grad(s, p, *T, H->h, theta, psi0, psi, lam, gdev, energy, grad && ng ? grad : nullptr, rest, st);
      return;
    } else {
      const UccWork u = carve_ucc(s, p, rest);
      const std::vector<double> th = theta_host(p, theta, st);
      term_weights(p, theta, u.w, st);
      const double nu = t_norm(s, p, th, u, st);
      expm_apply(s, p, u, nu, 1.0, psi0, psi, st);
      sigma_energy_dev(s, H->h, psi, lam, scal, rest, st);  // reuses the UCC work area
      if (grad && ng) {
        term_weights(p, theta, u.w, st);
        ucc_grad_impl(s, p, u, nu, psi, lam, gdev, st);
      }
    }
    if (grad && ng) SQ_HIP(hipMemcpyAsync(grad, gdev, sizeof(double) * ng, hipMemcpyDeviceToHost, st));
    SQ_HIP(hipMemcpyAsync(energy, scal, sizeof(double), hipMemcpyDeviceToHost, st));
    SQ_HIP(hipStreamSynchronize(st));
  });
}

int64_t sq_ucc_work_bytes(const sq_space* sp, const sq_program* pr) {
  if (!sp || !pr) return -1;
  const Space& s = sp->s;
  const int64_t ng = (int64_t)pr->p.gates.size() + 1;
  return 8 * (2 * s.dim + 64 + ng + 64 + ucc_work_doubles(s, pr->p));
}

}  // extern "C"
