// Whole gate sweeps of small spaces in one workgroup (replaces the gate loop
// of construct_ups_state and the gradient sweep, operator_state_algebra.py:
// 963-1412, ups_wavefunction.py:1060-1142, for spaces whose state vectors fit
// a CU's LDS).
//
// A gate outside the brick-wall layouts (factorised UCC: excitations between
// any orbitals) touches a few hundred determinant pairs of a small space, far
// too few to fill a launch: one launch per gate and direction is launch
// latency and nothing else ((8e,8o) fUCCSD: 360 gates, 1078 launches of
// 2-4 us, 4.0 ms per energy and gradient).  Here one block of 512 threads
// holds psi (and lambda in the reverse sweep) in LDS and runs every gate, one
// barrier per gate.
//
//   * A rotation (GC_ROT, each half of GC_SA_SINGLE) is a list of determinant
//     pairs, built once per program on the host: 13-bit indices i, j and the
//     sign, one 32-bit word per pair.  The words of a gate are loaded two
//     gates ahead into registers, by every thread on every path, so that the
//     number in flight is known at each wait and their L2 latency is off the
//     chain (loaded under a condition, each step waited for the words of the
//     next: (8e,8o) forward sweep 146 -> 126 us, reverse 260 -> 206).  512
//     threads: fewer idle waves to issue for (an evaluation 1024: 414 us, 512:
//     359, 256: 400).
//   * The other gates are polynomials in T (multi-frequency spin-adapted
//     doubles).  T couples a determinant to few others: its connected
//     components have at most kMaxComp members.  Members are ordered by their
//     occupation of the gate's orbitals and given signs that make the
//     component's matrix T_c one of a handful per program, so that the gate
//     is one small matrix-vector product per component, a thread per row:
//       M_c(theta) = 1 + sum_f sin(S_f theta) D_f + (cos(S_f theta) - 1) C_f,
//       D_f = sum_{k odd} K_kf T_c^k,  C_f = sum_{k even} K_kf T_c^k
//     with the polynomial's frequencies S_f and coefficients K; D_f and C_f
//     are summed on the host in long double.  T_c is antisymmetric, so the
//     inverse gate is the transpose.  The matrices of a chunk of gates are
//     made at once in the LDS that psi and lambda leave ((6e,6o) spin-adapted:
//     228 -> 187 us an evaluation; gate by gate their two dependent loads were
//     half of a step; a thread per row instead of one per component, whose m x m
//     products were one chain: 180 -> 123 us).  (The per-gate kernels take eight to ten passes of every
//     term over every determinant per polynomial gate and vector.)
//   * The gradient 2 <lambda|T psi> of a gate is summed per thread, reduced
//     in each wave and added over the waves by one of them during the next
//     gate: no extra barrier.
//
// Energy and gradient, per-gate kernels -> this sweep: fUCCSD (8e,8o) 3.86 ->
// 0.35 ms, spin-adapted fUCCSD (6e,6o) 11.1 -> 0.12 ms.

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <vector>

#include "sq_internal.h"

namespace sq {

namespace {

constexpr int kST = 512;                  // threads of the one block
constexpr int kSW = kST / 64;             // its waves
constexpr int kSmallDim = 8192;           // 13-bit determinant indices
constexpr int kMaxComp = 8;               // members of a component of T
constexpr int kChunk = 256;               // steps (and trig slots) staged in LDS at a time
constexpr size_t kSmallEntries = 1 << 25; // pair words per program (128 MB)
constexpr int kDiag = 1 << 16;            // flag of a diagonal matrix element
constexpr size_t kSmallLds = 160 * 1024 - 1024;

// One step: a rotation half (nf = 0: pair words [e0, e0 + n)) or a polynomial
// gate (rows of components [e0, e0 + n), its matrix elements from m0 in the chunk's).
// slot: first trig slot within the step's chunk.
struct SmallStep {
  int32_t gate, nf, e0, n, slot, m0, pad[2];
};

// A matrix element of a gate: its place in the type's coefficients, their
// stride (| kDiag), the gate's first trig slot and its frequencies.
struct MatElem {
  int32_t off, stride, slot, nf;
};

struct TrigSlot {
  double scale;
  int32_t gate, pad;
};

struct SmallChunk {
  int32_t s0, s1, t0, t1, m0, m1;  // steps [s0, s1), trig slots [t0, t1), matrix elements [m0, m1)
};

}  // namespace

struct SmallPlan {
  int nchunks = 0, maxmat = 0;
  bool poly = false;
  SmallStep* steps = nullptr;
  SmallChunk* chunks = nullptr;
  TrigSlot* slots = nullptr;
  uint32_t* pairs = nullptr;
  uint4* members = nullptr;  // per row of a component: its kMaxComp members (index | negative << 15)
  uint32_t* meta = nullptr;  // and size | row << 4 | matrix offset << 8
  MatElem* mel = nullptr;
  double* ctab = nullptr;    // per type: T | D_0 | C_0 | D_1 | ...
  uint8_t* nograd = nullptr; // per gate: 1 where the generator is zero (gradient 0)
  int ngates = 0;
  size_t lds_fwd = 0, lds_rev = 0;
  ~SmallPlan() {
    for (void* p : {(void*)steps, (void*)chunks, (void*)slots, (void*)pairs, (void*)members, (void*)meta, (void*)mel,
                    (void*)ctab, (void*)nograd})
      if (p) (void)hipFree(p);
  }
};

void small_plan_free(SmallPlan* P) { delete P; }

namespace {

template <class T>
T* put(const std::vector<T>& v) {
  T* d = nullptr;
  SQ_HIP(hipMalloc(&d, sizeof(T) * std::max<size_t>(v.size(), 1)));
  if (!v.empty()) SQ_HIP(hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
  return d;
}

size_t small_lds(int64_t dim, int maxmat, bool rev) {
  return (size_t)(dim + 1) / 2 * 16 * (rev ? 2 : 1) + (size_t)kChunk * (sizeof(double2) + sizeof(SmallStep) + 8) +
         (size_t)maxmat * 8 * (rev ? 2 : 1);
}

// Matrix elements per chunk: what the reverse sweep's LDS leaves, at most 64 KB.
int mat_room(int64_t dim) {
  const size_t base = small_lds(dim, 0, true);
  return base >= kSmallLds ? 0 : (int)std::min<size_t>((kSmallLds - base) / 16, 4096);
}

// A type of component: its size, polynomial and matrix.
struct CompType {
  int m, slot;
  std::vector<double> T;
  int off;  // into ctab
};

struct Builder {
  const Space& sp;
  const Program& P;
  std::vector<SmallStep> steps;
  std::vector<SmallChunk> chunks;
  std::vector<TrigSlot> slots;
  std::vector<uint32_t> pairs, meta;
  std::vector<uint4> members;
  std::vector<MatElem> mel;
  std::vector<double> ctab;
  std::vector<uint8_t> nograd;
  std::vector<CompType> types;
  std::vector<int2> lists;
  std::map<std::pair<const void*, std::vector<int>>, std::pair<int, int>> cache;
  int maxmat = 0;

  Builder(const Space& s, const Program& p) : sp(s), P(p) {}

  // (determinant, image, sign) of one operator product
  template <class F>
  void each(const Term& T, F&& f) {
    int ao, al, bo, bl;
    spin_part_list(sp.h_astr, T.a, lists, cache, ao, al);
    spin_part_list(sp.h_bstr, T.b, lists, cache, bo, bl);
    for (int r = 0; r < al; ++r) {
      const int2 A = ao < 0 ? int2{r, r} : lists[ao + r];
      for (int c = 0; c < bl; ++c) {
        const int2 B = bo < 0 ? int2{c, c} : lists[bo + c];
        f(A.x * sp.nsb + B.x, (A.y & 0x7fffffff) * sp.nsb + (B.y & 0x7fffffff), ((A.y ^ B.y) < 0) != (T.coef < 0));
      }
    }
  }

  // Opens a chunk when the running one has no room for a step of nt slots and
  // nm matrix elements.
  int open(int nt, int nm = 0) {
    if (chunks.empty() || chunks.back().s1 - chunks.back().s0 >= kChunk ||
        chunks.back().t1 - chunks.back().t0 + nt > kChunk ||
        chunks.back().m1 - chunks.back().m0 + nm > mat_room(sp.dim)) {
      const int s = (int)steps.size(), t = (int)slots.size(), m = (int)mel.size();
      chunks.push_back(SmallChunk{s, s, t, t, m, m});
    }
    SmallChunk& c = chunks.back();
    const int slot = c.t1 - c.t0;
    c.s1 += 1;
    c.t1 += nt;
    c.m1 += nm;
    maxmat = std::max(maxmat, c.m1 - c.m0);
    return slot;
  }

  void rotation(int g, const Term& T, double scale) {
    const int e0 = (int)pairs.size();
    each(T, [&](int i, int j, bool neg) { pairs.push_back((uint32_t)i | (uint32_t)j << 13 | (neg ? 0x80000000u : 0u)); });
    const int n = (int)pairs.size() - e0;
    const int slot = open(1);
    slots.push_back(TrigSlot{scale, g, 0});
    steps.push_back(SmallStep{g, 0, e0, n, slot, 0, {0, 0}});
  }

  int type_of(int m, int slot, const std::vector<double>& T, const GatePoly& poly) {
    for (size_t k = 0; k < types.size(); ++k) {
      if (types[k].m != m || types[k].slot != slot) continue;
      bool same = true;
      for (int e = 0; e < m * m && same; ++e) same = std::fabs(types[k].T[e] - T[e]) < 1e-14;
      if (same) return (int)k;
    }
    CompType t{m, slot, T, (int)ctab.size()};
    const int mm = m * m;
    ctab.insert(ctab.end(), T.begin(), T.end());
    std::vector<long double> pw(T.begin(), T.end()), nx(mm);
    std::vector<long double> acc((size_t)2 * poly.nf * mm, 0.0L);
    for (int k = 1; k <= poly.nk; ++k) {
      for (int f = 0; f < poly.nf; ++f) {
        long double* a = acc.data() + (size_t)(2 * f + ((k & 1) ? 0 : 1)) * mm;
        for (int e = 0; e < mm; ++e) a[e] += (long double)poly.K[k - 1][f] * pw[e];
      }
      for (int a = 0; a < m; ++a)
        for (int b = 0; b < m; ++b) {
          long double v = 0.0L;
          for (int c = 0; c < m; ++c) v += (long double)T[a * m + c] * pw[c * m + b];
          nx[a * m + b] = v;
        }
      pw.swap(nx);
    }
    for (long double v : acc) ctab.push_back((double)v);
    types.push_back(std::move(t));
    return (int)types.size() - 1;
  }

  // false: a component is too large or T is not antisymmetric
  bool polynomial(int g) {
    const GateDev& gd = P.gates[g];
    const GatePoly poly = gate_poly(gd);
    struct Ent {
      int i, j;
      double v;
    };
    std::vector<Ent> ent;
    uint32_t orbs = 0;
    for (int t = gd.term_begin; t < gd.term_end; ++t) {
      const Term& T = P.terms[t];
      for (int o = 0; o < T.a.n; ++o) orbs |= 1u << T.a.orb[o];
      for (int o = 0; o < T.b.n; ++o) orbs |= 1u << T.b.orb[o];
      // <j|T|i>
      each(T, [&](int i, int j, bool neg) { ent.push_back(Ent{j, i, neg ? -std::fabs(T.coef) : std::fabs(T.coef)}); });
    }
    std::vector<int> root(sp.dim, -1), comp(sp.dim, -1), loc(sp.dim, 0), touched;
    auto find = [&](int x) {
      while (root[x] != x) x = root[x] = root[root[x]];
      return x;
    };
    for (const Ent& e : ent) {
      for (int x : {e.i, e.j})
        if (root[x] < 0) {
          root[x] = x;
          touched.push_back(x);
        }
      const int a = find(e.i), b = find(e.j);
      if (a != b) root[std::max(a, b)] = std::min(a, b);
    }
    // members of a component by their occupation of the gate's orbitals
    auto code = [&](int x) {
      const uint64_t a = sp.h_astr[x / sp.nsb] & orbs, b = sp.h_bstr[x % sp.nsb] & orbs;
      return a << 32 | b;
    };
    std::sort(touched.begin(), touched.end(), [&](int x, int y) {
      const int rx = find(x), ry = find(y);
      if (rx != ry) return rx < ry;
      return code(x) < code(y);
    });
    struct Comp {
      int x0, m, type;
      uint32_t neg;
    };
    std::vector<Comp> comps;
    for (int k = 0; k < (int)touched.size(); ++k) {
      const int x = touched[k];
      if (k == 0 || find(touched[k - 1]) != find(x)) comps.push_back(Comp{k, 0, 0, 0});
      Comp& c = comps.back();
      loc[x] = c.m++;
      comp[x] = (int)comps.size() - 1;
      if (c.m > kMaxComp) return false;
    }
    std::vector<double> mats(comps.size() * kMaxComp * kMaxComp, 0.0);
    for (const Ent& e : ent) {
      const Comp& c = comps[comp[e.i]];
      mats[(size_t)comp[e.i] * kMaxComp * kMaxComp + loc[e.i] * c.m + loc[e.j]] += e.v;
    }
    for (size_t k = 0; k < comps.size(); ++k) {
      Comp& c = comps[k];
      double* T = mats.data() + k * kMaxComp * kMaxComp;
      for (int a = 0; a < c.m; ++a)
        for (int b = 0; b <= a; ++b)
          if (T[a * c.m + b] != -T[b * c.m + a]) return false;
      // signs: every member positive towards the member it is first reached from
      int order[kMaxComp], n = 0;
      bool seen[kMaxComp] = {false};
      for (int start = 0; start < c.m; ++start) {
        if (seen[start]) continue;
        seen[start] = true;
        int at = n;
        order[n++] = start;
        for (; at < n; ++at)
          for (int b = 0; b < c.m; ++b) {
            const double v = T[b * c.m + order[at]];
            if (seen[b] || v == 0.0) continue;
            seen[b] = true;
            order[n++] = b;
            const bool neg = (v < 0) != (((c.neg >> order[at]) & 1u) != 0);
            if (neg) c.neg |= 1u << b;
          }
      }
      std::vector<double> S(c.m * c.m);
      for (int a = 0; a < c.m; ++a)
        for (int b = 0; b < c.m; ++b) {
          const bool neg = (((c.neg >> a) ^ (c.neg >> b)) & 1u) != 0;
          S[a * c.m + b] = T[a * c.m + b] == 0.0 ? 0.0 : (neg ? -T[a * c.m + b] : T[a * c.m + b]);
        }
      c.type = type_of(c.m, gd.kind * 16 + gd.poly, S, poly);
    }
    std::stable_sort(comps.begin(), comps.end(), [](const Comp& a, const Comp& b) { return a.type < b.type; });
    const int c0 = (int)meta.size();
    int moff = -1, last = -1, used = 0;
    std::vector<MatElem> own;
    for (const Comp& c : comps) {
      const CompType& t = types[c.type];
      if (c.type != last) {
        last = c.type;
        moff = used;
        for (int e = 0; e < t.m * t.m; ++e)
          own.push_back(MatElem{t.off + e, t.m * t.m | (e % (t.m + 1) == 0 ? kDiag : 0), 0, poly.nf});
        used += t.m * t.m;
      }
      uint16_t w[kMaxComp] = {0};
      for (int a = 0; a < c.m; ++a)
        w[a] = (uint16_t)((uint32_t)touched[c.x0 + a] | ((c.neg >> a) & 1u) << 15);
      auto two = [&](int a) { return (uint32_t)w[a] | (uint32_t)w[a + 1] << 16; };
      if (c.m < 2) continue;
      while (((int)meta.size() - c0) % 64 + c.m > 64) {  // the rows of a component stay in one wave
        members.push_back(uint4{0u, 0u, 0u, 0u});
        meta.push_back(0u);
      }
      for (int a = 0; a < c.m; ++a) {
        members.push_back(make_uint4(two(0), two(2), two(4), two(6)));
        meta.push_back((uint32_t)c.m | (uint32_t)a << 4 | (uint32_t)moff << 8);
      }
    }
    const int slot = open(poly.nf, used);
    const int m0 = (int)mel.size() - chunks.back().m0;
    for (MatElem& e : own) e.slot = slot;
    mel.insert(mel.end(), own.begin(), own.end());
    for (int f = 0; f < poly.nf; ++f) slots.push_back(TrigSlot{poly.S[f], g, 0});
    steps.push_back(SmallStep{g, poly.nf, c0, (int)meta.size() - c0, slot, m0, {0, 0}});
    return true;
  }

  bool build() {
    nograd.assign(P.gates.size(), 0);
    for (int g = 0; g < (int)P.gates.size(); ++g) {
      const GateDev& gd = P.gates[g];
      if (gd.kind == GC_ROT) {
        rotation(g, P.terms[gd.term_begin], gd.scale);
      } else if (gd.kind == GC_SA_SINGLE) {
        rotation(g, P.terms[gd.term_begin], 1.0);
        rotation(g, P.terms[gd.term_begin + 2], 1.0);
      } else if (gd.term_end == gd.term_begin) {
        nograd[g] = 1;
      } else if (!polynomial(g)) {
        return false;
      }
      if (pairs.size() > kSmallEntries || meta.size() > kSmallEntries / 4) return false;
    }
    return true;
  }
};

// ---- device ---------------------------------------------------------------------

struct SmallDev {
  const SmallStep* steps;
  const SmallChunk* chunks;
  const TrigSlot* slots;
  const uint32_t* pairs;
  const uint4* members;
  const uint32_t* meta;
  const MatElem* mel;
  const double* ctab;
  const uint8_t* nograd;
  int nchunks, dim, maxmat, ngates;
};

constexpr int kAhead = 3;  // pairs of a step that a thread loads ahead

// What a thread needs of a step, loaded ahead: the step's record and trig
// values, and its first pairs or its first row of a component.
struct Ahead {
  int gate, nf, e0, n, m0;
  double c, sn, scale;
  uint32_t p[kAhead], meta;
  uint4 mem;
};

// One row of a component's matrix (M: the gate, T: its generator, both m x m in
// LDS) on its members; the transpose where inv.  The rows of a component are
// lanes of one wave, whose reads of the members all come before its writes.
// Returns the row's part of <lam|T psi> (REV).
template <int m, bool REV>
__device__ __forceinline__ double comp_row(double* X, double* L, const double* __restrict__ M,
                                           const double* __restrict__ T, const uint4& mem, int row, bool inv) {
  const uint32_t w[4] = {mem.x, mem.y, mem.z, mem.w};
  double x[m], l[m];
#pragma unroll
  for (int a = 0; a < m; ++a) {
    const uint32_t h = (w[a >> 1] >> (16 * (a & 1))) & 0xffffu;
    const double s = (h & 0x8000u) ? -1.0 : 1.0;
    x[a] = s * X[h & 0x7fffu];
    if (REV) l[a] = s * L[h & 0x7fffu];
  }
  const uint64_t half = m > 4 && row >= 4 ? (uint64_t)w[2] | (uint64_t)w[3] << 32 : (uint64_t)w[0] | (uint64_t)w[1] << 32;
  const uint32_t own = (uint32_t)(half >> (16 * (row & 3)));
  const int at = (int)(own & 0x7fffu);
  const double s = (own & 0x8000u) ? -1.0 : 1.0;
  const double mine = REV ? s * L[at] : 0.0;
  const double* Mr = M + (inv ? row : row * m);
  const int step = inv ? m : 1;
  double vx = 0.0, vl = 0.0, vt = 0.0;
#pragma unroll
  for (int b = 0; b < m; ++b) {
    const double e = Mr[b * step];
    vx += e * x[b];
    if (REV) {
      vl += e * l[b];
      vt += T[row * m + b] * x[b];
    }
  }
  X[at] = s * vx;
  if (REV) L[at] = s * vl;
  return mine * vt;
}

// meta: size | row << 4 | matrix offset << 8.
template <bool REV>
__device__ __forceinline__ double comp_any(double* X, double* L, const double* M, const double* T, uint32_t meta,
                                           const uint4& mem, bool inv) {
  const double* Mc = M + (meta >> 8);
  const double* Tc = T + (meta >> 8);
  const int row = (int)((meta >> 4) & 15u);
  switch (meta & 15u) {
    case 2: return comp_row<2, REV>(X, L, Mc, Tc, mem, row, inv);
    case 3: return comp_row<3, REV>(X, L, Mc, Tc, mem, row, inv);
    case 4: return comp_row<4, REV>(X, L, Mc, Tc, mem, row, inv);
    case 5: return comp_row<5, REV>(X, L, Mc, Tc, mem, row, inv);
    case 6: return comp_row<6, REV>(X, L, Mc, Tc, mem, row, inv);
    case 7: return comp_row<7, REV>(X, L, Mc, Tc, mem, row, inv);
    case 8: return comp_row<8, REV>(X, L, Mc, Tc, mem, row, inv);
    default: return 0.0;  // padding, or a single member: T = 0
  }
}

// What the launches of an energy and gradient call take along in further
// blocks, instead of launches and copies of their own ((6e,6o) spin-adapted 186
// -> 180 us an evaluation, (8e,8o) fUCCSD 358 -> 353): the forward sweep fills
// zero[0, nzero) with zeros and copies host theta to theta_out, the reverse
// sweep writes the sum of epart[0, nepart) to *e_out.
struct SmallExtra {
  double* zero = nullptr;
  double* theta_out = nullptr;
  const double* epart = nullptr;
  double* e_out = nullptr;
  int64_t nzero = 0, nepart = 0;
};

constexpr int kZeroBlocks = 4;

// REV = false: dst = U src (back: U^+ src).  REV = true: the reverse sweep on
// (src = psi, lam), gradients to grad; back is then true.
// Bound by the chain of barriers and LDS round trips, one per gate: the block
// uses one CU, and a gate's arithmetic is a few hundred cycles of it.
template <bool REV, bool POLY>
__global__ __launch_bounds__(kST) void k_small_sweep(SmallDev S, const double* theta, const double* src,
                                                     double* dst, const double* __restrict__ lam,
                                                     double* __restrict__ grad, int back, SmallExtra ex) {
  extern __shared__ double smem[];
  __shared__ double red[2][kSW];
  double* X = smem;
  const int dimp = (S.dim + 1) & ~1;  // 16-byte alignment of what follows
  double* L = X + (REV ? dimp : 0);
  double2* cs = reinterpret_cast<double2*>(L + dimp);
  SmallStep* steps = reinterpret_cast<SmallStep*>(cs + kChunk);
  double* scales = reinterpret_cast<double*>(steps + kChunk);
  double* mats = scales + kChunk;  // the chunk's gate matrices, [maxmat] | their generators
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool inv = REV || back;
  if (blockIdx.x != 0) {
    if (!REV) {
      for (int64_t i = (int64_t)(blockIdx.x - 1) * kST + tid; i < ex.nzero; i += (int64_t)(gridDim.x - 1) * kST)
        ex.zero[i] = 0.0;
    } else {
      double e = 0.0;
      for (int64_t i = tid; i < ex.nepart; i += kST) e += ex.epart[i];
      e = wave_sum63(e);
      if (lane == 63) red[0][wave] = e;
      __syncthreads();
      if (tid == 0) {
        e = 0.0;
        for (int w = 0; w < kSW; ++w) e += red[0][w];
        *ex.e_out = e;
      }
    }
    return;
  }
  if (!REV && ex.theta_out) {
    for (int g = tid; g < S.ngates; g += kST) ex.theta_out[g] = theta[g];
    theta = ex.theta_out;  // read again after the barrier below
  }
  for (int i = tid; i < S.dim; i += kST) {
    X[i] = src[i];
    if (REV) L[i] = lam[i];
  }
  if (REV)
    for (int g = tid; g < S.ngates; g += kST)
      if (S.nograd[g]) grad[g] = 0.0;
  // the running sum of the gate whose steps are being reduced
  int par = 0;
  int done_gate = -1;   // gate of the previous step
  int done_waves = 0;   // its waves with pairs or rows
  double done_sum = 0.0;
  SmallStep next{};     // the record of the step after the next but one
  for (int ci = 0; ci < S.nchunks; ++ci) {
    const SmallChunk C = S.chunks[inv ? S.nchunks - 1 - ci : ci];
    __syncthreads();
    for (int i = tid; i < C.s1 - C.s0; i += kST) steps[i] = S.steps[C.s0 + i];
    for (int i = tid; i < C.t1 - C.t0; i += kST) {
      const TrigSlot t = S.slots[C.t0 + i];
      const double th = theta[t.gate];
      double sn = 0.0, c = 1.0;
      if (!(fabs(th) < 1e-28)) sincos(t.scale * th, &sn, &c);  // NaN passes through
      cs[i] = double2{c, !POLY && inv ? -sn : sn};
      scales[i] = t.scale;
    }
    __syncthreads();
    if (POLY) {
      const int nm = C.m1 - C.m0;
      constexpr int U = 4;
      for (int e0 = tid; e0 < nm; e0 += U * kST) {
        MatElem me[U];
#pragma unroll
        for (int u = 0; u < U; ++u) me[u] = S.mel[C.m0 + min(e0 + u * kST, nm - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const double* __restrict__ c = S.ctab + me[u].off;
          const int mm = me[u].stride & (kDiag - 1);
          double v = (me[u].stride & kDiag) ? 1.0 : 0.0;
          for (int f = 0; f < me[u].nf; ++f) {
            const double2 x = cs[me[u].slot + f];
            v += x.y * c[(2 * f + 1) * mm] + (x.x - 1.0) * c[(2 * f + 2) * mm];
          }
          if (e0 + u * kST < nm) {
            mats[e0 + u * kST] = v;
            if (REV) mats[S.maxmat + e0 + u * kST] = c[0];
          }
        }
      }
    }
    const int ns = C.s1 - C.s0;
    auto step_at = [&](int k) { return inv ? ns - 1 - k : k; };
    // A step's record is read from LDS one step before it is used, and what it
    // points to is loaded two steps ahead: no LDS round trip but the
    // amplitudes' own lies between two barriers.  Every load is issued on every
    // path (the lists are padded, past the last step the last one again), so
    // that a step waits for its own words and not for those of the next.
    auto record = [&](int k) { return steps[step_at(min(k, ns - 1))]; };
    auto load = [&](const SmallStep& r, Ahead& a) {
      a.gate = __builtin_amdgcn_readfirstlane(r.gate);
      a.nf = POLY ? __builtin_amdgcn_readfirstlane(r.nf) : 0;
      a.e0 = __builtin_amdgcn_readfirstlane(r.e0);
      a.n = __builtin_amdgcn_readfirstlane(r.n);
      const double2 x = cs[r.slot];
      a.c = x.x;
      a.sn = POLY && inv ? -x.y : x.y;
      if (REV) a.scale = scales[r.slot];
      const uint32_t* __restrict__ p = S.pairs + (POLY && a.nf != 0 ? 0 : a.e0);
#pragma unroll
      for (int q = 0; q < kAhead; ++q) a.p[q] = p[tid + q * kST];
      if (POLY) {
        a.m0 = __builtin_amdgcn_readfirstlane(r.m0);
        const int e = (a.nf != 0 ? a.e0 : 0) + tid;
        a.meta = S.meta[e];
        a.mem = S.members[e];
      }
    };
    struct Amps {
      double xi, xj, li, lj;
    };
    auto fetch = [&](uint32_t p, Amps& v) {
      const int i = (int)(p & 8191u), j = (int)((p >> 13) & 8191u);
      v.xi = X[i], v.xj = X[j];
      if (REV) v.li = L[i], v.lj = L[j];
    };
    auto rotate = [&](uint32_t p, const Amps& v, double c, double sn, double& dot) {
      const int i = (int)(p & 8191u), j = (int)((p >> 13) & 8191u);
      const double sg = (p >> 31) ? -sn : sn;
      X[i] = c * v.xi - sg * v.xj;
      X[j] = sg * v.xi + c * v.xj;
      if (REV) {
        L[i] = c * v.li - sg * v.lj;
        L[j] = sg * v.li + c * v.lj;
        const double d = v.lj * v.xi - v.li * v.xj;
        dot += (p >> 31) ? -d : d;
      }
    };
    // one wave (the last, which has the fewest pairs) adds the previous step's
    // wave sums to its gate's gradient
    auto finish = [&](int gate_now) {
      if (!REV || done_gate < 0) return;
      if (wave == kSW - 1) {
        double v = lane < done_waves ? red[par ^ 1][lane & (kSW - 1)] : 0.0;
        v = row16_sum(v);
        done_sum += v;
        if (gate_now != done_gate) {
          if (lane == 15) grad[done_gate] = 2.0 * done_sum;
          done_sum = 0.0;
        }
      }
    };
    auto step = [&](int k, Ahead& cur, Ahead& fill) {
      if (k >= ns) return;
      lds_barrier();
      const int n = cur.n, gate = cur.gate, e0 = cur.e0;
      double dot = 0.0;
      if (!POLY || cur.nf == 0) {
        Amps v[kAhead];
        fetch(cur.p[0], v[0]);
#pragma unroll
        for (int q = 1; q < kAhead; ++q)
          if (n > q * kST) fetch(cur.p[q], v[q]);
        load(next, fill);
        next = record(k + 3);
#pragma unroll
        for (int q = 0; q < kAhead; ++q)
          if (tid + q * kST < n) rotate(cur.p[q], v[q], cur.c, cur.sn, dot);
        for (int i = tid + kAhead * kST; i < n; i += kST) {
          const uint32_t p = S.pairs[e0 + i];
          fetch(p, v[0]);
          rotate(p, v[0], cur.c, cur.sn, dot);
        }
        if (REV) dot *= cur.scale;
      } else {
        load(next, fill);
        next = record(k + 3);
        const double* M = mats + cur.m0;
        const double* T = M + S.maxmat;
        if (tid < n) dot += comp_any<REV>(X, L, M, T, cur.meta, cur.mem, inv);
        for (int i = tid + kST; i < n; i += kST)
          dot += comp_any<REV>(X, L, M, T, S.meta[e0 + i], S.members[e0 + i], inv);
      }
      if (REV) {
        finish(gate);
        if (wave * 64 < n) {
          dot = wave_sum63(dot);
          if (lane == 63) red[par][wave] = dot;
        }
        done_gate = gate;
        done_waves = min((n + 63) >> 6, kSW);
        par ^= 1;
      }
    };
    Ahead a, b, c;
    load(record(0), a);
    load(record(1), b);
    next = record(2);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the loop's waits then count its own loads
    for (int k = 0; k < ns; k += 3) {
      step(k, a, c);
      step(k + 1, b, a);
      step(k + 2, c, b);
    }
  }
  __syncthreads();
  if (REV) {
    if (done_gate >= 0 && wave == kSW - 1) {
      double v = lane < done_waves ? red[par ^ 1][lane & (kSW - 1)] : 0.0;
      v = row16_sum(v);
      if (lane == 15) grad[done_gate] = 2.0 * (done_sum + v);
    }
  } else {
    for (int i = tid; i < S.dim; i += kST) dst[i] = X[i];
  }
}

SmallDev device_view(const Space& s, const SmallPlan& P) {
  return SmallDev{P.steps, P.chunks, P.slots, P.pairs, P.members, P.meta, P.mel, P.ctab, P.nograd,
                  P.nchunks, (int)s.dim, P.maxmat, P.ngates};
}

}  // namespace

// The plan of a program whose state vectors fit one block's LDS, nullptr
// where the sweep does not apply: larger spaces, polynomial gates with larger
// components, or programs that run in tile stages from the first gate to the
// last (a stage spreads over many CUs and takes about 1 us per orbital pair).
const SmallPlan* small_for(const Space& s, const Program& p) {
  std::lock_guard<std::recursive_mutex> lock(p.plan_mu);
  if (!p.small_tried) {
    p.small_tried = true;
    const char* env = getenv("SQ_SMALL_SWEEP");
    if ((env && env[0] == '0') || s.dim == 0 || s.dim > kSmallDim || p.gates.empty()) return nullptr;
    if (tiles_cover(s, p)) return nullptr;
    Builder B(s, p);
    if (!B.build()) return nullptr;
    const bool poly = !B.meta.empty();
    // a step's loads take whole blocks of words
    B.pairs.resize(B.pairs.size() + kAhead * kST, 0u);
    B.meta.resize(B.meta.size() + kST, 0u);
    B.members.resize(B.members.size() + kST, uint4{0u, 0u, 0u, 0u});
    const size_t lds_rev = small_lds(s.dim, B.maxmat, true);
    if (lds_rev > kSmallLds) return nullptr;
    auto* P = new SmallPlan();
    try {
      P->nchunks = (int)B.chunks.size();
      P->maxmat = B.maxmat;
      P->poly = poly;
      P->steps = put(B.steps);
      P->chunks = put(B.chunks);
      P->slots = put(B.slots);
      P->pairs = put(B.pairs);
      P->members = put(B.members);
      P->meta = put(B.meta);
      P->mel = put(B.mel);
      P->ctab = put(B.ctab);
      P->nograd = put(B.nograd);
      P->ngates = (int)p.gates.size();
      P->lds_fwd = small_lds(s.dim, B.maxmat, false);
      P->lds_rev = lds_rev;
    } catch (...) {
      delete P;
      throw;
    }
    p.small = P;
  }
  return p.small;
}

void small_forward(const Space& s, const SmallPlan& P, const double* theta, const double* psi_in, double* psi,
                   bool dagger, hipStream_t st, double* zero, double* theta_out) {
  const SmallDev D = device_view(s, P);
  SmallExtra ex;
  ex.zero = zero;
  ex.nzero = zero ? s.dim : 0;
  ex.theta_out = theta_out;
  auto* kernel = P.poly ? k_small_sweep<false, true> : k_small_sweep<false, false>;
  allow_lds(kernel, P.lds_fwd);
  SQ_PROF(PC_SMALL, st, 16.0 * (double)s.dim, 0.0,
          kernel<<<zero ? 1 + kZeroBlocks : 1, kST, P.lds_fwd, st>>>(D, theta, psi_in, psi, nullptr, nullptr,
                                                                    dagger ? 1 : 0, ex));
}

void small_reverse(const Space& s, const SmallPlan& P, const double* theta, const double* psi, const double* lam,
                   double* grad, hipStream_t st, const double* epart, int64_t n_epart, double* e_out) {
  const SmallDev D = device_view(s, P);
  SmallExtra ex;
  ex.epart = epart;
  ex.nepart = n_epart;
  ex.e_out = e_out;
  auto* kernel = P.poly ? k_small_sweep<true, true> : k_small_sweep<true, false>;
  allow_lds(kernel, P.lds_rev);
  SQ_PROF(PC_SMALL, st, 16.0 * (double)s.dim, 0.0,
          kernel<<<e_out ? 2 : 1, kST, P.lds_rev, st>>>(D, theta, psi, nullptr, lam, grad, 1, ex));
}

}  // namespace sq
