// Fused brick-wall sweeps for gate layouts made of adjacent-pair gates
// (tUPS / QNP brick walls: sa_single(p,p+1), double(2p,2p+1,2p+2,2p+3)).
//
// Consecutive gates on one orbital pair (p, p+1) merge into a pair op.  Under
// the pair ops inside a window of w consecutive orbitals a determinant keeps
// its occupation outside the window and its electron count inside it, per
// spin: strings fall into groups of C(w, k) strings, in the canonical order of
// their window occupations.  A tile = (some alpha groups of one electron count)
// x (some beta groups of one count) is
// closed under every gate of the window, so one launch (a stage) loads each
// tile into LDS once, applies all the pair ops that are ready inside the
// window, whatever their depth in the brick wall, and writes it back.  The
// stages of a program are chosen greedily: the window position that takes
// the most pair ops next.  (12e,12o) tUPS with 4 layers has 8 brick columns
// and takes 3 stages of up to 22 pair ops at w = 8; (14e,14o) with 6 layers
// 12 columns and 5 stages.  Tiles gather rows and columns through tables, so
// state vectors never change layout.
//
// For one pair the gates only mix the <= 4 members of an "orbit" {alpha bit}
// x {beta bit} (other indices fixed), and their whole product is one small
// matrix per orbit type; a thread owns an orbit and applies it.  Signs come
// from the pair-local bits only: the environment parity cancels for
// number-conserving spin parts.  One barrier per pair op.
//
// The orbits of a tile depend on (w, electrons of both groups, pair position)
// only.  They are listed once per space as 32-bit words of LDS offsets, type
// after type; a thread loads its words two pair ops ahead into registers and
// the barriers wait for LDS only, so a pair op is LDS reads, the small matrix
// and LDS writes.  (Indices computed in the kernel from per-spin lists cost
// more than the matrices: 37 against 24 us for a (12e,12o) stage of 22 ops.)
//
// Per rotation string and orbit type (alpha part of the pair empty / doubly
// occupied / single, same for beta) the host precomputes a 12-bit code: for
// each of the 6 member pairs {0,1},{2,3},{0,2},{1,3},{0,3},{1,2} whether the
// string rotates it and with which sign.
//
// Kernels:
//   k_op_mats      per pair op and orbit type: the product of the op's gates
//                  (optionally with T_g inserted) from theta
//   k_win_fwd      one stage on one vector; dagger runs U^+
//   k_win_rev      reverse stage on (psi, lambda): antisymmetric orbit
//                  products, then un-apply the op matrices
//   k_op_grad      grad[g] from the orbit products summed over blocks

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <numeric>

#include "sq_internal.h"

namespace sq {

constexpr int kMaxWin = 8;          // orbitals per window
constexpr int kTileElems = 4900;    // amplitudes per tile: C(8,4)^2
constexpr int kMaxPairEntries = 8;  // entries per pair op (sa_single counts twice)
constexpr int kMaxOps = 64;         // pair ops per stage
constexpr int kTypes = 9;           // orbit types (alpha kind x beta kind)
constexpr int kTB = 256;            // threads per block of the gradient kernel

struct LocalOps {
  int8_t n;
  int8_t orb[4];  // 0 = p, 1 = p+1
  int8_t cre[4];
};

struct StageEntry {
  int32_t gate;   // program gate index
  double scale;   // angle multiplier (|coefficient|)
  uint32_t code[kTypes];
};

// Per pair op, the gates act on orbits of <= 4 amplitudes (member
// o = alpha bit | beta bit << 1).  Their combined action is one matrix per
// orbit type, stored compactly in kPairVals doubles:
//   [0..15]  type (alpha single, beta single): 4x4, row-major M[a][b]
//   [16..19] type (alpha single, beta empty):  2x2 on members {0, 1}
//   [20..23] type (alpha single, beta double): 2x2 on members {0, 1}
//   [24..27] type (alpha empty, beta single):  2x2 on members {0, 2}
//   [28..31] type (alpha double, beta single): 2x2 on members {0, 2}
// (types without a single pair are left alone by every gate).  A gate's
// gradient is sum over orbits of <lam|W T W^T|psi> with W the product of the
// op's later gates; W T W^T is antisymmetric, so the reverse sweep only
// accumulates Q[a<b] = sum (lam_a psi_b - lam_b psi_a):
//   Q[0..5]  type (single, single): pairs (0,1),(0,2),(0,3),(1,2),(1,3),(2,3)
//   Q[6..9]  the four two-member types, (member 0, second member)
constexpr int kPairVals = 32;
constexpr int kQVals = 10;
// Op matrices carry one more value, [32]: the factor for orbits of types
// without a single pair (1, or 0 when a derivative T_g is inserted on the
// op: T_g annihilates them); padded to 36.
constexpr int kMatVals = 36;

// One dispatch slot: rows arows[r0, r0 + R) of its alpha groups, columns
// bcol[c0, c0 + W) of its beta groups, electrons in the window and groups of
// each side (k | groups << 8), their orbit words.  R = 0 marks an empty slot.
struct TileRec {
  int32_t r0, R, c0, W, ka, kb, items, pad;
};

// Local strings of k electrons in the window: n4 have a given pair singly
// occupied (lower member; as many the upper one), ne have it empty, nd doubly
// occupied, at every pair position.
struct KInfo {
  int32_t n4, ne, nd;
};
// The same over a tile side's groups (g = k | groups << 8).
__host__ __device__ inline KInfo side_info(const KInfo* k, int g) {
  const KInfo i = k[g & 255];
  return KInfo{i.n4 * (g >> 8), i.ne * (g >> 8), i.nd * (g >> 8)};
}

// Orbit words of one pair position: five ranges and a sixth (alpha list x
// beta list), each filled up to whole waves of 64 words with kNone, so that a
// wave's 64 words are of one type: the type is a scalar branch and every
// matrix value a scalar operand.
//   [0, c1)  alpha and beta single: 4 members, m0 | dr << 13 | dc << 26
//   [c1, c2) alpha single, beta empty    [c2, c3) alpha single, beta double
//   [c3, c4) alpha empty, beta single    [c4, c5) alpha double, beta single:
//            2 members, m0 | d << 13
//   [c5, c6) neither single: m0
// (in waves; m0: first member, in doubles from the tile's first, which is
// preceded by a zero that kNone points to; dr, dc, d: distance of the others;
// swapping neighbouring orbitals moves a string by at most C(6, 3) = 20
// places within its group).
struct OpItems {
  int c1, c2, c3, c4, c5, c6;
};
__host__ __device__ inline OpItems op_items(const KInfo& A, const KInfo& B) {
  auto waves = [](int n) { return (n + 63) / 64; };
  OpItems o;
  o.c1 = waves(A.n4 * B.n4);
  o.c2 = o.c1 + waves(A.n4 * B.ne);
  o.c3 = o.c2 + waves(A.n4 * B.nd);
  o.c4 = o.c3 + waves(A.ne * B.n4);
  o.c5 = o.c4 + waves(A.nd * B.n4);
  o.c6 = o.c5 + waves((A.ne + A.nd) * (B.ne + B.nd));
  return o;
}
constexpr uint32_t kNone = 0u;  // the zero before the tile
constexpr int kMaxWaves = 27;   // c5 at most: k = 4 of 8 on both sides; merged tiles stay within it

struct OpRef {
  int32_t op, pos;  // program-wide pair op, pair position within the window
  int64_t poff;     // its gradient partials
};

struct StageDev {
  int nops, nsb, w, nb;  // nb: dispatch slots
  const int32_t* arows;
  const int32_t* bcol;
  const TileRec* tiles;
  const uint32_t* items;
  const OpRef* ops;      // program order
  KInfo k[kMaxWin + 1];
};

struct OpInfo {
  int32_t e0, e1;   // entries
  int32_t nblk;     // blocks of the reverse launch
  int32_t pad;
  int64_t poff;     // gradient partials [kQVals][nblk]
};

__host__ __device__ constexpr size_t align16(size_t b) { return (b + 15) / 16 * 16; }
// Dynamic LDS of one tile: zero, X (| zero, L) | rows | columns.  Two reverse tiles of
// 70 x 70 amplitudes fit a CU.
__host__ __device__ constexpr size_t tile_lds(int R, int W, int nvec) {
  return align16((size_t)R * W * 8 + 8) * nvec + align16(4 * (size_t)(R + W));
}

struct Stage {
  bool tiled = false;
  int g0 = 0;                // program gate of an untiled stage
  StageDev dev{};
  int rev_blocks = 0;        // grid of the reverse launch
  size_t lds_fwd = 0, lds_rev = 0;
};

// Rows, columns and tiles of one window position.
struct Window {
  int32_t *arows = nullptr, *bcol = nullptr;
  TileRec* tiles = nullptr;
  int nb = 0;
  size_t lds_fwd = 0, lds_rev = 0;
};

// Groups of k electrons per tile side, at most (0: none occurs).
struct Merge {
  int a[kMaxWin + 1] = {}, b[kMaxWin + 1] = {};
};

// What the windows of one width and tile target need on one space: the orbit
// words of the sides that occur, and the window positions used so far.
struct WidthTables {
  KInfo k[kMaxWin + 1] = {};
  Merge merge;
  uint32_t* items = nullptr;
  std::map<std::pair<int, int>, int> off;
  std::map<int, Window> at;
};

// Kept by the space (a space's programs share them) and freed with it.
struct WinCache {
  std::map<std::pair<int, int>, WidthTables> width;
  std::vector<void*> allocs;
  ~WinCache() {
    for (void* p : allocs) (void)hipFree(p);
  }
};

void win_cache_free(WinCache* c) { delete c; }

struct TilePlan {
  std::vector<Stage> stages;
  int nops = 0;
  int nt = 512;                 // threads per block of the stage kernels
  double* d_partial = nullptr;  // gradient partials of all ops
  int64_t partial_len = 0;
  double* d_mats = nullptr;     // [nops][kMatVals]
  OpInfo* d_info = nullptr;     // [nops]
  StageEntry* d_entries = nullptr;
  std::vector<void*> allocs;
  ~TilePlan() {
    for (void* p : allocs) (void)hipFree(p);
    if (d_partial) (void)hipFree(d_partial);
    if (d_mats) (void)hipFree(d_mats);
  }
};

// ---------------------------------------------------------------------------
// Host: stage construction.

static bool local_ops(const SpinOps& o, int p, LocalOps& out) {
  out.n = (int8_t)o.n;
  int nc = 0, na = 0;
  if (o.n > 4) return false;
  for (int j = 0; j < o.n; ++j) {
    int orb = o.orb[j];
    if (orb != p && orb != p + 1) return false;
    out.orb[j] = (int8_t)(orb - p);
    out.cre[j] = o.cre[j];
    (o.cre[j] ? nc : na)++;
  }
  return nc == na;
}

// Apply local ops to a 2-bit pair occupancy m (bit 0 = orbital p); false if zero.
static bool local_apply(const LocalOps& o, uint32_t& m, int& par) {
  for (int j = o.n - 1; j >= 0; --j) {
    uint32_t bit = 1u << o.orb[j];
    par += __builtin_popcount(m & (bit - 1u));
    if (o.cre[j]) {
      if (m & bit) return false;
      m |= bit;
    } else {
      if (!(m & bit)) return false;
      m &= ~bit;
    }
  }
  return true;
}

// Member pairs of an orbit (member o = alpha bit | beta bit << 1).
constexpr int kSlotA[6] = {0, 2, 0, 1, 0, 1};
constexpr int kSlotB[6] = {1, 3, 2, 3, 3, 2};

static int slot_of(int a, int b) {
  if (a > b) std::swap(a, b);
  for (int k = 0; k < 6; ++k)
    if (kSlotA[k] == a && kSlotB[k] == b) return k;
  return -1;
}

// Orbit-type codes of one rotation string with local spin parts la/lb.
static bool entry_codes(const LocalOps& la, const LocalOps& lb, double sgn, uint32_t* code) {
  for (int ta = 0; ta < 3; ++ta) {
    for (int tb = 0; tb < 3; ++tb) {
      uint32_t c = 0;
      for (int o = 0; o < 4; ++o) {
        const int ba = o & 1, bb = o >> 1;
        if ((ta != 2 && ba) || (tb != 2 && bb)) continue;
        uint32_t ma = ta == 2 ? (ba ? 2u : 1u) : (ta == 0 ? 0u : 3u);
        uint32_t mb = tb == 2 ? (bb ? 2u : 1u) : (tb == 0 ? 0u : 3u);
        const uint32_t ma0 = ma, mb0 = mb;
        int par = 0;
        if (!local_apply(la, ma, par) || !local_apply(lb, mb, par)) continue;
        if ((ta != 2 && ma != ma0) || (tb != 2 && mb != mb0)) return false;
        const int ba2 = ta == 2 ? (ma == 2u) : ba;
        const int bb2 = tb == 2 ? (mb == 2u) : bb;
        const int o2 = ba2 | (bb2 << 1);
        if (o2 == o) return false;
        const int sl = slot_of(o, o2);
        double sig = ((par & 1) ? -1.0 : 1.0) * sgn;
        if (o > o2) sig = -sig;  // orientation: slot rotations run from the lower member
        if (c & (3u << (2 * sl))) return false;
        c |= (1u | (sig < 0 ? 2u : 0u)) << (2 * sl);
      }
      code[ta * 3 + tb] = c;
    }
  }
  return true;
}

// Can gate g run inside a tile stage?  Fills its entries (pair index unset).
static bool tile_entries(const Program& P, int g, int& p_out, std::vector<StageEntry>& out) {
  const GateDev& gd = P.gates[g];
  int p = P.pair_p[g];
  if (p < 0) return false;
  if (gd.kind != GC_ROT && gd.kind != GC_SA_SINGLE) return false;
  int halves = gd.kind == GC_SA_SINGLE ? 2 : 1;
  out.clear();
  for (int h = 0; h < halves; ++h) {
    const Term& T = P.terms[gd.term_begin + 2 * h];
    StageEntry e{};
    e.gate = g;
    e.scale = halves == 2 ? 1.0 : gd.scale;
    LocalOps la, lb;
    if (!local_ops(T.a, p, la) || !local_ops(T.b, p, lb)) return false;
    if (!entry_codes(la, lb, T.coef < 0 ? -1.0 : 1.0, e.code)) return false;
    out.push_back(e);
  }
  p_out = p;
  return true;
}

template <class T>
static T* upload(std::vector<void*>& allocs, const std::vector<T>& v) {
  T* d = nullptr;
  SQ_HIP(hipMalloc(&d, sizeof(T) * std::max<size_t>(v.size(), 1)));
  allocs.push_back(d);
  if (!v.empty()) SQ_HIP(hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
  return d;
}

// Local strings of k of w orbitals, lexicographic by occupied orbitals, as the
// space orders its strings.
static std::vector<uint32_t> local_strings(int w, int k) {
  std::vector<uint32_t> strs;
  std::vector<int> c(k);
  std::iota(c.begin(), c.end(), 0);
  for (;;) {
    uint32_t s = 0;
    for (int p : c) s |= 1u << p;
    strs.push_back(s);
    int i = k - 1;
    while (i >= 0 && c[i] == w - k + i) --i;
    if (i < 0) break;
    ++c[i];
    for (int j = i + 1; j < k; ++j) c[j] = c[j - 1] + 1;
  }
  return strs;
}

// Per pair position: lower members, their upper partners, empty, double.
struct PairLists {
  std::vector<int> lo, up, em, db;
};
static std::vector<PairLists> pair_lists(int w, int k) {
  const std::vector<uint32_t> strs = local_strings(w, k);
  std::vector<int> rank((size_t)1 << w, -1);
  for (size_t i = 0; i < strs.size(); ++i) rank[strs[i]] = (int)i;
  std::vector<PairLists> out(w - 1);
  for (int j = 0; j + 1 < w; ++j)
    for (size_t i = 0; i < strs.size(); ++i) {
      const uint32_t loc = (strs[i] >> j) & 3u;
      if (loc == 0u) out[j].em.push_back((int)i);
      else if (loc == 3u) out[j].db.push_back((int)i);
      else if (loc == 1u) {
        out[j].lo.push_back((int)i);
        out[j].up.push_back(rank[strs[i] ^ (3u << j)]);
      }
    }
  return out;
}

// Orders the words items[from..] so that the 16 lanes which reach LDS together
// (8-byte accesses, 32 banks of 8 bytes) fall into different banks with every
// member of their orbits: each group of 16 takes the first words among the
// next 64 that still fit.  (By this model list order takes 1.9 times the
// conflict-free cycles and this order 1.04; the counters go from 2.2 to 1.8,
// a reverse stage from 37.6 to 36.0 us at 12 orbitals, 404 to 393 at 14.)
static void spread_banks(std::vector<uint32_t>& items, size_t from, bool four) {
  constexpr int kLook = 64;
  std::vector<uint32_t> out;
  out.reserve(items.size() - from);
  uint32_t look[kLook];
  int n = 0;
  size_t next = from;
  while (n > 0 || next < items.size()) {
    while (n < kLook && next < items.size()) look[n++] = items[next++];
    uint32_t used[4] = {0, 0, 0, 0};
    int taken = 0, kept = 0;
    uint32_t rest[kLook];
    for (int i = 0; i < n; ++i) {
      const uint32_t x = look[i], m0 = x & 8191u;
      const uint32_t d = four ? (x >> 13) & 8191u : x >> 13, dc = four ? x >> 26 : 0u;
      const uint32_t bit[4] = {1u << (m0 & 31u), 1u << ((m0 + d) & 31u), 1u << ((m0 + dc) & 31u),
                               1u << ((m0 + d + dc) & 31u)};
      bool fits = taken < 16;
      for (int a = 0; a < (four ? 4 : 2) && fits; ++a) fits = !(used[a] & bit[a]);
      if (fits) {
        for (int a = 0; a < (four ? 4 : 2); ++a) used[a] |= bit[a];
        out.push_back(x);
        ++taken;
      } else {
        rest[kept++] = x;
      }
    }
    // a group that found fewer takes the oldest of the others
    int i = 0;
    for (; taken < 16 && i < kept; ++i, ++taken) out.push_back(rest[i]);
    n = kept - i;
    std::copy(rest + i, rest + kept, look);
  }
  std::copy(out.begin(), out.end(), items.begin() + from);
}

static int binomial(int n, int k) {
  if (k < 0 || k > n) return 0;
  int b = 1;
  for (int i = 0; i < k; ++i) b = b * (n - i) / (i + 1);
  return b;
}

static KInfo window_info(int w, int k) {
  return KInfo{binomial(w - 2, k - 1), binomial(w - 2, k), binomial(w - 2, k - 2)};
}

// Windows of width w on a space: per electron count k inside, the strings of a
// group, the pair counts and the alpha and beta groups.
struct WinCounts {
  int w, len[kMaxWin + 1], a[kMaxWin + 1], b[kMaxWin + 1];
  KInfo info[kMaxWin + 1];
  WinCounts(const Space& sp, int width) : w(width) {
    for (int k = 0; k <= w; ++k) {
      len[k] = binomial(w, k);
      info[k] = window_info(w, k);
      a[k] = binomial(sp.n - w, sp.na - k);
      b[k] = binomial(sp.n - w, sp.nb - k);
    }
  }
};

// Group counts of the tile sides that hold all groups of k electrons, at most
// m a side, as evenly as they go: the larger count and how many sides have it,
// the others one less.
struct Split {
  int sides, big, nbig;
};
static Split split_groups(int groups, int m) {
  Split s;
  s.sides = (groups + m - 1) / m;
  s.big = (groups + s.sides - 1) / s.sides;
  s.nbig = groups - s.sides * (s.big - 1);
  return s;
}

// Groups per tile side for tiles of up to about target amplitudes.  With few
// electrons the groups are small and many ((16: 3,3), windows of 8: 93 of 1 to
// 56 strings per spin, 8649 pairs), and a block takes each pair op of its
// tile behind a barrier, 0.5 us however small the tile.
static Merge merge_groups(const WinCounts& C, int target) {
  Merge M;
  auto side = [&](const int* groups, int limit, int* m) {  // returns the longest side
    int most = 1;
    for (int k = 0; k <= C.w; ++k) {
      m[k] = 0;
      if (groups[k] == 0) continue;
      m[k] = split_groups(groups[k], std::max(1, std::min(limit / C.len[k], groups[k]))).big;
      most = std::max(most, m[k] * C.len[k]);
    }
    return most;
  };
  for (int e = std::min(target, kTileElems);; e = e * 3 / 4) {
    int rows = side(C.a, (int)std::sqrt((double)e), M.a);
    const int cols = side(C.b, e / rows, M.b);
    rows = side(C.a, e / cols, M.a);
    bool fits = true;
    for (int ka = 0; ka <= C.w && fits; ++ka)
      for (int kb = 0; kb <= C.w && fits; ++kb) {
        if (M.a[ka] * M.b[kb] <= 1) continue;
        const OpItems o = op_items(side_info(C.info, ka | M.a[ka] << 8), side_info(C.info, kb | M.b[kb] << 8));
        fits = M.a[ka] * C.len[ka] * M.b[kb] * C.len[kb] <= kTileElems && o.c5 <= kMaxWaves;
      }
    if (fits || e < 4) return M;
  }
}

// Tiles of one window of width w and the amplitudes of the largest.
struct Tiling {
  int64_t tiles;
  int most;
};
static Tiling merged_tiles(const WinCounts& C, const Merge& M) {
  auto sides = [&](const int* groups, const int* m, int& most) {
    int64_t c = 0;
    for (int k = 0; k <= C.w; ++k) {
      if (m[k] == 0) continue;
      c += split_groups(groups[k], m[k]).sides;
      most = std::max(most, m[k] * C.len[k]);
    }
    return std::max<int64_t>(c, 1);
  };
  int rows = 1, cols = 1;
  const int64_t a = sides(C.a, M.a, rows), b = sides(C.b, M.b, cols);
  return Tiling{a * b, rows * cols};
}

// Orbit words of the tile sides that occur in windows of width w.
static void build_width(const Space& sp, int w, int target, WidthTables& T, std::vector<void*>& allocs) {
  std::vector<std::vector<PairLists>> L(w + 1);
  const WinCounts C(sp, w);
  for (int k = 0; k <= w; ++k) {
    L[k] = pair_lists(w, k);
    T.k[k] = C.info[k];
  }
  T.merge = merge_groups(C, target);
  // the sides (k | groups << 8) of one spin
  auto sides = [&](const int* groups, const int* m) {
    std::vector<int> out;
    for (int k = 0; k <= w; ++k) {
      if (m[k] == 0) continue;
      const Split s = split_groups(groups[k], m[k]);
      out.push_back(k | s.big << 8);
      if (s.nbig < s.sides) out.push_back(k | (s.big - 1) << 8);
    }
    return out;
  };
  // a pair position's lists over all groups of a side
  auto over_groups = [&](int g, int j) {
    const PairLists& P = L[g & 255][j];
    const int len = C.len[g & 255];
    PairLists out;
    for (int i = 0; i < (g >> 8); ++i) {
      for (int x : P.lo) out.lo.push_back(x + i * len);
      for (int x : P.up) out.up.push_back(x + i * len);
      for (int x : P.em) out.em.push_back(x + i * len);
      for (int x : P.db) out.db.push_back(x + i * len);
    }
    return out;
  };
  std::vector<uint32_t> items;
  for (int ga : sides(C.a, T.merge.a))
    for (int gb : sides(C.b, T.merge.b)) {
      T.off[{ga, gb}] = (int)items.size();
      const int W = (gb >> 8) * C.len[gb & 255];
      for (int j = 0; j + 1 < w; ++j) {
        const PairLists A = over_groups(ga, j), B = over_groups(gb, j);
        auto at = [&](int r, int c) { return (uint32_t)(1 + r * W + c); };
        size_t from = items.size();
        auto fill = [&](bool four) {
          spread_banks(items, from, four);
          items.resize((items.size() + 63) / 64 * 64, kNone);
          from = items.size();
        };
        for (size_t r = 0; r < A.lo.size(); ++r)
          for (size_t c = 0; c < B.lo.size(); ++c)
            items.push_back(at(A.lo[r], B.lo[c]) | (uint32_t)((A.up[r] - A.lo[r]) * W) << 13 |
                            (uint32_t)(B.up[c] - B.lo[c]) << 26);
        fill(true);
        for (const std::vector<int>* q : {&B.em, &B.db}) {
          for (size_t r = 0; r < A.lo.size(); ++r)
            for (int c : *q) items.push_back(at(A.lo[r], c) | (uint32_t)((A.up[r] - A.lo[r]) * W) << 13);
          fill(false);
        }
        for (const std::vector<int>* q : {&A.em, &A.db}) {
          for (int r : *q)
            for (size_t c = 0; c < B.lo.size(); ++c)
              items.push_back(at(r, B.lo[c]) | (uint32_t)(B.up[c] - B.lo[c]) << 13);
          fill(false);
        }
        for (const std::vector<int>* q : {&A.em, &A.db})
          for (int r : *q)
            for (const std::vector<int>* x : {&B.em, &B.db})
              for (int c : *x) items.push_back(at(r, c));
        items.resize((items.size() + 63) / 64 * 64, kNone);
      }
    }
  T.items = upload(allocs, items);
}

// A tile side: electrons in the window and groups (k | groups << 8), strings.
struct Side {
  int g;
  std::vector<int32_t> str;
};

// Strings by electrons inside [lo, lo + w) and occupation outside (a group, in
// canonical order), the groups of one count dealt to tile sides.
static std::vector<Side> window_sides(const std::vector<uint32_t>& strs, int lo, int w, const int* m) {
  const uint32_t in = ((1u << w) - 1u) << lo;
  std::map<uint32_t, std::vector<int32_t>> g[kMaxWin + 1];
  for (size_t i = 0; i < strs.size(); ++i)
    g[__builtin_popcount(strs[i] & in)][strs[i] & ~in].push_back((int32_t)i);
  std::vector<Side> out;
  for (int k = 0; k <= w; ++k) {
    if (g[k].empty()) continue;
    const Split s = split_groups((int)g[k].size(), m[k]);
    auto it = g[k].begin();
    for (int x = 0; x < s.sides; ++x) {
      const int n = x < s.nbig ? s.big : s.big - 1;
      out.push_back(Side{k | n << 8, {}});
      for (int i = 0; i < n; ++i, ++it) out.back().str.insert(out.back().str.end(), it->second.begin(), it->second.end());
    }
  }
  return out;
}

// Tables and dispatch order of one window position.  Workgroups go to the
// XCDs round robin (slot b on XCD b % 8), each XCD with its own L2: tiles of
// one alpha side read the same rows of the state, so whole sides are given
// to one XCD (largest first, each to the XCD with the fewest elements so
// far), largest tiles first there.  Empty slots have R = 0.
static Window make_window(const Space& sp, int lo, int w, const WidthTables& T, std::vector<void*>& allocs) {
  const std::vector<Side> A = window_sides(sp.h_astr, lo, w, T.merge.a), B = window_sides(sp.h_bstr, lo, w, T.merge.b);
  Window W;
  std::vector<int32_t> arows, bcol;
  std::vector<int> a0, b0;
  for (const Side& g : A) {
    a0.push_back((int)arows.size());
    arows.insert(arows.end(), g.str.begin(), g.str.end());
  }
  for (const Side& g : B) {
    b0.push_back((int)bcol.size());
    bcol.insert(bcol.end(), g.str.begin(), g.str.end());
  }
  constexpr int kXcds = 8;
  std::vector<int> ao(A.size()), bo(B.size());
  std::iota(ao.begin(), ao.end(), 0);
  std::iota(bo.begin(), bo.end(), 0);
  std::stable_sort(ao.begin(), ao.end(), [&](int x, int y) { return A[x].str.size() > A[y].str.size(); });
  std::stable_sort(bo.begin(), bo.end(), [&](int x, int y) { return B[x].str.size() > B[y].str.size(); });
  std::vector<std::vector<TileRec>> bins(kXcds);
  std::vector<int64_t> load(kXcds, 0);
  // few alpha sides: single tiles are spread instead
  const bool whole = A.size() >= 2 * kXcds;
  for (int a : ao) {
    int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    for (int b : bo) {
      if (!whole) x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      const int R = (int)A[a].str.size(), C = (int)B[b].str.size();
      bins[x].push_back(TileRec{a0[a], R, b0[b], C, A[a].g, B[b].g, T.off.at({A[a].g, B[b].g}), 0});
      load[x] += (int64_t)R * C;
      W.lds_fwd = std::max(W.lds_fwd, tile_lds(R, C, 1));
      W.lds_rev = std::max(W.lds_rev, tile_lds(R, C, 2));
    }
  }
  size_t len = 0;
  for (auto& b : bins) {
    std::stable_sort(b.begin(), b.end(), [](const TileRec& x, const TileRec& y) {
      return (int64_t)x.R * x.W > (int64_t)y.R * y.W;
    });
    len = std::max(len, b.size());
  }
  std::vector<TileRec> slots(len * kXcds, TileRec{});
  for (int x = 0; x < kXcds; ++x)
    for (size_t k = 0; k < bins[x].size(); ++k) slots[k * kXcds + x] = bins[x][k];
  while (!slots.empty() && slots.back().R == 0) slots.pop_back();
  W.nb = (int)slots.size();
  W.arows = upload(allocs, arows);
  W.bcol = upload(allocs, bcol);
  W.tiles = upload(allocs, slots);
  return W;
}

struct PairOp {
  int p;
  std::vector<StageEntry> entries;
};

// The order in which stages of width w take the ops of one run: per stage its
// window position and the ops (indices into ops), program order kept.
static std::vector<std::pair<int, std::vector<int>>> schedule(const std::vector<PairOp>& ops, int n, int w) {
  std::vector<std::pair<int, std::vector<int>>> out;
  std::vector<char> done(ops.size(), 0);
  std::vector<int> t;
  size_t left = ops.size(), first = 0;
  while (left > 0) {
    int best = -1;
    std::vector<int> take;
    while (done[first]) ++first;
    for (int lo = 0; lo + w <= n; ++lo) {
      uint32_t blocked = ~(((1u << w) - 1u) << lo);
      t.clear();
      for (size_t i = first; i < ops.size() && t.size() < kMaxOps && blocked != ~0u; ++i) {
        if (done[i]) continue;
        const uint32_t m = 3u << ops[i].p;
        if (blocked & m) blocked |= m;
        else t.push_back((int)i);
      }
      if (t.size() > take.size()) {
        take.swap(t);
        best = lo;
      }
    }
    for (int i : take) done[i] = 1;
    left -= take.size();
    out.push_back({best, take});
  }
  return out;
}

// Window width and tile target.  A program's tile target (or SQ_TILE_TARGET)
// gives the widest window whose mean unmerged tile stays below it.  Otherwise
// the cheapest of a model of the sweep (us, mean of forward and reverse),
// fitted to 1- to 4-layer sweeps at 4 to 16 orbitals and all fillings: a stage
// costs 5.5 and 8.5 per million amplitudes (its passes over memory); a pair op
// 0.8 and 1 more per 11600 amplitudes of the largest tile and 34000 of the mean
// one, as often as the tiles go round the 256 CUs.  Narrow windows need more
// stages, small tiles more rounds, large ones leave CUs idle.  Its choices take
// 0.8 % more than the best ones on average, 7 % at most.  Measured, forward and
// reverse sweep of 4 layers with w = 6, 7, 8: (8e,8o) 110, 114, 114; (10e,10o)
// 145, 131, 157; (12e,12o) 1242, 384, 207 us.  Tiles of one pair of groups
// against merged ones: (16: 3,3) 3400 -> 270 us, (14: 3,7) 1510 -> 480,
// (14e,14o) 2450 -> 2350 (energy and gradient of (16: 3,3) 3550 -> 415, with
// stages of one brick column each 713).
struct WinShape {
  int width, target;  // target: of merge_groups
};
static WinShape window_shape(const Space& sp, const std::vector<PairOp>& ops, int target, int instances) {
  const int most = std::min(kMaxWin, sp.n);
  if (target <= 0)
    if (const char* env = getenv("SQ_TILE_TARGET")) target = atoi(env);
  if (target > 0) {
    int w = 2;
    auto pairs = [&](int width) {  // of groups
      const WinCounts C(sp, width);
      return merged_tiles(C, merge_groups(C, 1)).tiles;
    };
    while (w < most && sp.dim <= pairs(w + 1) * (int64_t)target) ++w;
    return WinShape{w, target};
  }
  WinShape best{most, kTileElems};
  double cost = -1.0;
  for (int w = std::min(4, most); w <= most; ++w) {
    const WinCounts C(sp, w);
    const double stages = (double)schedule(ops, sp.n, w).size();
    for (int fill : {512, 1024, 2048, 4096, kTileElems}) {
      const Tiling t = merged_tiles(C, merge_groups(C, fill));
      const double mean = (double)sp.dim / (double)t.tiles;
      const double op = 0.8 + (double)t.most / 11600.0 + mean / 34000.0;
      const double c = stages * (5.5 + 8.5e-6 * (double)sp.dim * instances) +
                       (double)ops.size() * op * std::max(1.0, (double)t.tiles * instances / 256.0);
      if (cost < 0.0 || c < cost) {
        cost = c;
        best = WinShape{w, fill};
      }
    }
  }
  return best;
}

TilePlan* build_tile_plan(const Space& sp, const Program& P, int instances) {
  auto* T = new TilePlan();
  try {
    const int n = (int)P.gates.size();
    std::vector<StageEntry> ent, all;
    std::vector<OpInfo> info;
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);  // the space's tables are shared
    if (!sp.win) sp.win = new WinCache;
    for (int g = 0; g < n;) {
      int p;
      if (!tile_entries(P, g, p, ent)) {
        Stage S;
        S.g0 = g++;
        T->stages.push_back(S);
        continue;
      }
      // the run of tileable gates from g, merged into pair ops
      std::vector<PairOp> ops;
      std::vector<int> last(sp.n, -1);  // latest op on each orbital
      for (; g < n && tile_entries(P, g, p, ent); ++g) {
        const int o = last[p];
        if (o >= 0 && o == last[p + 1] && ops[o].p == p &&
            ops[o].entries.size() + ent.size() <= (size_t)kMaxPairEntries) {
          ops[o].entries.insert(ops[o].entries.end(), ent.begin(), ent.end());
        } else {
          last[p] = last[p + 1] = (int)ops.size();
          ops.push_back(PairOp{p, ent});
        }
      }
      const WinShape shape = window_shape(sp, ops, P.tile_target, instances);
      const int w = shape.width;
      auto wt = sp.win->width.find({w, shape.target});
      if (wt == sp.win->width.end()) {
        WidthTables t;
        build_width(sp, w, shape.target, t, sp.win->allocs);
        wt = sp.win->width.emplace(std::make_pair(w, shape.target), std::move(t)).first;
      }
      WidthTables& wide = wt->second;
      for (auto& st : schedule(ops, sp.n, w)) {
        const int lo = st.first;
        auto it = wide.at.find(lo);
        if (it == wide.at.end()) it = wide.at.emplace(lo, make_window(sp, lo, w, wide, sp.win->allocs)).first;
        const Window& W = it->second;
        Stage S;
        S.tiled = true;
        S.rev_blocks = std::min(W.nb, 1024);
        std::vector<OpRef> refs;
        for (int i : st.second) {
          OpInfo I{};
          I.e0 = (int)all.size();
          all.insert(all.end(), ops[i].entries.begin(), ops[i].entries.end());
          I.e1 = (int)all.size();
          I.nblk = S.rev_blocks;
          I.poff = T->partial_len;
          T->partial_len += (int64_t)kQVals * I.nblk;
          refs.push_back(OpRef{(int)info.size(), ops[i].p - lo, I.poff});
          info.push_back(I);
        }
        StageDev d{};
        d.nops = (int)refs.size();
        d.nsb = sp.nsb;
        d.w = w;
        d.nb = W.nb;
        d.arows = W.arows;
        d.bcol = W.bcol;
        d.tiles = W.tiles;
        d.items = wide.items;
        d.ops = upload(T->allocs, refs);
        for (int k = 0; k <= w; ++k) d.k[k] = wide.k[k];
        S.dev = d;
        S.lds_fwd = W.lds_fwd;
        S.lds_rev = W.lds_rev;
        T->stages.push_back(S);
      }
    }
    T->nops = (int)info.size();
    // one block per CU and tile: more threads shorten every pair op; more
    // tiles than that keep the CUs full with smaller blocks
    int most = 0;
    for (auto& S : T->stages) most = std::max(most, S.dev.nb);
    T->nt = P.tile_threads ? P.tile_threads : (int64_t)most * instances <= 256 ? 1024 : 512;
    T->d_entries = upload(T->allocs, all);
    T->d_info = upload(T->allocs, info);
    SQ_HIP(hipMalloc(&T->d_partial, sizeof(double) * std::max<int64_t>(T->partial_len, 1)));
    SQ_HIP(hipMalloc(&T->d_mats, sizeof(double) * std::max<int64_t>((int64_t)T->nops * kMatVals, 1)));
  } catch (...) {
    delete T;
    throw;
  }
  return T;
}

void destroy_tile_plan(TilePlan* T) { delete T; }

// A plan with tiled stages, or nullptr.  They are used unless SQ_TILES=0.
static TilePlan* make_plan(const Space& s, const Program& p, int instances) {
  const char* env = getenv("SQ_TILES");
  if ((env && env[0] == '0') || s.dim == 0 || s.nsb > 65535) return nullptr;
  TilePlan* T = build_tile_plan(s, p, instances);
  if (T->nops > 0) return T;
  destroy_tile_plan(T);
  return nullptr;
}

const TilePlan* tiles_for(const Space& s, const Program& p) {
  std::lock_guard<std::recursive_mutex> lock(p.plan_mu);
  if (!p.tiles_built) {
    p.tiles_built = true;
    p.tiles = make_plan(s, p, 1);
  }
  return p.tiles;
}

// Groups of instances (sq_batch.hip) have a plan of their own: with many
// instances per launch the widest window is the best one.
std::shared_ptr<const TilePlan> group_tiles_for(const Space& s, const Program& p) {
  std::lock_guard<std::recursive_mutex> lock(p.plan_mu);
  if (!p.group_tiles_built) {
    p.group_tiles_built = true;
    p.group_tiles.reset(make_plan(s, p, 64));
    if (p.group_tiles && !tiles_whole(*p.group_tiles)) p.group_tiles.reset();
  }
  return p.group_tiles;
}

bool tiles_cover(const Space& s, const Program& p) {
  const TilePlan* T = tiles_for(s, p);
  if (!T) return false;
  for (const Stage& S : T->stages)
    if (!S.tiled) return false;
  return true;
}

// ---------------------------------------------------------------------------
// Device kernels.

// Orbit-type classes of the compact layout: type index (alpha kind * 3 +
// beta kind), offset, second member.
__device__ __constant__ int c_cls_type[5] = {8, 6, 7, 2, 5};
__device__ __constant__ int c_cls_off[5] = {0, 16, 20, 24, 28};

// An op's entries in LDS with their rotation cosine/sine.
struct EntryLds {
  int gate[kMaxPairEntries];
  double scale[kMaxPairEntries], c[kMaxPairEntries], s[kMaxPairEntries];
  uint32_t code[kMaxPairEntries][kTypes];
};

__device__ __forceinline__ void load_entries(const StageEntry* __restrict__ entries, int e0, int n,
                                             const double* __restrict__ theta, EntryLds& E,
                                             double* __restrict__ theta_out = nullptr) {
  for (int x = threadIdx.x; x < n * kTypes; x += blockDim.x) E.code[x / kTypes][x % kTypes] = entries[e0 + x / kTypes].code[x % kTypes];
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    const StageEntry& en = entries[e0 + e];
    const double th = theta[en.gate];
    if (theta_out) theta_out[en.gate] = th;
    double s = 0.0, c = 1.0;
    if (fabs(th) >= 1e-28) sincos(en.scale * th, &s, &c);
    E.gate[e] = en.gate;
    E.scale[e] = en.scale;
    E.c[e] = c;
    E.s[e] = s;
  }
}

// v = R v for the rotation of one entry code (disjoint member planes).
__device__ __forceinline__ void rot_vec(uint32_t code, double c, double s, double (&v)[4]) {
#pragma unroll
  for (int sl = 0; sl < 6; ++sl) {
    const uint32_t f = (code >> (2 * sl)) & 3u;
    const int a = kSlotA[sl], b = kSlotB[sl];
    const double cc = (f & 1u) ? c : 1.0, sg = (f & 1u) ? ((f & 2u) ? -s : s) : 0.0;
    const double x = v[a], y = v[b];
    v[a] = cc * x - sg * y;
    v[b] = sg * x + cc * y;
  }
}

// out += scale * T v, T|a> = sg|b>, T|b> = -sg|a> per active plane.
__device__ __forceinline__ void t_vec(uint32_t code, double scale, const double (&v)[4], double (&out)[4]) {
#pragma unroll
  for (int sl = 0; sl < 6; ++sl) {
    const uint32_t f = (code >> (2 * sl)) & 3u;
    const int a = kSlotA[sl], b = kSlotB[sl];
    const double sg = (f & 1u) ? ((f & 2u) ? -scale : scale) : 0.0;
    out[b] += sg * v[a];
    out[a] -= sg * v[b];
  }
}

// One block per pair op (the blocks after them clear nzero doubles at zero, the
// target of the sigma that follows): the op's gate product in forward order,
// with T_g
// inserted after gate g when deriv_gate is in this op.  A thread carries one
// column of one class's matrix through the rotations.
__global__ __launch_bounds__(64) void k_op_mats(const OpInfo* __restrict__ info, const StageEntry* __restrict__ entries,
                                                const double* __restrict__ theta, int deriv_gate,
                                                double* __restrict__ mats, int64_t th_stride, int64_t mats_stride,
                                                int nops, double* __restrict__ theta_out, double* __restrict__ zero,
                                                int64_t nzero) {
  __shared__ EntryLds E;
  if ((int)blockIdx.x >= nops) {
    zero += blockIdx.y * nzero;
    const int64_t step = (int64_t)(gridDim.x - nops) * blockDim.x;
    for (int64_t i = (int64_t)(blockIdx.x - nops) * blockDim.x + threadIdx.x; i < nzero; i += step) zero[i] = 0.0;
    return;
  }
  theta += blockIdx.y * th_stride;
  mats += blockIdx.y * mats_stride;
  const OpInfo I = info[blockIdx.x];
  const int n = I.e1 - I.e0;
  load_entries(entries, I.e0, n, theta, E, theta_out);
  __syncthreads();
  const int cls = threadIdx.x >> 2, q = threadIdx.x & 3;
  if (cls >= 5) return;
  const int t = c_cls_type[cls];
  double v[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) v[a] = a == q ? 1.0 : 0.0;
  bool has_deriv = false;
  for (int k = 0; k < n; ++k) {
    rot_vec(E.code[k][t], E.c[k], E.s[k], v);
    if (E.gate[k] == deriv_gate && (k + 1 == n || E.gate[k + 1] != deriv_gate)) {
      has_deriv = true;
      double o[4] = {0.0, 0.0, 0.0, 0.0};
      for (int x = k; x >= 0 && E.gate[x] == deriv_gate; --x) t_vec(E.code[x][t], E.scale[x], v, o);
#pragma unroll
      for (int a = 0; a < 4; ++a) v[a] = o[a];
    }
  }
  double* base = mats + (size_t)blockIdx.x * kMatVals;
  if (threadIdx.x == 0) base[kPairVals] = has_deriv ? 0.0 : 1.0;
  double* out = base + c_cls_off[cls];
  if (cls == 0) {
#pragma unroll
    for (int a = 0; a < 4; ++a) out[a * 4 + q] = v[a];
  } else {
    const int m1 = cls <= 2 ? 1 : 2;  // second member: alpha pair or beta pair
    if (q == 0 || q == m1) {
      out[q ? 1 : 0] = v[0];
      out[q ? 3 : 2] = m1 == 1 ? v[1] : v[2];
    }
  }
}

// One block per pair op: Q summed over the blocks of the reverse launch, then
// for every entry k of the op dot_k = sum_{a<b} (W T_k W^T)[a][b] Q[a<b] per
// class, W the product of the op's entries after k; grad[gate] = 2 sum over
// its entries of scale * dot.  A thread carries column q of W and of W T_k
// through the rotations: (W T_k W^T)[a][b] = sum_q (W T_k)[a][q] W[b][q].
constexpr int kQa[6] = {0, 0, 0, 1, 1, 2};
constexpr int kQb[6] = {1, 2, 3, 2, 3, 3};

__global__ __launch_bounds__(kTB) void k_op_grad(const OpInfo* __restrict__ info, const StageEntry* __restrict__ entries,
                                                 const double* __restrict__ theta, const double* __restrict__ partial,
                                                 double* __restrict__ grad, int64_t th_stride, int64_t part_stride,
                                                 int64_t grad_stride, int nops, const double* __restrict__ epart,
                                                 int64_t n_epart, double* __restrict__ e_out) {
  if ((int)blockIdx.x == nops) {  // the energy from the partials of the sigma
    __shared__ double ered[kTB / 64];
    double e = 0.0;
    for (int64_t i = threadIdx.x; i < n_epart; i += kTB) e += epart[i];
    for (int off = 32; off > 0; off >>= 1) e += __shfl_down(e, off, 64);
    if ((threadIdx.x & 63) == 0) ered[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
      double tot = 0.0;
      for (int w = 0; w < kTB / 64; ++w) tot += ered[w];
      e_out[0] = tot;
    }
    return;
  }
  theta += blockIdx.y * th_stride;
  partial += blockIdx.y * part_stride;
  grad += blockIdx.y * grad_stride;
  __shared__ double Q[kQVals];
  __shared__ double wt[kMaxPairEntries * 5 * 4][8];
  __shared__ double dots[kMaxPairEntries * 5];
  __shared__ double red[kQVals][kTB / 64];
  __shared__ EntryLds E;
  const OpInfo I = info[blockIdx.x];
  const int n = I.e1 - I.e0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double acc[kQVals];
#pragma unroll
  for (int v = 0; v < kQVals; ++v) acc[v] = 0.0;
  const double* src = partial + I.poff;
  for (int b = threadIdx.x; b < I.nblk; b += kTB)
#pragma unroll
    for (int v = 0; v < kQVals; ++v) acc[v] += src[(size_t)v * I.nblk + b];
  load_entries(entries, I.e0, n, theta, E);
  __syncthreads();
  if (threadIdx.x < n * 20) {
    const int k = threadIdx.x / 20, cls = (threadIdx.x % 20) >> 2, q = threadIdx.x & 3;
    const int t = c_cls_type[cls];
    double w[4], x[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < 4; ++a) w[a] = a == q ? 1.0 : 0.0;
    t_vec(E.code[k][t], 1.0, w, x);
    for (int e = k + 1; e < n; ++e) {
      rot_vec(E.code[e][t], E.c[e], E.s[e], w);
      rot_vec(E.code[e][t], E.c[e], E.s[e], x);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      wt[threadIdx.x][a] = w[a];
      wt[threadIdx.x][4 + a] = x[a];
    }
  }
#pragma unroll
  for (int v = 0; v < kQVals; ++v) {
    double a = acc[v];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
    if (lane == 0) red[v][wave] = a;
  }
  __syncthreads();
  if (threadIdx.x < kQVals) {
    double tot = 0.0;
    for (int w = 0; w < kTB / 64; ++w) tot += red[threadIdx.x][w];
    Q[threadIdx.x] = tot;
  }
  __syncthreads();
  if (threadIdx.x < n * 5) {
    const int k = threadIdx.x / 5, cls = threadIdx.x % 5;
    const double(*c)[8] = wt + k * 20 + cls * 4;
    double d = 0.0;
    if (cls == 0) {
#pragma unroll
      for (int x = 0; x < 6; ++x) {
        double m = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) m += c[q][4 + kQa[x]] * c[q][kQb[x]];
        d += m * Q[x];
      }
    } else {
      const int m1 = cls <= 2 ? 1 : 2;
      double m = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) m += c[q][4] * c[q][m1];
      d = m * Q[5 + cls];
    }
    dots[threadIdx.x] = d * E.scale[k];
  }
  __syncthreads();
  // one thread per gate: the first entry of each run of equal gates sums the run
  if (threadIdx.x < n && (threadIdx.x == 0 || E.gate[threadIdx.x - 1] != E.gate[threadIdx.x])) {
    const int g = E.gate[threadIdx.x];
    double tot = 0.0;
    for (int q = threadIdx.x; q < n && E.gate[q] == g; ++q)
      for (int cls = 0; cls < 5; ++cls) tot += dots[q * 5 + cls];
    grad[g] = 2.0 * tot;
  }
}

// ---- tile kernels -----------------------------------------------------------

struct TileLds {
  double* X;
  double* L;
  int32_t* rows;
  int32_t* cols;
};

__device__ __forceinline__ TileLds carve_lds(double* smem, int R, int W, bool rev) {
  TileLds m;
  char* p = reinterpret_cast<char*>(smem);
  const size_t v = align16((size_t)R * W * 8 + 8);
  m.X = smem;
  p += v;
  m.L = reinterpret_cast<double*>(p);
  if (rev) p += v;
  if (threadIdx.x == 0) {
    m.X[0] = 0.0;
    if (rev) m.L[0] = 0.0;
  }
  m.rows = reinterpret_cast<int32_t*>(p);
  m.cols = m.rows + R;
  return m;
}

// A tile's canonical rows and columns into LDS.
template <int NT>
__device__ __forceinline__ void tile_setup(const StageDev& S, const TileRec& T, const TileLds& m) {
  for (int r = threadIdx.x; r < T.R; r += NT) m.rows[r] = S.arows[T.r0 + r];
  for (int c = threadIdx.x; c < T.W; c += NT) m.cols[c] = S.bcol[T.c0 + c];
  __syncthreads();
}

// Data that no kernel in flight writes, read through the constant address
// space: uniform reads become scalar loads, also past the barriers' memory
// clobbers (which otherwise turn them into vector loads with a full wait).
template <class T>
using ConstPtr = const T __attribute__((address_space(4)))*;
template <class T>
__device__ __forceinline__ ConstPtr<T> as_const(const T* p) {
  return (ConstPtr<T>)(uintptr_t)p;
}

// A thread's orbit words of one pair op: wave v takes the wave-sized groups
// v, v + NT / 64, ...
template <int NT>
struct Words {
  static constexpr int P = (kMaxWaves + NT / 64 - 1) / (NT / 64);
  uint32_t w[P];
};

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

template <int NT>
__device__ __forceinline__ void load_words(const uint32_t* __restrict__ items, int n, Words<NT>& x) {
#pragma unroll
  for (int u = 0; u < Words<NT>::P; ++u) {
    const int g = wave_id() + u * (NT / 64);
    if (g < n) x.w[u] = items[g * 64 + (threadIdx.x & 63)];
  }
}

// Global <-> LDS copies of a tile for NV vectors (psi | lam), gathered
// through the row and column tables, U loads per vector in flight.
template <int NT, int NV>
__device__ __forceinline__ void tile_load(const StageDev& S, const TileRec& T, const TileLds& m,
                                          const double* __restrict__ g0, const double* __restrict__ g1) {
  constexpr int U = NT >= 1024 ? 5 : 8;
  const int E = T.R * T.W;
  const float invW = 1.0f / (float)T.W;
  for (int e0 = threadIdx.x; e0 < E; e0 += NT * U) {
    double v[NV][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * NT;
      if (e < E) {
        const int r = (int)(((float)e + 0.5f) * invW);
        const size_t idx = (size_t)m.rows[r] * S.nsb + m.cols[e - r * T.W];
        v[0][u] = g0[idx];
        if (NV > 1) v[NV - 1][u] = g1[idx];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * NT;
      if (e < E) {
        m.X[1 + e] = v[0][u];
        if (NV > 1) m.L[1 + e] = v[NV - 1][u];
      }
    }
  }
}

template <int NT, int NV>
__device__ __forceinline__ void tile_store(const StageDev& S, const TileRec& T, const TileLds& m, double* g0,
                                           double* g1) {
  const int E = T.R * T.W;
  const float invW = 1.0f / (float)T.W;
  for (int e = threadIdx.x; e < E; e += NT) {
    const int r = (int)(((float)e + 0.5f) * invW);
    const int c = e - r * T.W;
    const size_t idx = (size_t)m.rows[r] * S.nsb + m.cols[c];
    g0[idx] = m.X[1 + e];
    if (NV > 1) g1[idx] = m.L[1 + e];
  }
}

// o = M v (TR: M^T v), M row-major 4x4.
template <bool TR>
__device__ __forceinline__ void mat4(const double (&M)[16], const double (&v)[4], double (&o)[4]) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double acc = (TR ? M[a] : M[4 * a]) * v[0];
#pragma unroll
    for (int b = 1; b < 4; ++b) acc += (TR ? M[4 * b + a] : M[4 * a + b]) * v[b];
    o[a] = acc;
  }
}

template <bool TR>
__device__ __forceinline__ void orbit2(double* X, uint32_t w, const double (&B)[4]) {
  const int m0 = (int)(w & 8191u), m1 = m0 + (int)(w >> 13);
  const double v0 = X[m0], v1 = X[m1];
  X[m0] = B[0] * v0 + (TR ? B[2] : B[1]) * v1;
  X[m1] = (TR ? B[1] : B[2]) * v0 + B[3] * v1;
}

template <int NT, bool TR>
__device__ __forceinline__ void fwd_op(const OpItems& o, const Words<NT>& x, double* X, ConstPtr<double> Mp,
                                       const uint32_t* __restrict__ items) {
  double M[16], be[4], bd[4], ae[4], ad[4];
#pragma unroll
  for (int q = 0; q < 16; ++q) M[q] = Mp[q];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    be[q] = Mp[16 + q];
    bd[q] = Mp[20 + q];
    ae[q] = Mp[24 + q];
    ad[q] = Mp[28 + q];
  }
  const bool deriv = Mp[kPairVals] == 0.0;
#pragma unroll
  for (int u = 0; u < Words<NT>::P; ++u) {
    const int g = wave_id() + u * (NT / 64);
    const uint32_t w = x.w[u];
    if (g < o.c1) {
      const int m0 = (int)(w & 8191u), dr = (int)((w >> 13) & 8191u), dc = (int)(w >> 26);
      const double v[4] = {X[m0], X[m0 + dr], X[m0 + dc], X[m0 + dr + dc]};
      double y[4];
      mat4<TR>(M, v, y);
      X[m0] = y[0];
      X[m0 + dr] = y[1];
      X[m0 + dc] = y[2];
      X[m0 + dr + dc] = y[3];
    } else if (g < o.c2) {
      orbit2<TR>(X, w, be);
    } else if (g < o.c3) {
      orbit2<TR>(X, w, bd);
    } else if (g < o.c4) {
      orbit2<TR>(X, w, ae);
    } else if (g < o.c5) {
      orbit2<TR>(X, w, ad);
    }
  }
  if (deriv)  // T_g annihilates the amplitudes no gate moves
    for (int i = o.c5 * 64 + threadIdx.x; i < o.c6 * 64; i += NT) X[items[i]] = 0.0;
}

// Wave sums of four values on the matrix cores.  v_mfma_f64_4x4x4 contracts
// over the four rows of 16 lanes: A[i][k] at lane i + 4 b + 16 k, B[k][j] at
// lane j + 4 b + 16 k, D[i][j] at lane j + 4 b + 16 i.  With A[i][k] = 1 for
// i = q only, value q's sum over the rows lands in row q of D; the four
// products add into one register, whose rows are then summed.  Row q's last
// lane ends with the sum of value q.  (Four MFMAs and 12 vector instructions
// for four values, against about 44 with lane exchanges.)
__device__ __forceinline__ double rows_of(double acc, double one, double v) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(one, v, acc, 0, 0, 0);
}

// The pair ops of one stage on one vector (canonical order, in place).
// dagger: U^+ (transposed matrices, ops in reverse).  src may be dst (in
// place) or the sweep's input vector (first stage).
template <int NT, bool DAGGER>
__global__ __launch_bounds__(NT) void k_win_fwd(StageDev S, const double* __restrict__ mats, const double* src, double* dst, int64_t mats_stride,
                                                int64_t vec_stride) {
  extern __shared__ double smem[];
  mats += blockIdx.y * mats_stride;
  src += blockIdx.y * vec_stride;
  dst += blockIdx.y * vec_stride;
  for (int slot = blockIdx.x; slot < S.nb; slot += gridDim.x) {
    const ConstPtr<TileRec> tp = as_const(S.tiles) + slot;
    const TileRec T{tp->r0, tp->R, tp->c0, tp->W, tp->ka, tp->kb, tp->items, 0};
    if (T.R == 0) continue;
    const TileLds m = carve_lds(smem, T.R, T.W, false);
    const OpItems o = op_items(side_info(S.k, T.ka), side_info(S.k, T.kb));
    const uint32_t* items = S.items + T.items;
    auto at = [&](int j) { return as_const(S.ops) + (DAGGER ? S.nops - 1 - j : j); };
    auto load = [&](int j, Words<NT>& x) {
      if (j < S.nops) load_words<NT>(items + at(j)->pos * o.c6 * 64, o.c5, x);
    };
    auto step = [&](int j, const Words<NT>& cur, Words<NT>& fill) {
      if (j >= S.nops) return;
      lds_barrier();
      load(j + 2, fill);
      const int op = at(j)->op, pos = at(j)->pos;
      fwd_op<NT, DAGGER>(o, cur, m.X, as_const(mats) + op * kMatVals, items + pos * o.c6 * 64);
    };
    tile_setup<NT>(S, T, m);
    Words<NT> a, b, c;
    load(0, a);
    load(1, b);
    tile_load<NT, 1>(S, T, m, src, nullptr);
    for (int j = 0; j < S.nops; j += 3) {
      step(j, a, c);
      step(j + 1, b, a);
      step(j + 2, c, b);
    }
    __syncthreads();
    tile_store<NT, 1>(S, T, m, dst, nullptr);
    __syncthreads();  // the next tile overwrites the LDS tables
  }
}

// One 2-member orbit of the reverse sweep: returns its product
// lam_0 psi_1 - lam_1 psi_0 and un-applies the matrix (B^T) on both vectors.
__device__ __forceinline__ double rev_orbit2(double* X, double* L, uint32_t w, const double (&B)[4]) {
  const int m0 = (int)(w & 8191u), m1 = m0 + (int)(w >> 13);
  const double v0 = X[m0], v1 = X[m1], w0 = L[m0], w1 = L[m1];
  X[m0] = B[0] * v0 + B[2] * v1;
  X[m1] = B[1] * v0 + B[3] * v1;
  L[m0] = B[0] * w0 + B[2] * w1;
  L[m1] = B[1] * w0 + B[3] * w1;
  return w0 * v1 - w1 * v0;
}

// Reverse stage on (psi, lam), in place: per pair op, the antisymmetric orbit
// products Q[a<b] += lam_a psi_b - lam_b psi_a before un-applying the op's
// matrix (M^T) on both.  The wave sums of an op are added up by one wave
// during the next op and go to partial[poff + v * blocks + block], which a
// block that walks several tiles accumulates.
template <int NT>
__global__ __launch_bounds__(NT) void k_win_rev(StageDev S, const double* __restrict__ mats, double* __restrict__ psi,
                                                double* __restrict__ lam, double* __restrict__ partial, int write_back,
                                                int64_t mats_stride, int64_t vec_stride, int64_t part_stride) {
  mats += blockIdx.y * mats_stride;
  psi += blockIdx.y * vec_stride;
  lam += blockIdx.y * vec_stride;
  partial += blockIdx.y * part_stride;
  constexpr int kWaves = NT / 64;
  extern __shared__ double smem[];
  __shared__ double red[2][kQVals][kWaves];
  const int lane = threadIdx.x & 63, wave = wave_id();
  double sel[4];  // rows_of's selectors
#pragma unroll
  for (int q = 0; q < 4; ++q) sel[q] = (lane & 3) == q ? 1.0 : 0.0;
  bool first = true;
  for (int slot = blockIdx.x; slot < S.nb; slot += gridDim.x) {
    const ConstPtr<TileRec> tp = as_const(S.tiles) + slot;
    const TileRec T{tp->r0, tp->R, tp->c0, tp->W, tp->ka, tp->kb, tp->items, 0};
    if (T.R == 0) continue;
    const TileLds m = carve_lds(smem, T.R, T.W, true);
    const OpItems o = op_items(side_info(S.k, T.ka), side_info(S.k, T.kb));
    const uint32_t* items = S.items + T.items;
    double* X = m.X;
    double* L = m.L;
    auto load = [&](int j, Words<NT>& x) {
      if (j >= 0) load_words<NT>(items + as_const(S.ops)[j].pos * o.c6 * 64, o.c5, x);
    };
    auto finish = [&](int j) {  // op j's wave sums to the block's partial
      if (wave == (j & (kWaves - 1)) && lane < kQVals) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) v += red[j & 1][lane][w];
        double* dst = partial + as_const(S.ops)[j].poff + (size_t)lane * gridDim.x + blockIdx.x;
        *dst = first ? v : *dst + v;
      }
    };
    auto step = [&](int j, const Words<NT>& cur, Words<NT>& fill) {
      if (j < 0) return;
      lds_barrier();
      load(j - 2, fill);
      const ConstPtr<double> Mp = as_const(mats) + as_const(S.ops)[j].op * kMatVals;
      double M[16], be[4], bd[4], ae[4], ad[4];
#pragma unroll
      for (int q = 0; q < 16; ++q) M[q] = Mp[q];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        be[q] = Mp[16 + q];
        bd[q] = Mp[20 + q];
        ae[q] = Mp[24 + q];
        ad[q] = Mp[28 + q];
      }
      double Q[8], Qe = 0.0, Qd = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) Q[q] = 0.0;
#pragma unroll
      for (int u = 0; u < Words<NT>::P; ++u) {
        const int g = wave_id() + u * (NT / 64);
        const uint32_t x = cur.w[u];
        if (g < o.c1) {
          const int m0 = (int)(x & 8191u), dr = (int)((x >> 13) & 8191u), dc = (int)(x >> 26);
          const double v[4] = {X[m0], X[m0 + dr], X[m0 + dc], X[m0 + dr + dc]};
          const double w[4] = {L[m0], L[m0 + dr], L[m0 + dc], L[m0 + dr + dc]};
          Q[0] += w[0] * v[1] - w[1] * v[0];
          Q[1] += w[0] * v[2] - w[2] * v[0];
          Q[2] += w[0] * v[3] - w[3] * v[0];
          Q[3] += w[1] * v[2] - w[2] * v[1];
          Q[4] += w[1] * v[3] - w[3] * v[1];
          Q[5] += w[2] * v[3] - w[3] * v[2];
          double y[4];
          mat4<true>(M, v, y);
          X[m0] = y[0];
          X[m0 + dr] = y[1];
          X[m0 + dc] = y[2];
          X[m0 + dr + dc] = y[3];
          mat4<true>(M, w, y);
          L[m0] = y[0];
          L[m0 + dr] = y[1];
          L[m0 + dc] = y[2];
          L[m0 + dr + dc] = y[3];
        } else if (g < o.c2) {
          Q[6] += rev_orbit2(X, L, x, be);
        } else if (g < o.c3) {
          Q[7] += rev_orbit2(X, L, x, bd);
        } else if (g < o.c4) {
          Qe += rev_orbit2(X, L, x, ae);
        } else if (g < o.c5) {
          Qd += rev_orbit2(X, L, x, ad);
        }
      }
      // a wave's groups are wave, wave + kWaves, ...: the types it has
      const bool four = wave < o.c1;
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
      if (four) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s0 = rows_of(s0, sel[q], Q[q]);
        s1 = rows_of(s1, sel[0], Q[4]);
        s1 = rows_of(s1, sel[1], Q[5]);
        s0 = row16_sum(s0);
      }
      s1 = rows_of(s1, sel[2], Q[6]);
      s1 = rows_of(s1, sel[3], Q[7]);
      s2 = rows_of(s2, sel[0], Qe);
      s2 = rows_of(s2, sel[1], Qd);
      s1 = row16_sum(s1);
      s2 = row16_sum(s2);
      if ((lane & 15) == 15) {
        const int q = lane >> 4;
        red[j & 1][q][wave] = s0;
        red[j & 1][4 + q][wave] = s1;
        if (q < 2) red[j & 1][8 + q][wave] = s2;
      }
      if (j + 1 < S.nops) finish(j + 1);
    };
    tile_setup<NT>(S, T, m);
    Words<NT> a, b, c;
    load(S.nops - 1, a);
    load(S.nops - 2, b);
    tile_load<NT, 2>(S, T, m, psi, lam);
    for (int j = S.nops - 1; j >= 0; j -= 3) {
      step(j, a, c);
      step(j - 1, b, a);
      step(j - 2, c, b);
    }
    __syncthreads();
    finish(0);
    first = false;
    if (write_back)  // not for the first stage of the program: the un-applied states are not needed
      tile_store<NT, 2>(S, T, m, psi, lam);
    __syncthreads();  // the next tile overwrites the LDS tables and red
  }
  if (first)  // no tile: empty sums
    for (int x = threadIdx.x; x < S.nops * kQVals; x += NT)
      partial[S.ops[x / kQVals].poff + (size_t)(x % kQVals) * gridDim.x + blockIdx.x] = 0.0;
}

// ---------------------------------------------------------------------------
// Host orchestration.

static double stage_bytes(const Space& s, int vectors) { return 16.0 * (double)s.dim * vectors; }

static void launch_mats(const TilePlan& T, const double* theta, int deriv_gate, double* mats, const Multi& M,
                        hipStream_t st, double* theta_out = nullptr, double* zero = nullptr, int64_t nzero = 0) {
  const int zb = zero ? (int)std::min<int64_t>((nzero + 1023) / 1024, 512) : 0;
  SQ_PROF(PC_OTHER, st, 8.0 * (double)(zero ? nzero : 0) * M.n, 0.0,
          k_op_mats<<<dim3(T.nops + zb, M.n), 64, 0, st>>>(T.d_info, T.d_entries, theta, deriv_gate, mats, M.theta,
                                                          M.mats, T.nops, theta_out, zero, nzero));
}

// One block per dispatch slot, up to 2048 (more slots are walked by the same
// blocks; 2048 is a multiple of 8, so a block stays on one XCD's slots).
static void launch_fwd(const TilePlan& T, const Stage& S, const double* mats, bool dagger, const double* src,
                       double* dst, const Multi& M, hipStream_t st) {
  auto* kernel = dagger ? (T.nt == 256 ? k_win_fwd<256, true> : T.nt == 512 ? k_win_fwd<512, true> : k_win_fwd<1024, true>)
                        : (T.nt == 256 ? k_win_fwd<256, false> : T.nt == 512 ? k_win_fwd<512, false> : k_win_fwd<1024, false>);
  allow_lds(kernel, S.lds_fwd + 1024);
  const dim3 grid((unsigned)std::max(1, std::min(S.dev.nb, 2048)), (unsigned)M.n);
  kernel<<<grid, T.nt, S.lds_fwd, st>>>(S.dev, mats, src, dst, M.mats, M.vec);
  SQ_HIP(hipGetLastError());
}

static void launch_rev(const TilePlan& T, const Stage& S, const double* mats, double* psi, double* lam,
                       double* partial, int wb, const Multi& M, hipStream_t st) {
  auto* kernel = T.nt == 256 ? k_win_rev<256> : T.nt == 512 ? k_win_rev<512> : k_win_rev<1024>;
  allow_lds(kernel, S.lds_rev + 4096);
  const dim3 grid((unsigned)std::max(1, S.rev_blocks), (unsigned)M.n);
  kernel<<<grid, T.nt, S.lds_rev, st>>>(S.dev, mats, psi, lam, partial, wb, M.mats, M.vec, M.part);
  SQ_HIP(hipGetLastError());
}

static void launch_grad(const TilePlan& T, const double* theta, const double* partial, double* grad, const Multi& M,
                        hipStream_t st, const double* epart = nullptr, int64_t n_epart = 0, double* e_out = nullptr) {
  SQ_PROF(PC_REDUCE, st, 8.0 * ((double)T.partial_len * M.n + (double)n_epart), 0.0,
          k_op_grad<<<dim3(T.nops + (e_out ? 1 : 0), M.n), kTB, 0, st>>>(T.d_info, T.d_entries, theta, partial, grad,
                                                                        M.theta, M.part, M.grad, T.nops, epart,
                                                                        n_epart, e_out));
}

bool tiles_whole(const TilePlan& T) {
  if (T.nops == 0) return false;
  for (const Stage& S : T.stages)
    if (!S.tiled) return false;
  return true;
}

// Forward sweep (dagger: U^+, gates reversed with -theta) over the whole
// program, tiles where possible, psi = U psi_in (canonical order; psi_in may
// be psi).  A first tiled stage reads psi_in itself (its tiles cover every
// amplitude), otherwise psi_in is copied first.
// scratch >= dim doubles (derivative insertion on per-gate stages);
// gwork >= 2*dim doubles for gates that run through the per-gate kernels.
// deriv_gate >= 0 inserts T_g right after gate g (plain gradient; forward only).
void tiles_forward(const Space& s, const Program& p, const TilePlan& T, const double* theta, const double* psi_in,
                   double* psi, double* scratch, double* gwork, int deriv_gate, bool dagger, hipStream_t st,
                   double* zero, double* theta_out) {
  const Multi one;
  launch_mats(T, theta, dagger ? -1 : deriv_gate, T.d_mats, one, st, theta_out, zero, zero ? s.dim : 0);
  const int ns = (int)T.stages.size();
  const double* src = psi_in;
  for (int ii = 0; ii < ns; ++ii) {
    const int i = dagger ? ns - 1 - ii : ii;
    const Stage& S = T.stages[i];
    if (!S.tiled) {
      if (src != psi) copy_vec(src, psi, s.dim, st);
      src = psi;
      apply_gate_impl(s, p, S.g0, theta, dagger, psi, gwork, st);
      if (S.g0 == deriv_gate) {
        grad_action_impl(s, p, S.g0, psi, scratch, st);
        copy_vec(scratch, psi, s.dim, st);
      }
      continue;
    }
    SQ_PROF(PC_TILE_FWD, st, stage_bytes(s, 1), 0.0, launch_fwd(T, S, T.d_mats, dagger, src, psi, one, st));
    src = psi;
  }
  if (src != psi) copy_vec(src, psi, s.dim, st);
}

// Reverse sweep on (psi, lam) with gradient dots into grad_dev[g] (device).
// gwork >= 2*dim; partial: reduction scratch of the per-gate kernels.
// mats_ready: the op matrices of theta (no derivative insertion) are still
// in place from a forward sweep on this stream.
void tiles_reverse(const Space& s, const Program& p, const TilePlan& T, const double* theta, double* psi, double* lam,
                   double* gwork, double* partial, double* grad_dev, bool mats_ready, hipStream_t st,
                   const double* epart, int64_t n_epart, double* e_out) {
  const Multi one;
  if (!mats_ready) launch_mats(T, theta, -1, T.d_mats, one, st);
  for (int i = (int)T.stages.size() - 1; i >= 0; --i) {
    const Stage& S = T.stages[i];
    if (!S.tiled) {
      reverse_step_impl(s, p, S.g0, theta, psi, lam, grad_dev, gwork, partial, st);
      continue;
    }
    const int wb = i > 0 ? 1 : 0;
    SQ_PROF(PC_TILE_REV, st, stage_bytes(s, wb ? 2 : 1), 0.0,
            launch_rev(T, S, T.d_mats, psi, lam, T.d_partial, wb, one, st));
  }
  if (T.nops > 0) launch_grad(T, theta, T.d_partial, grad_dev, one, st, epart, n_epart, e_out);
}

// ---- groups of instances of one program ------------------------------------

int64_t tiles_mats_doubles(const TilePlan& T) { return (int64_t)T.nops * kMatVals; }

int64_t tiles_partial_doubles(const TilePlan& T) { return std::max<int64_t>(T.partial_len, 1); }

void tiles_forward_group(const Space& s, const TilePlan& T, const double* theta, double* psi, double* mats,
                         const Multi& M, double* zero, hipStream_t st) {
  SQ_CHECK(M.n > 0 && M.n <= 65535, SQ_ERR_ARG, "too many instances in one batched group");
  launch_mats(T, theta, -1, mats, M, st, nullptr, zero, s.dim);
  for (const Stage& S : T.stages)
    SQ_PROF(PC_TILE_FWD, st, stage_bytes(s, 1) * M.n, 0.0, launch_fwd(T, S, mats, false, psi, psi, M, st));
}

void tiles_reverse_group(const Space& s, const TilePlan& T, const double* theta, double* psi, double* lam,
                         const double* mats, double* partial, double* grad, const Multi& M, hipStream_t st) {
  for (int i = (int)T.stages.size() - 1; i >= 0; --i) {
    const Stage& S = T.stages[i];
    const int wb = i > 0 ? 1 : 0;
    SQ_PROF(PC_TILE_REV, st, stage_bytes(s, wb ? 2 : 1) * M.n, 0.0,
            launch_rev(T, S, mats, psi, lam, partial, wb, M, st));
  }
  launch_grad(T, theta, partial, grad, M, st);
}

}  // namespace sq
