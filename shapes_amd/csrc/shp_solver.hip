// shp_solver.hip - ordered FP64 (drop-in) solve: the sequential sweep run
// as a schedule of independent items.
//
// The reference applies the cached lagrangians in descending key order
// (applyCachedSlns, shapes/src/Physics/Solvers/Contact.hs:74-121) and then
// sweeps the contacts `iterations` times in the same order (improveWorld,
// :146-157).  A pair's one or two contacts (a manifold) are adjacent in that
// order, so the sequence is a sequence of items (p, m): pass p of manifold m
// (pass 0 is the warm start), both contacts one after the other.  An item
// reads and writes the velocities of its two bodies and its own lagrangians
// only, so it depends on nothing but the latest earlier item on each of its
// dynamic bodies.  Running every item as early as that allows - level by
// level, an item one level after the later of its two predecessors, whatever
// their passes - performs exactly the sequential floating-point operations
// on the same inputs: the result is the sequential one bit for bit.  Static
// bodies (both inverse masses 0) are read-only and order nothing.
//
// What bounds it is the chain of levels, so the levels run across the
// passes (an 8192-polygon pile of 11.5-14.6 k manifolds and 9 passes has
// about 200 of them where pass after pass has 1060, a column scene of 900
// boxes 166 instead of 444), and a level costs the instructions of one
// wavefront, 4.4 cycles each, hardly any latency beside them: so two lanes
// share an item, and one wavefront in four makes the schedule beside the
// others, which run it.
//
// One workgroup per world:
//   1. links: per body the manifolds on it in sequence order; a manifold's
//      link on a body is the next manifold there, after the last one the
//      first (of the next pass)
//   2. the schedule (integer work only): a manifold holds a token count; an
//      item that runs passes a token to the next manifold on each of its
//      dynamic bodies, and a manifold with the tokens of all its dynamic
//      sides is an item of the next level.  Three levels ahead of
//   3. the items, level by level, a barrier after each: entry and record of
//      the next level are loaded while the current one runs; velocities and
//      lagrangians are in LDS when they fit
//   4. velocities and lagrangians are written back
// The links and tokens are 16-bit LDS arrays when they fit (6 bytes a
// contact), else 32-bit arrays in global memory: the same code.
//
// A large world with CUs to spare is solved by many workgroups instead, whose
// items wait for their bodies rather than for a level (k_solve_flow).
//
// Measured (this kernel; before, items waited on per-body counters or ran
// pass after pass): 55-box pyramid 72 us (159), 900 boxes 61 us (741), 512
// worlds of 8-1024 bodies 183 us (752), 8192 polygons 1.48 ms (3.45; there
// the state is in global memory and its line accesses bound a level).
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "shp_engine.h"
#include "shp_flow.h"
#include "shp_geom.h"
#include "shp_records.h"
#include "shp_solve_common.h"

using namespace shp;

// levels in flight: level l runs while level l + 3 is made from level l + 2
#define RING 4
// LDS of the levels' items (more go to global memory): 1016 (2040 with more
// lanes) 16-bit items a level
constexpr int front_bytes(int threads) { return RING * (threads > 256 ? 4096 : 2048); }

// ---- items ------------------------------------------------------------------
// Two lanes per item: the even lane has body a and the friction row's
// lagrangian, the odd lane body b and the normal row's.

__device__ __forceinline__ double dpp_pair(double x, bool from_odd) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return from_odd ? __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0xF5, 0xf, 0xf, true),
                                     __builtin_amdgcn_mov_dpp(lo, 0xF5, 0xf, 0xf, true))
                  : __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0xA0, 0xf, 0xf, true),
                                     __builtin_amdgcn_mov_dpp(lo, 0xA0, 0xf, 0xf, true));
}
// the value of the pair's odd / even lane, in both
__device__ __forceinline__ double from_b(double x) { return dpp_pair(x, true); }
__device__ __forceinline__ double from_a(double x) { return dpp_pair(x, false); }

// An item: its manifold's first contact (world-local), top bit: pass 0.
#define ITEM_WARM 0x80000000u

// One lane's half of an item's record (shp_records.h), as loaded: nothing is
// computed from it before the item runs, so that no instruction waits for
// the loads of the next item.
struct ORec {
  uint32_t item;
  uint16_t warm;     // the contacts' warm flags, a byte each
  double2 u, m, q;   // row normal; this side's inverse masses; mu, ids
  double2 a[2];      // per contact: this side's angular entries of the rows
  double2 f[2];      // per contact: bias and effective mass of this lane's row
};

__device__ __forceinline__ void load_orec(const Ctx& c, int c0, uint32_t item, int side, ORec& r) {
  const int k = c0 + (int)(item & ~ITEM_WARM);
  const double2* h = flow_rec(c, k);
  const double2* hs = h + side;
  r.item = item;
  r.u = h[0];
  r.q = h[3];
  r.m = hs[1];
  r.a[0] = hs[4];
  r.f[0] = hs[6];
  r.a[1] = hs[FLOW_WORDS + 4];  // the next slot, also when there is one contact
  r.f[1] = hs[FLOW_WORDS + 6];
  __builtin_memcpy(&r.warm, c.warm + k, 2);
}

__device__ __forceinline__ int orec_id(const ORec& r, int side) {
  const long long ids = __double_as_longlong(r.q.y);
  return (int)(side ? ids >> 32 : ids);
}

__device__ __forceinline__ double flip_sign(double x, int mask) {
  return __hiloint2double(__double2hiint(x) ^ mask, __double2loint(x));
}

// Velocities (3 doubles per local body in LDS, or gvel) and lagrangians (two
// doubles per contact, normal first, in LDS or glam).  In global memory a
// compute unit's loads and stores cost a cycle per line each instruction
// touches, so there the pair's lanes share every access: lane 0 takes the
// first 16 bytes of a body's word, lane 1 the rest, first body a's, then b's.
template <bool VLDS, bool LLDS>
struct OState {
  double* vel;
  double* lam;
  const Ctx* c;
  int b0, c0;
  // la, lb: the item's bodies; v: this lane's own
  __device__ __forceinline__ void load(int la, int lb, int side, double* v) const {
    if (VLDS) {
      const double* p = vel + 3 * (side ? lb : la);
      v[0] = p[0];
      v[1] = p[1];
      v[2] = p[2];
    } else {
      const double2 a = ((const double2*)(c->gvel + b0 + la))[side];
      const double2 b = ((const double2*)(c->gvel + b0 + lb))[side];
      const double bx = from_a(b.x), by = from_a(b.y), aw = from_b(a.x);
      v[0] = side ? bx : a.x;
      v[1] = side ? by : a.y;
      v[2] = side ? b.x : aw;
    }
  }
  __device__ __forceinline__ void store(int la, int lb, int side, bool fixed, const double* v) const {
    if (VLDS) {
      double* p = vel + 3 * (side ? lb : la);
      if (fixed) return;
      p[0] = v[0];
      p[1] = v[1];
      p[2] = v[2];
    } else {
      // a static body's word gets its own velocity (no other item changes it)
      const double bx = from_b(v[0]), by = from_b(v[1]), aw = from_a(v[2]);
      ((double2*)(c->gvel + b0 + la))[side] = side ? make_double2(aw, 0.0) : make_double2(v[0], v[1]);
      ((double2*)(c->gvel + b0 + lb))[side] = side ? make_double2(v[2], 0.0) : make_double2(bx, by);
    }
  }
  // this lane's lagrangian of contact k + j: the normal one in lane 1
  __device__ __forceinline__ double load_lam(int k, int j, int side) const {
    k += j;
    if (LLDS) return lam[2 * k + 1 - side];
    const double2 l = c->glam[c0 + k];
    return side ? l.x : l.y;
  }
  __device__ __forceinline__ void store_lam(int k, int j, int side, double l) {
    k += j;
    if (LLDS)
      lam[2 * k + 1 - side] = l;
    else
      ((double*)(c->glam + c0 + k))[1 - side] = l;
  }
};

// One item.  Pass 0: useCache (Solvers/Contact.hs:
// 100-114), applySln with the cached lambdas.  Later passes:
// improveContactSln (:124-143), i.e. contactLagrangian with bounceB
// (Constraints/Contact.hs:74-95, Restitution.hs:34-47), solutionProcessor =
// positive / clampAbs (Constraints/Contact.hs:101-110,
// SolutionProcessors.hs:33-53), applySln.  The contacts' rows are jn =
// (-u, jn2, u, jn5) and jt = (-cw(u), jt2, cw(u), jt5): (sx, sy, jn) and
// (sy, -sx, jt) on one side.  The rows' products are folded from index 0
// on: the even lane folds body a's three, the odd lane goes on with body
// b's.  Without restitution the bounce term is min 0 (0 * x) = 0.
// GENERAL: some lane of the wavefront is in pass 0 or has restitution.
template <bool GENERAL, class State>
__device__ __forceinline__ void run_item(const ORec& r, int side, State& S) {
  double v[3], lam[2];
  const int k = (int)(r.item & ~ITEM_WARM);
  const bool warm = GENERAL && (r.item & ITEM_WARM);
  const int id = orec_id(r, side), la = orec_id(r, 0) & FLOW_BODY, lb = orec_id(r, 1) & FLOW_BODY;
  const bool fixed = id < 0, two = (id & FLOW_TWO) != 0;  // FLOW_STATIC is the sign bit
  S.load(la, lb, side, v);
  lam[0] = S.load_lam(k, 0, side);
  lam[1] = two ? S.load_lam(k, 1, side) : 0.0;
  const int neg_a = side ? 0 : (int)0x80000000;
  const double sx = flip_sign(r.u.x, neg_a), sy = flip_sign(r.u.y, neg_a);
  const double iml = r.m.x, imr = r.m.y;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j && !two) break;
    const double l = lam[j];
    const double n0 = sx, n1 = sy, n2 = r.a[j].x, t0 = sy, t1 = -sx, t2 = r.a[j].y;
    const double pn0 = n0 * v[0], pn1 = n1 * v[1], pn2 = n2 * v[2];
    const double pt0 = t0 * v[0], pt1 = t1 * v[1], pt2 = t2 * v[2];
    const double an = from_a((pn0 + pn1) + pn2), at = from_a((pt0 + pt1) + pt2);
    const double dn = ((an + pn0) + pn1) + pn2;  // odd lane
    const double dt = from_b(((at + pt0) + pt1) + pt2);
    double bias = r.f[j].x;
    if (GENERAL && (id & FLOW_BOUNCE)) {
      // closing = ((-va + zcross(-wa, ra)) + vb) + zcross(wb, rb)
      const Ctx& c = *S.c;
      const int kg = S.c0 + k + j;
      const double es = c.e[S.b0 + (side ? lb : la)], e = hs_min(from_a(es), from_b(es));
      const double rx = (side ? c.rbx : c.rax)[kg], ry = (side ? c.rby : c.ray)[kg];
      const double w = side ? v[2] : -v[2];
      const double zx = -(w * ry), zy = w * rx;
      const double ax = from_a(-v[0] + zx), ay = from_a(-v[1] + zy);
      const double cx = (ax + v[0]) + zx, cy = (ay + v[1]) + zy;  // odd lane
      const double bb = hs_min(0.0, e * (cx * sx + cy * sy));
      if (side) bias = bias + bb;
    }
    const double q = (-((side ? dn : dt) + bias)) / r.f[j].y;
    const double m = hs_max(q, -l);
    const double z = side ? m : q;
    const double tot = l + z;
    const double thr = from_b(tot * r.q.x);
    double acc = tot;
    if (!side) acc = tot > thr ? thr : (tot < -thr ? -thr : tot);
    double app = side ? z : acc - l;
    bool apply = !fixed;
    if (warm) {  // the lagrangians as they are
      acc = l;
      app = l;
      apply = apply && ((r.warm >> (8 * j)) & 0xFF) != 0;
    }
    S.store_lam(k, j, side, acc);
    const double gn = from_b(app), gt = from_a(app);
    // applyLagrangian (Constraint.hs:182-221), normal first; a static side
    // keeps its velocity (the reference adds +-0 to it)
    if (apply) {
      v[0] = (v[0] + ((n0 * gn) * iml)) + ((t0 * gt) * iml);
      v[1] = (v[1] + ((n1 * gn) * iml)) + ((t1 * gt) * iml);
      v[2] = (v[2] + ((n2 * gn) * imr)) + ((t2 * gt) * imr);
    }
  }
  S.store(la, lb, side, fixed, v);
}

// ---- schedule ---------------------------------------------------------------

// Exclusive prefix sum over the T threads of one value each.  wsum holds T / 64 ints of LDS.
template <int T>
__device__ __forceinline__ int block_exclusive(int s, int* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  int x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  __syncthreads();  // wsum may still be read from an earlier call
  if (lane == 63) wsum[wid] = x;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int q = 0; q < T / 64; ++q) before += q < wid ? wsum[q] : 0;
  return before + x - s;
}

// All LDS accesses of the workgroup before this point precede all after it;
// global loads and stores stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Schedule state of one world.  A manifold is named by its first contact
// (world-local index).  L: 16-bit entries in LDS, else 32-bit ones in global
// memory.  A link is a manifold, with its top bit set when that manifold has
// one dynamic side only; NONE ends a static side.
template <bool L>
struct Sched {
  using E = std::conditional_t<L, uint16_t, uint32_t>;
  static constexpr uint32_t NONE = L ? 0xFFFFu : 0xFFFFFFFFu;
  static constexpr uint32_t ONE = L ? 0x8000u : 0x80000000u;
  E* next;   // 2 per contact slot: the next manifold on body a, on body b
  E* cnt;    // tokens received, a one-sided manifold's counting twice; the
             // per-body lists while the links are built
  E* off;    // per body (build): end of its list of manifolds it is body b of
  E* first;  // per body (build): the first manifold it is body a of
  // adds v to p[i], returns the old value
  __device__ __forceinline__ static uint32_t add(E* p, uint32_t i, uint32_t v) {
    if constexpr (L) {  // half of an LDS word (no half ever overflows)
      const uint32_t sh = 16u * (i & 1u);
      const uint32_t o = __hip_atomic_fetch_add((uint32_t*)p + (i >> 1), v << sh, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WORKGROUP);
      return (o >> sh) & 0xFFFFu;
    } else {
      return __hip_atomic_fetch_add(p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __device__ __forceinline__ uint32_t count(uint32_t m) const {
    const uint32_t* p = L ? (const uint32_t*)cnt + (m >> 1) : (const uint32_t*)cnt + m;
    const uint32_t x = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return L ? (x >> (16u * (m & 1u))) & 0xFFFFu : x;
  }
  // the manifolds body x is body b of: cnt[lo, hi), unordered
  __device__ __forceinline__ uint32_t lo(int x) const { return x ? off[x - 1] : 0u; }
  __device__ __forceinline__ uint32_t list_min(int x, int above) const {
    uint32_t best = NONE;
    for (uint32_t q = lo(x), hi = off[x]; q < hi; ++q) {
      const uint32_t t = cnt[q];
      if ((int)(t & ~ONE) > above && (t & ~ONE) < (best & ~ONE)) best = t;
    }
    return best;
  }
  // the first manifold on body x: the pairs of larger bodies come first
  __device__ __forceinline__ uint32_t first_of(int x) const {
    const uint32_t t = list_min(x, -1);
    return t != NONE ? t : (uint32_t)first[x];
  }
};

// Links of the world's manifolds and the tokens of pass 0.  ab: per contact
// its local bodies (FLOW_STATIC set for a static one), -1 for the second
// contact of a manifold.
template <int T, bool L>
__device__ __forceinline__ void build_links(const Sched<L>& S, const int2* ab, int n, int nb,
                                            int* wsum) {
  using E = typename Sched<L>::E;
  constexpr uint32_t NONE = Sched<L>::NONE, ONE = Sched<L>::ONE;
  const int tid = threadIdx.x;
  for (int i = tid; i < nb; i += T) {
    S.first[i] = (E)NONE;
    if constexpr (!L) S.off[i] = 0;
  }
  if constexpr (L)
    for (int i = tid; i < (nb + 1) / 2; i += T) ((uint32_t*)S.off)[i] = 0u;
  __syncthreads();
  // per body: how many manifolds it is body b of, the first it is body a of
  // (a body's pairs as a are adjacent)
  for (int k = tid; k < n; k += T) {
    const int2 g = ab[k];
    if (g.x == -1) continue;
    const int2 p = k > 0 ? ab[k - 1] : make_int2(-2, -2);
    const int pa = p.x == -1 ? ab[k - 2].x : p.x;  // a second contact has a first
    if (g.y >= 0) (void)S.add(S.off, (uint32_t)g.y, 1u);
    if (g.x >= 0 && pa != g.x) S.first[g.x] = (E)((uint32_t)k | (g.y < 0 ? ONE : 0u));
  }
  __syncthreads();
  {  // counts -> starts
    const int chunk = (nb + T - 1) / T;
    const int x0 = min(nb, tid * chunk), x1 = min(nb, x0 + chunk);
    int s = 0;
    for (int x = x0; x < x1; ++x) s += (int)S.off[x];
    int run = block_exclusive<T>(s, wsum);
    for (int x = x0; x < x1; ++x) {
      const int t = (int)S.off[x];
      S.off[x] = (E)run;
      run += t;
    }
  }
  __syncthreads();
  for (int k = tid; k < n; k += T) {  // the lists; off becomes their ends
    const int2 g = ab[k];
    if (g.x == -1 || g.y < 0) continue;
    S.cnt[S.add(S.off, (uint32_t)g.y, 1u)] = (E)((uint32_t)k | (g.x < 0 ? ONE : 0u));
  }
  __syncthreads();
  for (int k = tid; k < n; k += T) {
    const int2 g = ab[k];
    if (g.x == -1) continue;
    uint32_t na = NONE, nx = NONE;
    if (g.x >= 0) {
      // the next pair of the same body a, or its first manifold (next pass)
      int k1 = k + 1;
      int2 f = k1 < n ? ab[k1] : make_int2(-2, -2);
      if (f.x == -1) {
        ++k1;
        f = k1 < n ? ab[k1] : make_int2(-2, -2);
      }
      na = f.x == g.x ? (uint32_t)k1 | (f.y < 0 ? ONE : 0u) : S.first_of(g.x);
    }
    if (g.y >= 0) {
      // the next manifold that has it as body b, the first that has it as
      // body a, or its first one (next pass)
      nx = S.list_min(g.y, k);
      if (nx == NONE) nx = S.first[g.y];
      if (nx == NONE) nx = S.first_of(g.y);
    }
    S.next[2 * k] = (E)na;
    S.next[2 * k + 1] = (E)nx;
  }
  __syncthreads();
  for (int x = tid; x < nb; x += T) S.first[x] = (E)S.first_of(x);
  __syncthreads();
  if constexpr (L) {
    for (int i = tid; i < (n + 1) / 2; i += T) ((uint32_t*)S.cnt)[i] = 0u;
  } else {
    for (int i = tid; i < n; i += T) S.cnt[i] = 0u;
  }
  __syncthreads();
}

// The items of the last levels (a ring): CAP of each in LDS (16-bit entries
// when the schedule is in LDS, its manifolds then being below 2^15), the rest
// in global memory; one spare slot a level.  Slots beyond a level's width
// hold older items or 0.  width: the levels' widths, a ring of twice the size.
template <int T, bool L>
struct Front {
  using E = std::conditional_t<L, uint16_t, uint32_t>;
  static constexpr int STRIDE = front_bytes(T) / RING / (int)sizeof(E), CAP = STRIDE - 8;
  static constexpr uint32_t TOP = L ? 0x8000u : 0x80000000u;
  E* lds;
  uint32_t* spill;  // RING x cap
  int* width;       // 2 * RING
  int cap;
  __device__ __forceinline__ static uint32_t item(uint32_t m) {
    return L ? ((m & TOP) << 16) | (m & ~TOP) : m;
  }
  __device__ __forceinline__ E* row(int l) const { return lds + (l & (RING - 1)) * STRIDE; }
  __device__ __forceinline__ uint32_t* far(int l, int i) const {
    return spill + (long)(l & (RING - 1)) * cap + i;
  }
  __device__ __forceinline__ uint32_t near(int l, int i) const { return item(row(l)[i]); }
  // item i of level l, any i below its width
  __device__ __forceinline__ uint32_t get(int l, int i) const {
    uint32_t m = near(l, min(i, CAP - 1));
    // (an atomic load, so that the two do not become one flat load of a
    // selected address, which would wait for every load in flight)
    if (i >= CAP)
      m = __hip_atomic_load(far(l, i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return m;
  }
  __device__ __forceinline__ void put(int l, int i, uint32_t k, bool warm) const {
    if (i < CAP)
      row(l)[i] = (E)(k | (warm ? TOP : 0u));
    else
      *far(l, i) = k | (warm ? ITEM_WARM : 0u);
  }
  __device__ __forceinline__ int n(int l) const {
    return __builtin_amdgcn_readfirstlane(width[l & (2 * RING - 1)]);
  }
};

// Makes level l + 1 from level l with NS wavefronts (sw: this one's number
// among them): every item passes its tokens on.  passes: the last pass.  A
// lane without a token to pass adds 0 to its own item's count, and one
// without an item to list writes the spare slot, so that the common case
// has no branches (a taken one costs as much as six instructions).
template <int NS, int T, bool L>
__device__ __forceinline__ void make_level(const Sched<L>& S, const Front<T, L>& fr, int l, int sw,
                                           int passes) {
  using F = Front<T, L>;
  constexpr uint32_t NONE = Sched<L>::NONE, ONE = Sched<L>::ONE;
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int width = fr.n(l);
  int* out = fr.width + ((l + 1) & (2 * RING - 1));
  auto* row = fr.row(l + 1);
  int made = 0;  // NS == 1
  for (int i0 = sw * 64; i0 < width; i0 += NS * 64) {
    const int i = i0 + lane;
    const bool act = i < width;
    uint32_t k = width <= F::CAP ? fr.near(l, min(i, F::CAP - 1)) : fr.get(l, act ? i : 0);
    k &= ~ITEM_WARM;
    uint32_t t0, t1;
    if constexpr (L) {
      const uint32_t x = ((const uint32_t*)S.next)[k];
      t0 = x & 0xFFFFu;
      t1 = x >> 16;
    } else {
      t0 = S.next[2 * k];
      t1 = S.next[2 * k + 1];
    }
    // a link that does not lead forward leads to the next pass
    const bool last = (int)(S.count(k) >> 1) - 1 >= passes;
    const bool go0 = act && t0 != NONE && !(last && (t0 & ~ONE) <= k);
    const bool go1 = act && t1 != NONE && !(last && (t1 & ~ONE) <= k);
    const uint32_t v0 = go0 ? ((t0 & ONE) ? 2u : 1u) : 0u, v1 = go1 ? ((t1 & ONE) ? 2u : 1u) : 0u;
    const uint32_t n0 = S.add(S.cnt, go0 ? t0 & ~ONE : k, v0) + v0;
    const uint32_t n1 = S.add(S.cnt, go1 ? t1 & ~ONE : k, v1) + v1;
    // an even count: all tokens of a pass, 2 those of pass 0
    const bool r0 = go0 && (n0 & 1u) == 0u, r1 = go1 && (n1 & 1u) == 0u;
    const unsigned long long b0 = __ballot(r0), b1 = __ballot(r1);
    const int c0 = (int)__popcll(b0), all = c0 + (int)__popcll(b1);
    int base = made;
    if constexpr (NS > 1) {
      if (all) {
        if (lane == 0) base = atomicAdd(out, all);
        base = __builtin_amdgcn_readfirstlane(base);
      }
    }
    const int p0 = base + (int)__popcll(b0 & below), p1 = base + c0 + (int)__popcll(b1 & below);
    if (base + all <= F::CAP) {
      row[r0 ? p0 : F::CAP] = (typename F::E)((t0 & ~ONE) | (n0 == 2u ? F::TOP : 0u));
      row[r1 ? p1 : F::CAP] = (typename F::E)((t1 & ~ONE) | (n1 == 2u ? F::TOP : 0u));
    } else {
      if (r0) fr.put(l + 1, p0, t0 & ~ONE, n0 == 2u);
      if (r1) fr.put(l + 1, p1, t1 & ~ONE, n1 == 2u);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    }
    made += all;
  }
  if constexpr (NS == 1) {
    if (lane == 0) *out = made;
  } else {
    // the ring's entry after next, free by now
    if (sw == 0 && lane == 0) fr.width[(l + 2) & (2 * RING - 1)] = 0;
  }
}

// All levels: the last NS wavefronts make the schedule, the others run it,
// STEP items of a level at a time.
template <int T, bool L, bool VLDS, bool LLDS>
__device__ __forceinline__ void run_levels(const Ctx& c, const Sched<L>& Q,
                                           OState<VLDS, LLDS> S, const Front<T, L>& fr) {
  constexpr int NS = T / 256, NE = T / 64 - NS, STEP = NE * 32;
  static_assert(STEP <= Front<T, L>::CAP, "a level's first step reads its LDS slots");
  const int wave = threadIdx.x >> 6;
  auto sync = [] {
    if (VLDS && LLDS)
      lds_barrier();
    else
      __syncthreads();
  };
  // Both loops end at the first empty level: a manifold sends tokens into
  // its next pass only before the last one, and else only forward.
  const int passes = c.iterations;
  for (int l = 0; l < RING - 2; ++l) {  // levels 1 and 2
    if (wave >= NE) make_level<NS, T, L>(Q, fr, l, wave - NE, passes);
    __syncthreads();
  }
  if (wave >= NE) {
    for (int l = 0; fr.n(l) != 0; ++l) {
      make_level<NS, T, L>(Q, fr, l + RING - 2, wave - NE, passes);
      sync();
    }
    return;
  }
  const int side = threadIdx.x & 1, e = (int)threadIdx.x >> 1;
  int l = 0, base = 0, width = fr.n(0);
  ORec x, y;
  load_orec(c, S.c0, fr.near(0, e), side, x);
  auto step = [&](const ORec& now, ORec& nxt) {
    // the next step's item: of this level, or of the next level (a lane
    // beyond the width loads some item's record and does not run it)
    const bool more = base + STEP < width;
    const uint32_t item = more ? fr.get(l, min(base + STEP + e, width - 1))
                               : fr.near(l + 1, e);
    load_orec(c, S.c0, item, side, nxt);
    const bool act = base + e < width;
    if (__ballot(act && ((now.item & ITEM_WARM) || (orec_id(now, side) & FLOW_BOUNCE)))) {
      if (act) run_item<true>(now, side, S);
    } else {
      if (act) run_item<false>(now, side, S);
    }
    base += STEP;
    if (!more) {
      const int w = fr.width[(l + 1) & (2 * RING - 1)];
      sync();
      ++l;
      base = 0;
      width = __builtin_amdgcn_readfirstlane(w);
    }
  };
  while (width > 0) {
    step(x, y);
    if (width == 0) break;
    step(y, x);
  }
}

template <int T, bool L>
__device__ __forceinline__ void solve_world(const Ctx& c, const Sched<L>& Q, unsigned char* pool,
                                            long pool_bytes, int w, int c0, int n, int b0, int nb,
                                            const Front<T, L>& fr, int* wsum) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int2* ab = c.sch_ab + c0;
  build_links<T, L>(Q, ab, n, nb, wsum);
  // a token to the first manifold of every body; the ready ones are level 0
  for (int x0 = 0; x0 < nb; x0 += T) {
    const int x = x0 + tid;
    const uint32_t t = x < nb ? (uint32_t)Q.first[x] : Sched<L>::NONE;
    bool ready = false;
    if (t != Sched<L>::NONE) {
      const uint32_t v = (t & Sched<L>::ONE) ? 2u : 1u;
      ready = ((Q.add(Q.cnt, t & ~Sched<L>::ONE, v) + v) & 1u) == 0u;
    }
    const unsigned long long bal = __ballot(ready);
    int base = 0;
    if (bal) {
      if (lane == 0) base = atomicAdd(&fr.width[0], (int)__popcll(bal));
      base = __builtin_amdgcn_readfirstlane(base);
    }
    if (ready)
      fr.put(0, base + (int)__popcll(bal & ((1ull << lane) - 1ull)), t & ~Sched<L>::ONE, true);
  }
  __syncthreads();
  tmark(c, w, 1);
  // velocities, then lagrangians, in the rest of the LDS pool (over the
  // build's per-body arrays)
  const bool vlds = 24L * nb <= pool_bytes;
  const long vbytes = vlds ? 24L * nb : 0;
  const bool llds = vlds && vbytes + 16L * n <= pool_bytes;
  double* vel = (double*)pool;
  double* lam = vel + 3L * nb;
  for (int i = tid; i < nb; i += T) {
    const double x = c.vx[b0 + i], y = c.vy[b0 + i], w = c.w[b0 + i];
    if (vlds) {
      vel[3 * i] = x;
      vel[3 * i + 1] = y;
      vel[3 * i + 2] = w;
    } else {
      c.gvel[b0 + i] = make_double4(x, y, w, 0.0);
    }
  }
  for (int k = tid; k < n; k += T) {
    const double2 l = make_double2(c.ln[c0 + k], c.lt[c0 + k]);
    if (llds) {
      lam[2 * k] = l.x;
      lam[2 * k + 1] = l.y;
    } else {
      c.glam[c0 + k] = l;
    }
  }
  __syncthreads();
  tmark(c, w, 2);
  tmark(c, w, 3);
  if (llds)
    run_levels<T, L, true, true>(c, Q, OState<true, true>{vel, lam, &c, b0, c0}, fr);
  else if (vlds)
    run_levels<T, L, true, false>(c, Q, OState<true, false>{vel, lam, &c, b0, c0}, fr);
  else
    run_levels<T, L, false, false>(c, Q, OState<false, false>{vel, lam, &c, b0, c0}, fr);
  __syncthreads();
  tmark(c, w, 4);
  for (int k = tid; k < n; k += T) {
    double2 l;
    if (llds)
      l = make_double2(lam[2 * k], lam[2 * k + 1]);
    else
      l = c.glam[c0 + k];
    c.ln[c0 + k] = l.x;
    c.lt[c0 + k] = l.y;
  }
  for (int i = tid; i < nb; i += T) {
    const int g = b0 + i;
    if (c.is_static[g]) continue;
    if (vlds) {
      c.vx[g] = vel[3 * i];
      c.vy[g] = vel[3 * i + 1];
      c.w[g] = vel[3 * i + 2];
    } else {
      const double4 v = c.gvel[g];
      c.vx[g] = v.x;
      c.vy[g] = v.y;
      c.w[g] = v.z;
    }
  }
  __syncthreads();
  tmark(c, w, 5);
}

// ---- one world on several CUs ----------------------------------------------
//
// Two lanes to a manifold for the whole solve, its record and lagrangians in
// their registers, and no schedule: a lane of a manifold waits for the
// manifold's turn on its body (flow_pack's words: pass * the body's manifolds +
// the manifold's place among them in sequence order, from the lists k_sat
// made), and the two run the item when both have it.  So the items run as in
// the levels above, each as early as the latest earlier item on each of its
// bodies allows, and a level costs a hand-over from CU to CU (about 1 us with
// the item) whatever its width, where one CU runs the 600 items of a level of
// an 8192-polygon pile in 7.5 us.  A lane that has seen its body several turns
// away looks again only that many rounds later, and keeps the address of its
// body's words (350 us without).  That pile, 8 iterations: 330 us, 1610 on one
// CU, and 2600 there once its schedule outgrew the LDS (from about 19 k
// contacts).  Looking in every round took 11 us more; workgroups of 64 or 128
// lanes instead of 256 the same.
struct OFlow {
  const Ctx* c;
  int b0, c0;
  u32x4 x, y;  // the body's words as loaded
  double lam[2];
  int g, last;  // the body; its last manifold's pass, else -1
  unsigned long long* word;  // the body's words
  int pass;
  __device__ __forceinline__ void load(int, int, int, double* v) const {
    flow_unpack(x, y, v);
  }
  __device__ __forceinline__ void store(int, int, int, bool fixed, const double* v) const {
    if (fixed) return;
    u32x4 n[2];
    flow_pack(v, (x[1] >> 16) + 1u, n);
    store_16(word, n[0]);
    store_16(word + 2, n[1]);
    if (pass == last) {
      c->vx[g] = v[0];
      c->vy[g] = v[1];
      c->w[g] = v[2];
    }
  }
  __device__ __forceinline__ double load_lam(int, int j, int) const { return lam[j]; }
  __device__ __forceinline__ void store_lam(int, int j, int, double l) { lam[j] = l; }
};

__global__ __launch_bounds__(256) void k_solve_flow(Ctx c) {
  __shared__ int s_tmp[2];
  const int blk = blockIdx.x % c.flow_groups, w = c.world_order[blockIdx.x / c.flow_groups];
  const int b0 = c.body_off[w];
  const int p0 = c.wpair_off[w], np = c.wpair_off[w + 1] - p0;
  int* ctl = c.flow_ctl + (long)w * FLOW_CTL;
  const int want = (np + FLOW_ORDERED_PAIRS - 1) / FLOW_ORDERED_PAIRS;
  if (np == 0) return;
  // bodies of too many manifolds, too many pairs, or contacts beyond the
  // capacity: k_solve_ordered
  if (ctl[FC_FULL] != 0 || want > c.flow_groups || c.coff[p0 + np] > c.contact_cap) {
    if (blk == 0 && threadIdx.x == 0) ctl[FS_ALONE] = 1;
    return;
  }
  if (blk >= want) return;
  int groups;
  const int seat = flow_join(c, ctl + FS_SEATS, ctl + FS_GROUPS, blk, want, s_tmp, &groups);
  if (seat < 0) return;
  if (groups < want) {
    if (seat == 0 && threadIdx.x == 0) ctl[FS_ALONE] = 1;
    return;
  }
  if (seat == 0) tmark(c, w, 0);
  const int side = threadIdx.x & 1, q = seat * FLOW_ORDERED_PAIRS + ((int)threadIdx.x >> 1);
  const int p = p0 + q, passes = c.iterations + 1, shift = c.flow_shift[w];
  ORec r;
  OFlow S;
  S.c = &c;
  S.b0 = b0;
  S.c0 = c.wcont_off[w];
  S.pass = 0;
  bool alive = q < np && c.ccount[p] > 0;
  int k = 0, at = 0, of = 0, id = 0;
  if (alive) {
    k = c.coff[p] - S.c0;
    load_orec(c, S.c0, (uint32_t)k, side, r);
    id = orec_id(r, side);
    S.g = b0 + (id & FLOW_BODY);
    const double *ln = c.ln + S.c0 + k, *lt = c.lt + S.c0 + k;
    S.lam[0] = side ? ln[0] : lt[0];
    S.lam[1] = (id & FLOW_TWO) == 0 ? 0.0 : side ? ln[1] : lt[1];
    if (id >= 0) {
      of = c.adj_n[S.g + shift];
      const int4* row = (const int4*)(c.adj + (long)(S.g + shift) * FLOW_DEGREE);
      for (int e = 0; e < of; e += 4) {
        const int4 x = row[e / 4];
        at += x.x < p;
        at += e + 1 < of && x.y < p;
        at += e + 2 < of && x.z < p;
        at += e + 3 < of && x.w < p;
      }
    } else {
      const double v[3] = {c.vx[S.g], c.vy[S.g], c.w[S.g]};
      u32x4 n[2];
      flow_pack(v, 0, n);
      S.x = n[0];
      S.y = n[1];
    }
    S.last = at == of - 1 ? passes - 1 : -1;
  }
  S.word = c.flow_vel + FLOW_LINE * (long)((alive ? S.g : b0) + shift);
  int rest = 0;
  if (seat == 0)
    for (int k = 1; k < 4; ++k) tmark(c, w, k);
  for (int polls = 1; __ballot(alive); ++polls) {
    bool ready = alive && id < 0;
    if (alive && id >= 0) {
      if (rest > 0) {
        --rest;
      } else {
        const uint32_t turn = (uint32_t)(S.pass * of + at) & 0xFFFFu;
        load_pair(S.word, S.word + 2, S.x, S.y);
        ready = S.x[1] >> 16 == turn && S.x[3] >> 16 == turn && S.y[1] >> 16 == turn &&
                S.y[3] >> 16 == turn;
        rest = ready ? 0 : min(((int)(turn - (S.x[1] >> 16)) & 0xFFFF) - 1, 7);
      }
    }
    const int other = __builtin_amdgcn_mov_dpp((int)ready, 0xB1, 0xf, 0xf, true);
    const bool run = ready && other;
    r.item = (uint32_t)k | (S.pass == 0 ? ITEM_WARM : 0u);
    if (__ballot(run)) {
      if (__ballot(run && (S.pass == 0 || (id & FLOW_BOUNCE)))) {
        if (run) run_item<true>(r, side, S);
      } else {
        if (run) run_item<false>(r, side, S);
      }
      if (run && ++S.pass == passes) {
        alive = false;
        double* l = (side ? c.ln : c.lt) + S.c0 + k;
        l[0] = S.lam[0];
        if (id & FLOW_TWO) l[1] = S.lam[1];
      }
      polls = 0;  // what remains to wait for has come nearer
    }
    if (polls % 256 == 255) {
      if (polls >= c.flow_polls - 1) {
        atomicOr(&c.counters[CNT_FLAGS], SHP_FLAG_STALL);
        poke(ctl + FS_ABORT, 1);
      }
      if (peek(ctl + FS_ABORT) != 0) return;
    }
  }
  tmark_last(c, w, 4);  // (a manifold's last item has written its results back)
  tmark_last(c, w, 5);
}

template <int T>
__global__ __launch_bounds__(T) void k_solve_ordered(Ctx c, int pool_bytes) {
  extern __shared__ __align__(16) unsigned char pool[];
  __shared__ int wsum[T / 64];
  __shared__ int s_front[front_bytes(T) / 4];
  __shared__ int s_width[2 * RING];
  const int w = c.world_order[blockIdx.x];
  const int tid = threadIdx.x;
  const int c0 = c.wcont_off[w], c1 = c.wcont_off[w + 1];
  if (c1 <= c0) return;
  // solved by k_solve_flow?
  if ((int)blockIdx.x < c.flow_worlds && c.flow_ctl[(long)w * FLOW_CTL + FS_ALONE] == 0) return;
  const int n = c1 - c0;
  const int b0 = c.body_off[w], nb = c.body_off[w + 1] - b0;
  tmark(c, w, 0);
  if (tid < 2 * RING) s_width[tid] = 0;
  for (int i = tid; i < front_bytes(T) / 4; i += T) s_front[i] = 0;
  uint32_t* glob = c.sch_glob + (3L + RING) * c0;
  // LDS: links 4 B and tokens 2 B a contact, then 4 B a body while they are
  // built (then the velocities)
  const long hot = (4L * n + 2L * ((n + 1) & ~1) + 15) & ~15L;
  const long body2 = 2L * ((nb + 1) & ~1);
  if (n < 0x7FFF && c.iterations < 0x7FF0 && nb < 0x7FFF && hot + 2 * body2 <= pool_bytes) {
    Sched<true> Q;
    Q.next = (uint16_t*)pool;
    Q.cnt = Q.next + 2 * n;
    Q.off = (uint16_t*)(pool + hot);
    Q.first = (uint16_t*)(pool + hot + body2);
    solve_world<T, true>(c, Q, pool + hot, pool_bytes - hot, w, c0, n, b0, nb,
                         Front<T, true>{(uint16_t*)s_front, glob + 3L * n, s_width, n}, wsum);
  } else {
    Sched<false> Q;
    Q.next = glob;
    Q.cnt = glob + 2L * n;
    Q.off = (uint32_t*)c.sch_off + b0;
    Q.first = (uint32_t*)c.sch_first + b0;
    solve_world<T, false>(c, Q, pool, pool_bytes, w, c0, n, b0, nb,
                          Front<T, false>{(uint32_t*)s_front, glob + 3L * n, s_width, n}, wsum);
  }
}

// static LDS: wsum, s_front, s_width
size_t ordered_static_lds(int threads) {
  return lds16((size_t)(threads / 64) * 4) + lds16(front_bytes(threads)) + lds16(2 * RING * 4);
}

// LDS per world: velocities 24 B a body, about 2.2 contacts of 22 B a body,
// as far as it goes.  4 waves per world; a world of more than
// 512 bodies gets 8 (with 16, at 128 registers a lane, an 8192-polygon pile
// took 1.93 ms instead of 1.64).
void plan_ordered_solver(StepPlan* P, int solver_threads, const std::vector<int32_t>& body_off,
                         const std::vector<int32_t>& order) {
  P->solve_threads = solver_threads ? solver_threads : (P->max_nb > 512 ? 512 : 256);
  const size_t room = LDS_BYTES_PER_CU - ordered_static_lds(P->solve_threads) - 256;
  P->solve_lds = std::min<size_t>(room, 72UL * P->max_nb + 1024);
  // Worlds on several CUs, while the lanes (two to a pair) fit the GPU at 110
  // registers: us a step, 6 iterations, on several CUs against one: one world
  // of 1024 bodies 327 / 246, 2048 412 / 333, 4096 527 / 681, 8192 653 / 1211,
  // 16384 870 / 2751, 32768 1152 / 5004; 4 of 8192 754 / 1317.
  int big = 0;
  while (big < P->W && body_off[order[big] + 1] - body_off[order[big]] > FLOW_ORDERED_MIN_BODIES)
    ++big;
  if (big > 0) {
    const long groups = std::min<long>((3 * P->max_nb + FLOW_ORDERED_PAIRS - 1) / FLOW_ORDERED_PAIRS,
                                       FLOW_ORDERED_GROUPS / big);
    if (groups * FLOW_ORDERED_PAIRS >= 2 * P->max_nb) {
      P->flow_worlds = big;
      P->flow_groups = (int)groups;
    }
  }
}

static const void* ordered_kernel(int threads) {
  return threads == 512 ? (const void*)k_solve_ordered<512> : (const void*)k_solve_ordered<256>;
}

shp_status solver_alloc(shp_batch* b) {
  const StepPlan& P = b->plan;
  if (P.solver != SHP_SOLVER_ORDERED_F64) return colored_alloc(b);
  const void* fn = ordered_kernel(P.solve_threads);
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)P.solve_lds) !=
      hipSuccess) {
    shp_set_error("hipFuncSetAttribute (ordered solver LDS) failed");
    return SHP_E_HIP;
  }
  hipFuncAttributes a{};
  if (hipFuncGetAttributes(&a, fn) != hipSuccess ||
      a.sharedSizeBytes > ordered_static_lds(P.solve_threads)) {
    shp_set_error("ordered solver: static LDS above the plan's");
    return SHP_E_HIP;
  }
  return SHP_OK;
}

void launch_ordered_solver(shp_batch* b) {
  const StepPlan& P = b->plan;
  const Ctx& c = b->ctx;
  if (P.flow_worlds > 0)
    k_solve_flow<<<(unsigned)(P.flow_worlds * P.flow_groups), 256, 0, b->stream>>>(c);
  if (P.solve_threads == 512)
    k_solve_ordered<512><<<c.W, 512, P.solve_lds, b->stream>>>(c, (int)P.solve_lds);
  else
    k_solve_ordered<256><<<c.W, 256, P.solve_lds, b->stream>>>(c, (int)P.solve_lds);
}
