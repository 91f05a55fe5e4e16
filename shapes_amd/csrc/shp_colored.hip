// shp_colored.hip - graph-coloured Gauss-Seidel solver (FP32 math, FP64
// impulse accumulators) and the per-step solve-quality measurements.
//
// The reference solves contacts strictly one after another
// (improveWorld, shapes/src/Physics/Solvers/Contact.hs:146-157).  This mode
// keeps the same per-contact update (lagrangian2, positive, clampAbs,
// applySln) but reorders the sweep: a world's manifolds (pairs with
// contacts; one lane solves a pair's <= 2 points in key order) are coloured
// so that no two manifolds of a colour share a dynamic body, then each
// colour is solved in parallel.  Colours come from deterministic
// Jones-Plassmann rounds: in each round every uncoloured manifold whose
// hashed priority is the largest among the uncoloured manifolds on each of
// its dynamic bodies is selected (the selected manifolds share no dynamic
// body) and takes the smallest colour that no manifold on its dynamic
// bodies has (a 16-bit mask per body; past 16 colours, colour 16 + round).
// Velocities and constraint rows are FP32 (velocities staged in LDS when they
// fit); the accumulated lagrangians stay FP64; each body's FP64 velocity
// receives the FP32 change of the solve, so bodies without contacts keep their
// FP64 velocity exactly.
//
// Records are per manifold: the normal, materials, inverse masses and
// bodies once, then per contact the two cross terms of each row, bias,
// lever arms, effective masses and the FP64 lagrangians; a second contact
// has a record of its own (a manifold with one contact reads nothing of
// it).  Records are interleaved word by word in blocks of four manifolds
// (shp_records.h): a wavefront reading 64 consecutive manifolds reads each
// word as 16 runs of 64 bytes, the rest of each 128-byte line being the
// next word, which its next load reads, with 16-byte loads from one
// address per lane; one manifold's record spans about four lines, which
// is what its writer stores to (blocks of 64: seven).  The rows are
// rebuilt from them exactly (jn = (-u, jn2, u, jn5), jt = (-cw(u), jt2,
// cw(u), jt5) with u the row normal; negation commutes with rounding to
// FP32).  A lane keeps its slot of a colour in every pass, so the record
// of its manifold of the next colour (lagrangians included) is loaded
// before the barrier that ends the current colour.
//
// A large world with CUs to spare is coloured and swept by many workgroups
// instead, whose manifolds wait for the bodies they need, not for each other
// (colour_flow, sweep_flow): the same colours and the same updates of each
// body in the same order, so the same results.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "shp_engine.h"
#include "shp_flow.h"
#include "shp_geom.h"
#include "shp_records.h"
#include "shp_solve_common.h"

using namespace shp;

// colours 0..15 are assigned smallest-free from the per-body masks; a
// manifold whose bodies already use all 16 takes GREEDY_COLOURS + round,
// so the Jones-Plassmann rounds stop at JP_ROUNDS to keep every colour and
// the serial tail below COLOR_CAP (and below the uint8 sentinel 0xFF)
#define GREEDY_COLOURS 16
#define JP_ROUNDS (COLOR_CAP - GREEDY_COLOURS - 3)


__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

// a . b as a product and five fused multiply-adds, in index order
__device__ __forceinline__ float dot6f(const float* a, const float* b) {
  float d = a[0] * b[0];
#pragma unroll
  for (int q = 1; q < 6; ++q) d = fmaf(a[q], b[q], d);
  return d;
}

struct ConF {
  float jn2, jn5, jt2, jt5, bn, icn, ict, wn2, wn5, wt2, wt5;
  double ln, lt;
};

struct ManF {
  float ux, uy, mu, e, ax, ay, bx, by;
  int ga, gb, flags, turns;
  ConF k[2];
};

// The records and the first manifold of one world.
struct RecW {
  float4* rec;
  float4* rec2;
  int p0;
};

__device__ __forceinline__ RecW recw(const Ctx& c, const PackF& P, int p0) {
  RecW r;
  r.rec = P.rec;
  r.rec2 = P.rec2;
  r.p0 = p0;
  return r;
}

// Words 3-6 of a record, `step` apart: one contact.
__device__ __forceinline__ void load_contact(const float4* w, int step, ConF& k) {
  const float4 a = w[0], b = w[step], d = w[2 * step];
  const double2 l = *(const double2*)(w + 3 * step);
  k.jn2 = a.x;
  k.jn5 = a.y;
  k.jt2 = a.z;
  k.jt5 = a.w;
  k.bn = b.x;
  k.icn = b.y;
  k.ict = b.z;
  k.wn2 = b.w;
  k.wn5 = d.x;
  k.wt2 = d.y;
  k.wt5 = d.z;
  k.ln = l.x;
  k.lt = l.y;
}

// Words 0-2: the manifold.
__device__ __forceinline__ void load_head(const float4* r, int step, ManF& m) {
  const float4 a = r[0], b = r[step];
  const int4 g = *(const int4*)(r + 2 * step);
  m.ux = a.x;
  m.uy = a.y;
  m.mu = a.z;
  m.e = a.w;
  m.ax = b.x;
  m.ay = b.y;
  m.bx = b.z;
  m.by = b.w;
  m.ga = g.x;
  m.gb = g.y;
  m.flags = g.z;
  m.turns = g.w;
}

// Manifold m of the world (local index) and its contacts; the second
// contact's record loads only when the manifold has one.
__device__ __forceinline__ void load_man(const RecW& R, int m_loc, ManF& m) {
  const float4* r = rec_of(R.rec, R.p0 + m_loc);
  load_head(r, RB, m);
  load_contact(r + 3 * RB, RB, m.k[0]);
  if (m.flags & MFL_TWO) load_contact(rec2_of(R.rec2, R.p0 + m_loc), RB, m.k[1]);
}

// Where contact j's lagrangians of manifold m_loc are.
__device__ __forceinline__ double2* lambda_of(const RecW& R, int m_loc, int j) {
  return (double2*)(j ? rec2_of(R.rec2, R.p0 + m_loc) + 3 * RB : rec_of(R.rec, R.p0 + m_loc) + 6 * RB);
}

// v += l * w, fused per entry (w: a row times the inverse masses)
__device__ __forceinline__ void applyw(float l, const float* w, float* v) {
#pragma unroll
  for (int q = 0; q < 6; ++q) v[q] = fmaf(l, w[q], v[q]);
}

// FP32 velocities: LDS (3 floats per local body) or fv (global memory).
template <bool VLDS>
struct VelF {
  float* lds;
  const Ctx* c;
  int b0;
  // the velocities of a manifold's bodies, and back
  __device__ __forceinline__ void load(const ManF& m, float* v) const {
    load(m.ga, v);
    load(m.gb, v + 3);
  }
  __device__ __forceinline__ void store(const ManF& m, const float* v, bool changed) const {
    if (!changed) return;
    if (!(m.flags & MFL_A_STATIC)) store(m.ga, v);
    if (!(m.flags & MFL_B_STATIC)) store(m.gb, v + 3);
  }
  __device__ __forceinline__ void load(int g, float* v) const {
    if (VLDS) {
      const float* p = lds + 3 * (g - b0);
      v[0] = p[0];
      v[1] = p[1];
      v[2] = p[2];
    } else {
      const float4 x = c->fv[g];
      v[0] = x.x;
      v[1] = x.y;
      v[2] = x.z;
    }
  }
  __device__ __forceinline__ void store(int g, const float* v) const {
    if (VLDS) {
      float* p = lds + 3 * (g - b0);
      p[0] = v[0];
      p[1] = v[1];
      p[2] = v[2];
    } else {
      c->fv[g] = make_float4(v[0], v[1], v[2], 0.0f);
    }
  }
};

// Velocities of a world swept by several workgroups: two words per body in
// global memory, vx | omega's low half << 32 | turn << 48 and vy | omega's
// high half << 32 | turn << 48, where `turn` counts the manifolds that have
// had the body.  A manifold takes its bodies when the count is its own turn,
// pass * (the body's manifolds) + its place among them by colour, and hands
// them on by writing the words with the count raised: the data carry their
// own flag, so that no barrier, fence or acknowledged store lies between two
// colours, only one store and the load that sees it (0.54 us between CUs of
// an XCD, 0.68 across XCDs; a barrier of 256 workgroups alone takes 3.5).
// (No word can be a whole 2^16 turns behind: the manifold itself has had the
// body in the last pass.)  Both words move in one 16-byte access, each with
// its own count, past the L1 cache (sc1, as agent-scope atomics compile to;
// there is none of 16 bytes): as two accesses of 8 bytes a hand-over takes
// 0.70 and 0.86 us.  A body has a line of 128 bytes to itself: accesses to one
// line from many CUs wait for each other (8192 polygons 114 us with 8 bodies to
// a line, 96 with one; with the 16-byte accesses 88).
struct VelFlow {
  const Ctx* c;
  unsigned long long* vel;  // the line of body 0, whose world's bodies have theirs
  int* abort;
  mutable bool dead;
  mutable unsigned long long w[4];  // the words as loaded

  static __device__ __forceinline__ void unpack(unsigned long long x, unsigned long long y, float* v) {
    v[0] = __uint_as_float((uint32_t)x);
    v[1] = __uint_as_float((uint32_t)y);
    v[2] = __uint_as_float(((uint32_t)(x >> 32) & 0xFFFFu) | (uint32_t)(y >> 32) << 16);
  }
  static __device__ __forceinline__ void pack(const float* v, uint32_t turn, unsigned long long* w) {
    const uint32_t o = __float_as_uint(v[2]);
    w[0] = __float_as_uint(v[0]) | (unsigned long long)((o & 0xFFFFu) | turn << 16) << 32;
    w[1] = __float_as_uint(v[1]) | (unsigned long long)((o >> 16) | turn << 16) << 32;
  }
  // waits for the manifold's turn on both its bodies
  __device__ __forceinline__ void wait(const ManF& m, int pass) const {
    const Turns t = unpack_turns(m.turns);
    const uint32_t ta = (uint32_t)(pass * t.of_a + t.at_a) & 0xFFFFu,
                   tb = (uint32_t)(pass * t.of_b + t.at_b) & 0xFFFFu;
    const unsigned long long *pa = vel + FLOW_LINE * (long)m.ga, *pb = vel + FLOW_LINE * (long)m.gb;
    for (int n = 1;; ++n) {
      u32x4 x, y;
      load_pair(pa, pb, x, y);
      w[0] = x[0] | (unsigned long long)x[1] << 32;
      w[1] = x[2] | (unsigned long long)x[3] << 32;
      w[2] = y[0] | (unsigned long long)y[1] << 32;
      w[3] = y[2] | (unsigned long long)y[3] << 32;
      const bool a = t.of_a == 0 || ((uint32_t)(w[0] >> 48) == ta && (uint32_t)(w[1] >> 48) == ta);
      const bool b = t.of_b == 0 || ((uint32_t)(w[2] >> 48) == tb && (uint32_t)(w[3] >> 48) == tb);
      if ((a && b) || dead) break;
      if (n % 256 == 0) {
        if (n >= c->flow_polls) {
          atomicOr(&c->counters[CNT_FLAGS], SHP_FLAG_STALL);
          poke(abort, 1);
        }
        dead = peek(abort) != 0;
      }
    }
  }
  __device__ __forceinline__ void load(const ManF&, float* v) const {
    unpack(w[0], w[1], v);
    unpack(w[2], w[3], v + 3);
  }
  __device__ __forceinline__ void store(const ManF& m, const float* v, bool changed) const {
    const Turns t = unpack_turns(m.turns);
    auto hand_on = [&](int g, const unsigned long long* old, const float* x, bool keep) {
      const uint32_t turn = ((uint32_t)(old[0] >> 48) + 1u) & 0xFFFFu;
      unsigned long long n[2];
      float y[3];
      unpack(old[0], old[1], y);
      pack(keep ? y : x, turn, n);
      const u32x4 x4 = {(uint32_t)n[0], (uint32_t)(n[0] >> 32), (uint32_t)n[1], (uint32_t)(n[1] >> 32)};
      store_16(vel + FLOW_LINE * (long)g, x4);
    };
    if (t.of_a) hand_on(m.ga, w, v, !changed || (m.flags & MFL_A_STATIC));
    if (t.of_b) hand_on(m.gb, w + 2, v + 3, !changed || (m.flags & MFL_B_STATIC));
  }
};

// One manifold: warm start (pass 0: useCache's applySln) or one sweep
// (improveContactSln with FP32 velocities/rows and FP64 accumulators) of
// its contacts in key order.  lambda(j): where contact j's lagrangians go.
// The FP32 arithmetic is this solver's own: the bounce
// term's closing velocity is the normal row times the velocities (the same
// quantity as bounceB's, Solvers/Contact.hs), the effective masses enter as
// reciprocals, and products with velocities are fused.
template <class Lambda, class Vel>
__device__ __forceinline__ void solve_man(Lambda lambda, ManF& m, bool warm, const Vel& V) {
  float v[6];
  V.load(m, v);
  const int nk = (m.flags & MFL_TWO) ? 2 : 1;
  bool changed = false;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j >= nk) break;
    ConF& k = m.k[j];
    // rows (the friction row's direction is clockwise(u)) and the rows
    // times the inverse masses
    const float jn[6] = {-m.ux, -m.uy, k.jn2, m.ux, m.uy, k.jn5};
    const float jt[6] = {-m.uy, m.ux, k.jt2, m.uy, -m.ux, k.jt5};
    const float wn[6] = {-m.ax, -m.ay, k.wn2, m.bx, m.by, k.wn5};
    const float wt[6] = {-m.ay, m.ax, k.wt2, m.by, -m.bx, k.wt5};
    if (warm) {
      if (!(m.flags & (j == 0 ? MFL_WARM0 : MFL_WARM1))) continue;
      applyw((float)k.ln, wn, v);
      applyw((float)k.lt, wt, v);
      changed = true;
      continue;
    }
    const float dn = dot6f(jn, v), dt = dot6f(jt, v);
    float bb = m.e * dn;  // bounce term
    bb = 0.0f <= bb ? 0.0f : bb;
    const float new_n = -(dn + (k.bn + bb)) * k.icn;
    const float new_t = -dt * k.ict;
    double app_n = hs_max((double)new_n, -k.ln);
    double acc_n = k.ln + app_n;
    double thr = acc_n * (double)m.mu;
    double acc_t = k.lt + (double)new_t;
    double accp = acc_t > thr ? thr : (acc_t < -thr ? -thr : acc_t);
    double app_t = accp - k.lt;
    applyw((float)app_n, wn, v);
    applyw((float)app_t, wt, v);
    k.ln = acc_n;
    k.lt = accp;
    changed = true;
  }
  V.store(m, v, changed);
  if (changed && !warm) {  // the solved contacts' lagrangians
    *lambda(0) = make_double2(m.k[0].ln, m.k[0].lt);
    if (nk > 1) *lambda(1) = make_double2(m.k[1].ln, m.k[1].lt);
  }
}

// The colouring's parts are inlined whatever their size: as a call, one of them
// takes the kernel's arguments (1 KB) and its register arrays through scratch
// memory (4097 worlds' step with k_colour<1024> 1930 us, 1300 inlined).

// Colours per pair, in global memory: -1 uncoloured, -2 no contacts.
__device__ __forceinline__ int colour_of(int x) { return x; }

// Colour of a manifold selected in Jones-Plassmann round r whose dynamic
// bodies use the colours in `used`.
__device__ __forceinline__ int greedy_colour(uint32_t used, int r) {
  return used != 0xFFFFu ? __builtin_ctz(~used) : GREEDY_COLOURS + r;
}

__device__ __forceinline__ int wave_sum(int x) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
__device__ __forceinline__ int wave_max(int x) {
  for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o));
  return x;
}

// atomicAdd(&ctr[key], 1) for every lane with key >= 0, one atomic per
// distinct key of the wavefront (lanes of equal key take consecutive
// values); returns the lane's old value, or -1.  Every lane of the
// wavefront calls it.
__device__ __forceinline__ int wave_count(int* ctr, int key) {
  const int lane = threadIdx.x & 63;
  unsigned long long pending = __ballot(key >= 0);
  int res = -1;
  while (pending) {
    const int leader = __ffsll((long long)pending) - 1;
    const int k = __shfl(key, leader);
    const unsigned long long grp = __ballot(key == k) & pending;
    int base = 0;
    if (lane == leader) base = atomicAdd(&ctr[k], (int)__popcll(grp));
    base = __shfl(base, leader);
    if ((grp >> lane) & 1ull) res = base + (int)__popcll(grp & ((1ull << lane) - 1ull));
    pending &= ~grp;
  }
  return res;
}

// Slots of the coloured manifolds: colour l owns manifold indices
// [p0 + s_off[l], p0 + s_off[l + 1]); scur holds the colour cursors;
// slot[q] (pair q of the world) gets its manifold index, or -1.  The order
// inside a colour is free, except in the serial tail colour (tail >= 0),
// whose manifolds may share bodies: thread 0 places those in pair order.
template <int T, class CT>
__device__ __forceinline__ void assign_slots(int p0, int np, const CT* colour, int* scur, int tail,
                                             int32_t* slot) {
  for (int q0 = 0; q0 < np; q0 += T) {
    const int q = q0 + threadIdx.x;
    const int cl = q < np ? colour_of(colour[q]) : -1;
    const bool in_tail = cl == tail && tail >= 0;
    const int m = wave_count(scur, in_tail ? -1 : cl);
    if (q < np && !in_tail) slot[q] = cl < 0 ? -1 : p0 + m;
  }
  if (tail >= 0 && threadIdx.x == 0) {
    int m = scur[tail];
    for (int q = 0; q < np; ++q)
      if (colour_of(colour[q]) == tail) slot[q] = p0 + m++;
  }
}

// Warm-start pass and sweeps, colour by colour, with prefetching.  Phase
// h = pass * ncol + l; lane t of `step` takes manifolds off[l] + t, + step,
// ... of colour l (the last colour serially by lane 0 when colouring
// stopped after JP_ROUNDS), and `sync` ends each phase.  Two records per
// lane: the lane's next manifold of a colour loads into the other record
// while the current one solves, and its first manifold of the next colour
// loads before the phase ends (not with one colour: that is the manifold
// just solved, whose lagrangians the pass changes).  The colour bounds of
// this phase (cs, ce) and the next (ns, ne) stay in registers; those of
// the phase after next are read early in the phase.
template <class Vel, class Sync>
__device__ __forceinline__ void sweep_prefetched(const Ctx& c, const RecW& R, int ncol,
                                                 bool serial_tail, const int* off, int lane,
                                                 const int step, const Vel& V, Sync sync) {
  const int phases = (c.iterations + 1) * ncol;
  auto first_of = [&](int l, int b0_, int b1_) {
    const bool tail = serial_tail && l == ncol - 1;
    return tail ? (lane == 0 ? b0_ : b1_) : b0_ + lane;
  };
  auto next = [&](int l) { return l + 1 == ncol ? 0 : l + 1; };
  int l = 0, l1 = next(0);
  int cs = off[0], ce = off[1];
  int ns = off[l1], ne = off[l1 + 1];
  ManF m, n;
  bool loaded = false;
  for (int h = 0; h < phases; ++h) {
    const int l2 = next(l1);
    const int s2 = off[l2], e2 = off[l2 + 1];
    const bool warm = h < ncol;
    const int di = serial_tail && l == ncol - 1 ? 1 : step;
    const int end = ce;
    int i = first_of(l, cs, ce);
    if (i < end && !loaded) load_man(R, i, m);
    while (i < end) {
      int inext = i + di;
      bool more = inext < end;
      if (more) load_man(R, inext, n);
      solve_man([&](int j) { return lambda_of(R, i, j); }, m, warm, V);
      if (!more) break;
      i = inext;
      inext = i + di;
      more = inext < end;
      if (more) load_man(R, inext, m);
      solve_man([&](int j) { return lambda_of(R, i, j); }, n, warm, V);
      if (!more) break;
      i = inext;
    }
    loaded = false;
    if (ncol > 1 && h + 1 < phases) {
      const int j = first_of(l1, ns, ne);
      if (j < ne) {
        load_man(R, j, m);
        loaded = true;
      }
    }
    sync();
    cs = ns;
    ce = ne;
    ns = s2;
    ne = e2;
    l = l1;
    l1 = l2;
  }
}

// Warm-start pass and sweeps of one world by one workgroup.
template <bool VLDS, int T>
__device__ void sweep_colours(const Ctx& c, const RecW& R, int ncol, bool serial_tail,
                              const int* s_off, const VelF<VLDS>& V) {
  sweep_prefetched(c, R, ncol, serial_tail, s_off, (int)threadIdx.x, T, V,
                   [] { __syncthreads(); });
}

// Colour-order bookkeeping shared by both kernels: per-colour counts of the
// coloured manifolds -> s_off (exclusive) and s_cur (cursors).
template <int T, class CT>
__device__ __forceinline__ void colour_offsets(const CT* colour, int np, int ncol, int* s_off, int* s_cur) {
  const int tid = threadIdx.x;
  for (int i = tid; i <= ncol + 1; i += T) s_cur[i] = 0;
  __syncthreads();
  for (int q0 = 0; q0 < np; q0 += T) {
    const int q = q0 + tid;
    (void)wave_count(s_cur, q < np ? colour_of(colour[q]) : -1);
  }
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int l = 0; l <= ncol; ++l) {
      int h = s_cur[l];
      s_off[l] = acc;
      s_cur[l] = acc;
      acc += h;
    }
    s_off[ncol + 1] = acc;
  }
  __syncthreads();
}

// Colouring in LDS: local body ids and pair indices fit 16 and 15 bits and
// the colouring (6 B per body, 7 B per manifold) fits the pool.
__device__ __forceinline__ bool colour_fits_lds(int nb, int np, int nm, int pool_bytes) {
  return nb < (int)NO_BODY && np <= 32767 && 4L * nb + 2L * ((nb + 1) & ~1) + 7L * nm <= pool_bytes;
}
// FP32 velocities in LDS: 12 B per body.
__device__ __forceinline__ bool vel_fits_lds(int nb, int pool_bytes) { return 12L * nb <= pool_bytes; }

// Pair indices below this fit prio32 (17 bits, prio32 - 1 below 2^32).
#define PRIO32_PAIRS 131071
// Colouring with the per-body priorities (4 B per body) and, when they fit
// too, colour masks (2 B) in LDS and the manifold lists in global memory.
__device__ __forceinline__ bool colour_fits_hybrid(int nb, int np, int pool_bytes) {
  return nb < (int)NO_BODY && np <= PRIO32_PAIRS && 4L * nb <= pool_bytes;
}
__device__ __forceinline__ bool colour_masks_fit(int nb, int pool_bytes) {
  return 4L * nb + 2L * ((nb + 1) & ~1) <= pool_bytes;
}

// Hashed priority of manifold q of world w: 15 hash bits, then the index
// (distinct within a world).  prio32 packs it for q < PRIO32_PAIRS (LDS
// colouring), prio64 for any q (global colouring); both order manifolds
// alike, so the colours do not depend on which path colours a world.
__device__ __forceinline__ uint32_t prio32(int q, int w) {
  return (((mix32((uint32_t)q * 0x9E3779B9u + (uint32_t)w) & 0x7FFFu) << 17) | (uint32_t)q) + 1u;
}
__device__ __forceinline__ unsigned long long prio64(int q, int w) {
  return ((unsigned long long)(mix32((uint32_t)q * 0x9E3779B9u + (uint32_t)w) & 0x7FFFu) << 32) |
         (unsigned long long)((uint32_t)q + 1u);
}

// After colouring world w (colours 0..top-1, then the serial tail colour
// top if any): per-colour offsets into col_off[w], the colour count into
// col_info[w], and each pair's manifold slot into sched_order (pair index).
template <int T, class CT>
__device__ __forceinline__ void colour_finish(const Ctx& c, int w, int p0, int np, const CT* colour, int top,
                              bool serial_tail, int* s_off, int* s_cur) {
  const int ncol = top + (serial_tail ? 1 : 0);
  if (threadIdx.x == 0) atomicMax(&c.counters[CNT_LEVELS], ncol);
  colour_offsets<T>(colour, np, ncol, s_off, s_cur);
  assign_slots<T>(p0, np, colour, s_cur, serial_tail ? ncol - 1 : -1, c.sched_order + p0);
  int* off = c.col_off + (long)w * (COLOR_CAP + 3);
  for (int l = threadIdx.x; l <= ncol; l += T) off[l] = s_off[l];
  if (threadIdx.x == 0) c.col_info[w] = ncol | (serial_tail ? COL_TAIL : 0);
}

// Number of manifolds (pairs with stored contacts) of a world, summed over
// the workgroup; every thread gets it.
template <int T>
__device__ __forceinline__ int count_manifolds(const Ctx& c, int p0, int np, int* s_cnt) {
  if (threadIdx.x == 0) *s_cnt = 0;
  __syncthreads();
  int mine = 0;
  for (int q = threadIdx.x; q < np; q += T) mine += c.pair_ab[p0 + q] != NO_PAIR;
  mine = wave_sum(mine);
  if ((threadIdx.x & 63) == 0) atomicAdd(s_cnt, mine);
  __syncthreads();
  return *s_cnt;
}

// The rounds of colour_world_lds with each lane's manifolds (m = lane,
// lane + T, ...) held in registers with their bodies, priorities and
// colours: a round reads only the bodies' priorities and colour masks, a
// lane's coloured manifolds drop out of its later rounds, and the
// per-colour counts and manifold slots come from the registers.  The taken
// count is double-buffered, so a round needs three barriers.  Returns false
// (colours written to `colour` per pair instead) when the rounds stopped at
// JP_ROUNDS: the caller then places the serial tail in pair order.
#define COLOUR_REG_ITEMS 16
template <int T>
__device__ __forceinline__ bool colour_regs(const Ctx& c, int w, int p0, int nm, int nb, uint32_t* s_best,
                            uint16_t* s_used, const uint32_t* m_ab, const uint16_t* m_q,
                            int32_t* colour, int* s_off, int* s_cur, int* sm) {
  int* s_tk = sm;  // [2]: taken this round, next round
  int& s_top = sm[2];
  const int tid = threadIdx.x;
  // pair index q = (prio32 - 1) & 0x1FFFF
  uint32_t pr[COLOUR_REG_ITEMS], ab[COLOUR_REG_ITEMS];
  uint32_t col[COLOUR_REG_ITEMS / 4];  // colour of manifold k in byte k % 4
  uint32_t alive = 0;
#pragma unroll
  for (int k = 0; k < COLOUR_REG_ITEMS; ++k) {
    const int m = tid + k * T;
    pr[k] = 0;
    ab[k] = 0;
    if (k % 4 == 0) col[k / 4] = 0;
    if (m < nm) {
      pr[k] = prio32(m_q[m], w);
      ab[k] = m_ab[m];
      alive |= 1u << k;
    }
  }
  if (tid == 0) {
    s_tk[0] = 0;
    s_tk[1] = 0;
  }
  int left = nm, rounds = 0;
  while (left > 0 && rounds < JP_ROUNDS) {
    for (int i = tid; i < nb; i += T) s_best[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < COLOUR_REG_ITEMS; ++k) {
      if (!((alive >> k) & 1u)) continue;
      const uint32_t a = ab[k] & 0xFFFF, b = ab[k] >> 16;
      if (a != NO_BODY) atomicMax(&s_best[a], pr[k]);
      if (b != NO_BODY) atomicMax(&s_best[b], pr[k]);
    }
    __syncthreads();
    // the selected manifolds share no dynamic body: each updates the masks
    // of its own bodies
    int taken = 0;
#pragma unroll
    for (int k = 0; k < COLOUR_REG_ITEMS; ++k) {
      if (!((alive >> k) & 1u)) continue;
      const uint32_t a = ab[k] & 0xFFFF, b = ab[k] >> 16;
      if ((a == NO_BODY || s_best[a] == pr[k]) && (b == NO_BODY || s_best[b] == pr[k])) {
        const uint32_t used = (a != NO_BODY ? s_used[a] : 0u) | (b != NO_BODY ? s_used[b] : 0u);
        const int l = greedy_colour(used, rounds);
        col[k / 4] |= (uint32_t)l << (8 * (k % 4));
        if (l < GREEDY_COLOURS) {
          if (a != NO_BODY) s_used[a] = (uint16_t)(s_used[a] | (1u << l));
          if (b != NO_BODY) s_used[b] = (uint16_t)(s_used[b] | (1u << l));
        }
        alive &= ~(1u << k);
        ++taken;
      }
    }
    taken = wave_sum(taken);
    if ((tid & 63) == 0) atomicAdd(&s_tk[rounds & 1], taken);
    // every lane read last round's count before this round's first barrier
    if (tid == 0) s_tk[(rounds + 1) & 1] = 0;
    __syncthreads();
    left -= s_tk[rounds & 1];
    ++rounds;
  }
  auto colour_at = [&](int k) { return (int)((col[k / 4] >> (8 * (k % 4))) & 0xFFu); };
  {  // the colour count: the highest colour of a coloured manifold, plus one
    int top = 0;
#pragma unroll
    for (int k = 0; k < COLOUR_REG_ITEMS; ++k)
      if (tid + k * T < nm && !((alive >> k) & 1u)) top = max(top, colour_at(k) + 1);
    top = wave_max(top);
    if ((tid & 63) == 0) atomicMax(&s_top, top);
    __syncthreads();
  }
  const int ncol = s_top;
  if (left > 0) {
    // serial tail: colours per pair, the tail (colour ncol) for the rest
#pragma unroll
    for (int k = 0; k < COLOUR_REG_ITEMS; ++k)
      if (tid + k * T < nm) colour[(pr[k] - 1u) & 0x1FFFFu] = (alive >> k) & 1u ? ncol : colour_at(k);
    __syncthreads();
    return false;
  }
  // per-colour counts -> offsets, then each manifold's slot in its colour
  // (LDS atomics; the order inside a colour is free, since its manifolds
  // share no dynamic body)
  for (int i = tid; i <= ncol + 1; i += T) s_cur[i] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < COLOUR_REG_ITEMS; ++k)
    if (tid + k * T < nm) atomicAdd(&s_cur[colour_at(k)], 1);
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int l = 0; l <= ncol; ++l) {
      const int h = s_cur[l];
      s_off[l] = acc;
      s_cur[l] = acc;
      acc += h;
    }
    s_off[ncol + 1] = acc;
    atomicMax(&c.counters[CNT_LEVELS], ncol);
    c.col_info[w] = ncol;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < COLOUR_REG_ITEMS; ++k)
    if (tid + k * T < nm) {
      const int m = atomicAdd(&s_cur[colour_at(k)], 1);
      c.sched_order[p0 + ((pr[k] - 1u) & 0x1FFFFu)] = p0 + m;
    }
  int* off = c.col_off + (long)w * (COLOR_CAP + 3);
  for (int l = tid; l <= ncol; l += T) off[l] = s_off[l];
  return true;
}

// Jones-Plassmann colouring of world w's manifolds in LDS.  The world's
// manifolds are first gathered into a list (any order: the colours depend
// only on the priorities).  LDS pool: s_best (4 B/body), s_used (2 B/body),
// per manifold its local bodies (4 B), pair index (2 B) and colour (1 B:
// 0xFF uncoloured), room for `cap` manifolds.  Colours go to sched_level per
// pair (-2 for pairs without contacts).
template <int T>
__device__ __forceinline__ void colour_world_lds(const Ctx& c, int w, int p0, int np, int b0, int nb,
                                 int cap, unsigned char* pool, int* s_off, int* s_cur, int* sm) {
  int &s_left = sm[0], &s_taken = sm[1], &s_top = sm[2], &s_fill = sm[3];
  const int tid = threadIdx.x;
  uint32_t* s_best = (uint32_t*)pool;
  uint16_t* s_used = (uint16_t*)(s_best + nb);                  // nb: colours taken at the body
  uint32_t* m_ab = (uint32_t*)(s_used + ((nb + 1) & ~1));       // cap: local a | local b << 16
  uint16_t* m_q = (uint16_t*)(m_ab + cap);                      // cap: pair index
  uint8_t* m_col = (uint8_t*)(m_q + cap);                       // cap
  int32_t* colour = c.sched_level + p0;                         // per pair
  if (tid == 0) {
    s_top = 0;
    s_fill = 0;
  }
  for (int i = tid; i < nb; i += T) s_used[i] = 0;
  __syncthreads();
  // the manifold list: four pairs per lane in flight, one atomic per
  // wavefront per batch
  constexpr int LB = 4;
  const unsigned long long below = (1ull << (tid & 63)) - 1ull;
  for (int q0 = 0; q0 < np; q0 += LB * T) {
    uint32_t abv[LB];
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      const int q = q0 + u * T + tid;
      abv[u] = q < np ? c.pair_ab[p0 + q] : NO_PAIR;
    }
    unsigned long long bal[LB];
    int tot = 0;
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      bal[u] = __ballot(abv[u] != NO_PAIR);
      tot += (int)__popcll(bal[u]);
    }
    int base = 0;
    if ((tid & 63) == 0 && tot) base = atomicAdd(&s_fill, tot);
    base = __shfl(base, 0);
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      const int q = q0 + u * T + tid;
      if (abv[u] != NO_PAIR) {
        const int m = base + (int)__popcll(bal[u] & below);
        m_ab[m] = abv[u];
        m_q[m] = (uint16_t)q;
        m_col[m] = 0xFFu;
      } else if (q < np) {
        colour[q] = -2;
        c.sched_order[p0 + q] = -1;
      }
      base += (int)__popcll(bal[u]);
    }
  }
  __syncthreads();
  const int nm = s_fill;
  if (tid == 0) s_left = nm;
  __syncthreads();
  if constexpr (T >= 1024) {
    if (nm <= COLOUR_REG_ITEMS * T) {
      if (!colour_regs<T>(c, w, p0, nm, nb, s_best, s_used, m_ab, m_q, colour, s_off, s_cur,
                          sm))
        colour_finish<T>(c, w, p0, np, colour, s_top, true, s_off, s_cur);
      return;
    }
  }
  int rounds = 0;
  while (s_left > 0 && rounds < JP_ROUNDS) {
    for (int i = tid; i < nb; i += T) s_best[i] = 0;
    if (tid == 0) s_taken = 0;
    __syncthreads();
    for (int m = tid; m < nm; m += T) {
      if (m_col[m] != 0xFFu) continue;
      const uint32_t prio = prio32(m_q[m], w);
      const uint32_t ab = m_ab[m], a = ab & 0xFFFF, b = ab >> 16;
      if (a != NO_BODY) atomicMax(&s_best[a], prio);
      if (b != NO_BODY) atomicMax(&s_best[b], prio);
    }
    __syncthreads();
    // the selected manifolds share no dynamic body: each updates the masks
    // of its own bodies
    int taken = 0, top = 0;
    for (int m = tid; m < nm; m += T) {
      if (m_col[m] != 0xFFu) continue;
      const uint32_t prio = prio32(m_q[m], w);
      const uint32_t ab = m_ab[m], a = ab & 0xFFFF, b = ab >> 16;
      if ((a == NO_BODY || s_best[a] == prio) && (b == NO_BODY || s_best[b] == prio)) {
        const uint32_t used = (a != NO_BODY ? s_used[a] : 0u) | (b != NO_BODY ? s_used[b] : 0u);
        const int l = greedy_colour(used, rounds);
        m_col[m] = (uint8_t)l;
        if (l < GREEDY_COLOURS) {
          if (a != NO_BODY) s_used[a] = (uint16_t)(s_used[a] | (1u << l));
          if (b != NO_BODY) s_used[b] = (uint16_t)(s_used[b] | (1u << l));
        }
        top = max(top, l + 1);
        ++taken;
      }
    }
    taken = wave_sum(taken);
    top = wave_max(top);
    if ((tid & 63) == 0) {
      atomicAdd(&s_taken, taken);
      atomicMax(&s_top, top);
    }
    __syncthreads();
    if (tid == 0) s_left -= s_taken;
    ++rounds;
    __syncthreads();
  }
  const bool serial_tail = s_left > 0;
  const int top = s_top;
  for (int m = tid; m < nm; m += T) colour[m_q[m]] = m_col[m] == 0xFFu ? top : (int)m_col[m];
  __syncthreads();
  colour_finish<T>(c, w, p0, np, colour, top, serial_tail, s_off, s_cur);
}

// The same colouring for worlds whose colouring does not fit in LDS:
// 64-bit priorities and colour masks per body (col_bu) and colours per
// pair (sched_level) in global memory (L2-resident).  The uncoloured
// manifolds of a round are kept as a list of (pair index, body word)
// entries (col_list, two buffers of the world's pair range), so a round
// reads no pair or body arrays beside it: a round visits only them, clears
// only their bodies' priorities, and passes the manifolds it does not
// colour on to the next round's list.  The selection of a round depends
// only on which manifolds are uncoloured and on their priorities, so the
// colours are those of a round over every pair.
template <int T>
__device__ __forceinline__ void colour_world_global(const Ctx& c, int w, int p0, int np, int b0, int nb,
                                    int* s_off, int* s_cur, int* sm) {
  int &s_left = sm[0], &s_taken = sm[1], &s_top = sm[2], &s_fill = sm[3];
  const int tid = threadIdx.x;
  // per body: the round's largest priority (x) and the colours taken (y),
  // one 16-byte word, so a body's test reads one cache line
  ulonglong2* bu = c.col_bu + b0;
  int32_t* colour = c.sched_level + p0;  // per pair: colour, -1 uncoloured, -2 none
  // list entries: the pair index and its pair_ab word (world-local bodies)
  uint2* list[2] = {c.col_list + p0, c.col_list + c.pair_cap + p0};
  const unsigned long long below = (1ull << (tid & 63)) - 1ull;
  if (tid == 0) {
    s_top = 0;
    s_fill = 0;
  }
  for (int i = tid; i < nb; i += T) bu[i].y = 0ull;
  __syncthreads();
  // the first list: every pair with contacts
  for (int q0 = 0; q0 < np; q0 += T) {
    const int q = q0 + tid;
    const uint32_t ab = q < np ? c.pair_ab[p0 + q] : NO_PAIR;
    const bool has = ab != NO_PAIR;
    if (q < np) colour[q] = has ? -1 : -2;
    const unsigned long long bal = __ballot(has);
    int base = 0;
    if ((tid & 63) == 0 && bal) base = atomicAdd(&s_fill, (int)__popcll(bal));
    base = __shfl(base, 0);
    if (has) list[0][base + (int)__popcll(bal & below)] = make_uint2((uint32_t)q, ab);
  }
  __syncthreads();
  if (tid == 0) s_left = s_fill;
  __syncthreads();
  int rounds = 0, cur = 0;
  while (s_left > 0 && rounds < JP_ROUNDS) {
    const int n = s_left;
    const uint2* in = list[cur];
    uint2* out = list[cur ^ 1];
    for (int k = tid; k < n; k += T) {
      const uint32_t ab = in[k].y, a = ab & 0xFFFFu, b = ab >> 16;
      if (a != NO_BODY) bu[a].x = 0ull;
      if (b != NO_BODY) bu[b].x = 0ull;
    }
    if (tid == 0) {
      s_taken = 0;
      s_fill = 0;
    }
    __syncthreads();
    for (int k = tid; k < n; k += T) {
      const uint2 e = in[k];
      const unsigned long long prio = prio64((int)e.x, w);
      const uint32_t a = e.y & 0xFFFFu, b = e.y >> 16;
      if (a != NO_BODY) atomicMax(&bu[a].x, prio);
      if (b != NO_BODY) atomicMax(&bu[b].x, prio);
    }
    __syncthreads();
    int taken = 0, top = 0;
    for (int k0 = 0; k0 < n; k0 += T) {
      const int k = k0 + tid;
      bool keep = false;
      uint2 e = make_uint2(0u, 0u);
      if (k < n) {
        e = in[k];
        const unsigned long long prio = prio64((int)e.x, w);
        const uint32_t a = e.y & 0xFFFFu, b = e.y >> 16;
        const bool sa = a == NO_BODY, sb = b == NO_BODY;
        const ulonglong2 ra = sa ? make_ulonglong2(0ull, 0ull) : bu[a];
        const ulonglong2 rb = sb ? make_ulonglong2(0ull, 0ull) : bu[b];
        if ((sa || ra.x == prio) && (sb || rb.x == prio)) {
          const uint32_t used = (uint32_t)ra.y | (uint32_t)rb.y;
          const int l = greedy_colour(used, rounds);
          colour[e.x] = l;
          if (l < GREEDY_COLOURS) {
            if (!sa) bu[a].y = ra.y | (1ull << l);
            if (!sb) bu[b].y = rb.y | (1ull << l);
          }
          top = max(top, l + 1);
          ++taken;
        } else {
          keep = true;
        }
      }
      const unsigned long long bal = __ballot(keep);
      int base = 0;
      if ((tid & 63) == 0 && bal) base = atomicAdd(&s_fill, (int)__popcll(bal));
      base = __shfl(base, 0);
      if (keep) out[base + (int)__popcll(bal & below)] = e;
    }
    taken = wave_sum(taken);
    top = wave_max(top);
    if ((tid & 63) == 0) {
      atomicAdd(&s_taken, taken);
      atomicMax(&s_top, top);
    }
    __syncthreads();
    if (tid == 0) s_left = s_fill;
    cur ^= 1;
    ++rounds;
    __syncthreads();
  }
  const bool serial_tail = s_left > 0;
  const int top = s_top;
  // the manifolds the rounds did not reach form the serial tail colour
  for (int k = tid; k < s_left; k += T) colour[list[cur][k].x] = top;
  __syncthreads();
  colour_finish<T>(c, w, p0, np, colour, top, serial_tail, s_off, s_cur);
}

// The same colouring with the per-body priorities (prio32) in LDS, the
// colour masks in LDS (MASKS_LDS) or in col_bu, and the uncoloured
// manifolds' lists in global memory (as in colour_world_global): for
// worlds whose bodies fit LDS but whose manifolds do not.  A mask is read
// and written only by the manifold a round selects on the body.
template <int T, bool MASKS_LDS>
__device__ __forceinline__ void colour_world_hybrid(const Ctx& c, int w, int p0, int np, int b0, int nb,
                                    unsigned char* pool, int* s_off, int* s_cur, int* sm) {
  int &s_left = sm[0], &s_taken = sm[1], &s_top = sm[2], &s_fill = sm[3];
  const int tid = threadIdx.x;
  uint32_t* s_best = (uint32_t*)pool;
  uint16_t* s_used = (uint16_t*)(s_best + nb);  // MASKS_LDS
  unsigned long long* g_used = &c.col_bu[b0].y;  // else: body i's mask at g_used[2 i]
  auto used_of = [&](uint32_t i) -> uint32_t {
    return MASKS_LDS ? (uint32_t)s_used[i] : (uint32_t)g_used[2 * i];
  };
  auto set_used = [&](uint32_t i, uint32_t m) {
    if (MASKS_LDS)
      s_used[i] = (uint16_t)m;
    else
      g_used[2 * i] = m;
  };
  int32_t* colour = c.sched_level + p0;  // per pair: colour, -1 uncoloured, -2 none
  uint2* list[2] = {c.col_list + p0, c.col_list + c.pair_cap + p0};
  const unsigned long long below = (1ull << (tid & 63)) - 1ull;
  if (tid == 0) {
    s_top = 0;
    s_fill = 0;
  }
  for (int i = tid; i < nb; i += T) set_used(i, 0u);
  __syncthreads();
  for (int q0 = 0; q0 < np; q0 += T) {
    const int q = q0 + tid;
    const uint32_t ab = q < np ? c.pair_ab[p0 + q] : NO_PAIR;
    const bool has = ab != NO_PAIR;
    if (q < np) colour[q] = has ? -1 : -2;
    const unsigned long long bal = __ballot(has);
    int base = 0;
    if ((tid & 63) == 0 && bal) base = atomicAdd(&s_fill, (int)__popcll(bal));
    base = __shfl(base, 0);
    if (has) list[0][base + (int)__popcll(bal & below)] = make_uint2((uint32_t)q, ab);
  }
  __syncthreads();
  if (tid == 0) s_left = s_fill;
  __syncthreads();
  int rounds = 0, cur = 0;
  while (s_left > 0 && rounds < JP_ROUNDS) {
    const int n = s_left;
    const uint2* in = list[cur];
    uint2* out = list[cur ^ 1];
    for (int k = tid; k < n; k += T) {
      const uint32_t ab = in[k].y, a = ab & 0xFFFFu, b = ab >> 16;
      if (a != NO_BODY) s_best[a] = 0u;
      if (b != NO_BODY) s_best[b] = 0u;
    }
    if (tid == 0) {
      s_taken = 0;
      s_fill = 0;
    }
    __syncthreads();
    for (int k = tid; k < n; k += T) {
      const uint2 e = in[k];
      const uint32_t prio = prio32((int)e.x, w);
      const uint32_t a = e.y & 0xFFFFu, b = e.y >> 16;
      if (a != NO_BODY) atomicMax(&s_best[a], prio);
      if (b != NO_BODY) atomicMax(&s_best[b], prio);
    }
    __syncthreads();
    int taken = 0, top = 0;
    for (int k0 = 0; k0 < n; k0 += T) {
      const int k = k0 + tid;
      bool keep = false;
      uint2 e = make_uint2(0u, 0u);
      if (k < n) {
        e = in[k];
        const uint32_t prio = prio32((int)e.x, w);
        const uint32_t a = e.y & 0xFFFFu, b = e.y >> 16;
        const bool sa = a == NO_BODY, sb = b == NO_BODY;
        if ((sa || s_best[a] == prio) && (sb || s_best[b] == prio)) {
          const uint32_t ua = sa ? 0u : used_of(a), ub = sb ? 0u : used_of(b);
          const int l = greedy_colour(ua | ub, rounds);
          colour[e.x] = l;
          if (l < GREEDY_COLOURS) {
            if (!sa) set_used(a, ua | (1u << l));
            if (!sb) set_used(b, ub | (1u << l));
          }
          top = max(top, l + 1);
          ++taken;
        } else {
          keep = true;
        }
      }
      const unsigned long long bal = __ballot(keep);
      int base = 0;
      if ((tid & 63) == 0 && bal) base = atomicAdd(&s_fill, (int)__popcll(bal));
      base = __shfl(base, 0);
      if (keep) out[base + (int)__popcll(bal & below)] = e;
    }
    taken = wave_sum(taken);
    top = wave_max(top);
    if ((tid & 63) == 0) {
      atomicAdd(&s_taken, taken);
      atomicMax(&s_top, top);
    }
    __syncthreads();
    if (tid == 0) s_left = s_fill;
    cur ^= 1;
    ++rounds;
    __syncthreads();
  }
  const bool serial_tail = s_left > 0;
  const int top = s_top;
  for (int k = tid; k < s_left; k += T) colour[list[cur][k].x] = top;
  __syncthreads();
  colour_finish<T>(c, w, p0, np, colour, top, serial_tail, s_off, s_cur);
}

// The LDS accesses of a wavefront before this point are done before any of
// its accesses after it (the wavefront's lanes run together).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Small worlds (world_order[first_world, W), at most SWEEP_WAVE_MAX_BODIES
// bodies, FP32 velocities in the world's slice of LDS), SWEEP_WAVES of them to
// a workgroup: the warm pass and the sweeps of sweep_prefetched, colour by
// colour, by one wavefront with its own ordering of its LDS accesses between
// colours, or, above SWEEP_ONE_WAVE_BODIES bodies, by PARTS wavefronts that
// meet at a counter in LDS (PARTS = 1: no world of the launch is that large).
// The same updates in the same colour order as sweep_world, so the same
// results.  2048 worlds of 8 to 1024 bodies: 184 us, 254 with one wavefront for
// each, the largest world's time; the rest is the records, read again in each
// of 7 passes (0.6 GB).  Two wavefronts for the larger worlds take 187; the
// line at 128 or 256 bodies makes no difference there.  Without larger worlds
// the other wavefronts would only hold places on the CUs: 4096 worlds of 64
// bodies 95 us with PARTS = 1, 210 with 4.
template <int PARTS>
__global__ __launch_bounds__(64 * SWEEP_WAVES * PARTS) void k_sweep_waves(Ctx c, int first_world,
                                                                         int slice_floats) {
  extern __shared__ __align__(16) int lds[];
  __shared__ int s_met[SWEEP_WAVES];
  if (threadIdx.x < SWEEP_WAVES) s_met[threadIdx.x] = 0;
  __syncthreads();
  const int wave = threadIdx.x >> 6, slot = wave % SWEEP_WAVES, part = wave / SWEEP_WAVES;
  const int k = first_world + (int)blockIdx.x * SWEEP_WAVES + slot;
  if (k >= c.W) return;  // this wavefront only: no workgroup barrier follows
  const int w = c.world_order[k];
  const int info = c.col_info[w];
  const int ncol = info & 0xFFFF;
  if (ncol == 0) return;
  const bool serial_tail = info & COL_TAIL;
  const int p0 = c.wpair_off[w];
  const int b0 = c.body_off[w], nb = c.body_off[w + 1] - b0;
  const int parts = nb > SWEEP_ONE_WAVE_BODIES ? PARTS : 1;
  if (part >= parts) return;
  const int lane = 64 * part + (int)(threadIdx.x & 63), lanes = 64 * parts;
  const int* off = c.col_off + (long)w * (COLOR_CAP + 3);
  VelF<true> V;
  V.lds = (float*)lds + slot * slice_floats;
  V.c = &c;
  V.b0 = b0;
  int meet = 0;
  auto sync = [&] {
    if (parts == 1) {
      wave_sync();
      return;
    }
    // every wavefront of the world runs (they are one workgroup's) and comes
    // here as often
    meet += PARTS;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    if ((threadIdx.x & 63) == 0)
      __hip_atomic_fetch_add(&s_met[slot], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (__hip_atomic_load(&s_met[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < meet)
      __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  for (int i = lane; i < nb; i += lanes) {
    const int g = b0 + i;
    const float v[3] = {(float)c.vx[g], (float)c.vy[g], (float)c.w[g]};
    V.store(g, v);
  }
  sync();
  const PackF P = packf(c);
  sweep_prefetched(c, recw(c, P, p0), ncol, serial_tail, off, lane, lanes, V, sync);
  for (int i = lane; i < nb; i += lanes) {
    float v[3];
    V.load(b0 + i, v);
    c.fv[b0 + i] = make_float4(v[0], v[1], v[2], 0.0f);
  }
}

// Colouring of world w by one workgroup: in LDS when the world's colouring
// fits (by its pair count, else by its manifold count), else with the bodies
// in LDS and the manifold lists in global memory when the bodies fit, else in
// global memory.
template <int T>
__device__ __forceinline__ void colour_world(const Ctx& c, int w, int p0, int np, int pool_bytes,
                                             int* lds, int* sm) {
  int* s_off = lds;                      // COLOR_CAP + 3
  int* s_cur = lds + (COLOR_CAP + 3);    // COLOR_CAP + 3
  unsigned char* pool = (unsigned char*)(lds + 2 * (COLOR_CAP + 3) + 2);
  const int b0 = c.body_off[w], nb = c.body_off[w + 1] - b0;
  // room for every pair as a manifold, or else for the manifolds counted
  int cap = np;
  bool in_lds = colour_fits_lds(nb, np, np, pool_bytes);
  if (!in_lds) {
    cap = count_manifolds<T>(c, p0, np, &sm[0]);
    in_lds = colour_fits_lds(nb, np, cap, pool_bytes);
  }
  if (in_lds)
    colour_world_lds<T>(c, w, p0, np, b0, nb, cap, pool, s_off, s_cur, sm);
  else if (colour_fits_hybrid(nb, np, pool_bytes) && colour_masks_fit(nb, pool_bytes))
    colour_world_hybrid<T, true>(c, w, p0, np, b0, nb, pool, s_off, s_cur, sm);
  else if (colour_fits_hybrid(nb, np, pool_bytes))
    colour_world_hybrid<T, false>(c, w, p0, np, b0, nb, pool, s_off, s_cur, sm);
  else
    colour_world_global<T>(c, w, p0, np, b0, nb, s_off, s_cur, sm);
}

// ---- one world on several CUs ----------------------------------------------

// The rounds' colouring of a world without rounds, by several workgroups of T
// lanes with FLOW_ITEMS / T pairs each.  In the rounds a manifold is coloured
// once every manifold of higher priority on its bodies is; here it waits for
// just those.  The lists k_sat made give each manifold its rank by priority
// among its body's; a body's word (colours used | manifolds coloured << 32 |
// round << 48) says whose turn it is and holds all that the colour depends
// on: the next manifold of both its bodies takes the same colour as in the
// rounds, and its round is one past the latest on its bodies.  A lane keeps
// its manifolds in registers and looks at all that are left in turn, so the
// time is that of the longest chain of priorities (about 20 hand-overs)
// instead of 3 barriers and a scan of the lists for each of the rounds, on
// one CU: one pile of 32768 polygons 40 us (about 20 of them joining, ranking
// and the places in the colours), 496 before; of 8192 30, 113 before.
//
// The world's last workgroup writes col_off, col_info and flow_cnt when all of
// its colours are there; sched_level then holds each pair's colour and its place
// among those of its workgroup, from which the packing pass makes its slot in
// sched_order.  (Not written here: the workgroup that colours the world alone
// after all writes sched_order, and what another XCD's L2 still holds of an
// array could come after it.)  A world with a body of more than FLOW_DEGREE
// manifolds, more pairs than the lanes hold, or colours past FLOW_DEGREE is left
// to one workgroup: *last tells the one that has to colour it.
constexpr int FLOW_ITEMS = 8192, FLOW_COLOUR_LANES = 256;

__device__ __forceinline__ void colour_flow(const Ctx& c, int w, int p0, int np, int seat, int groups,
                                            int rows, int* lds, bool* last) {
  constexpr int AGENT = __HIP_MEMORY_SCOPE_AGENT, T = FLOW_COLOUR_LANES;
  int* s_cnt = lds;                 // FLOW_DEGREE
  int* s_last = lds + FLOW_DEGREE;
  // per pair its bodies, rank on a | rank on b << 8, and its colour; the first
  // T lanes wait for them, tid + k T each
  uint32_t* s_ab = (uint32_t*)(lds + 2 * FLOW_DEGREE);
  uint16_t* s_rank = (uint16_t*)(s_ab + FLOW_ITEMS);
  uint8_t* s_col = (uint8_t*)(s_rank + FLOW_ITEMS);
  int* ctl = c.flow_ctl + (long)w * FLOW_CTL;
  const int tid = threadIdx.x, f0 = c.body_off[w] + c.flow_shift[w];
  const int per = ((np + groups - 1) / groups + 63) & ~63;
  const int q0 = seat * per, n = min(per, np - q0);
  // The same for all wavefronts, whose barriers depend on it: FC_FULL is k_sat's
  // and stays as it is during this kernel, while FC_BAD is set by any workgroup
  // of the world at any time.
  const bool fits = per <= FLOW_ITEMS && ctl[FC_FULL] == 0;
  if (tid < FLOW_DEGREE) s_cnt[tid] = 0;
  if (fits) {
    auto key = [&](uint32_t q) {  // orders like prio64
      return (unsigned long long)(mix32(q * 0x9E3779B9u + (uint32_t)w) & 0x7FFFu) << 32 | q;
    };
    const int lanes = (int)blockDim.x;
    for (int i = tid; i < n; i += lanes) {
      const uint32_t ab = c.pair_ab[p0 + q0 + i];
      s_ab[i] = ab;
      s_col[i] = 0xFFu;
      if (ab == NO_PAIR) continue;
      const unsigned long long mine = key((uint32_t)(q0 + i));
      int r[2], m[2];
      const int4* row[2];
      int4 e[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint32_t loc = s ? ab >> 16 : ab & 0xFFFFu;
        const int g = f0 + (loc == NO_BODY ? 0 : (int)loc);
        row[s] = (const int4*)(c.adj + (long)g * FLOW_DEGREE);
        m[s] = loc == NO_BODY ? 0 : c.adj_n[g];
        e[s][0] = row[s][0];
        e[s][1] = row[s][1];
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        r[s] = 0;
        auto count = [&](int4 x, int at) {
          const int y[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (at + j < m[s] && key((uint32_t)(y[j] - p0)) > mine) ++r[s];
        };
        count(e[s][0], 0);
        if (m[s] > 4) count(e[s][1], 4);
        for (int at = 8; at < m[s]; at += 4) count(row[s][at / 4], at);
      }
      s_rank[i] = (uint16_t)(r[0] | r[1] << 8);
    }
    __syncthreads();
    uint32_t alive = 0;
    static_assert(FLOW_ITEMS / T <= 32, "a lane's pairs are bits of a word");
    if (tid < T)
      for (int i = tid, k = 0; i < n; i += T, ++k) alive |= (s_ab[i] != NO_PAIR ? 1u : 0u) << k;
    bool bad = false;
    for (int polls = 1; alive; ++polls) {
      // the lane's next manifolds, two at a time
      for (uint32_t rest = alive; rest;) {
        int k[2];
        uint32_t ab[2], rank[2];
        unsigned long long wa[2], wb[2];
        k[0] = __builtin_ctz(rest);
        rest &= rest - 1;
        k[1] = rest ? __builtin_ctz(rest) : k[0];
        rest &= rest - 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int i = tid + k[j] * T;
          ab[j] = s_ab[i];
          rank[j] = s_rank[i];
          const uint32_t a = ab[j] & 0xFFFFu, b = ab[j] >> 16;
          wa[j] = a != NO_BODY ? peek(c.flow_col + FLOW_LINE * (long)(f0 + a)) : 0ull;
          wb[j] = b != NO_BODY ? peek(c.flow_col + FLOW_LINE * (long)(f0 + b)) : 0ull;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (j == 1 && k[1] == k[0]) continue;
          if (((uint32_t)(wa[j] >> 32) & 0xFFFFu) != (rank[j] & 0xFFu) ||
              ((uint32_t)(wb[j] >> 32) & 0xFFFFu) != rank[j] >> 8)
            continue;
          const int round = max((int)(wa[j] >> 48), (int)(wb[j] >> 48));
          const int l = greedy_colour((uint32_t)(wa[j] | wb[j]) & 0xFFFFu, round);
          const bool ok = l < FLOW_DEGREE && round < JP_ROUNDS;
          bad |= !ok;
          s_col[tid + k[j] * T] = (uint8_t)(ok ? l : 0);
          alive &= ~(1u << k[j]);
          const unsigned long long up = (unsigned long long)min(round + 1, JP_ROUNDS) << 48;
          auto hand_on = [&](uint32_t loc, unsigned long long x) {
            if (loc == NO_BODY) return;
            poke(c.flow_col + FLOW_LINE * (long)(f0 + loc),
                 up | ((((x >> 32) & 0xFFFFull) + 1ull) << 32) | (uint32_t)(x | (ok ? 1ull << l : 0ull)));
          };
          hand_on(ab[j] & 0xFFFFu, wa[j]);
          hand_on(ab[j] >> 16, wb[j]);
        }
      }
      if (polls % 64 == 0) {
        if (polls >= c.flow_polls) {
          atomicOr(&c.counters[CNT_FLAGS], SHP_FLAG_STALL);
          bad = true;
        }
        if (bad || peek(ctl + FC_BAD) != 0) break;
      }
    }
    if (bad) poke(ctl + FC_BAD, 1);
    __syncthreads();
    // places within the colours: consecutive for a wavefront's pairs of a
    // colour, so that the sweeps' lanes stay near each other
    for (int i0 = 0; i0 < n; i0 += lanes) {
      const int i = i0 + tid;
      const int at = wave_count(s_cnt, i < n && s_col[i] != 0xFFu ? (int)s_col[i] : -1);
      if (i < n) s_ab[i] = (uint32_t)at;
    }
    __syncthreads();
    if (tid < FLOW_DEGREE) poke(c.flow_cnt + (rows + seat) * FLOW_DEGREE + tid, s_cnt[tid]);
    for (int i = tid; i < n; i += lanes) {
      const int l = s_col[i];
      c.sched_level[p0 + q0 + i] = l == 0xFF ? -1 : (int)s_ab[i] << 5 | l;
    }
  }
  // the last workgroup (the others' counts and flags are in: their stores were
  // complete before their additions)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0)
    *s_last = __hip_atomic_fetch_add(ctl + FC_DONE, 1, __ATOMIC_RELAXED, AGENT) == groups - 1
                  ? 1 + (fits && peek(ctl + FC_BAD) == 0)
                  : 0;
  __syncthreads();
  const int what = *s_last;
  __syncthreads();
  *last = what == 1;
  if (what != 2) return;
  // the colours' offsets, and within each those of the workgroups' manifolds,
  // in the order of the seats: FLOW_DEGREE columns, a run of seats to a lane
  const int l = tid % FLOW_DEGREE, runs = (int)blockDim.x / FLOW_DEGREE, run = tid / FLOW_DEGREE;
  const int len = (groups + runs - 1) / runs, s0 = min(run * len, groups), s1 = min(s0 + len, groups);
  int* s_run = (int*)s_ab;  // runs x FLOW_DEGREE
  int32_t* cnt = c.flow_cnt + rows * FLOW_DEGREE + l;
  int sum = 0;
  for (int s = s0; s < s1; ++s) sum += peek(cnt + s * FLOW_DEGREE);
  s_run[tid] = sum;
  __syncthreads();
  int before = 0, all = 0;
  for (int r = 0; r < runs; ++r) {
    const int x = s_run[r * FLOW_DEGREE + l];
    before += r < run ? x : 0;
    all += x;
  }
  for (int s = s0; s < s1; ++s) {
    const int x = peek(cnt + s * FLOW_DEGREE);
    cnt[s * FLOW_DEGREE] = before;
    before += x;
  }
  if (tid >= 64) return;
  const int have = tid < FLOW_DEGREE ? all : 0;
  int upto = have;
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(upto, o);
    if (tid >= o) upto += x;
  }
  const unsigned long long used = __ballot(have > 0);
  const int ncol = used ? 64 - __builtin_clzll(used) : 0;
  int* off = c.col_off + (long)w * (COLOR_CAP + 3);
  if (tid <= ncol) off[tid] = upto - have;
  if (tid == 0) {
    ctl[FC_ROWS] = rows;
    ctl[FC_SHARE] = per;
    c.col_info[w] = ncol | COL_FLOW;  // also without a manifold: sched_level says so
    atomicMax(&c.counters[CNT_LEVELS], ncol);
    tmark(c, w, 1);
  }
}

// Colouring: the flow worlds' workgroups, then one per world, the largest
// worlds first.
template <int T>
__global__ __launch_bounds__(T) void k_colour(Ctx c, int pool_bytes) {
  extern __shared__ __align__(16) int lds[];
  __shared__ int sm[4];
  const int flow_blocks = c.flow_worlds * c.flow_groups, blk = blockIdx.x;
  const bool flow = blk < flow_blocks;
  const int w = c.world_order[flow ? blk / c.flow_groups : blk - flow_blocks + c.flow_worlds];
  // the world's pairs (k_contacts writes the same offsets beside this kernel)
  const int b0 = c.body_off[w], b1 = c.body_off[w + 1];
  const int p0 = min(c.off_rank[b0], c.pair_cap), p1 = min(c.off_rank[b1], c.pair_cap);
  const int np = p1 - p0;
  if (np == 0) {  // nothing to solve
    if (threadIdx.x == 0) c.col_info[w] = 0;
    return;
  }
  if (blk == 0) tmark(c, w, 0);
  if (flow) {
    int* ctl = c.flow_ctl + (long)w * FLOW_CTL;
    const int want = flow_want(c, w, c.flow_groups);
    if (blk % c.flow_groups >= want) return;
    int groups;
    const int seat = flow_join(c, ctl + FC_SEATS, ctl + FC_GROUPS, blk % c.flow_groups, want, sm,
                               &groups);
    if (seat < 0) return;
    bool last;
    colour_flow(c, w, p0, np, seat, groups, blk / c.flow_groups * c.flow_groups, lds, &last);
    if (!last) return;
  }
  colour_world<T>(c, w, p0, np, pool_bytes, lds, sm);
  tmark(c, w, 1);
}

// Every coloured pair's <= 2 contacts become its manifold record, over the
// whole batch at once, when the contact kernel ran beside the colouring.
// Every value is loaded before the first store.
__global__ void k_pack_manifolds(Ctx c) {
  const int tp = c.wpair_off[c.W];
  const PackF P = packf(c);
  if (c.flow_worlds)  // the bodies' first velocity words
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < c.flow_bodies; i += gridDim.x * blockDim.x) {
      const int g = c.flow_body[i];
      const float v[3] = {(float)c.vx[g], (float)c.vy[g], (float)c.w[g]};
      unsigned long long x[2];
      VelFlow::pack(v, 0, x);
      *(ulonglong2*)(c.flow_vel + FLOW_LINE * (long)i) = make_ulonglong2(x[0], x[1]);
    }
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < tp; p += gridDim.x * blockDim.x) {
    int M, turns = 0;
    const int w = c.flow_worlds ? c.body_world[c.pa[p]] : 0;
    if (c.flow_worlds && c.col_info[w] == 0) {  // nothing to solve, or its colouring gave up
      c.sched_order[p] = -1;
      continue;
    }
    if (c.flow_worlds && (c.col_info[w] & COL_FLOW)) {
      const int s = c.sched_level[p], l = s & 31;
      const int* ctl = c.flow_ctl + (long)w * FLOW_CTL;
      const int p0 = c.wpair_off[w], row = ctl[FC_ROWS] + (p - p0) / ctl[FC_SHARE];
      M = s < 0 ? -1
                : p0 + c.col_off[(long)w * (COLOR_CAP + 3) + l] +
                      c.flow_cnt[row * FLOW_DEGREE + l] + (s >> 5);
      c.sched_order[p] = M;
      const int shift = c.flow_shift[w];
      auto turn = [&](int g, int& at, int& of) {
        const uint32_t used = c.is_static[g] ? 0u : (uint32_t)c.flow_col[FLOW_LINE * (long)(g + shift)];
        at = __popc(used & ((1u << l) - 1u));
        of = __popc(used);
      };
      Turns t;
      turn(c.pa[p], t.at_a, t.of_a);
      turn(c.pb[p], t.at_b, t.of_b);
      turns = pack_turns(t);
    } else {
      M = c.sched_order[p];
    }
    if (M < 0) continue;
    const int k0 = c.coff[p];
    if (k0 >= c.contact_cap) {
      write_null_record(P, M, c.pa[p], c.pb[p], turns);
      continue;
    }
    const int cap = c.contact_cap - k0, nk = c.ccount[p] < cap ? c.ccount[p] : cap;
    const int ga = c.ga[k0], gb = c.gb[k0];
    const d2 u = row_normal(c, k0);
    const double ima = c.iml[ga], ira = c.imr[ga], imb = c.iml[gb], irb = c.imr[gb];
    double4 x[2];
    double bn[2], mcn[2], mct[2], ln[2], lt[2];
    int warm = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (j >= nk) break;
      const int k = k0 + j;
      x[j] = c.jx[k];
      bn[j] = c.bn[k];
      mcn[j] = c.mcn[k];
      mct[j] = c.mct[k];
      ln[j] = c.ln[k];
      lt[j] = c.lt[k];
      warm |= (c.warm[k] ? 1 : 0) << j;
    }
    write_record_head(c, P, M, ga, gb, u, ima, imb, nk, warm, turns);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (j >= nk) break;
      write_record_rows(P, M, j, ira, irb, x[j].x, x[j].y, x[j].z, x[j].w, bn[j], mcn[j], mct[j]);
      write_record_lambda(P, M, j, ln[j], lt[j]);
    }
  }
}

// Warm-start pass, sweeps and write-back of world w, with FP32 velocities
// in LDS (VLDS) or in global memory.
template <bool VLDS, int T>
__device__ void sweep_world(const Ctx& c, int w, int ncol, bool serial_tail, float* vlds,
                            int* s_off) {
  const int tid = threadIdx.x;
  const int p0 = c.wpair_off[w];
  const int b0 = c.body_off[w], nb = c.body_off[w + 1] - b0;
  const int* off = c.col_off + (long)w * (COLOR_CAP + 3);
  for (int l = tid; l <= ncol; l += T) s_off[l] = off[l];
  VelF<VLDS> V;
  V.lds = vlds;
  V.c = &c;
  V.b0 = b0;
  // FP32 velocities; a lane has the loads of four bodies in flight
  for (int i0 = tid; i0 < nb; i0 += 4 * T) {
    float x[4][3];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int g = b0 + i0 + u * T;
      if (i0 + u * T < nb) {
        x[u][0] = (float)c.vx[g];
        x[u][1] = (float)c.vy[g];
        x[u][2] = (float)c.w[g];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * T < nb) V.store(b0 + i0 + u * T, x[u]);
  }
  __syncthreads();
  tmark(c, w, 2);
  tmark(c, w, 3);
  const PackF P = packf(c);
  sweep_colours<VLDS, T>(c, recw(c, P, p0), ncol, serial_tail, s_off, V);
  tmark(c, w, 4);
  // (every phase ends with a barrier) the final FP32 velocities to global
  // memory, for k_colour_unpack
  if (VLDS) {
    for (int i = tid; i < nb; i += T) {
      float v[3];
      V.load(b0 + i, v);
      c.fv[b0 + i] = make_float4(v[0], v[1], v[2], 0.0f);
    }
  }
  tmark(c, w, 5);
}

// The sweeps of a world by several workgroups, one wavefront of each, whose
// manifolds wait for their own bodies only (VelFlow).  A wavefront has an even
// share of every colour and takes its manifolds in colour order, so that what
// any of its lanes waits for comes before all that the wavefront has left to
// do.  Its records stay in LDS over the passes (its other wavefronts help to
// bring them in and the lagrangians out), so that between two colours there
// is only the velocities' way from CU to CU.  Few lanes to a CU, on many CUs:
// the scattered velocity words cost a CU's address unit a cycle each.  One
// pile of 32768 polygons, 4 iterations: 67 us (45 colours in turn, 1.4 us
// each: a hand-over, 0.3 us of arithmetic, the slowest of a wavefront's
// lanes), 1121 by one workgroup of 1024 lanes with a barrier after each
// colour; of 8192, 8 iterations: 91 (72 colours), 270 before (velocities in
// LDS).  With 256 lanes to a CU and the records read from L2 in each pass it
// took 172 and 209.
constexpr int FLOW_REC_BYTES = 16 * (REC_WORDS + REC2_WORDS);

// The share of colour `lane` that seat `seat` has: [first, last), the
// manifolds before it in the wavefront's records, and all of them; the most
// that any seat has.
struct FlowShare {
  int first, last, start, all, most;
};

__device__ __forceinline__ FlowShare flow_share(const Ctx& c, int w, int ncol, int seat, int groups) {
  const int lane = threadIdx.x & 63;
  const int* offs = c.col_off + (long)w * (COLOR_CAP + 3) + min(lane, ncol - 1);
  const int o0 = offs[0], o1 = offs[1], share = (o1 - o0 + groups - 1) / groups;
  FlowShare f;
  f.first = min(o0 + seat * share, o1);
  f.last = min(f.first + share, o1);
  const int n = lane < ncol ? f.last - f.first : 0;
  int sum = n;
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(sum, o);
    if (lane >= o) sum += x;
  }
  f.start = sum - n;
  f.all = __shfl(sum, 63);
  f.most = wave_sum(lane < ncol ? share : 0);
  return f;
}

__device__ void sweep_flow(const Ctx& c, int w, int ncol, const FlowShare f, float4* recs) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int step = f.all;  // between a record's words
  const PackF P = packf(c);
  const RecW R = recw(c, P, c.wpair_off[w]);
  for (int l = wave; l < ncol; l += waves) {
    const int i0 = __builtin_amdgcn_readlane(f.first, l), i1 = __builtin_amdgcn_readlane(f.last, l);
    const int s0 = __builtin_amdgcn_readlane(f.start, l) - i0;
    for (int i = i0 + lane; i < i1; i += 64) {
      const float4 *r = rec_of(R.rec, R.p0 + i), *r2 = rec2_of(R.rec2, R.p0 + i);
      float4 x[REC_WORDS + REC2_WORDS];
#pragma unroll
      for (int q = 0; q < REC_WORDS; ++q) x[q] = r[q * RB];
#pragma unroll
      for (int q = 0; q < REC2_WORDS; ++q) x[REC_WORDS + q] = r2[q * RB];
#pragma unroll
      for (int q = 0; q < REC_WORDS + REC2_WORDS; ++q) recs[q * step + s0 + i] = x[q];
    }
  }
  __syncthreads();
  if (wave == 0) {
    const int passes = c.iterations + 1;
    VelFlow V;
    V.c = &c;
    V.vel = c.flow_vel + FLOW_LINE * (long)c.flow_shift[w];
    V.abort = c.flow_ctl + (long)w * FLOW_CTL + FS_ABORT;
    V.dead = false;
    for (int pass = 0; pass < passes; ++pass)
      for (int l = 0; l < ncol; ++l) {
        const int i0 = __builtin_amdgcn_readlane(f.first, l);
        const int n = __builtin_amdgcn_readlane(f.last, l) - i0;
        float4* r0 = recs + __builtin_amdgcn_readlane(f.start, l);
        for (int i = lane; i < n; i += 64) {
          ManF m;
          load_head(r0 + i, step, m);
          load_contact(r0 + i + 3 * step, step, m.k[0]);
          load_contact(r0 + i + REC_WORDS * step, step, m.k[1]);
          V.wait(m, pass);
          solve_man([&](int j) { return (double2*)(r0 + i + (j ? REC_WORDS + 3 : 6) * step); }, m,
                    pass == 0, V);
        }
      }
  }
  __syncthreads();
  for (int l = wave; l < ncol; l += waves) {
    const int i0 = __builtin_amdgcn_readlane(f.first, l), i1 = __builtin_amdgcn_readlane(f.last, l);
    const int s0 = __builtin_amdgcn_readlane(f.start, l) - i0;
    for (int i = i0 + lane; i < i1; i += 64) {
      *(float4*)lambda_of(R, i, 0) = recs[6 * step + s0 + i];
      *(float4*)lambda_of(R, i, 1) = recs[(REC_WORDS + 3) * step + s0 + i];
    }
  }
}

// The flow worlds' workgroups, then one workgroup per world, the largest
// worlds first; velocities in LDS when they fit.
template <int T>
__global__ __launch_bounds__(T) void k_sweep_colours(Ctx c, int pool_bytes) {
  extern __shared__ __align__(16) int lds[];
  __shared__ int s_off[COLOR_CAP + 3];
  const int flow_blocks = c.flow_worlds * c.flow_groups, blk = blockIdx.x;
  const bool flow = blk < flow_blocks;
  const int w = c.world_order[flow ? blk / c.flow_groups : blk - flow_blocks + c.flow_worlds];
  const int info = c.col_info[w];
  const int ncol = info & 0xFFFF;
  if (ncol == 0) return;
  // (a shared world's sweeps are timed from here to the next kernel's start:
  // stamps inside them took 2 us)
  if (blk == 0)
    for (int k = 2; k < 4; ++k) tmark(c, w, k);
  if (flow && (info & COL_FLOW)) {
    int* ctl = c.flow_ctl + (long)w * FLOW_CTL;
    const int want = flow_want(c, w, c.flow_groups);
    if (blk % c.flow_groups >= want) return;
    int groups;
    const int seat = flow_join(c, ctl + FS_SEATS, ctl + FS_GROUPS, blk % c.flow_groups, want, s_off,
                               &groups);
    if (seat < 0) return;
    const FlowShare f = flow_share(c, w, ncol, seat, groups);
    if ((long)f.most * FLOW_REC_BYTES <= pool_bytes) {
      sweep_flow(c, w, ncol, f, (float4*)lds);
      return;
    }
    // records that do not fit in LDS: one workgroup
    if (seat != 0) return;
    if (threadIdx.x == 0) ctl[FS_ALONE] = 1;
  } else if (flow && blk % c.flow_groups != 0) {
    return;
  }
  const bool serial_tail = info & COL_TAIL;
  const int nb = c.body_off[w + 1] - c.body_off[w];
  if (vel_fits_lds(nb, pool_bytes))
    sweep_world<true, T>(c, w, ncol, serial_tail, (float*)lds, s_off);
  else
    sweep_world<false, T>(c, w, ncol, serial_tail, nullptr, s_off);
}

// After the sweeps, over the whole batch: the lagrangians back to contact
// order, and each swept world's FP32 velocity change into the FP64
// velocities (a body whose world had nothing to solve keeps its own).
__global__ void k_colour_unpack(Ctx c) {
  const long tp = c.wpair_off[c.W];
  const long n = tp > c.NB ? tp : (long)c.NB;
  const PackF P = packf(c);
  if (c.tstamp && blockIdx.x == 0 && (c.col_info[c.world_order[0]] & COL_FLOW) &&
      !c.flow_ctl[(long)c.world_order[0] * FLOW_CTL + FS_ALONE])
    for (int k = 4; k < 6; ++k) tmark(c, c.world_order[0], k);
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < n;
       t += (long)gridDim.x * blockDim.x) {
    if (t < tp) {
      const int M = c.sched_order[t];
      if (M >= 0) {
        const int k0 = c.coff[t];
        const int nk = min(c.ccount[t], c.contact_cap - k0);  // contacts that were stored
        for (int j = 0; j < nk; ++j) {
          const double2 l =
              *(const double2*)(j ? rec2_of(P.rec2, M) + 3 * RB : rec_of(P.rec, M) + 6 * RB);
          c.ln[k0 + j] = l.x;
          c.lt[k0 + j] = l.y;
        }
      }
    }
    if (t < c.NB) {
      const int g = (int)t;
      const int info = c.col_info[c.body_world[g]];
      if (!c.is_static[g] && (info & 0xFFFF) != 0) {
        float f[3];
        const int w = c.body_world[g];
        if ((info & COL_FLOW) && !c.flow_ctl[(long)w * FLOW_CTL + FS_ALONE]) {
          const ulonglong2 x = *(const ulonglong2*)(c.flow_vel + FLOW_LINE * (long)(g + c.flow_shift[w]));
          VelFlow::unpack(x.x, x.y, f);
        } else {
          const float4 x = c.fv[g];
          f[0] = x.x;
          f[1] = x.y;
          f[2] = x.z;
        }
        c.vx[g] = c.vx[g] + (double)(f[0] - (float)c.vx[g]);
        c.vy[g] = c.vy[g] + (double)(f[1] - (float)c.vy[g]);
        c.w[g] = c.w[g] + (double)(f[2] - (float)c.w[g]);
      }
    }
  }
}


// LDS of the colouring: colour offsets and cursors, then a pool for the
// per-body priorities and colour masks and the manifold list (pairs per
// world are unknown before a step: budgeted at 8 per body; a world that
// needs more is coloured in global memory); the sweeps use the pool for
// the FP32 velocities.  4 waves per world; a large world gets 8, and its
// colouring 16 (light on registers).
void plan_colored_solver(StepPlan* P, int solver_threads, const std::vector<int32_t>& body_off,
                         const std::vector<int32_t>& order) {
  const long nb = P->max_nb;
  const long np = std::min<long>(32767, 8 * nb + 64);
  const long need = std::max(6 * nb + 2 + 7 * np, 12 * nb);
  const size_t fixed = (2 * (COLOR_CAP + 3) + 2) * 4;
  P->color_lds = std::min<size_t>(fixed + need, LDS_MAX_BYTES);
  P->color_pool = P->color_lds - fixed;
  // 64: worlds of up to SWEEP_WAVE_MAX_BODIES sweep several to a workgroup, one
  // wavefront each or a few, the others (and the colouring) with 256 lanes
  P->color_threads = solver_threads == 64 ? 256
                     : solver_threads     ? solver_threads
                                          : (nb > 2048 ? 512 : 256);
  // A colouring workgroup of 1024 lanes takes a whole CU; with at least as
  // many worlds as CUs the colouring fills the GPU and gains little beside
  // the contact kernel (1024 piles: 6.60 ms for both plus the packing pass,
  // 6.04 ms in turn with the records from the contact kernel), while a few
  // worlds' colouring costs nothing there (one world: the contact kernel's
  // time) and smaller workgroups share CUs with it.
  P->records_in_contacts = P->color_threads >= 512 && P->W >= RECORDS_IN_CONTACTS_MIN_WORLDS;
  // Worlds on several CUs, as many as there are CUs for: us a step, 6
  // iterations, on several CUs against one (1024 lanes): one world of 1024
  // bodies 183 / 181, 2048 193 / 217, 4096 210 / 268, 8192 223 / 364, 16384
  // 265 / 765, 32768 325 / 1690; 8 of 4096 332 / 365, 16 of them 440 / 431,
  // 4 of 8192 326 / 441, 8 429 / 509, 4 of 16384 414 / 889, 2 of 32768
  // 417 / 1761.  (A workgroup's records fill its LDS at about 450 bodies, at
  // 2 manifolds each.)
  int big = 0;
  while (big < P->W && body_off[order[big] + 1] - body_off[order[big]] > FLOW_MIN_BODIES) ++big;
  if (big > 0 && !P->records_in_contacts) {
    const long groups = std::min<long>((nb + FLOW_GROUP_BODIES - 1) / FLOW_GROUP_BODIES,
                                       FLOW_MAX_GROUPS / big);
    if (groups * FLOW_GROUP_MAX >= nb) {
      P->flow_worlds = big;
      P->flow_groups = (int)groups;
      P->color_lds = LDS_MAX_BYTES;
      P->color_pool = P->color_lds - fixed;
    }
  }
}

// k_colour: sm[4]; k_sweep_colours: s_off[COLOR_CAP + 3]
size_t colored_static_lds(bool sweep) { return sweep ? lds16((COLOR_CAP + 3) * 4) : lds16(4 * 4); }

shp_status colored_alloc(shp_batch* b) {
  const StepPlan& P = b->plan;
  const int t = P.color_threads;
  const void* fns[] = {t >= 512 ? (const void*)k_colour<1024> : (const void*)k_colour<256>,
                       t == 1024  ? (const void*)k_sweep_colours<1024>
                       : t == 512 ? (const void*)k_sweep_colours<512>
                                  : (const void*)k_sweep_colours<256>};
  const size_t ldsz[] = {P.color_lds, P.color_pool};
  const void* waves = P.sweep_parts > 1 ? (const void*)k_sweep_waves<SWEEP_PARTS>
                                        : (const void*)k_sweep_waves<1>;
  if (P.g_sweep_waves > 0 &&
      hipFuncSetAttribute(waves, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)std::max<size_t>((size_t)SWEEP_WAVES * P.sweep_slice * 4, 16)) !=
          hipSuccess) {
    shp_set_error("hipFuncSetAttribute (wavefront sweeps LDS) failed");
    return SHP_E_HIP;
  }
  for (int k = 0; k < 2; ++k) {
    if (hipFuncSetAttribute(fns[k], hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsz[k]) !=
        hipSuccess) {
      shp_set_error("hipFuncSetAttribute (coloured solver LDS) failed");
      return SHP_E_HIP;
    }
    hipFuncAttributes a{};
    if (hipFuncGetAttributes(&a, fns[k]) != hipSuccess ||
        a.sharedSizeBytes > colored_static_lds(k == 1)) {
      shp_set_error("coloured solver: static LDS above the plan's");
      return SHP_E_HIP;
    }
  }
  return SHP_OK;
}

void launch_colored_pack(shp_batch* b) {
  k_pack_manifolds<<<b->plan.g_pack, 256, 0, b->stream>>>(b->ctx);
}

void launch_colouring(shp_batch* b, hipStream_t s) {
  const Ctx& c = b->ctx;
  const StepPlan& P = b->plan;
  const int pool = (int)P.color_pool;
  const unsigned grid = (unsigned)(c.W + c.flow_worlds * (c.flow_groups - 1));
  if (P.color_threads >= 512)
    k_colour<1024><<<grid, 1024, P.color_lds, s>>>(c, pool);
  else
    k_colour<256><<<grid, 256, P.color_lds, s>>>(c, pool);
}


void launch_colored_sweep(shp_batch* b) {
  const Ctx& c = b->ctx;
  const StepPlan& P = b->plan;
  const int pool = (int)P.color_pool;
  const unsigned big = (unsigned)P.sweep_big;
  if (big > 0) {
    const unsigned grid = big + (unsigned)(c.flow_worlds * (c.flow_groups - 1));
    if (P.color_threads == 1024)
      k_sweep_colours<1024><<<grid, 1024, P.color_pool, b->stream>>>(c, pool);
    else if (P.color_threads == 512)
      k_sweep_colours<512><<<grid, 512, P.color_pool, b->stream>>>(c, pool);
    else
      k_sweep_colours<256><<<grid, 256, P.color_pool, b->stream>>>(c, pool);
  }
  if (P.g_sweep_waves > 0) {
    const size_t lds = (size_t)SWEEP_WAVES * P.sweep_slice * 4;
    const unsigned grid = (unsigned)P.g_sweep_waves;
    if (P.sweep_parts > 1)
      k_sweep_waves<SWEEP_PARTS><<<grid, 64 * SWEEP_WAVES * SWEEP_PARTS, lds, b->stream>>>(
          c, (int)big, P.sweep_slice);
    else
      k_sweep_waves<1><<<grid, 64 * SWEEP_WAVES, lds, b->stream>>>(c, (int)big, P.sweep_slice);
  }
}

void launch_colored_unpack(shp_batch* b) {
  k_colour_unpack<<<b->plan.g_unpack, 256, 0, b->stream>>>(b->ctx);
}
