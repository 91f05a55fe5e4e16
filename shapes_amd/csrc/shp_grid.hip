// shp_grid.hip - uniform-grid broadphase for large worlds.
//
// Output contract (identical to the wavefront scan in shp_engine.hip and to
// culledKeys, shapes/src/Physics/Broadphase/Aabb.hs:168-183 / Grid.hs:67-86):
// for every body i of a world, all j < i of the same world with inclusive
// AABB overlap and not both static, segments in descending i, each segment
// in descending j.
//
// Each world has a cell size h >= the AABB extent of any of its "small"
// bodies (2 * the largest vertex radius of its dynamic bodies, plus a
// margin), fixed at creation.  Static bodies larger than that ("large",
// e.g. floors) are listed per world and tested explicitly.  A small body is
// binned by the cell of its AABB's min corner into a per-world hash table
// (counting sort, per-step), which stores a 48-byte record per body in
// bucket order (AABB, cell, index, static flag), so a bucket's candidates
// are read contiguously.  Any small j overlapping small i has its min
// corner in cells [cell(min_i) - 1, cell(max_i)] on each axis (at most 3x3
// cells), because max_j >= min_i and extent_j < h.  A large body i scans
// every j < i of its world.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "shp_engine.h"

__device__ __forceinline__ int cell_of(double x, double h) {
  double q = floor(x / h);
  if (!(q == q)) return 0;
  if (q > 1073741824.0) return 1073741824;
  if (q < -1073741824.0) return -1073741824;
  return (int)q;
}

// Bucket of cell (cx, cy): a row's cells are consecutive buckets, rows lie
// spread over the world's table (a golden-ratio step), so the 3 cells of a
// row that hold a body's partners are one run of records, and bodies in
// bucket order walk the same runs; cells that alias share a bucket and are
// told apart by their stored cell coordinates.
__device__ __forceinline__ uint32_t cell_hash(int cx, int cy, uint32_t mask) {
  const uint32_t step = (uint32_t)(((uint64_t)mask * 40503u) >> 16) | 1u;
  return ((uint32_t)cx + (uint32_t)cy * step) & mask;
}

__device__ __forceinline__ bool aabb_hit(const Ctx& c, double aminx, double amaxx, double aminy,
                                         double amaxy, int gj) {
  double bminx = c.bminx[gj], bmaxx = c.bmaxx[gj];
  double bminy = c.bminy[gj], bmaxy = c.bmaxy[gj];
  return !(bminx > amaxx || bmaxx < aminx) && !(bminy > amaxy || bmaxy < aminy);
}

// gravity (applyExternal) + binning of small bodies; empty slots
// (World.delete) get neither
__global__ void k_grid_assign(Ctx c) {
  begin_step(c);
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= c.NB) return;
  if (c.dead[g]) {
    const int w = c.body_world[g];
    c.cnt_rank[c.body_off[w + 1] - 1 - (g - c.body_off[w])] = 0;
    return;
  }
  if (c.iml[g] != 0.0 && !c.probe) {
    c.vx[g] = c.vx[g] + c.gx * c.dt;
    c.vy[g] = c.vy[g] + c.gy * c.dt;
  }
  if (c.is_large[g]) return;
  int w = c.body_world[g];
  double h = c.cell_h[w];
  int cx = cell_of(c.bminx[g], h), cy = cell_of(c.bminy[g], h);
  c.body_cell[2 * g] = cx;
  c.body_cell[2 * g + 1] = cy;
  int t0 = c.tab_off[w];
  uint32_t mask = (uint32_t)(c.tab_off[w + 1] - t0 - 1);
  c.body_slot[g] = atomicAdd(&c.bucket_cnt[t0 + cell_hash(cx, cy, mask)], 1);
}

struct GridRec {
  double minx, maxx, miny, maxy;
  int cx, cy, g, st;
};

__device__ __forceinline__ GridRec load_rec(const Ctx& c, int q) {
  const double2* p = (const double2*)(c.grid_rec + 6L * q);
  const double2 x = p[0], y = p[1];
  const int4 m = *(const int4*)(p + 2);
  return GridRec{x.x, x.y, y.x, y.y, m.x, m.y, m.z, m.w};
}

__global__ void k_grid_fill(Ctx c) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  // the next step's bucket counts (this one's are summed)
  for (long i = g; i <= c.grid_buckets; i += (long)gridDim.x * blockDim.x) c.bucket_cnt[i] = 0;
  if (g >= c.NB || c.is_large[g] || c.dead[g]) return;
  int w = c.body_world[g];
  int t0 = c.tab_off[w];
  uint32_t mask = (uint32_t)(c.tab_off[w + 1] - t0 - 1);
  const int cx = c.body_cell[2 * g], cy = c.body_cell[2 * g + 1];
  int b = t0 + cell_hash(cx, cy, mask);
  int pos = c.bucket_start[b] + c.body_slot[g];
  double2* p = (double2*)(c.grid_rec + 6L * pos);
  p[0] = make_double2(c.bminx[g], c.bmaxx[g]);
  p[1] = make_double2(c.bminy[g], c.bmaxy[g]);
  *(int4*)(p + 2) = make_int4(cx, cy, g, c.is_static[g] != 0);
}

// The body whose pairs are sought, its cell (that of its min corner).
struct GridBody {
  double minx, maxx, miny, maxy;
  int g, cx, cy;
  bool st, large;
};

// LANES lanes per body i (1, 4 or 16) visit every j < i of its world with
// which it makes a pair.  A small body's partners have their min corner in at
// most 3 rows of 3 cells, each row one run of records: 5 lanes to a row (16
// lanes), or one (4), and the last lane the world's large bodies; one lane
// does all of it.  A large body's lanes stride over every j < i.
template <int LANES, class F>
__device__ __forceinline__ void grid_visit(const Ctx& c, const GridBody& a, int sl, F&& hit) {
  constexpr int ROW_LANES = LANES == 16 ? 5 : 1;
  const int g = a.g;
  const int w = c.body_world[g];
  const int b0 = c.body_off[w];
  const double h = c.cell_h[w], slack = 1e-6 * h;
  // A large body scans every j < i of its world.  So does a body whose AABB
  // is not finite or, from rounding far out, wider than a cell (a small body's
  // AABB spans at most 3 x 3 candidate cells; a non-finite one would span up
  // to 2^62 of them): the same bounded work as a large body, by all lanes.
  const double span = (a.maxx - a.minx) + (a.maxy - a.miny);
  // does it reach n cells on? (within the rounding of x / h; a cell too many
  // only costs its candidates' tests)
  auto reaches = [&](double max, int cell, int n) { return max >= (double)(cell + n) * h - slack; };
  if (a.large || !(span - span == 0.0) || reaches(a.maxx, a.cx, 2) || reaches(a.maxy, a.cy, 2)) {
    for (int gj = g - 1 - sl; gj >= b0; gj -= LANES)
      if (!(a.st && c.is_static[gj]) && !c.dead[gj] &&
          aabb_hit(c, a.minx, a.maxx, a.miny, a.maxy, gj))
        hit(gj);
    return;
  }
  const int cx0 = a.cx - 1, cx1 = a.cx + reaches(a.maxx, a.cx, 1);
  const int cy0 = a.cy - 1, ncx = cx1 - cx0 + 1, ncy = 2 + reaches(a.maxy, a.cy, 1);
  if (sl == LANES - 1) {
    for (int q = c.large_off[w]; q < c.large_off[w + 1]; ++q) {
      const int gj = c.large_ids[q];
      if (gj >= g) break;  // ascending
      if (!(a.st && c.is_static[gj]) && !c.dead[gj] &&
          aabb_hit(c, a.minx, a.maxx, a.miny, a.maxy, gj))
        hit(gj);
    }
    if (LANES > 1) return;
  }
  const int t0 = c.tab_off[w];
  const uint32_t mask = (uint32_t)(c.tab_off[w + 1] - t0 - 1);
  const int* at = c.bucket_start + t0;
  for (int row = LANES == 1 ? 0 : sl / ROW_LANES; row < ncy; row += LANES == 1 ? 1 : 3) {
    const int cy = cy0 + row;
    const uint32_t first = cell_hash(cx0, cy, mask), last = first + (uint32_t)ncx - 1u;
    int from = at[first], to = at[min(last, mask) + 1];
    bool past = last > mask;  // the run goes on at the start of the world's table
    for (;;) {
      // four records' cells and indices in flight, then the boxes of those
      // that are in the row and below the body
      for (int q = from + sl % ROW_LANES; q < to; q += 4 * ROW_LANES) {
        int4 m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          m[k] = *(const int4*)(c.grid_rec + 6L * min(q + k * ROW_LANES, to - 1) + 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (q + k * ROW_LANES >= to || m[k].z >= g || m[k].y != cy || m[k].x < cx0 || m[k].x > cx1)
            continue;
          const double2* p = (const double2*)(c.grid_rec + 6L * (q + k * ROW_LANES));
          const double2 x = p[0], y = p[1];
          if (!(a.st && m[k].w) && !(x.x > a.maxx || x.y < a.minx) &&
              !(y.x > a.maxy || y.y < a.miny))
            hit(m[k].z);
        }
      }
      if (!past) break;
      past = false;
      from = at[0];
      to = at[last - mask];
    }
  }
}

// The pairs' counts (fill = 0, 4 or 16 lanes per body) and the pairs (fill =
// 1, 1 or 16 lanes).  The count pass takes the bodies in bucket order, in
// which a wavefront's bodies walk the same few runs of records (in body order,
// a cell to a lane or two and 2 bucket bounds to a cell, it took 307 us for
// 1.14 M bodies, bound by its 8.8 M scattered loads; 157 now), then the large
// bodies, and keeps each body's first GRID_SLOTS partners; the emit pass
// writes those without a second visit when they are all, and in descending j
// either way.
// Workgroups go to the 8 XCDs in turn: workgroup b of n as the one that makes
// those of an XCD consecutive, so that the records of a region are in one L2.
__device__ __forceinline__ int xcd_block(int b, int n) {
  return b % 8 * (n / 8) + min(b % 8, n % 8) + b / 8;
}

template <int LANES>
__global__ void k_grid_pairs(Ctx c, int fill) {
  const long t = (long)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const int sl = (int)(t % LANES);
  int g = (int)(t / LANES);  // the same for the LANES lanes of a group
  if (g >= c.NB) return;
  auto rank_of = [&](int body) {
    const int w = c.body_world[body];
    return c.body_off[w + 1] - 1 - (body - c.body_off[w]);
  };
  auto body_of = [&](int body) {
    const bool large = c.is_large[body];  // not binned: no cell
    return GridBody{c.bminx[body], c.bmaxx[body], c.bminy[body], c.bmaxy[body], body,
                    large ? 0 : c.body_cell[2 * body], large ? 0 : c.body_cell[2 * body + 1],
                    c.is_static[body] != 0, large};
  };
  auto upto = [&](int n) {  // the sum over the group's lanes up to this one
    for (int o = 1; o < LANES; o <<= 1) {
      const int y = __shfl_up(n, o, LANES);
      if (sl >= o) n += y;
    }
    return n;
  };
  if (!fill) {
    if constexpr (LANES > 1) {
      const int binned = c.bucket_start[c.grid_buckets];
      GridBody a;
      if (g < binned) {
        const GridRec r = load_rec(c, g);
        a = GridBody{r.minx, r.maxx, r.miny, r.maxy, r.g, r.cx, r.cy, r.st != 0, false};
      } else {
        if (g - binned >= c.large_off[c.W]) return;
        g = c.large_ids[g - binned];
        if (c.dead[g]) return;  // k_grid_assign counts none
        a = body_of(g);
      }
      int count = 0, kept[GRID_SLOTS];
      grid_visit<LANES>(c, a, sl, [&](int gj) {
#pragma unroll
        for (int k = 0; k < GRID_SLOTS; ++k)
          if (k == count) kept[k] = gj;
        ++count;
      });
      const int incl = upto(count), first = incl - count;
      const int total = __shfl(incl, LANES - 1, LANES);
      // the first GRID_SLOTS partners of the body, lane by lane
      int32_t* slots = c.grid_slots + (long)a.g * GRID_SLOTS;
#pragma unroll
      for (int k = 0; k < GRID_SLOTS; ++k)
        if (k < count && first + k < GRID_SLOTS) slots[first + k] = kept[k];
      if (sl == 0) c.cnt_rank[rank_of(a.g)] = total;
    }
    return;
  }
  // Past the capacity the step reports an overflow; the slots below it are
  // still all written (a segment that straddles the capacity keeps its
  // first pairs), so no later kernel of the step reads an unwritten slot.
  const int rank = rank_of(g);
  const int base = c.off_rank[rank], all = c.cnt_rank[rank];
  if ((long)base + all > c.pair_cap && sl == 0)
    atomicOr(&c.counters[CNT_FLAGS], SHP_FLAG_PAIR_OVERFLOW);
  if (all == 0 || base >= c.pair_cap) return;  // the same for the group's lanes
  const int total = min(all, c.pair_cap - base), end = base + total;
  if (all <= GRID_SLOTS) {  // the kept partners, in descending order
    const int32_t* slots = c.grid_slots + (long)g * GRID_SLOTS;
    if constexpr (LANES == 1) {
      int v[GRID_SLOTS];
#pragma unroll
      for (int k = 0; k < GRID_SLOTS; ++k) v[k] = k < all ? slots[k] : -1;
#pragma unroll
      for (int a = 1; a < GRID_SLOTS; ++a)
#pragma unroll
        for (int q = a; q > 0; --q)
          if (v[q - 1] < v[q]) {
            const int t = v[q - 1];
            v[q - 1] = v[q];
            v[q] = t;
          }
#pragma unroll
      for (int k = 0; k < GRID_SLOTS; ++k)
        if (k < total) {
          c.pa[base + k] = g;
          c.pb[base + k] = v[k];
        }
    } else {
      const int v = sl < all ? slots[sl] : -1;
      int at = 0;
#pragma unroll
      for (int k = 0; k < GRID_SLOTS; ++k) at += __shfl(v, k, LANES) > v ? 1 : 0;
      if (sl < all && at < total) {
        c.pa[base + at] = g;
        c.pb[base + at] = v;
      }
    }
    return;
  }
  const GridBody a = body_of(g);
  int pos = base;
  if constexpr (LANES > 1) {
    int count = 0;
    grid_visit<LANES>(c, a, sl, [&](int) { ++count; });
    pos += upto(count) - count;
  }
  grid_visit<LANES>(c, a, sl, [&](int gj) {
    if (pos < end) {
      c.pa[pos] = g;
      c.pb[pos] = gj;
    }
    ++pos;
  });
  // the group's stores precede lane 0's sort in this wavefront's program
  // order; the fence keeps the compiler from moving them
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  if (sl != 0) return;
  // the segment in descending j (insertion sort; segments are short)
  for (int k = base + 1; k < end; ++k) {
    const int v = c.pb[k];
    int q = k - 1;
    while (q >= base && c.pb[q] < v) {
      c.pb[q + 1] = c.pb[q];
      --q;
    }
    c.pb[q + 1] = v;
  }
}

// 16 lanes per body while that still fits about one wave of work per SIMD
// slot of the GPU several times over (batches up to 131072 bodies); beyond
// (the plan's grid_wide false), 4 lanes per body count and keep the first
// partners, one lane per body emits.
// The wide schedule gives each body 16 lanes in both passes.  Otherwise the
// count pass splits a body's cells over 4 lanes (their gathers overlap, and
// the pass is bound by their latency) and the emit pass takes 1 lane, which
// for most bodies only copies the partners the count pass kept.
static void launch_grid_pairs(shp_batch* b, int fill) {
  const Ctx& c = b->ctx;
  const StepPlan& P = b->plan;
  if (P.grid_wide)
    k_grid_pairs<16><<<P.g_pairs, 256, 0, b->stream>>>(c, fill);
  else if (!fill)
    k_grid_pairs<4><<<P.g_pairs_count, 256, 0, b->stream>>>(c, 0);
  else
    k_grid_pairs<1><<<P.g_pairs, 256, 0, b->stream>>>(c, 1);
}

// Grid broadphase, first half: binning and per-body pair counts into
// cnt_rank (the caller then scans cnt_rank into off_rank).
hipError_t launch_grid_count(shp_batch* b) {
  Ctx& c = b->ctx;
  hipStream_t s = b->stream;
  k_grid_assign<<<b->plan.g_bodies, 256, 0, s>>>(c);
  hipError_t e = scan_grid_buckets(b);
  if (e != hipSuccess) return e;
  k_grid_fill<<<b->plan.g_bodies, 256, 0, s>>>(c);
  launch_grid_pairs(b, 0);
  return hipGetLastError();
}

// Second half: emit the pairs at off_rank.
hipError_t launch_grid_emit(shp_batch* b) {
  launch_grid_pairs(b, 1);
  return hipGetLastError();
}
