// shp_records.h - the solvers' records: their layout, and how one is written
// from a pair's contacts (by the contact kernel, which has every value in
// registers); the coloured solver's are patched by the learned warm start.
#pragma once

#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "shp_engine.h"
#include "shp_geom.h"

namespace shp {

// Manifold M's record: 7 words of 16 bytes, word q at
// rec[(M / RB) * 7 * RB + q * RB + M % RB] (blocks of RB manifolds)
//   0  ux, uy, mu, e       the row normal (flip applied), materials
//   1  ax, ay, bx, by      the normal times the inverse masses of a / b
//   2  ga, gb, flags, turns  bodies (global ids), flags, and for a world
//                          solved on several CUs the manifold's turns
//   3  jn2, jn5, jt2, jt5  the first contact: angular entries of the
//                          normal / friction rows
//   4  bn, icn, ict, wn2   bias, reciprocal effective masses, angular
//   5  wn5, wt2, wt5, 0      entries times the inverse inertias
//   6  ln, lt              its lagrangians (FP64)
// and the second contact's 4 words (3-6 above) at
// rec2[(M / RB) * 4 * RB + q * RB + M % RB].  Products and reciprocals are
// formed in FP64 and rounded once.
enum { REC_WORDS = 7, REC2_WORDS = 4 };
// manifolds per block, a power of two dividing 64: 4 against 64 and 8, a
// step of 1024 piles 21.23 against 21.36 ms and of 4096 small worlds 1.599
// against 1.613 (2: 21.68 / 1.647)
constexpr int RB = 4;
static_assert(16 * 64 * (REC_WORDS + REC2_WORDS) == 4 * COLOR_PACK_FLOATS(64),
              "record words differ from the buffer size");
// a manifold's turn on a dynamic body: its place among the body's manifolds by
// colour, and their number (0: a static body)
struct Turns {
  int at_a, of_a, at_b, of_b;
};
__host__ __device__ __forceinline__ int pack_turns(Turns t) {
  return t.at_a | t.of_a << 8 | t.at_b << 16 | t.of_b << 24;
}
__host__ __device__ __forceinline__ Turns unpack_turns(int x) {
  return Turns{x & 0xFF, (x >> 8) & 0xFF, (x >> 16) & 0xFF, (int)((unsigned)x >> 24)};
}
// manifold flags: 1 a static, 2 b static, 4 first contact warm, 8 second
// contact present, 16 second contact warm
enum { MFL_A_STATIC = 1, MFL_B_STATIC = 2, MFL_WARM0 = 4, MFL_TWO = 8, MFL_WARM1 = 16 };

struct PackF {
  float4* rec;   // REC_WORDS x PC (PC rounded up to blocks)
  float4* rec2;  // REC2_WORDS x PC
};

__device__ __forceinline__ PackF packf(const Ctx& c) {
  PackF p;
  p.rec = (float4*)c.pk;
  p.rec2 = p.rec + (long)REC_WORDS * ((c.pair_cap + 63) / 64 * 64);
  return p;
}

// Word 0 of manifold M's record (words q at + RB q) and of its second
// contact's.
__device__ __forceinline__ float4* rec_of(float4* rec, int M) {
  return rec + (long)((unsigned)M / RB) * (REC_WORDS * RB) + ((unsigned)M % RB);
}
__device__ __forceinline__ float4* rec2_of(float4* rec2, int M) {
  return rec2 + (long)((unsigned)M / RB) * (REC2_WORDS * RB) + ((unsigned)M % RB);
}

// Word 3 of manifold M's record (its first contact) or of its second
// contact's (words at + RB q).
__device__ __forceinline__ float4* rec_contact(const PackF& P, int M, int j) {
  return j ? rec2_of(P.rec2, M) : rec_of(P.rec, M) + 3 * RB;
}

// Contact j (0 or 1) of manifold M as the contact generation computes it:
// the rows' angular entries, bias and effective masses, with the inverse
// inertias ira / irb of the two bodies ...
__device__ __forceinline__ void write_record_rows(const PackF& P, int M, int j, double ira,
                                                  double irb, double jn2, double jn5, double jt2,
                                                  double jt5, double bn, double mcn, double mct) {
  float4* w = rec_contact(P, M, j);
  w[0] = make_float4((float)jn2, (float)jn5, (float)jt2, (float)jt5);
  w[RB] = make_float4((float)bn, (float)(1.0 / mcn), (float)(1.0 / mct), (float)(ira * jn2));
  w[2 * RB] = make_float4((float)(irb * jn5), (float)(ira * jt2), (float)(irb * jt5), 0.0f);
}

// ... and its warm-start lagrangians.
__device__ __forceinline__ void write_record_lambda(const PackF& P, int M, int j, double ln,
                                                    double lt) {
  *(double2*)(rec_contact(P, M, j) + 3 * RB) = make_double2(ln, lt);
}

// The rest of manifold M's record: row normal u (flip applied), materials,
// the normal times the inverse masses ima / imb, bodies and flags for its
// nk (1 or 2) stored contacts, bit j of `warm` set when contact j is warm.
__device__ __forceinline__ void write_record_head(const Ctx& c, const PackF& P, int M, int ga,
                                                  int gb, d2 u, double ima, double imb, int nk,
                                                  int warm, int turns) {
  const int flags = (c.is_static[ga] ? MFL_A_STATIC : 0) | (c.is_static[gb] ? MFL_B_STATIC : 0) |
                    ((warm & 1) ? MFL_WARM0 : 0) | (nk > 1 ? MFL_TWO : 0) |
                    (nk > 1 && (warm & 2) ? MFL_WARM1 : 0);
  float4* r = rec_of(P.rec, M);
  r[0] = make_float4((float)u.x, (float)u.y, (float)((c.mu[ga] + c.mu[gb]) / 2.0),
                     (float)hs_min(c.e[ga], c.e[gb]));
  r[RB] = make_float4((float)(ima * u.x), (float)(ima * u.y), (float)(imb * u.x),
                      (float)(imb * u.y));
  *(int4*)(r + 2 * RB) = make_int4(ga, gb, flags, turns);
}

// A manifold whose contacts lie beyond the contact capacity (the step then
// reports the overflow): a record that touches no velocity and no contact.
__device__ __forceinline__ void write_null_record(const PackF& P, int M, int ga, int gb,
                                                  int turns) {
  float4* r = rec_of(P.rec, M);
  const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  r[0] = z;
  r[RB] = z;
  *(int4*)(r + 2 * RB) = make_int4(ga, gb, MFL_A_STATIC | MFL_B_STATIC, turns);
  r[3 * RB] = z;
  r[4 * RB] = z;
  r[5 * RB] = z;
  r[6 * RB] = z;
}

// Contact j of manifold M given a warm start after its record was written
// (the learned one): its lagrangians and warm flag.
__device__ __forceinline__ void patch_record_warm(const PackF& P, int M, int j, double ln, double lt) {
  write_record_lambda(P, M, j, ln, lt);
  atomicOr((int*)(rec_of(P.rec, M) + 2 * RB) + 2, j ? MFL_WARM1 : MFL_WARM0);
}

// The ordered solver's FP64 records, 8 words of 16 bytes per contact slot:
// a manifold's head at its first contact,
//   0 ux, uy (row normal, flip applied)  1 iml_a, imr_a  2 iml_b, imr_b
//   3 mu, local bodies a | b << 32 with flags
// and every contact's rows, for the lane of body a and the lane of body b
//   4 jn2, jt2  5 jn5, jt5  6 0, mct  7 bn, mcn
// The contact kernel writes them (it has every value in registers), so that
// the solve, one workgroup per world, need not gather them: on one
// 8192-polygon world that took 0.3 ms of one CU, here it adds 3 us.
enum { FLOW_BODY = 0x1FFFFFFF, FLOW_BOUNCE = 0x20000000, FLOW_TWO = 0x40000000,
       FLOW_STATIC = (int)0x80000000 };

__device__ __forceinline__ double2* flow_rec(const Ctx& c, int k) {
  return (double2*)c.pk + (long)k * FLOW_WORDS;
}

__device__ __forceinline__ void write_flow_head(const Ctx& c, int k, int ga, int gb, int b0, d2 u,
                                                const double* im, bool two) {
  double2* h = flow_rec(c, k);
  const int la = (ga - b0) | (c.is_static[ga] ? FLOW_STATIC : 0);
  const int lb = (gb - b0) | (c.is_static[gb] ? FLOW_STATIC : 0);
  const int fl = (two ? FLOW_TWO : 0) | (hs_min(c.e[ga], c.e[gb]) != 0.0 ? FLOW_BOUNCE : 0);
  h[0] = make_double2(u.x, u.y);
  h[1] = make_double2(im[0], im[2]);
  h[2] = make_double2(im[3], im[5]);
  // pairMu (Friction.hs:46-48)
  h[3] = make_double2((c.mu[ga] + c.mu[gb]) / 2.0,
                      __longlong_as_double((long long)(uint32_t)(la | fl) |
                                           ((long long)(lb | fl) << 32)));
  c.sch_ab[k] = make_int2(la, lb);
}

// bn + 0: the bias with a bounce term of 0 (turns -0 into 0)
__device__ __forceinline__ void write_flow_con(const Ctx& c, int k, double jn2, double jn5,
                                               double jt2, double jt5, double bn, double mcn,
                                               double mct) {
  double2* w = flow_rec(c, k) + 4;
  w[0] = make_double2(jn2, jt2);
  w[1] = make_double2(jn5, jt5);
  w[2] = make_double2(0.0, mct);
  w[3] = make_double2(bn + 0.0, mcn);
}

}  // namespace shp
