// Helpers of the dGamma kernels that evaluate their frequency integrals in
// independent waves (SU(2), XYZ and TRI cores): lane exchanges, wave-private
// LDS, bracket searches, unit decoding, and the sums of a LanePlan.
#pragma once
#include "frg_common.h"
#include "lane_plan.h"

namespace frg {

constexpr int kRhsWaves = 4;    // waves (independent work units) per workgroup
constexpr int kRhsPoints = 16;  // points described per production pass: 64 lanes, four per point
// byte offsets past every vertex (smaller than 2 GiB): buffer loads return 0.
// Rows of points past the list, and sites past L.  Nothing is added to the sum
// of the two; to a row past the list, offsets within a row are
constexpr unsigned kNoRow = 0x80000000u, kNoSite = 0x7ffffff0u;
static_assert((unsigned long long)kNoRow + kNoSite + 16 <= 1ull << 32, "a 16-byte load at the sum does not wrap");

// value of the other lane of an even/odd lane pair
__device__ __forceinline__ int pair_swap(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ double pair_swap(double v) {
  int2 q;
  __builtin_memcpy(&q, &v, 8);
  q.x = pair_swap(q.x);
  q.y = pair_swap(q.y);
  __builtin_memcpy(&v, &q, 8);
  return v;
}
// lanes i and i ^ 8 of every row of 16 exchanged
__device__ __forceinline__ double half_row_swap(double v) {
  int2 q;
  __builtin_memcpy(&q, &v, 8);
  q.x = __builtin_amdgcn_mov_dpp(q.x, 0x128, 0xf, 0xf, true);  // row_ror:8
  q.y = __builtin_amdgcn_mov_dpp(q.y, 0x128, 0xf, 0xf, true);
  __builtin_memcpy(&v, &q, 8);
  return v;
}
// a DPP move of a double; banks (fours of lanes of a row) outside the mask keep v
template <int CTRL, int BANKS = 0xf> __device__ __forceinline__ double row_move(double v) {
  int2 q;
  __builtin_memcpy(&q, &v, 8);
  q.x = __builtin_amdgcn_update_dpp(q.x, q.x, CTRL, 0xf, BANKS, BANKS == 0xf);
  q.y = __builtin_amdgcn_update_dpp(q.y, q.y, CTRL, 0xf, BANKS, BANKS == 0xf);
  __builtin_memcpy(&v, &q, 8);
  return v;
}
// block (four lanes) b of every row of 16 reads block b + 1, b + 2, b + 3 (mod 4)
__device__ __forceinline__ double block_next(double v) { return row_move<0x12c>(v); }   // row_ror:12
__device__ __forceinline__ double block_cross(double v) { return row_move<0x128>(v); }  // row_ror:8
__device__ __forceinline__ double block_prev(double v) { return row_move<0x124>(v); }   // row_ror:4
// the lanes of every half row in reverse order: blocks exchanged, and reversed
__device__ __forceinline__ double half_mirror(double v) { return row_move<0x141>(v); }
// orders a wave's LDS writes before its later reads of other lanes' data (the
// LDS executes one wave's accesses in order; this keeps the compiler from
// moving them)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// keeps the descriptors of a point out of registers between its uses: tiles
// and sites of one point read them again from LDS (broadcast reads, cheap
// next to the gathers) where the compiler would otherwise hold some 50
// registers of them
__device__ __forceinline__ void reread_lds() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// computes a and b here: the compiler would otherwise sink their sums to the
// last use, across the branches between, and hold the gathered supports until
// then (more than 100 spilled registers)
template <class T> __device__ __forceinline__ void settle(T &a, T &b) { asm volatile("" : "+v"(a), "+v"(b)); }

struct Bracket {
  int lo, step;  // support indices lo and lo + step (step 0: clamped, weight 0)
  double b;
};
__device__ __forceinline__ Bracket bracket_of(const double *m, int nw, double w, int geo, float ga, float gb) {
  int lo, hi;
  double b;
  interp_sel(m, nw, w, geo, ga, gb, lo, hi, b);
  return Bracket{lo, hi - lo, b};
}

__device__ __forceinline__ int tri_decode(int q) {
  int s = (int)((sqrt(8.0 * q + 1.0) - 1.0) * 0.5);
  while ((s + 1) * (s + 2) / 2 <= q) ++s;
  while (s * (s + 1) / 2 > q) --s;
  return s;
}

using d4 = __attribute__((ext_vector_type(4))) double;

// Update of a 16 x 16 matrix by four points: lane 16 k + r of a and b holds rows
// (columns) r at point k.  Done by 4 x 4 x 4 matrix instructions, four blocks
// each, b rotated by blocks: 17 cycles of a SIMD each where the 16 x 16 x 4
// instruction takes some 130 (measured 73 against 38 TFLOP/s).  c[z] of lane
// 16 i + 4 b + j is the element (4 b + i, 4 ((b + z) % 4) + j).
__device__ __forceinline__ double mfma_blocks(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void outer_update(d4 &c, double a, double b) {
  const double b1 = block_next(b), b2 = block_cross(b), b3 = block_prev(b);
  c[0] = mfma_blocks(a, b, c[0]);
  c[1] = mfma_blocks(a, b1, c[1]);
  c[2] = mfma_blocks(a, b2, c[2]);
  c[3] = mfma_blocks(a, b3, c[3]);
}

// XCD-aware order of workgroups (dispatched round-robin over the 8 XCDs): runs
// of chunk consecutive positions go to the XCDs in turn
__device__ __forceinline__ long long xcd_position(unsigned block, int chunk) {
  const long long j = block >> 3;
  return ((j / chunk) * 8 + (block & 7)) * chunk + (j % chunk);
}

// Units of the S and U channels: (X, a >= b), the bundles of transfer
// frequency X serving the results (t = b, o = a) and (t = a, o = b); and per
// (X, t) the second result of the diagonal item (X, t, X).
inline long long su_units(long long nw) { return nw * (nw * (nw + 1) / 2 + nw); }
struct SuUnit {
  int X, a, b;
  int kind;  // 0: S rule (diagonal supports +) for both results, 1: U rule (-) for both, 2: first U, second S
  int outs;  // bit 0: the result (t = b, o = a), bit 1: (t = a, o = b)
  // result r is item (o, t, X) for the U rule, else (X, t, o)
  __device__ __forceinline__ bool u_rule(int r) const { return kind == 1 || (kind == 2 && r == 0); }
  __device__ __forceinline__ int item(int r, int nw) const {
    const int t = r ? a : b, o = r ? b : a;
    return (u_rule(r) ? tri(o, X) : tri(X, o)) * nw + t;
  }
};
__device__ __forceinline__ SuUnit su_unit(int unit, int nw) {
  const int npair = nw * (nw + 1) / 2, per = npair + nw;
  SuUnit u;
  u.X = unit / per;
  const int q = unit - u.X * per;
  if (q < npair) {
    u.a = __builtin_amdgcn_readfirstlane(tri_decode(q));
    u.b = q - u.a * (u.a + 1) / 2;
    u.kind = u.a <= u.X ? 0 : (u.b >= u.X ? 1 : 2);
    u.outs = u.a == u.b ? 1 : 3;
  } else {
    const int t = q - npair;
    u.a = t <= u.X ? u.X : t;
    u.b = t <= u.X ? t : u.X;
    u.kind = t <= u.X ? 1 : 0;
    u.outs = t <= u.X ? 1 : 2;
  }
  return u;
}

// A lane's access buffer of an S / U unit's point (lanes four per point: pair
// pp, argument pj): t slot its own argument, o slot the other lane's.  x, y:
// row byte offsets at the first t support and the two o supports, z: byte step
// to the second t support; wa, wb: weights with the density sign of the rule
// (rule 1: diagonal supports negated); diag: bits 2, 3 for diagonal o supports.
struct SuBuffer {
  int x, y, z, diag;
  double2 wa, wb;
};
__device__ __forceinline__ SuBuffer su_buffer(const Bracket &t, const Bracket &o, int X, int nw, int rowbytes, int rule) {
  SuBuffer d;
  const int ol = o.lo, oh = o.lo + o.step;
  const int rl = ol > X ? tri(ol, X) : tri(X, ol), rh = oh > X ? tri(oh, X) : tri(X, oh);
  d.x = (rl * nw + t.lo) * rowbytes;
  d.y = (rh * nw + t.lo) * rowbytes;
  d.z = t.step * rowbytes;
  d.diag = (ol == X ? 4 : 0) | (oh == X ? 8 : 0);
  const bool nl = rule ? ol >= X : ol > X, nh = rule ? oh >= X : oh > X;
  const double bl = nl ? -(1.0 - o.b) : 1.0 - o.b, bh = nh ? -o.b : o.b;
  d.wa = make_double2((1.0 - t.b) * bl, t.b * bl);
  d.wb = make_double2((1.0 - t.b) * bh, t.b * bh);
  return d;
}

// a lane's sum over its entries of a plan (ent: the lane's first quadruple);
// the next quadruple is loaded while one is summed
__device__ __forceinline__ double plan_sum(const uint4 *ent, int lanes, int cnt, const double *m) {
  double sum = 0.0;
  uint4 next = cnt > 0 ? ent[0] : make_uint4(0, 0, 0, 0);
  for (int k = 0; k < cnt; k += 4) {
    const uint4 q = next;
    ent += lanes;
    if (k + 4 < cnt) next = *ent;
    sum = fma((double)(q.x >> 16), m[q.x & 0xffff], sum);
    if (k + 1 < cnt) sum = fma((double)(q.y >> 16), m[q.y & 0xffff], sum);
    if (k + 2 < cnt) sum = fma((double)(q.z >> 16), m[q.z & 0xffff], sum);
    if (k + 3 < cnt) sum = fma((double)(q.w >> 16), m[q.w & 0xffff], sum);
  }
  return sum;
}

}  // namespace frg
