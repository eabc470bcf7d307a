// Device helpers shared by the SU(2), XYZ and TRI flow kernels: the frequency
// mesh (bracket searches, interpolation), the self-energy interpolation, the
// trapezoid evaluation points of ImplicitIntegrator, the per-cutoff tables of
// evaluation points and propagator weights, and the access-buffer descriptors
// (support rows, bilinear weights, density signs) of the SU(2) and XYZ vertex
// layouts.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace frg {

constexpr double kPi = 3.14159265358979323846;
constexpr double kTwoPi = 2.0 * kPi;

// ---------------------------------------------------------------------------
// frequency mesh (positive half m[0..n) ascending; signed index i in [-n, n))
// ---------------------------------------------------------------------------
__device__ __forceinline__ double mesh_at(const double *m, int i) { return i >= 0 ? m[i] : -m[-i - 1]; }

// number of mesh points <= w (branch-free binary lifting)
__device__ __forceinline__ int count_le(const double *m, int n, double w) {
  int pos = 0;
  for (int step = 1 << (31 - __clz(n)); step > 0; step >>= 1) {
    const int p = pos + step;
    if (p <= n && m[p - 1] <= w) pos = p;
  }
  return pos;
}

// first mesh point > w, and the one before it, within [0, n)
__device__ inline int greater_pos(const double *m, int n, double w) {
  if (w <= m[0]) return 0;
  const int c = count_le(m, n, w);
  return c < n ? c : n - 1;
}

__device__ inline int lesser_pos(const double *m, int n, double w) { return w <= m[0] ? 0 : count_le(m, n, w) - 1; }

// FrequencyDiscretization::lesser / greater (src/FrequencyDiscretization.hpp:253-296)
__device__ inline int mesh_lesser(const double *m, int n, double w) { return w < 0 ? -(greater_pos(m, n, -w) + 1) : lesser_pos(m, n, w); }
__device__ inline int mesh_greater(const double *m, int n, double w) { return w < 0 ? -(lesser_pos(m, n, -w) + 1) : greater_pos(m, n, w); }

// FrequencyDiscretization::interpolateOffset (src/FrequencyDiscretization.hpp:326-356)
// (written as !(w > m[0]) so that a NaN argument clamps to index 0 instead of
// producing index -1; identical to the reference for every non-NaN w)
__device__ __forceinline__ void interp(const double *m, int n, double w, int &lo, int &hi, double &bias) {
  if (!(w > m[0])) { lo = 0; hi = 0; bias = 0.0; return; }
  const int c = count_le(m, n, w);
  if (c >= n) { lo = n - 1; hi = n - 1; bias = 0.0; return; }
  lo = c - 1;
  hi = c;
  bias = (w - m[lo]) / (m[hi] - m[lo]);
}

// SU2VertexSingleParticle::getValue (src/SU2/SU2VertexSingleParticle.hpp:73-87)
__device__ inline double sigma_at(const double *m, int n, const double *data, double w) {
  double sign = 1.0;
  if (w < 0) { w = -w; sign = -1.0; }
  int lo, hi; double b;
  interp(m, n, w, lo, hi, b);
  return sign * ((1 - b) * data[lo] + b * data[hi]);
}

__device__ __forceinline__ int tri(int a, int b) { return a * (a + 1) / 2 + b; }

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// ---------------------------------------------------------------------------
// trapezoid windows: evaluation points and weights (0.5 folded in), in the
// order ImplicitIntegrator visits them (src/lib/Integrator.hpp:137-287).  A
// window is its two end indices and its number of points; every point follows
// from its position, so that lanes form them side by side.
// ---------------------------------------------------------------------------
struct PointWeight {
  double x, w;
};
struct Window {
  double min, max;
  int lo, hi, cnt;
};

// (-inf, max]
__device__ inline Window window_right(const double *m, int n, double max) {
  const int hi = mesh_lesser(m, n, max);
  return Window{0.0, max, -n, hi, hi != -n ? hi + n + 2 : 2};
}
__device__ inline PointWeight right_point(const double *m, const Window &w, int k) {
  const double first = mesh_at(m, w.lo);
  if (w.hi == w.lo) return PointWeight{k == 0 ? w.max : first, 0.5 * (w.max - first)};
  const int i = w.lo + k;
  if (i > w.hi) return PointWeight{w.max, 0.5 * (w.max - mesh_at(m, w.hi))};
  const double up = i == w.hi ? w.max : mesh_at(m, i + 1), down = mesh_at(m, i == w.lo ? i : i - 1);
  return PointWeight{mesh_at(m, i), 0.5 * (up - down)};
}
// [min, max]
__device__ inline Window window_both(const double *m, int n, double min, double max) {
  const int lo = mesh_greater(m, n, min), hi = mesh_lesser(m, n, max);
  return Window{min, max, lo, hi, hi >= lo ? hi - lo + 3 : 2};
}
__device__ inline PointWeight both_point(const double *m, const Window &w, int k) {
  if (w.hi < w.lo) return PointWeight{k == 0 ? w.max : w.min, 0.5 * (w.max - w.min)};
  if (k == 0) return PointWeight{w.min, 0.5 * (mesh_at(m, w.lo) - w.min)};
  const int i = w.lo + k - 1;
  if (i > w.hi) return PointWeight{w.max, 0.5 * (w.max - mesh_at(m, w.hi))};
  const double up = i == w.hi ? w.max : mesh_at(m, i + 1), down = i == w.lo ? w.min : mesh_at(m, i - 1);
  return PointWeight{mesh_at(m, i), 0.5 * (up - down)};
}
// [min, inf)
__device__ inline Window window_left(const double *m, int n, double min) {
  const int lo = mesh_greater(m, n, min);
  return Window{min, 0.0, lo, n - 1, lo != n - 1 ? n - lo + 1 : 2};
}
__device__ inline PointWeight left_point(const double *m, const Window &w, int k) {
  if (k == 0) return PointWeight{w.min, 0.5 * (mesh_at(m, w.lo) - w.min)};
  const int i = w.lo + k - 1;
  if (w.lo == w.hi) return PointWeight{mesh_at(m, i), 0.5 * (mesh_at(m, i) - w.min)};
  const double up = mesh_at(m, i == w.hi ? i : i + 1), down = i == w.lo ? w.min : mesh_at(m, i - 1);
  return PointWeight{mesh_at(m, i), 0.5 * (up - down)};
}

// Evaluation points and weights of one channel with exact transfer frequency
// m[x] at cutoff cut: the conventional points +-cut with p(cut, cut +- X)
// (src/SU2/SU2FrgCore.cpp:349-371, src/TRI/TRIFrgCore.cpp:2917-2940), then the
// three Katanin windows (src/SU2/SU2FrgCore.cpp:378-392) with
// dSigma(w') G(w')^2 G(X + w') folded into the trapezoid weight
// (src/SU2/SU2FrgCore.cpp:343-347,373-424).  Depends on (x, cut) only, so every
// item of a flow shares the table.
//
// weight_tables_wave: one 64-lane workgroup per table, x < nw a channel list,
// x == nw the plain trapezoid list of the correlation integrals at nu = 0 (the
// windows with X = 0; src/SU2/SU2MeasurementCorrelation.cpp:145-159,
// src/TRI/TRIMeasurementCorrelation.cpp:270-284).  s_m is LDS space for the
// nw mesh values.  *overflow is raised if a list exceeds emax entries.  What
// bounds it is latency: one lane that walked the windows in turn took 18 us
// (32 frequencies).
__device__ inline void weight_tables_wave(int x, const double *mesh, int nw, double cut, const double *v2,
                                          const double *dv2, double *Wwp, double *Wc, int *Wn, double *Cwp,
                                          double *Cw, int *Cn, int emax, int *overflow, double *s_m) {
  const int lane = threadIdx.x;
  for (int i = lane; i < nw; i += 64) s_m[i] = mesh[i];
  __syncthreads();
  const double *m = s_m;
  const bool plain = x == nw;
  const double X = plain ? 0.0 : m[x];
  double *wp = plain ? Cwp : Wwp + (size_t)x * emax, *w = plain ? Cw : Wc + (size_t)x * emax;
  const int k0 = plain ? 0 : (X > 2.0 * cut ? 2 : 1);
  const bool right = -(X + cut) > mesh_at(m, -nw), both = X - cut > cut, left = cut < mesh_at(m, nw - 1);
  Window R{}, B{}, Lw{};
  if (right) R = window_right(m, nw, -(X + cut));
  if (both) B = window_both(m, nw, cut - X, -cut);
  if (left) Lw = window_left(m, nw, cut);
  const int k1 = k0 + R.cnt, k2 = k1 + B.cnt, cnt = k2 + Lw.cnt;
  const int kend = cnt < emax ? cnt : emax;
  for (int k = lane; k < kend; k += 64) {
    if (k < k0) {
      const double b = k ? cut - X : cut + X;
      wp[k] = k ? -cut : cut;
      w[k] = 1.0 / ((cut + sigma_at(m, nw, v2, cut)) * (b + sigma_at(m, nw, v2, b)));
      continue;
    }
    const PointWeight q = k < k1 ? right_point(m, R, k - k0) : (k < k2 ? both_point(m, B, k - k1) : left_point(m, Lw, k - k2));
    wp[k] = q.x;
    if (plain) {
      w[k] = q.w;
    } else {
      const double d1 = q.x + sigma_at(m, nw, v2, q.x);
      w[k] = q.w * (sigma_at(m, nw, dv2, q.x) / (d1 * d1 * (X + q.x + sigma_at(m, nw, v2, X + q.x))));
    }
  }
  if (lane == 0) {
    (plain ? *Cn : Wn[x]) = kend;
    if (cnt > emax) atomicOr(overflow, 1);
  }
}

constexpr int kSigmaThreads = 320;  // workgroup of the dSigma kernels: four waves of the range sum and one

// correlation kernels: workgroup, of which the first threads evaluate the
// site-local vertices and the rest (point, site) pairs
constexpr int kCorrThreads = 1024, kCorrEggs = 128, kCorrPoints = kCorrThreads - kCorrEggs;

// out[q] = sum over o < n of partial[o * nq + q] by a workgroup (nq <= 1024):
// the points dealt to the threads of an output, so that one waits for n / 8
// loads or fewer where there are threads for it
__device__ inline void sum_partials(const double *partial, int n, int nq, double *out) {
  __shared__ double part[1024];
  const int nt = blockDim.x, tid = threadIdx.x;
  const int parts = nq < nt ? (nt / nq < 1024 / nq ? nt / nq : 1024 / nq) : 1;
  for (int k = tid; k < parts * nq; k += nt) {
    const int q = k % nq;
    double v = 0.0;
    for (int o = k / nq; o < n; o += parts) v += partial[(size_t)o * nq + q];
    part[k] = v;
  }
  __syncthreads();
  for (int q = tid; q < nq; q += nt) {
    double v = part[q];
    for (int p = 1; p < parts; ++p) v += part[p * nq + q];
    out[q] = v;
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// access-buffer descriptors (SU(2) and XYZ layouts: one element per (row, site))
// ---------------------------------------------------------------------------
// row index of a support point with the s <-> u exchange of
// _generateAccessBufferOffset (src/SU2/SU2VertexTwoParticle.hpp:616-632,
// src/XYZ/XYZVertexTwoParticle.hpp:637-653); neg = density sign flip
__device__ __forceinline__ int support_row(int so, int to, int uo, int nw, bool &neg) {
  if (so < uo) { neg = true; return tri(uo, so) * nw + to; }
  neg = false;
  return tri(so, uo) * nw + to;
}

struct Interp {
  int lo, hi;
  double b;
};

__device__ __forceinline__ Interp interp_of(const double *m, int nw, double x) {
  Interp r;
  interp(m, nw, x, r.lo, r.hi, r.b);
  return r;
}

// interpolateOffset from the bracket position c = count_le(m, n, w)
__device__ __forceinline__ void interp_finish(const double *m, int n, int c, double w, Interp &r) {
  if (!(w > m[0])) { r.lo = 0; r.hi = 0; r.b = 0.0; return; }
  if (c >= n) { r.lo = n - 1; r.hi = n - 1; r.b = 0.0; return; }
  r.lo = c - 1;
  r.hi = c;
  r.b = (w - m[r.lo]) / (m[r.hi] - m[r.lo]);
}

// two interpolateOffset calls whose bracket searches run in one binary-lifting
// loop, so that the two chains of dependent mesh reads overlap; each result
// equals interp_of(m, n, x)
__device__ __forceinline__ void interp_pair(const double *m, int n, double x0, double x1, Interp &a, Interp &b) {
  int p0 = 0, p1 = 0;
  for (int step = 1 << (31 - __clz(n)); step > 0; step >>= 1) {
    const int q0 = p0 + step, q1 = p1 + step;
    if (q0 <= n && m[q0 - 1] <= x0) p0 = q0;
    if (q1 <= n && m[q1 - 1] <= x1) p1 = q1;
  }
  interp_finish(m, n, p0, x0, a);
  interp_finish(m, n, p1, x1, b);
}

// Bracket positions on a geometric mesh (the exponential discretisation,
// m[i] close to m[0] r^i): the guess floor(log2(w) ga + gb) + 1 from the
// hardware FP32 logarithm is within one of count_le, and the comparisons with
// the mesh that follow make the position exact for any mesh.  ga = 1 / log2 r,
// gb = -log2(m[0]) / log2 r (geo_mesh_params).
__device__ __forceinline__ int count_le_geo(const double *m, int n, double w, float ga, float gb) {
  float t = fmaf(__log2f((float)w), ga, gb) + 1.0f;
  t = fminf(fmaxf(t, 0.0f), (float)n);  // NaN (w <= 0) -> 0
  int c = (int)t;
  while (c < n && m[c] <= w) ++c;
  while (c > 0 && m[c - 1] > w) --c;
  return c;
}

__device__ __forceinline__ void interp_pair_geo(const double *m, int n, double x0, double x1, float ga, float gb,
                                                Interp &a, Interp &b) {
  const int p0 = count_le_geo(m, n, x0, ga, gb), p1 = count_le_geo(m, n, x1, ga, gb);
  interp_finish(m, n, p0, x0, a);
  interp_finish(m, n, p1, x1, b);
}

// interpolateOffset with the bracket from count_le_geo (geo != 0) or from the
// binary search
__device__ __forceinline__ void interp_sel(const double *m, int n, double w, int geo, float ga, float gb, int &lo,
                                           int &hi, double &bias) {
  Interp r;
  interp_finish(m, n, geo ? count_le_geo(m, n, w, ga, gb) : count_le(m, n, w), w, r);
  lo = r.lo;
  hi = r.hi;
  bias = r.b;
}

// Host: parameters of count_le_geo when every log2(m[i] / m[0]) lies within a
// quarter step of i log2 r (on = 0 otherwise: use the binary search).
inline void geo_mesh_params(const double *m, int n, int &on, float &ga, float &gb) {
  on = 0;
  ga = gb = 0.0f;
  if (n < 2 || !(m[0] > 0.0)) return;
  const double l2r = std::log2(m[n - 1] / m[0]) / (n - 1);
  if (!(l2r > 0.0) || !std::isfinite(l2r)) return;
  for (int i = 0; i < n; ++i)
    if (!(std::fabs(std::log2(m[i] / m[0]) - i * l2r) <= 0.25)) return;
  on = 1;
  ga = (float)(1.0 / l2r);
  gb = (float)(-std::log2(m[0]) / l2r);
}

template <class V2> __device__ __forceinline__ V2 buf_load(__amdgpu_buffer_rsrc_t r, int byte_off);

template <> __device__ __forceinline__ double2 buf_load<double2>(__amdgpu_buffer_rsrc_t r, int byte_off) {
  auto v = __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0);
  double2 d;
  __builtin_memcpy(&d, &v, 16);
  return d;
}

template <> __device__ __forceinline__ float2 buf_load<float2>(__amdgpu_buffer_rsrc_t r, int byte_off) {
  auto v = __builtin_amdgcn_raw_buffer_load_b64(r, byte_off, 0, 0);
  float2 d;
  __builtin_memcpy(&d, &v, 8);
  return d;
}

// Access-buffer descriptor of generateAccessBuffer(s, t, u, channel)
// (src/SU2/SU2VertexTwoParticle.hpp:399-490, src/XYZ/XYZVertexTwoParticle.hpp:419-496)
// from the two interpolations it needs: chan 0 = s exact (I1 on t, I2 on u),
// 1 = t exact (I1 on s, I2 on u), 2 = u exact (I1 on s, I2 on t).  Support byte
// offsets are row * rowbytes; the density weight carries the sign of the
// s <-> u exchange.
struct Desc4 {
  int off[4];
  double ws[4];
  double wd[4];
  int neg;  // bit q: support q is stored s <-> u exchanged (density weight negated)
};

__device__ __forceinline__ Desc4 assemble(int chan, int ex, Interp i1, Interp i2, int nw, int rowbytes) {
  Desc4 d;
  const int l1[4] = {i1.lo, i1.hi, i1.lo, i1.hi};
  const int l2[4] = {i2.lo, i2.lo, i2.hi, i2.hi};
  const double b1 = i1.b, b2 = i2.b;
  const double w[4] = {(1 - b2) * (1 - b1), (1 - b2) * b1, b2 * (1 - b1), b2 * b1};
  d.neg = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    int so, to, uo;
    if (chan == 0) { so = ex; to = l1[q]; uo = l2[q]; }
    else if (chan == 1) { so = l1[q]; to = ex; uo = l2[q]; }
    else { so = l1[q]; to = l2[q]; uo = ex; }
    bool neg;
    const int row = support_row(so, to, uo, nw, neg);
    d.off[q] = row * rowbytes;
    d.ws[q] = w[q];
    d.wd[q] = neg ? -w[q] : w[q];
    if (neg) d.neg |= 1 << q;
  }
  return d;
}

// one access buffer of a pair: the signed s and u arguments decide the site
// exchange (exactly one of them negative); swap says whether the
// pair's interpolations (I0, I1) feed the descriptor's (slot 1, slot 2) or
// (slot 2, slot 1)
struct PairBuf {
  int k;
  double a, c;
  bool swap;
  int chan;
};

}  // namespace frg
