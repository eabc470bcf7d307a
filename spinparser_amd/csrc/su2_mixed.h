// Mixed-precision dGamma/dLambda of the SU(2) core by independent waves: FP32
// vertex shadow, bundles and products, FP64 sums.  Included by su2_flow.hip
// after su2_rhs.h, whose structure it has: a unit (X, {a, b}) serves two items,
// a gather both buffers of a T pair.
//
// Every term of an integral is formed by the same FP32 operations as in the
// general kernel, in the same order, so that sharing the gathers changes no
// rounding: a bundle sums its four supports in the order of the access buffer
// (its two interpolations change places between the S and the U rule, and
// between the buffers of a T pair), and the products take the bundles in the
// order of the rule.  Signs are exact: a U bundle differs from the S one by the
// sign of the density, its result by the sign of the density result.  The sums
// over points are FP64 sums of the FP32 terms.
//
// What bounds it: the gathers (8 bytes a lane) and the vector instructions about
// equally.  Simple cubic J1-J2, 48 frequencies, 23 sites, mean over the cutoffs
// 100 to 3: 1095 -> 494 us per evaluation (k_su32 238, k_t32 256) against one
// 256-thread workgroup per item with a producer wave.  Kagome, 26 sites, bonds
// not equivalent to their reverse, 48 frequencies: 950 -> 590 us at cutoff 20,
// 2336 -> 1859 us at 0.3.
#pragma once

// spin and density of an access buffer from its supports v in the order (lo lo),
// (hi lo), (lo hi), (hi hi) of its two interpolations
__device__ __forceinline__ float spin_chain(float w0, float w1, float w2, float w3, float2 v0, float2 v1, float2 v2,
                                            float2 v3) {
  return fmaf(fabsf(w3), v3.x, fmaf(fabsf(w2), v2.x, fmaf(fabsf(w1), v1.x, fabsf(w0) * v0.x)));
}
__device__ __forceinline__ float density_chain(float w0, float w1, float w2, float w3, float2 v0, float2 v1, float2 v2,
                                               float2 v3) {
  return fmaf(w3, v3.y, fmaf(w2, v2.y, fmaf(w1, v1.y, w0 * v0.y)));
}
struct Bundle32 {
  float s, d;
};
// integralKernelS (src/SU2/SU2FrgCore.cpp:199-227) of a point's four buffers,
// added to the sums with the point's weight
__device__ __forceinline__ void add_ladder32(double &as, double &ad, float c, Bundle32 a0, Bundle32 a1, Bundle32 a2,
                                             Bundle32 a3) {
  const float h = fmaf(a0.s, a1.s, a2.s * a3.s);
  const float x = fmaf(a0.d, a1.s, fmaf(a2.d, a3.s, fmaf(a0.s, a1.d, a2.s * a3.d)));
  as += (double)(c * fmaf(-0.5f, h, x));
  ad += (double)(c * fmaf(0.1875f, h, fmaf(a0.d, a1.d, a2.d * a3.d)));
}

constexpr int kSu32WaveBytes = 64 * 16 + 64 * 16 + kRhsPoints * 8;

template <int RHO, bool ASYM>
__global__ __launch_bounds__(64 * kRhsWaves, 4) void k_su32(const FlowDev *__restrict__ fl, int nflows, long long total) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const long long blk = xcd_position(blockIdx.x, kChunk);
  if (blk >= total) return;
  int f = 0;
  {
    int lo = 0, hi = nflows - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (fl[mid].su_base <= blk) lo = mid;
      else hi = mid - 1;
    }
    f = lo;
  }
  const FlowDev &F = fl[f];
  const int nw = F.nw, L = F.L;
  double *s_mesh = reinterpret_cast<double *>(lds_raw);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < nw; i += 64 * kRhsWaves) s_mesh[i] = F.mesh[i];
  __syncthreads();
  const int unit = (int)(blk - F.su_base) * kRhsWaves + wave;
  if (unit >= nw * (nw * (nw + 1) / 2 + nw)) return;
  const SuUnit un = su_unit(unit, nw);
  const int X = un.X, a = un.a, b = un.b, kind = un.kind, outs = un.outs;
  const SuShape sh = su_shape_of(L, RHO);
  const int sums = sh.slots * L * 16;
  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * (kSu32WaveBytes > sums ? kSu32WaveBytes : sums);
  int4 *s_off = reinterpret_cast<int4 *>(wl);
  float4 *s_w = reinterpret_cast<float4 *>(wl + 64 * 16);
  double *s_c = reinterpret_cast<double *>(wl + 64 * 32);

  const __amdgpu_buffer_rsrc_t rG =
      __builtin_amdgcn_make_buffer_rsrc((void *)F.G32, (short)0, (int)F.g32_bytes, 0x00020000);
  const int rowbytes = L * 8;
  const int slot0 = lane / sh.lps;
  const int lj = lane - slot0 * sh.lps;
  const bool active = slot0 < sh.slots;
  const int slot = active ? slot0 : sh.slots - 1;
  unsigned sr[RHO], sx[RHO];  // byte offsets of the sites, plain and exchanged
#pragma unroll
  for (int i = 0; i < RHO; ++i) {
    const int r = lj + i * sh.lps;
    const bool ok = active && r < L;
    sr[i] = ok ? (unsigned)F.site_rid[r] * 8u : kNoSite;
    sx[i] = ASYM ? (ok ? (unsigned)F.inv_rid[r] * 8u : kNoSite) : sr[i];
  }
  double a1s[RHO], a1d[RHO], a2s[RHO], a2d[RHO];
#pragma unroll
  for (int i = 0; i < RHO; ++i) a1s[i] = a1d[i] = a2s[i] = a2d[i] = 0.0;

  // producer role of a lane: point pe, pair pp (0: V0 / V2, 1: V1 / V3), argument pj
  const int pe = lane >> 2, pp = (lane >> 1) & 1, pj = lane & 1;
  double half;
  {
    const double xm = s_mesh[X], am = s_mesh[a], bm = s_mesh[b];
    half = 0.5 * (xm + ((pp ^ pj) ? am : -am) + (pj ? -bm : bm));
  }
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;

  auto points = [&](auto kind_c) {
    constexpr int KIND = decltype(kind_c)::value;
    constexpr bool U1 = KIND != 0, U2 = KIND == 1;  // U rule in the first, second result
    double wp_next = pe < n ? Wwp[pe] : 0.0, c_next = pe < n ? Wc[pe] : 0.0;
    for (int e0 = 0; e0 < n; e0 += sh.nb) {
      const int nvalid = n - e0 < sh.nb ? n - e0 : sh.nb;
      {
        const double v = half + wp_next, c = c_next;
        const Bracket t = bracket_of(s_mesh, nw, fabs(v), F.geo, F.ga, F.gb);
        Bracket o;
        o.lo = pair_swap(t.lo);
        o.step = pair_swap(t.step);
        o.b = pair_swap(t.b);
        const bool ok = pe < nvalid;
        int4 d = make_int4((int)kNoRow, (int)kNoRow, 0, 0);
        float4 w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (ok) {
          const SuBuffer sb = su_buffer(t, o, X, nw, rowbytes, KIND == 1 ? 1 : 0);
          d = make_int4(sb.x, sb.y, sb.z, sb.diag);
          w = make_float4((float)sb.wa.x, (float)sb.wa.y, (float)sb.wb.x, (float)sb.wb.y);
          if (ASYM) {
            const double vo = pair_swap(v);
            const bool pos = vo > 0, neg = vo < 0;
            d.w |= (pj ? neg : pos) ? 1 : 0;
            d.w |= (pj ? pos : neg) ? 2 : 0;  // the exchange of the first result's V0 / V2
          }
        }
        wave_lds_fence();
        s_off[lane] = d;
        s_w[lane] = w;
        if (pp == 0 && pj == 0) s_c[pe] = ok ? c : 0.0;
        const int en = e0 + sh.nb + pe;
        wp_next = en < n ? Wwp[en] : 0.0;
        c_next = en < n ? Wc[en] : 0.0;
        wave_lds_fence();
      }
      for (int eb = 0; eb < nvalid; eb += sh.slots) {
        const int e = eb + slot;
        const float c = (float)s_c[e];
#pragma unroll
        for (int i = 0; i < RHO; ++i) {
          // all supports of the point's buffers V0, V2, V1, V3 (second result's names)
          float2 v[4][4], x[ASYM ? 2 : 1][4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int4 d = s_off[4 * e + k];
            const unsigned site = ASYM && (d.w & 1) ? sx[i] : sr[i];
            v[k][0] = buf_load<float2>(rG, d.x + site);
            v[k][1] = buf_load<float2>(rG, d.x + site + d.z);
            v[k][2] = buf_load<float2>(rG, d.y + site);
            v[k][3] = buf_load<float2>(rG, d.y + site + d.z);
            if (ASYM && k < 2) {
              const unsigned other = (d.w & 2) ? sx[i] : sr[i];
              x[k][0] = buf_load<float2>(rG, d.x + other);
              x[k][1] = buf_load<float2>(rG, d.x + other + d.z);
              x[k][2] = buf_load<float2>(rG, d.y + other);
              x[k][3] = buf_load<float2>(rG, d.y + other + d.z);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          // bundles of the second and of the first result
          Bundle32 b2[4], b1[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float4 w = s_w[4 * e + k];
            auto of = [&](const float2 (&q)[4], const float4 &g, bool u) {
              return u ? Bundle32{spin_chain(g.x, g.z, g.y, g.w, q[0], q[2], q[1], q[3]),
                                  density_chain(g.x, g.z, g.y, g.w, q[0], q[2], q[1], q[3])}
                       : Bundle32{spin_chain(g.x, g.y, g.z, g.w, q[0], q[1], q[2], q[3]),
                                  density_chain(g.x, g.y, g.z, g.w, q[0], q[1], q[2], q[3])};
            };
            b2[k] = of(v[k], w, U2);
            if constexpr (KIND == 2) {
              // the first result's rule on diagonal supports
              const int dg = s_off[4 * e + k].w;
              float4 g = w;
              if (dg & 4) {
                g.x = -g.x;
                g.y = -g.y;
              }
              if (dg & 8) {
                g.z = -g.z;
                g.w = -g.w;
              }
              b1[k] = ASYM && k < 2 ? of(x[ASYM ? k & 1 : 0], g, true) : of(v[k], g, true);
            } else {
              b1[k] = ASYM && k < 2 ? of(x[ASYM ? k & 1 : 0], w, U1) : b2[k];
            }
          }
          if (outs & 2) {
            if (U2) add_ladder32(a2s[i], a2d[i], c, b2[1], b2[3], b2[0], b2[2]);
            else add_ladder32(a2s[i], a2d[i], c, b2[0], b2[2], b2[1], b2[3]);
          }
          if (outs & 1) {
            if (U1) add_ladder32(a1s[i], a1d[i], c, b1[0], b1[3], b1[1], b1[2]);
            else add_ladder32(a1s[i], a1d[i], c, b1[1], b1[2], b1[0], b1[3]);
          }
          reread_lds();
        }
      }
    }
  };
  if (kind == 0) points(std::integral_constant<int, 0>{});
  else if (kind == 1) points(std::integral_constant<int, 1>{});
  else points(std::integral_constant<int, 2>{});

  // sum over the slots; results: (t = b, o = a), then (t = a, o = b)
  double *s_red = reinterpret_cast<double *>(wl);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (!(outs & (r ? 2 : 1))) continue;
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < RHO; ++i) {
      const int site = lj + i * sh.lps;
      if (active && site < L)
        reinterpret_cast<double2 *>(s_red)[slot * L + site] =
            r ? make_double2(a2s[i], a2d[i]) : make_double2(a1s[i], a1d[i]);
    }
    wave_lds_fence();
    const bool urule = un.u_rule(r);
    double *out = reinterpret_cast<double *>(F.dG + (size_t)un.item(r, nw) * L);
    for (int k = lane; k < 2 * L; k += 64) {
      double v = 0.0;
      for (int z = 0; z < sh.slots; ++z) v += s_red[z * 2 * L + k];
      unsafeAtomicAdd(out + k, (urule && (k & 1)) ? -v : v);
    }
  }
}
inline int su32_wave_bytes(int L, int rho) {
  const int sums = su_shape_of(L, rho).slots * L * 16;
  return kSu32WaveBytes > sums ? kSu32WaveBytes : sums;
}

// T channel and the final sum, eight points at a time in the operand layout
// of the matrix instructions (k_t); the bubble's products are exact in FP64
template <int FT, int HT, bool ASYM>
__global__ __launch_bounds__(64 * kRhsWaves, FT + HT == 1 ? 4 : 3) void k_t32(const FlowDev *__restrict__ fl, int nflows, long long total) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  constexpr int NT = FT + HT;
  const long long blk = xcd_position(blockIdx.x, kChunk);
  if (blk >= total) return;
  int f = 0;
  {
    int lo = 0, hi = nflows - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (fl[mid].t_base <= blk) lo = mid;
      else hi = mid - 1;
    }
    f = lo;
  }
  const FlowDev &F = fl[f];
  const int nw = F.nw, L = F.L;
  double *s_mesh = reinterpret_cast<double *>(lds_raw);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < nw; i += 64 * kRhsWaves) s_mesh[i] = F.mesh[i];
  __syncthreads();
  // items t-major: neighbouring waves share the mesh slab of their exact t
  const int nsu = nw * (nw + 1) / 2;
  const int pos = (int)(blk - F.t_base) * kRhsWaves + wave;
  if (pos >= nsu * nw) return;
  const int X = pos / nsu, su = pos - X * nsu;
  const int so = __builtin_amdgcn_readfirstlane(tri_decode(su));
  const int uo = su - so * (so + 1) / 2;
  const int item = su * nw + X;

  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * t_wave_bytes(L);
  int4 *s_off = reinterpret_cast<int4 *>(wl);              // [(point, pair)]
  float4 *s_w = reinterpret_cast<float4 *>(wl + 512);      // [(point, pair)]
  float4 *s_loc = reinterpret_cast<float4 *>(wl + 1024);   // [point][2]: factors of k = 4, 5; 6, 7
  int2 *s_fl = reinterpret_cast<int2 *>(wl + 1536);        // [(point, pair)]
  double *s_c = reinterpret_cast<double *>(wl + 1792);

  const __amdgpu_buffer_rsrc_t rG =
      __builtin_amdgcn_make_buffer_rsrc((void *)F.G32, (short)0, (int)F.g32_bytes, 0x00020000);
  const int rowbytes = L * 8;
  unsigned sr[NT], sx[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    const int r = k < FT ? 16 * k + (lane & 15) : 16 * FT + (lane & 7);
    sr[k] = r < L ? (unsigned)F.site_rid[r] * 8u : kNoSite;
    sx[k] = ASYM ? (r < L ? (unsigned)F.inv_rid[r] * 8u : kNoSite) : sr[k];
  }
  double rs[NT], rd[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) rs[k] = rd[k] = 0.0;
  BubbleTiles<FT, HT> C;
  C.clear();

  // producer role: point pe, pair pp, argument pj: A (pj 0) and B (pj 1) of
  // pair 0: A = w1 - w', B = w1p + w'; pair 1: A = w2p - w', B = w2 + w'
  const int pe = lane >> 2, pp = (lane >> 1) & 1, pj = lane & 1;
  double half;
  {
    const double s = s_mesh[so], t = s_mesh[X], u = s_mesh[uo];
    half = 0.5 * (s + (pj ? t : -t) + (pp ? -u : u));
  }
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;
  double wp_next = pe < n ? Wwp[pe] : 0.0, c_next = pe < n ? Wc[pe] : 0.0;

  for (int e0 = 0; e0 < n; e0 += kRhsPoints) {
    const int nvalid = n - e0 < kRhsPoints ? n - e0 : kRhsPoints;
    {
      const double c = c_next;
      const double v = pj ? half + wp_next : half - wp_next;
      const Bracket me = bracket_of(s_mesh, nw, fabs(v), F.geo, F.ga, F.gb);
      Bracket ot;
      ot.lo = pair_swap(me.lo);
      ot.step = pair_swap(me.step);
      ot.b = pair_swap(me.b);
      const double vo = pair_swap(v);
      const bool ok = pe < nvalid;
      int2 off = make_int2((int)kNoRow, (int)kNoRow);
      float2 w = make_float2(0.0f, 0.0f);
      int flag = 0;
      float fs = 0.0f, fd = 0.0f;
      if (ok) {
        // the pair's second buffer (s slot |B|, u slot |A|); lane pj describes
        // the supports of A's index pj
        const Bracket A = pj ? ot : me, B = pj ? me : ot;
        const int ia = A.lo + (pj ? A.step : 0), b0 = B.lo, b1 = B.lo + B.step;
        off.x = ((b0 > ia ? tri(b0, ia) : tri(ia, b0)) * nw + X) * rowbytes;
        off.y = ((b1 > ia ? tri(b1, ia) : tri(ia, b1)) * nw + X) * rowbytes;
        const double wa = pj ? A.b : 1.0 - A.b;
        const float w0 = (float)(wa * (1.0 - B.b)), w1 = (float)(wa * B.b);
        w.x = b0 < ia ? -w0 : w0;
        w.y = b1 < ia ? -w1 : w1;
        flag = (b0 == ia ? 4 : 0) | (b1 == ia ? 8 : 0);
        if (ASYM) {
          const double av = pj ? vo : v, bv = pj ? v : vo;
          const bool ex0 = (av < 0) != (pp ? bv > 0 : bv < 0);  // the pair's first buffer
          const bool ex1 = (bv < 0) != (pp ? av > 0 : av < 0);
          flag |= (ex1 ? 1 : 0) | (ex0 != ex1 ? 2 : 0);
        }
        // site-local vertex (u slot exact) with the same brackets: s slot this
        // lane's argument, t slot the other's; site 0, no exchange
        // (SU2VertexTwoParticle::getValueLocal, src/SU2/SU2VertexTwoParticle.hpp:347-360)
        float vs = 0.0f, vd = 0.0f;
        float2 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int is = me.lo + ((q & 1) ? me.step : 0), it = ot.lo + ((q & 2) ? ot.step : 0);
          x[q] = buf_load<float2>(rG, ((is > X ? tri(is, X) : tri(X, is)) * nw + it) * rowbytes);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int is = me.lo + ((q & 1) ? me.step : 0);
          const float wl = (float)(((q & 2) ? ot.b : 1.0 - ot.b) * ((q & 1) ? me.b : 1.0 - me.b));
          vs = fmaf(wl, x[q].x, vs);
          vd = fmaf(is < X ? -wl : wl, x[q].y, vd);
        }
        fs = fmaf(0.25f, vs, -vd);
        fd = -fmaf(0.75f, vs, vd);
      }
      wave_lds_fence();
      reinterpret_cast<int2 *>(s_off)[lane] = off;
      reinterpret_cast<float2 *>(s_w)[lane] = w;
      reinterpret_cast<int *>(s_fl)[lane] = flag;
      // factors of the first buffers (k = 4, 5: pj 0 of pair 1, pair 0), then of the second ones
      reinterpret_cast<float2 *>(s_loc)[4 * pe + 2 * pj + 1 - pp] = make_float2(fs, fd);
      if (pp == 0 && pj == 0) s_c[pe] = ok ? c : 0.0;
      const int en = e0 + kRhsPoints + pe;
      wp_next = en < n ? Wwp[en] : 0.0;
      c_next = en < n ? Wc[en] : 0.0;
      wave_lds_fence();
    }
    for (int eb = 0; eb < nvalid; eb += 8) {
      // gathers one tile of sites, e the lane's point: (c A2, A3) per channel
      auto gather = [&](int k, int e, double (&P)[2], double (&Q)[2]) {
        float2 v[2][4];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int4 o = s_off[2 * e + p];
          const unsigned site = ASYM && (s_fl[2 * e + p].x & 1) ? sx[k] : sr[k];
          v[p][0] = buf_load<float2>(rG, o.x + site);
          v[p][1] = buf_load<float2>(rG, o.y + site);
          v[p][2] = buf_load<float2>(rG, o.z + site);
          v[p][3] = buf_load<float2>(rG, o.w + site);
        }
        __builtin_amdgcn_sched_barrier(0);
        const float c = (float)s_c[e];
        Bundle32 first[2], second[2];
        // the pair's first buffer: the interpolations in the other order, the
        // density sign of the other exchange
        auto image = [&](int p, const float4 &w, const float2 (&x)[4]) {
          const int2 g = s_fl[2 * e + p];
          const float m0 = (g.x & 4) ? w.x : -w.x, m1 = (g.x & 8) ? w.y : -w.y;
          const float m2 = (g.y & 4) ? w.z : -w.z, m3 = (g.y & 8) ? w.w : -w.w;
          return Bundle32{spin_chain(m0, m2, m1, m3, x[0], x[2], x[1], x[3]),
                          density_chain(m0, m2, m1, m3, x[0], x[2], x[1], x[3])};
        };
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float4 w = s_w[2 * e + p];
          second[p] = Bundle32{spin_chain(w.x, w.y, w.z, w.w, v[p][0], v[p][1], v[p][2], v[p][3]),
                               density_chain(w.x, w.y, w.z, w.w, v[p][0], v[p][1], v[p][2], v[p][3])};
          first[p] = image(p, w, v[p]);
          if (ASYM) {
            settle(second[p].s, second[p].d);
            settle(first[p].s, first[p].d);
          }
        }
        if (ASYM) {
          // an argument of exactly zero: the first buffer exchanges the sites
          // the other way.  After the rest and as a branch of the whole wave: a
          // lane's own branch that replaced supports still in use kept both
          // gathers of every tile in registers (157 spilled at 26 sites)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const int gx = s_fl[2 * e + p].x;
            if (__any(gx & 2)) {
              const int4 o = s_off[2 * e + p];
              const unsigned site = (gx & 1) ? sr[k] : sx[k];
              const float2 x[4] = {buf_load<float2>(rG, o.x + site), buf_load<float2>(rG, o.y + site),
                                   buf_load<float2>(rG, o.z + site), buf_load<float2>(rG, o.w + site)};
              const Bundle32 f = image(p, s_w[2 * e + p], x);
              if (gx & 2) first[p] = f;
            }
          }
        }
        const float4 l0 = s_loc[2 * e], l1 = s_loc[2 * e + 1];
        rs[k] += (double)(c * fmaf(l0.x, first[0].s, fmaf(l0.z, first[1].s, fmaf(l1.x, second[0].s, l1.z * second[1].s))));
        rd[k] += (double)(c * fmaf(l0.y, first[0].d, fmaf(l0.w, first[1].d, fmaf(l1.y, second[0].d, l1.w * second[1].d))));
        P[0] = (double)(c * second[0].s);
        P[1] = (double)(c * second[0].d);
        Q[0] = (double)second[1].s;
        Q[1] = (double)second[1].d;
        reread_lds();
      };
      double ph[2], qh[2];
      if (HT) {
        gather(FT, eb + (lane >> 3), ph, qh);
        C.half(ph, qh);
      }
      // the full tiles' even points, then the odd ones
#pragma unroll
      for (int par = 0; par < (FT ? 2 : 0); ++par) {
        double P[FT ? FT : 1][2], Q[FT ? FT : 1][2];
#pragma unroll
        for (int i = 0; i < FT; ++i) gather(i, eb + 2 * (lane >> 4) + par, P[i], Q[i]);
        C.full(par, P, Q, ph, qh);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  t_finish<true, FT, HT>(F, C, rs, rd, wl, item, 2 * F.flags[4]);
}
