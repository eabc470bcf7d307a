// dGamma/dLambda of the XYZ core by waves.  Included by xyz_flow.hip after the
// flow descriptor XyzDev (wave_rhs.h before it).
//
// The S, T and U integrals have the structure described in su2_rhs.h: the U
// integrals are images of the S ones, the bundles of a unit (X, {a, b}) serve
// two items (V0 and V2 with the site exchange inverted in the first), and the
// buffers of a T pair are images of each other.  Exchanged bundles read site
// rid' = inv_rid of a site through another spin permutation.  Every stored
// site is gathered once, and the lanes hold a site together with its inverse,
// so that both exchange states of a bundle come from the lane's registers.
// This needs site_rid[r] = r and inv_rid to be an involution, which every
// lattice of the factory has; other tables run the general kernels.
//
// What bounds it: the gathers (k_xyz_su: 86 % of its time at 16.5 cycles each), and
// in k_xyz_t the alternation of gathers (44 %) and matrix instructions (28 % of its
// time) between barriers.  Honeycomb Heisenberg-Kitaev, 23 sites, 64
// frequencies, against one workgroup per item with a producer wave: 8.78 ->
// 3.86 ms at cutoff 20, 23.5 -> 10.2 ms at 0.7, 38.3 -> 15.6 ms at 0.02 (k_xyz_su
// 6.1 ms, k_xyz_t 9.4 ms).
#pragma once

constexpr int kMaxXyzRhsL = 32;
constexpr int kXyzMaxTiles = 10;  // bubble tiles per wave of k_xyz_t

// lanes of a point: a pair of sites each, r and its inverse where they differ
struct XyzLane {
  int a, b;    // sites (-1: none)
  int pa, pb;  // spin permutations of a and b: plain | exchanged << 6 (2 bits per component); bit 12 of pb: b is a's inverse
};

struct XyzShape {
  int lps, slots, nb;
};
__host__ __device__ inline XyzShape xyz_shape(int lps) {
  XyzShape s;
  s.lps = lps;
  s.slots = 64 / lps < kRhsPoints ? 64 / lps : kRhsPoints;
  s.nb = s.slots * (kRhsPoints / s.slots);
  return s;
}

struct Vec4 {
  double x, y, z, d;
};
// the four supports of a buffer at one site (components X, Y and Z, D).  Lanes
// without a point or without a second site read what a neighbour reads and keep
// nothing of it: an offset past the vertex could wrap with the half row added.
struct Quad4 {
  double2 a[4], b[4];
};
__device__ __forceinline__ Quad4 load_quad4(__amdgpu_buffer_rsrc_t r, int o0, int o1, int o2, int o3, unsigned site,
                                            unsigned half) {
  const unsigned o[4] = {o0 + site, o1 + site, o2 + site, o3 + site};
  Quad4 q;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q.a[i] = buf_load<double2>(r, o[i]);
    q.b[i] = buf_load<double2>(r, o[i] + half);
  }
  return q;
}
__device__ __forceinline__ void settle4(Vec4 &v) {
  settle(v.x, v.y);
  settle(v.z, v.d);
}
// stored weights carry the density sign; spin weights are their absolute values
__device__ __forceinline__ Vec4 interpolate4(double2 wa, double2 wb, const Quad4 &q) {
  const double w[4] = {wa.x, wa.y, wb.x, wb.y};
  Vec4 v{fabs(w[0]) * q.a[0].x, fabs(w[0]) * q.a[0].y, fabs(w[0]) * q.b[0].x, w[0] * q.b[0].y};
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    v.x = fma(fabs(w[i]), q.a[i].x, v.x);
    v.y = fma(fabs(w[i]), q.a[i].y, v.y);
    v.z = fma(fabs(w[i]), q.b[i].x, v.z);
    v.d = fma(w[i], q.b[i].y, v.d);
  }
  settle4(v);
  return v;
}
__device__ __forceinline__ double pick3v(const Vec4 &v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }
// bundle of one site of a lane: raw its stored values, inv those of its inverse
__device__ __forceinline__ Vec4 bundle4(const Vec4 &raw, const Vec4 &inv, bool ex, int perms) {
  const Vec4 s{ex ? inv.x : raw.x, ex ? inv.y : raw.y, ex ? inv.z : raw.z, ex ? inv.d : raw.d};
  const int pm = ex ? perms >> 6 : perms;
  return Vec4{pick3v(s, pm & 3), pick3v(s, (pm >> 2) & 3), pick3v(s, (pm >> 4) & 3), s.d};
}
__device__ __forceinline__ Vec4 scaled(const Vec4 &v, double c) { return Vec4{c * v.x, c * v.y, c * v.z, c * v.d}; }
// ladder of two bundles (src/XYZ/XYZFrgCore.cpp:223-275): spin output c gets
// a_d b_c + a_c b_d - (a_c1 b_c2 + a_c2 b_c1), the density the scalar product
__device__ __forceinline__ void add_ladder(Vec4 &s, const Vec4 &a, const Vec4 &b) {
  s.x = fma(a.d, b.x, fma(a.x, b.d, fma(-a.z, b.y, fma(-a.y, b.z, s.x))));
  s.y = fma(a.d, b.y, fma(a.y, b.d, fma(-a.z, b.x, fma(-a.x, b.z, s.y))));
  s.z = fma(a.d, b.z, fma(a.z, b.d, fma(-a.x, b.y, fma(-a.y, b.x, s.z))));
  s.d = fma(a.d, b.d, fma(a.x, b.x, fma(a.y, b.y, fma(a.z, b.z, s.d))));
}

constexpr int kXyzSuWaveBytes = 64 * 64;  // descriptors (3200 bytes), then the sums of a result

// adds the S and U integrals of all items to dG (zeroed before); two additions
// to each value, so their order does not matter.  The second site's loads are
// issued after the first site's are used: 162 registers, three waves per SIMD,
// 1 to 5 % faster than both at once with two.
__global__ __launch_bounds__(64 * kRhsWaves, 3) void k_xyz_su(XyzDev F, long long total) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const long long blk = xcd_position(blockIdx.x, kXyzChunk);
  if (blk >= total) return;
  const int nw = F.nw, L = F.L;
  double *s_mesh = reinterpret_cast<double *>(lds_raw);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < nw; i += 64 * kRhsWaves) s_mesh[i] = F.mesh[i];
  __syncthreads();
  const int unit = (int)blk * kRhsWaves + wave;
  if (unit >= nw * (nw * (nw + 1) / 2 + nw)) return;
  const SuUnit un = su_unit(unit, nw);
  const int X = un.X, kind = un.kind, outs = un.outs;
  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * kXyzSuWaveBytes;
  int4 *s_off = reinterpret_cast<int4 *>(wl);
  double2 *s_wa = reinterpret_cast<double2 *>(wl + 64 * 16);
  double2 *s_wb = s_wa + 64;
  double *s_c = reinterpret_cast<double *>(wl + 64 * 48);

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 32;
  const unsigned halfrow = L * 16;  // the Z, D half of a row
  const XyzShape sh = xyz_shape(F.lps);
  const int slot0 = lane / sh.lps, lj = lane - slot0 * sh.lps;
  const bool active = slot0 < sh.slots;
  const int slot = active ? slot0 : sh.slots - 1;
  const XyzLane ln = F.lanes[lj];
  const bool cyc = (ln.pb >> 12) & 1;
  const unsigned sa = (unsigned)ln.a * 16u, sb = ln.b >= 0 ? (unsigned)ln.b * 16u : sa;
  // first result (t = b, o = a), second (t = a, o = b); sites a, b of the lane
  Vec4 r1[2], r2[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) r1[i] = r2[i] = Vec4{0.0, 0.0, 0.0, 0.0};

  const int pe = lane >> 2, pp = (lane >> 1) & 1, pj = lane & 1;
  double half;
  {
    const double xm = s_mesh[X], am = s_mesh[un.a], bm = s_mesh[un.b];
    half = 0.5 * (xm + ((pp ^ pj) ? am : -am) + (pj ? -bm : bm));
  }
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;
  const int rule = kind == 1 ? 1 : 0;

  auto points = [&](auto mixed_c) {
    constexpr bool MIXEDKIND = decltype(mixed_c)::value;
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
        const double vo = pair_swap(v);
        const bool ok = pe < nvalid;
        int4 d = make_int4((int)kNoRow, (int)kNoRow, 0, 0);
        double2 wa = make_double2(0.0, 0.0), wb = wa;
        if (ok) {
          const SuBuffer b = su_buffer(t, o, X, nw, rowbytes, rule);
          // bit 0: site exchange of the second result, bit 1: of the first one's V0 / V2
          const bool pos = vo > 0, neg = vo < 0;
          d = make_int4(b.x, b.y, b.z, b.diag | ((pj ? neg : pos) ? 1 : 0) | ((pj ? pos : neg) ? 2 : 0));
          wa = b.wa;
          wb = b.wb;
        }
        wave_lds_fence();
        s_off[lane] = d;
        s_wa[lane] = wa;
        s_wb[lane] = wb;
        if (pp == 0 && pj == 0) s_c[pe] = ok ? c : 0.0;
        const int en = e0 + sh.nb + pe;
        wp_next = en < n ? Wwp[en] : 0.0;
        c_next = en < n ? Wc[en] : 0.0;
        wave_lds_fence();
      }
      for (int eb = 0; eb < nvalid; eb += sh.slots) {
        const int e = eb + slot;
        const double c = s_c[e];
        Vec4 p[2][2];     // V1, V3 times the point's coefficient, per site
        double g[2][2];   // their density under the first result's rule
        // V1 and V3 (k = 2, 3) first: factors of V0 and V2 (k = 0, 1)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int k = kk ^ 2;
          reread_lds();
          const int4 d = s_off[4 * e + k];
          const Quad4 qa = load_quad4(rG, d.x, d.x + d.z, d.y, d.y + d.z, sa, halfrow);
          __builtin_amdgcn_sched_barrier(0);
          const double2 wa = s_wa[4 * e + k], wb = s_wb[4 * e + k];
          const Vec4 va = interpolate4(wa, wb, qa);
          double fa = va.d;
          bool dg = false;
          if (MIXEDKIND) {
            dg = __any(d.w & 12);
            if (dg)
              fa = fma(-2.0, ((d.w & 4) ? fma(wa.y, qa.b[1].y, wa.x * qa.b[0].y) : 0.0) +
                                 ((d.w & 8) ? fma(wb.y, qa.b[3].y, wb.x * qa.b[2].y) : 0.0), fa);
          }
          __builtin_amdgcn_sched_barrier(0);
          const Quad4 qb = load_quad4(rG, d.x, d.x + d.z, d.y, d.y + d.z, sb, halfrow);
          const Vec4 vb = interpolate4(wa, wb, qb);
          double fb = vb.d;
          if (MIXEDKIND) {
            if (dg)
              fb = fma(-2.0, ((d.w & 4) ? fma(wa.y, qb.b[1].y, wa.x * qb.b[0].y) : 0.0) +
                                 ((d.w & 8) ? fma(wb.y, qb.b[3].y, wb.x * qb.b[2].y) : 0.0), fb);
          }
          const Vec4 &ia = cyc ? vb : va, &ib = cyc ? va : vb;
          const bool ex = d.w & 1;
          if (kk < 2) {
            p[kk][0] = scaled(bundle4(va, ia, ex, ln.pa), c);
            p[kk][1] = scaled(bundle4(vb, ib, ex, ln.pb), c);
            if (MIXEDKIND) {
              g[kk][0] = c * (ex && cyc ? fb : fa);
              g[kk][1] = c * (ex && cyc ? fa : fb);
            }
          } else {
            if (outs & 2) {
              add_ladder(r2[0], bundle4(va, ia, ex, ln.pa), p[k][0]);
              add_ladder(r2[1], bundle4(vb, ib, ex, ln.pb), p[k][1]);
            }
            if (outs & 1) {
              const bool ef = d.w & 2;
              Vec4 x = bundle4(va, ia, ef, ln.pa), y = bundle4(vb, ib, ef, ln.pb);
              Vec4 px = p[1 - k][0], py = p[1 - k][1];
              if (MIXEDKIND) {
                x.d = ef && cyc ? fb : fa;
                y.d = ef && cyc ? fa : fb;
                px.d = g[1 - k][0];
                py.d = g[1 - k][1];
              }
              add_ladder(r1[0], x, px);
              add_ladder(r1[1], y, py);
            }
          }
        }
      }
    }
  };
  if (kind == 2) points(std::true_type{});
  else points(std::false_type{});

  double *s_red = reinterpret_cast<double *>(wl);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (!(outs & (r ? 2 : 1))) continue;
    wave_lds_fence();
    if (active) {
      const Vec4 &x = r ? r2[0] : r1[0], &y = r ? r2[1] : r1[1];
      double2 *o = reinterpret_cast<double2 *>(s_red) + 2 * slot * L;
      o[ln.a] = make_double2(x.x, x.y);
      o[L + ln.a] = make_double2(x.z, x.d);
      if (ln.b >= 0) {
        o[ln.b] = make_double2(y.x, y.y);
        o[L + ln.b] = make_double2(y.z, y.d);
      }
    }
    wave_lds_fence();
    const bool urule = un.u_rule(r);
    double *out = F.dG + (size_t)un.item(r, nw) * L * 4;
    for (int k = lane; k < 4 * L; k += 64) {
      double v = 0.0;
      for (int z = 0; z < sh.slots; ++z) v += s_red[z * 4 * L + k];
      unsafeAtomicAdd(out + k, (urule && k >= 2 * L && (k & 1)) ? -v : v);
    }
  }
}

// ---------------------------------------------------------------------------
// T channel and the final sum
// ---------------------------------------------------------------------------
// A workgroup of four waves evaluates the T channel of an item, the points
// dealt to the waves in turn.  The lattice bubble is linear in the products
// P[a][r1] Q[b][r2] of the pair's bundles (spin components a, b): the waves
// write P = c A0 and Q = A1 of their points to LDS and accumulate the 16 x 16
// tiles of the 4 L x 4 L product matrix that the overlap lists refer to, each
// wave its own tiles, on the matrix cores.  Three waves per SIMD although up to
// 28 tiles then spill 23 registers and more 96: 2 to 15 % faster than two.
// density of a T buffer on its diagonal supports
__device__ __forceinline__ double diagonal4(int2 fl, double2 wa, double2 wb, const Quad4 &q) {
  const double m0 = (fl.x & 4) ? wa.x : 0.0, m1 = (fl.x & 8) ? wa.y : 0.0;
  const double m2 = (fl.y & 4) ? wb.x : 0.0, m3 = (fl.y & 8) ? wb.y : 0.0;
  return fma(m3, q.b[3].y, fma(m2, q.b[2].y, fma(m1, q.b[1].y, m0 * q.b[0].y)));
}
constexpr int kXyzTDesc = 512 + 1024 + 1024 + 1024 + 256 + 128;  // off, w, factors, images, flags, c
__host__ __device__ inline int xyz_t_stride(int L) {  // row stride of P, Q (doubles): an odd multiple of 16
  const int t = (4 * L + 15) / 16;
  return 16 * (t | 1);
}
// The tiles pass through LDS sixteen at a time for the overlap sums: all at
// once would leave one workgroup per CU (28 tiles at L = 23).
constexpr int kXyzPassTiles = 16;
// bytes of LDS: mesh, then descriptors and P, Q; after the points the sums of
// the lanes, then a pass of tiles and the partial overlap sums
__host__ __device__ inline int xyz_t_lds(int nw, int L, int lps) {
  const int slots = xyz_shape(lps).slots;
  const int pq = kRhsWaves * kXyzTDesc + 2 * kRhsWaves * slots * xyz_t_stride(L) * 8;
  const int c = kXyzPassTiles * 256 * 8 + 256 * 8, acc = kRhsWaves * slots * L * 32;
  return ((nw * 8 + 15) & ~15) + (pq > c ? (pq > acc ? pq : acc) : (c > acc ? c : acc));
}

template <int TPW>
__global__ __launch_bounds__(64 * kRhsWaves, 3) void k_xyz_t(XyzDev F) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int nw = F.nw, L = F.L;
  const int nsu = nw * (nw + 1) / 2;
  const long long pos = xcd_position(blockIdx.x, kXyzChunk);
  if (pos >= (long long)nsu * nw) return;
  // items t-major: neighbouring workgroups share the mesh slab of their exact t
  const int X = (int)(pos / nsu), su = (int)(pos - (long long)X * nsu);
  const int so = __builtin_amdgcn_readfirstlane(tri_decode(su)), uo = su - so * (so + 1) / 2;
  const size_t item = (size_t)su * nw + X;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double *s_mesh = reinterpret_cast<double *>(lds_raw);
  const int pe = lane >> 2;
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;
  const int pt = kRhsWaves * pe + wave;  // point of the lane within the team's batch
  double wp_next = pt < n ? Wwp[pt] : 0.0, c_next = pt < n ? Wc[pt] : 0.0;
  for (int i = tid; i < nw; i += 64 * kRhsWaves) s_mesh[i] = F.mesh[i];
  __syncthreads();

  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * kXyzTDesc;
  int2 *s_off = reinterpret_cast<int2 *>(wl);               // [(point, pair) * 2 + half]
  double2 *s_w = reinterpret_cast<double2 *>(wl + 512);     // [(point, pair) * 2 + half]
  double4 *s_f = reinterpret_cast<double4 *>(wl + 1536);    // [(point, pair)] factors of the bundle
  double4 *s_g = reinterpret_cast<double4 *>(wl + 2560);    // [(point, pair)] factors of its image
  int *s_fl = reinterpret_cast<int *>(wl + 3584);
  double *s_c = reinterpret_cast<double *>(wl + 3840);
  const int stride = xyz_t_stride(L);
  const XyzShape sh = xyz_shape(F.lps);
  const int team = kRhsWaves * sh.slots;  // points per step of the workgroup
  double *s_P = reinterpret_cast<double *>(lds_raw + ((nw * 8 + 15) & ~15) + kRhsWaves * kXyzTDesc);
  double *s_Q = s_P + team * stride;

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 32;
  const unsigned halfrow = L * 16;  // the Z, D half of a row
  const int slot0 = lane / sh.lps, lj = lane - slot0 * sh.lps;
  const bool active = slot0 < sh.slots;
  const int slot = active ? slot0 : sh.slots - 1;
  const XyzLane ln = F.lanes[lj];
  const bool cyc = (ln.pb >> 12) & 1;
  const unsigned sa = (unsigned)ln.a * 16u, sb = ln.b >= 0 ? (unsigned)ln.b * 16u : sa;
  Vec4 acc[2];
  acc[0] = acc[1] = Vec4{0.0, 0.0, 0.0, 0.0};
  d4 C[TPW];
#pragma unroll
  for (int k = 0; k < TPW; ++k) C[k] = d4{0.0, 0.0, 0.0, 0.0};
  const int ntiles = F.ntiles;
  // the wave's tiles (uniform): rows and columns of their first elements
  int row[TPW], col[TPW];
#pragma unroll
  for (int k = 0; k < TPW; ++k) {
    const int tc = k * kRhsWaves + wave < ntiles ? F.tiles[k * kRhsWaves + wave] : 0;
    row[k] = __builtin_amdgcn_readfirstlane(tc & 0xffff);
    col[k] = __builtin_amdgcn_readfirstlane(tc >> 16);
  }
  const int kr = (lane >> 4) * stride + (lane & 15);

  // producer role: point pe of the wave, pair pp, argument pj: A (pj 0) and B
  // of pair 0: A = w1 - w', B = w1p + w'; pair 1: A = w2p - w', B = w2 + w'
  const int pp = (lane >> 1) & 1, pj = lane & 1;
  double half;
  {
    const double s = s_mesh[so], t = s_mesh[X], u = s_mesh[uo];
    half = 0.5 * (s + (pj ? t : -t) + (pp ? -u : u));
  }

  for (int e0 = 0; e0 < n; e0 += kRhsWaves * sh.nb) {
    {
      const double c = c_next;
      const double v = pj ? half + wp_next : half - wp_next;
      const Bracket me = bracket_of(s_mesh, nw, fabs(v), F.geo, F.ga, F.gb);
      Bracket ot;
      ot.lo = pair_swap(me.lo);
      ot.step = pair_swap(me.step);
      ot.b = pair_swap(me.b);
      const double vo = pair_swap(v);
      const bool ok = pe < sh.nb && e0 + pt < n;
      int2 off = make_int2((int)kNoRow, (int)kNoRow);
      double2 w = make_double2(0.0, 0.0);
      int flag = 0;
      Vec4 f{0.0, 0.0, 0.0, 0.0};
      if (ok) {
        // the pair's first buffer: s slot |A|, u slot |B|; lane pj describes
        // the supports of A's index pj
        const Bracket A = pj ? ot : me, B = pj ? me : ot;
        const int ia = A.lo + (pj ? A.step : 0), b0 = B.lo, b1 = B.lo + B.step;
        off.x = ((b0 > ia ? tri(b0, ia) : tri(ia, b0)) * nw + X) * rowbytes;
        off.y = ((b1 > ia ? tri(b1, ia) : tri(ia, b1)) * nw + X) * rowbytes;
        const double wa = pj ? A.b : 1.0 - A.b;
        const double w0 = wa * (1.0 - B.b), w1 = wa * B.b;
        w.x = ia < b0 ? -w0 : w0;
        w.y = ia < b1 ? -w1 : w1;
        const double av = pj ? vo : v, bv = pj ? v : vo;
        const bool ex0 = (av < 0) != (pp ? bv > 0 : bv < 0);  // the pair's first buffer
        const bool ex1 = (bv < 0) != (pp ? av > 0 : av < 0);  // its image
        flag = (b0 == ia ? 4 : 0) | (b1 == ia ? 8 : 0) | (ex0 ? 1 : 0) | (ex0 != ex1 ? 2 : 0);
        // site-local vertex (u slot exact) with the same brackets: s slot this
        // lane's argument, t slot the other's; site 0, no exchange
        // (XYZVertexTwoParticle.hpp:355-376), as chalice factors scaled by the
        // point's weight (XYZFrgCore.cpp:333-416): spin output k gets the two
        // other spin components with +, the component itself and the density
        // with -; the density output minus the sum
        Vec4 l{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int is = me.lo + (q ? me.step : 0);
          const double ws = q ? me.b : 1.0 - me.b;
          const int row = ((is > X ? tri(is, X) : tri(X, is)) * nw + ot.lo) * rowbytes;
          const double wl0 = ws * (1.0 - ot.b), wl1 = ws * ot.b;
          const double2 x0 = buf_load<double2>(rG, row), y0 = buf_load<double2>(rG, row + halfrow);
          const double2 x1 = buf_load<double2>(rG, row + ot.step * rowbytes);
          const double2 y1 = buf_load<double2>(rG, row + ot.step * rowbytes + halfrow);
          l.x = fma(wl1, x1.x, fma(wl0, x0.x, l.x));
          l.y = fma(wl1, x1.y, fma(wl0, x0.y, l.y));
          l.z = fma(wl1, y1.x, fma(wl0, y0.x, l.z));
          const double d = fma(wl1, y1.y, wl0 * y0.y);
          l.d += is < X ? -d : d;
        }
        const double spin = (l.x + l.y) + l.z;
        f = Vec4{c * (fma(-2.0, l.x, spin) - l.d), c * (fma(-2.0, l.y, spin) - l.d), c * (fma(-2.0, l.z, spin) - l.d),
                 -c * (l.d + spin)};
      }
      const Vec4 g{pair_swap(f.x), pair_swap(f.y), pair_swap(f.z), pair_swap(f.d)};
      wave_lds_fence();
      s_off[lane] = off;
      s_w[lane] = w;
      s_fl[lane] = flag;
      if (pj == 0) {
        // the other pair's first buffer A and its image (spin equal, density
        // negated): factors f + g for the spin, f - g for the density
        s_f[2 * pe + (1 - pp)] = make_double4(f.x + g.x, f.y + g.y, f.z + g.z, f.d - g.d);
        s_g[2 * pe + (1 - pp)] = make_double4(g.x, g.y, g.z, g.d);
        if (pp == 0) s_c[pe] = ok ? c : 0.0;
      }
      const int en = e0 + kRhsWaves * sh.nb + pt;
      wp_next = en < n ? Wwp[en] : 0.0;
      c_next = en < n ? Wc[en] : 0.0;
      wave_lds_fence();
    }
    const int left = (n - e0 + kRhsWaves - 1) / kRhsWaves;  // points of a wave, at most
    const int steps = ((left < sh.nb ? left : sh.nb) + sh.slots - 1) / sh.slots;
    for (int it = 0; it < steps; ++it) {
      const int e = it * sh.slots + slot;
      double *P = s_P + (wave * sh.slots + slot) * stride, *Q = s_Q + (wave * sh.slots + slot) * stride;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        reread_lds();
        const int4 o = reinterpret_cast<const int4 *>(s_off)[2 * e + p];
        const Quad4 qa = load_quad4(rG, o.x, o.y, o.z, o.w, sa, halfrow);
        __builtin_amdgcn_sched_barrier(0);
        const double2 wa = s_w[4 * e + 2 * p], wb = s_w[4 * e + 2 * p + 1];
        const int2 fl2 = reinterpret_cast<const int2 *>(s_fl)[2 * e + p];
        const bool special = __any((fl2.x | fl2.y) & 14);
        const Vec4 va = interpolate4(wa, wb, qa);
        double da = 0.0, db = 0.0;  // density on diagonal supports
        if (special) da = diagonal4(fl2, wa, wb, qa);
        __builtin_amdgcn_sched_barrier(0);
        const Quad4 qb = load_quad4(rG, o.x, o.y, o.z, o.w, sb, halfrow);
        const Vec4 vb = interpolate4(wa, wb, qb);
        if (special) db = diagonal4(fl2, wa, wb, qb);
        const double4 f = s_f[2 * e + p];
        const Vec4 &ia = cyc ? vb : va, &ib = cyc ? va : vb;
        const bool ex = fl2.x & 1;
        const Vec4 x = bundle4(va, ia, ex, ln.pa), y = bundle4(vb, ib, ex, ln.pb);
        acc[0].x = fma(f.x, x.x, acc[0].x);
        acc[0].y = fma(f.y, x.y, acc[0].y);
        acc[0].z = fma(f.z, x.z, acc[0].z);
        acc[0].d = fma(f.w, x.d, acc[0].d);
        acc[1].x = fma(f.x, y.x, acc[1].x);
        acc[1].y = fma(f.y, y.y, acc[1].y);
        acc[1].z = fma(f.z, y.z, acc[1].z);
        acc[1].d = fma(f.w, y.d, acc[1].d);
        if (special) {
          // the image's density is -d + 2 (diagonal supports, which keep their
          // sign); with an argument of exactly zero it exchanges the sites the
          // other way
          const double4 gf = s_g[2 * e + p];
          const bool ei = (fl2.x & 2) ? !ex : ex;
          acc[0].d = fma(2.0 * gf.w, ei && cyc ? db : da, acc[0].d);
          acc[1].d = fma(2.0 * gf.w, ei && cyc ? da : db, acc[1].d);
          if (fl2.x & 2) {
            const Vec4 xi = bundle4(va, ia, ei, ln.pa), yi = bundle4(vb, ib, ei, ln.pb);
            acc[0].x = fma(gf.x, xi.x - x.x, acc[0].x);
            acc[0].y = fma(gf.y, xi.y - x.y, acc[0].y);
            acc[0].z = fma(gf.z, xi.z - x.z, acc[0].z);
            acc[0].d = fma(-gf.w, xi.d - x.d, acc[0].d);
            acc[1].x = fma(gf.x, yi.x - y.x, acc[1].x);
            acc[1].y = fma(gf.y, yi.y - y.y, acc[1].y);
            acc[1].z = fma(gf.z, yi.z - y.z, acc[1].z);
            acc[1].d = fma(-gf.w, yi.d - y.d, acc[1].d);
          }
        }
        if (active) {
          double *D = p ? Q : P;
          const double c = p ? 1.0 : s_c[e];
          D[ln.a] = c * x.x;
          D[L + ln.a] = c * x.y;
          D[2 * L + ln.a] = c * x.z;
          D[3 * L + ln.a] = c * x.d;
          if (ln.b >= 0) {
            D[ln.b] = c * y.x;
            D[L + ln.b] = c * y.y;
            D[2 * L + ln.b] = c * y.z;
            D[3 * L + ln.b] = c * y.d;
          }
        }
      }
      __syncthreads();
      // four points at a time, a wave's tiles one after the other: their sums
      // are independent, so the matrix instructions follow one another
      for (int e4 = 0; e4 < team; e4 += 4) {
        const double *p = s_P + e4 * stride + kr, *q = s_Q + e4 * stride + kr;
        double x[TPW], y[TPW];
#pragma unroll
        for (int k = 0; k < TPW; ++k) {
          x[k] = p[row[k]];
          y[k] = q[col[k]];
        }
#pragma unroll
        for (int k = 0; k < TPW; ++k)
          if (k * kRhsWaves + wave < ntiles) C[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], y[k], C[k], 0, 0, 0);
      }
      __syncthreads();
    }
  }

  // lattice bubble (XYZFrgCore.cpp:295-322): 4 times the sum over the overlap
  // lists, then the points, the S and U values and the prefactor 1/(2 pi)
  // (XYZFrgCore.cpp:564-570)
  __syncthreads();
  unsigned char *area = lds_raw + ((nw * 8 + 15) & ~15);
  double *s_acc = reinterpret_cast<double *>(area);
  if (active) {
    double2 *o = reinterpret_cast<double2 *>(s_acc) + 2 * (wave * sh.slots + slot) * L;
    o[ln.a] = make_double2(acc[0].x, acc[0].y);
    o[L + ln.a] = make_double2(acc[0].z, acc[0].d);
    if (ln.b >= 0) {
      o[ln.b] = make_double2(acc[1].x, acc[1].y);
      o[L + ln.b] = make_double2(acc[1].z, acc[1].d);
    }
  }
  double *out = F.dG + item * L * 4 + tid;
  const double su_sum = tid < 4 * L ? *out : 0.0;
  __syncthreads();
  double v = 0.0, rpa = 0.0;
  if (tid < 4 * L)
    for (int z = 0; z < team; ++z) v += s_acc[z * 4 * L + tid];
  double *s_C = reinterpret_cast<double *>(area), *s_part = s_C + kXyzPassTiles * 256;
  const int *plan = F.plan;
#pragma unroll
  for (int k0 = 0; k0 < TPW; k0 += kXyzPassTiles / kRhsWaves) {
    if (k0 * kRhsWaves >= ntiles) break;
    __syncthreads();
#pragma unroll
    for (int k = k0; k < k0 + kXyzPassTiles / kRhsWaves && k < TPW; ++k) {
      if (k * kRhsWaves + wave >= ntiles) break;
#pragma unroll
      for (int z = 0; z < 4; ++z)
        s_C[((k - k0) * kRhsWaves + wave) * 256 + (4 * z + (lane >> 4)) * 16 + (lane & 15)] = C[k][z];
    }
    // the pass's plan: quadruples, lane_of (4 L + 1), count (256), entries
    const int quads = plan[0], *lane_of = plan + 1, *count = lane_of + 4 * L + 1;
    const uint4 *ent = reinterpret_cast<const uint4 *>(plan + ((4 * L + 2 + 64 * kRhsWaves + 3) & ~3));
    const int cnt = count[tid];
    __syncthreads();
    s_part[tid] = plan_sum(ent + tid, 64 * kRhsWaves, cnt, s_C);
    __syncthreads();
    if (tid < 4 * L)
      for (int l = lane_of[tid], l1 = lane_of[tid + 1]; l < l1; ++l) rpa += s_part[l];
    plan = reinterpret_cast<const int *>(ent + (size_t)quads * 64 * kRhsWaves);
  }
  if (tid < 4 * L) {
    v = (fma(4.0, rpa, v) + su_sum) * (1.0 / kTwoPi);
    *out = v;
    if (isnan(v)) atomicOr(&F.flags[0], 1);
  }
}
