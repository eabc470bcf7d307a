// FP64 dGamma/dLambda of the SU(2) core: the frequency integrals of the three
// channels evaluated by independent waves.  Included by su2_flow.hip after the
// flow descriptor FlowDev.
//
// Structure used (X = the transfer frequency of a channel, on the mesh):
//
//  * S and U are images of each other.  With Gamma_X(t, o) the vertex whose
//    first outer frequency sits on the mesh point X, the reference's S kernel
//    of item (s, t, u) (src/SU2/SU2FrgCore.cpp:199-227) is a function
//    R(X = s; t, o = u) of four bundles Gamma_X,
//      V0 = Gamma_X(|al|, |be|)   al = (X + o - t) / 2 + w'
//      V2 = Gamma_X(|be|, |al|)   be = (X - o + t) / 2 + w'
//      V1 = Gamma_X(|ga|, |ep|)   ga = (X + o + t) / 2 + w'
//      V3 = Gamma_X(|ep|, |ga|)   ep = (X - o - t) / 2 + w'
//    and its U kernel (:305-334) is the same function at X = u, o = s, with the
//    density result negated: the U buffers hold V2, V3, V0, V1, under which the
//    products V0 V1 + V2 V3 do not change.
//  * R(X; t, o) and R(X; o, t) use the same bundles: exchanging t and o swaps
//    V0 with V2 (with the site exchange flag inverted) and leaves V1 and V3.
//    One evaluation of the bundles of (X, {a, b}) therefore serves two items:
//    half the gathers and descriptors of evaluating every item's S and U.
//  * The two access buffers of a T pair (:229-303) hold the same support rows
//    with the outer frequencies exchanged, so they differ by the density sign:
//    one gather serves both.
//
// The density sign of exchanged storage treats rows with equal outer indices
// ("diagonal" supports) as not exchanged from either side, so the mirrored
// value differs from the sign rule there; those supports are flagged in the
// descriptors and corrected explicitly.
//
// Frequency arguments: the sums s +- t +- u of float mesh values are exact in
// FP64, so regrouping them does not change any argument or bracket.
//
// What bounds it: a 16-byte gather of a wave costs the vector cache 16.8 cycles of
// its CU where the lanes read whole cache lines, 21 with 19 neighbouring sites of
// three rows, however near the data, so the work was arranged to issue few of
// them with full lanes.  Every wave evaluates a unit of its own and describes
// its own points, without barriers: no producer wave to wait for, and a unit's
// points fill the wave.  Simple cubic J1-J2, 64 frequencies, 23 sites: one
// evaluation 2.28 -> 0.99 ms at cutoff 60 and 9.80 -> 4.83 ms at cutoff 0.02
// (k_su 2.56 ms, k_t 2.15 ms; over the whole flow the gathers of k_su take 94 % of
// its time at 16.5 cycles each) against one 256-thread
// workgroup per item with a producer wave; 31 sites, 45 frequencies at cutoff
// 0.05: 3.0 -> 1.5 ms; square, 9 sites, 32 frequencies, whole flow 142 -> 87 ms.
#pragma once

constexpr int kMaxRhsL = 32;    // largest lattice of the T kernel's register tiles

// the four supports of an access buffer at one site: (t lo, t hi) of the first
// and of the second o index
struct Quad {
  double2 v0, v1, v2, v3;
};
__device__ __forceinline__ Quad load_quad(__amdgpu_buffer_rsrc_t r, int4 d, unsigned site) {
  Quad q;
  q.v0 = buf_load<double2>(r, d.x + site);
  q.v1 = buf_load<double2>(r, d.x + site + d.z);
  q.v2 = buf_load<double2>(r, d.y + site);
  q.v3 = buf_load<double2>(r, d.y + site + d.z);
  return q;
}
// the bilinear weights are not negative and the stored ones carry the density
// sign: the spin weights are their absolute values (free on the FMA)
__device__ __forceinline__ double spin_sum(double2 wa, double2 wb, const Quad &q) {
  return fma(fabs(wb.y), q.v3.x, fma(fabs(wb.x), q.v2.x, fma(fabs(wa.y), q.v1.x, fabs(wa.x) * q.v0.x)));
}
__device__ __forceinline__ double density_sum(double2 wa, double2 wb, const Quad &q) {
  return fma(wb.y, q.v3.y, fma(wb.x, q.v2.y, fma(wa.y, q.v1.y, wa.x * q.v0.y)));
}
// the part of density_sum on diagonal supports (flag bits 2 and 3)
__device__ __forceinline__ double diagonal_sum(int flags, double2 wa, double2 wb, const Quad &q) {
  return ((flags & 4) ? fma(wa.y, q.v1.y, wa.x * q.v0.y) : 0.0) + ((flags & 8) ? fma(wb.y, q.v3.y, wb.x * q.v2.y) : 0.0);
}

// ---------------------------------------------------------------------------
// S and U channels
// ---------------------------------------------------------------------------
// A wave evaluates a unit (X, {a, b}): lanes are slots x site groups, a lane
// holding RHO sites of its point.  RHO is chosen for the lane use (points at a
// time x sites / lanes; at L = 23 72 %, 90 % and 96 % for RHO 1, 2, 3).  Four
// waves per SIMD: 90 to 112 registers; five were 0-2 % faster for RHO = 1 only.
struct SuShape {
  int rho, lps, slots, nb;  // sites per lane, lanes per point, points at a time, points per descriptor batch
};
__host__ __device__ inline SuShape su_shape_of(int L, int rho) {
  SuShape s;
  s.rho = rho;
  s.lps = (L + rho - 1) / rho;
  s.slots = 64 / s.lps < kRhsPoints ? 64 / s.lps : kRhsPoints;
  s.nb = s.slots * (kRhsPoints / s.slots);
  return s;
}
inline SuShape su_shape(int L) {
  SuShape best = su_shape_of(L, 1);
  for (int rho = 2; rho <= 3; ++rho) {
    const SuShape s = su_shape_of(L, rho);
    if (s.slots * best.rho * 20 > best.slots * s.rho * 21) best = s;  // at least 5 % more lanes in use
  }
  return best;
}
constexpr int kSuWaveBytes = 64 * 16 + 64 * 32 + kRhsPoints * 8;

// adds the S and U integrals of all items to dG (zeroed before): every item
// receives one S and one U value, so the sum does not depend on their order
template <int RHO, bool ASYM>
__global__ __launch_bounds__(64 * kRhsWaves, 4) void k_su(const FlowDev *__restrict__ fl, int nflows, long long total) {
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
  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * kSuWaveBytes;
  int4 *s_off = reinterpret_cast<int4 *>(wl);
  double2 *s_wa = reinterpret_cast<double2 *>(wl + 64 * 16);
  double2 *s_wb = s_wa + 64;
  double *s_c = reinterpret_cast<double *>(wl + 64 * 48);

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 16;
  const SuShape sh = su_shape_of(L, RHO);
  const int slot0 = lane / sh.lps;
  const int lj = lane - slot0 * sh.lps;
  const bool active = slot0 < sh.slots;
  const int slot = active ? slot0 : sh.slots - 1;
  unsigned sr[RHO], sx[RHO];  // byte offsets of the sites, plain and exchanged
#pragma unroll
  for (int i = 0; i < RHO; ++i) {
    const int r = lj + i * sh.lps;
    const bool ok = active && r < L;
    sr[i] = ok ? (unsigned)F.site_rid[r] * 16u : kNoSite;
    sx[i] = ASYM ? (ok ? (unsigned)F.inv_rid[r] * 16u : kNoSite) : sr[i];
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
  const int rule = kind == 1 ? 1 : 0;

  auto points = [&](auto mixed_c) {
    constexpr bool MIXEDKIND = decltype(mixed_c)::value;
    double wp_next = pe < n ? Wwp[pe] : 0.0, c_next = pe < n ? Wc[pe] : 0.0;
    for (int e0 = 0; e0 < n; e0 += sh.nb) {
      const int nvalid = n - e0 < sh.nb ? n - e0 : sh.nb;
      // descriptors of the batch: one bracket search per lane, shared with the
      // other lane of its pair; lane (pe, pp, pj) describes V0, V2, V1, V3
      {
        const double v = half + wp_next, c = c_next;
        const Bracket t = bracket_of(s_mesh, nw, fabs(v), F.geo, F.ga, F.gb);
        Bracket o;
        o.lo = pair_swap(t.lo);
        o.step = pair_swap(t.step);
        o.b = pair_swap(t.b);
        const bool ok = pe < nvalid;
        int4 d = make_int4((int)kNoRow, (int)kNoRow, 0, 0);
        double2 wa = make_double2(0.0, 0.0), wb = wa;
        if (ok) {
          // bits 2, 3 of w: the support's outer indices are equal
          const SuBuffer sb = su_buffer(t, o, X, nw, rowbytes, rule);
          d = make_int4(sb.x, sb.y, sb.z, sb.diag);
          wa = sb.wa;
          wb = sb.wb;
          if (ASYM) {
            const double vo = pair_swap(v);
            const bool pos = vo > 0, neg = vo < 0;
            d.w |= (pj ? neg : pos) ? 1 : 0;
            d.w |= (pj ? pos : neg) ? 2 : 0;  // the exchange of the second result's V0 / V2
          }
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
#pragma unroll
        for (int i = 0; i < RHO; ++i) {
          // V1 and V3 first: their products with the point's coefficient are
          // the factors of V0 and V2, which are added up as they arrive.  The
          // next buffer's loads are issued before the present one is used, and
          // nothing more (the scheduling barriers).  With
          // h = V0 V1 + V2 V3 over the spin parts the results are
          // spin -h/2 + D0 S1 + S0 D1 + D2 S3 + S2 D3, density 3/16 h + D0 D1 + D2 D3
          reread_lds();
          double s1, s3, d1, d3, g1, g3;  // g: the density factors of the first result
          int4 d = s_off[4 * e + 2];
          Quad v = load_quad(rG, d, ASYM ? ((d.w & 1) ? sx[i] : sr[i]) : sr[i]);
#pragma unroll
          for (int k = 2; k < 4; ++k) {
            const int dw = d.w;
            const Quad q = v;
            d = s_off[4 * e + (k == 2 ? 3 : 0)];
            v = load_quad(rG, d, ASYM ? ((d.w & 1) ? sx[i] : sr[i]) : sr[i]);
            __builtin_amdgcn_sched_barrier(0);
            const double2 wa = s_wa[4 * e + k], wb = s_wb[4 * e + k];
            double S = c * spin_sum(wa, wb, q), D = c * density_sum(wa, wb, q);
            settle(S, D);
            double Df = D;
            if (MIXEDKIND) {
              if (__any(dw & 12)) Df = fma(-2.0 * c, diagonal_sum(dw, wa, wb, q), D);
            }
            if (k == 2) { s1 = S; d1 = D; g1 = Df; }
            else { s3 = S; d3 = D; g3 = Df; }
            __builtin_amdgcn_sched_barrier(0);
          }
          // k = 0: V0, partner V1 in the second result, V3 in the first; k = 1: V2
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int4 dk = d;
            Quad q = v;
            if (ASYM) v = load_quad(rG, dk, (dk.w & 2) ? sx[i] : sr[i]);
            if (!ASYM && k == 0) {
              d = s_off[4 * e + 1];
              v = load_quad(rG, d, sr[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
            const double2 wa = s_wa[4 * e + k], wb = s_wb[4 * e + k];
            double S = spin_sum(wa, wb, q), D = density_sum(wa, wb, q);
            settle(S, D);
            if (outs & 2) {
              const double sp = k ? s3 : s1, dp = k ? d3 : d1;
              a2s[i] = fma(S, fma(-0.5, sp, dp), fma(D, sp, a2s[i]));
              a2d[i] = fma(S, 0.1875 * sp, fma(D, dp, a2d[i]));
            }
            if (ASYM) {
              q = v;
              if (k == 0) {
                d = s_off[4 * e + 1];
                v = load_quad(rG, d, (d.w & 1) ? sx[i] : sr[i]);
              }
              __builtin_amdgcn_sched_barrier(0);
              S = spin_sum(wa, wb, q);
              D = density_sum(wa, wb, q);
            }
            if (MIXEDKIND) {
              if (__any(dk.w & 12)) D = fma(-2.0, diagonal_sum(dk.w, wa, wb, q), D);
            }
            if (outs & 1) {
              const double sp = k ? s1 : s3, dp = k ? g1 : g3;
              a1s[i] = fma(S, fma(-0.5, sp, dp), fma(D, sp, a1s[i]));
              a1d[i] = fma(S, 0.1875 * sp, fma(D, dp, a1d[i]));
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
  };
  if (kind == 2) points(std::true_type{});
  else points(std::false_type{});

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
    const int item = un.item(r, nw);
    double *out = reinterpret_cast<double *>(F.dG + (size_t)item * L);
    for (int k = lane; k < 2 * L; k += 64) {
      double v = 0.0;
      for (int z = 0; z < sh.slots; ++z) v += s_red[z * 2 * L + k];
      unsafeAtomicAdd(out + k, (urule && (k & 1)) ? -v : v);
    }
  }
}

// ---------------------------------------------------------------------------
// T channel and the final sum
// ---------------------------------------------------------------------------
// A wave evaluates the T channel of an item, eight points at a time, its lanes
// in the operand layout of the FP64 matrix instructions (lane l =
// row l % 16 of point l / 16): the gathered values are the operands of the
// lattice-bubble update C[a][b] += sum_e P_e[a] Q_e[b] without a pass through
// LDS.  Sites come in FT full tiles of 16 and, with HT, a half tile of 8 whose
// lanes take eight points at once; in the matrix operands its even points sit
// in rows 0-7 and its odd points in rows 8-15.  The blocks of 4 x 4 that the
// overlap lists need are updated and no others: 36 instructions for eight points
// and both channels at L = 23 (612 cycles of a SIMD; 14 of 16 x 16 x 4 took 1800,
// cubic r6 at cutoff 60 0.987 -> 0.967 ms).  The matrix instructions run at
// the vector FP64 rate; what they save is the LDS traffic of a rank update from
// shared factors.  Two tiles: three waves per SIMD (two: 5 to 8 % slower at
// L = 23), single tiles four.
struct TShape {
  int ft, ht, lp;  // full tiles, half tile, row stride of the bubble matrix
};
__host__ __device__ inline TShape t_shape(int L) {
  TShape s;
  s.ft = L <= 8 ? 0 : (L <= 24 ? 1 : 2);
  s.ht = (L <= 8 || (L > 16 && L <= 24)) ? 1 : 0;
  s.lp = 16 * s.ft + 8 * s.ht;
  return s;
}
constexpr int kTDescBytes = 32 * 16 + 32 * 32 + 32 * 32 + 64 * 4 + kRhsPoints * 8;
__host__ __device__ inline int t_wave_bytes(int L) {
  const int lp = t_shape(L).lp;
  const int c = lp * lp * 8 + 64 * 8;
  return c > kTDescBytes ? c : kTDescBytes;
}

// distinct (rid1, rid2) pairs of every site's overlap list, with their
// multiplicities, dealt to the lanes of a wave
template <class PLAN>
inline void build_overlap_plan(PLAN &plan, int L, const int *off, const int *rid1, const int *rid2) {
  const int lp = t_shape(L).lp;
  plan.begin((size_t)lp * lp, L);
  for (int r = 0; r < L; ++r) {
    const int *r1 = rid1 + off[r], *r2 = rid2 + off[r];
    plan.add_list(off[r + 1] - off[r], [=](size_t i) { return (unsigned)(r1[i] * lp + r2[i]); });
    plan.end_output();
  }
  plan.deal(64);
}

// the bubble matrix of both channels in a wave's registers: full tiles, full
// rows x half columns, half rows x full columns, half tile
template <int FT, int HT> struct BubbleTiles {
  d4 c[2][FT ? FT * FT : 1];
  double2 r[2][FT ? FT : 1], l[2][FT ? FT : 1], h[2];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
      for (int k = 0; k < FT * FT; ++k) c[ch][k] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < FT; ++k) r[ch][k] = l[ch][k] = make_double2(0.0, 0.0);
      h[ch] = make_double2(0.0, 0.0);
    }
  }
  // half tile: even and odd points in blocks of their own
  __device__ __forceinline__ void half(const double (&ph)[2], const double (&qh)[2]) {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
      h[ch].x = mfma_blocks(ph[ch], qh[ch], h[ch].x);
      h[ch].y = mfma_blocks(ph[ch], half_mirror(qh[ch]), h[ch].y);
    }
  }
  // the even (par 0) or odd points of the full tiles, and of the half tile with them
  __device__ __forceinline__ void full(int par, const double (&P)[FT ? FT : 1][2], const double (&Q)[FT ? FT : 1][2],
                                       const double (&ph)[2], const double (&qh)[2]) {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
      for (int i = 0; i < FT; ++i)
#pragma unroll
        for (int j = 0; j < FT; ++j) outer_update(c[ch][i * FT + j], P[i][ch], Q[j][ch]);
      if (HT) {
        // the half tile at these points in both halves of the rows
        const double p = par ? row_move<0x128, 0x3>(ph[ch]) : row_move<0x128, 0xc>(ph[ch]);
        const double q = par ? row_move<0x128, 0x3>(qh[ch]) : row_move<0x128, 0xc>(qh[ch]);
        const double pm = half_mirror(p), qm = half_mirror(q);
#pragma unroll
        for (int i = 0; i < FT; ++i) {
          r[ch][i].x = mfma_blocks(P[i][ch], q, r[ch][i].x);
          r[ch][i].y = mfma_blocks(P[i][ch], qm, r[ch][i].y);
          l[ch][i].x = mfma_blocks(p, Q[i][ch], l[ch][i].x);
          l[ch][i].y = mfma_blocks(pm, Q[i][ch], l[ch][i].y);
        }
      }
    }
  }
  // channel ch into LDS, rows of 16 FT + 8 HT
  __device__ __forceinline__ void store(int ch, double *s_C, int lane) const {
    constexpr int LP = 16 * FT + 8 * HT;
    // lane (ri, b, rj) holds elements (4 b + ri, rj of another block of columns)
    const int ri = lane >> 4, cb = (lane >> 2) & 3, rj = lane & 3;
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      const int row = (16 * i + 4 * cb + ri) * LP;
#pragma unroll
      for (int j = 0; j < FT; ++j)
#pragma unroll
        for (int z = 0; z < 4; ++z) s_C[row + 16 * j + 4 * ((cb + z) & 3) + rj] = c[ch][i * FT + j][z];
      if (HT) {
        const int h0 = 16 * FT, lo = 4 * (cb & 1), hi = 4 * (1 - (cb & 1)) + 3;
        s_C[row + h0 + lo + rj] = r[ch][i].x;
        s_C[row + h0 + hi - rj] = r[ch][i].y;
        s_C[(h0 + lo + ri) * LP + 16 * i + 4 * cb + rj] = l[ch][i].x;
        s_C[(h0 + hi - ri) * LP + 16 * i + 4 * cb + rj] = l[ch][i].y;
      }
    }
    if (HT) {
      const double x = h[ch].x + half_row_swap(h[ch].x), y = h[ch].y + half_row_swap(h[ch].y);
      if (cb < 2) {
        double *o = s_C + (16 * FT + 4 * cb + ri) * LP + 16 * FT;
        o[4 * cb + rj] = x;
        o[4 * (1 - cb) + 3 - rj] = y;
      }
    }
  }
};

// the end of an item: the overlap sums of the bubble matrix, the sums over the
// points (rs, rd: per tile of sites), S and U values, prefactor and 2^scale.
// wl: the wave's LDS.  MIXED: an FP32 term that overflowed makes the value NaN,
// as it does a compensated FP32 sum, so that the flow counts as diverged.
template <bool MIXED, int FT, int HT>
__device__ __forceinline__ void t_finish(const FlowDev &F, const BubbleTiles<FT, HT> &C, const double (&rs)[FT + HT],
                                         const double (&rd)[FT + HT], unsigned char *wl, int item, int scale) {
  // RPA(rid) = sum over getOverlap(rid) of C[rid1][rid2] (src/SU2/SU2FrgCore.cpp:250-266)
  constexpr int LP = 16 * FT + 8 * HT, NT = FT + HT;
  const int L = F.L, lane = threadIdx.x & 63;
  double *s_C = reinterpret_cast<double *>(wl);
  double *s_part = s_C + LP * LP;
  const int cnt = F.plan_count[lane];
  double rpa[2] = {0.0, 0.0};
#pragma unroll
  for (int ch = 0; ch < 2; ++ch) {
    wave_lds_fence();
    C.store(ch, s_C, lane);
    wave_lds_fence();
    s_part[lane] = plan_sum(reinterpret_cast<const uint4 *>(F.plan_ent) + lane, 64, cnt, s_C);
    wave_lds_fence();
    if (lane < L) {
      const int l1 = F.plan_lane[lane + 1];
      for (int l = F.plan_lane[lane]; l < l1; ++l) rpa[ch] += s_part[l];
    }
  }
  // sum over the points, S and U values, prefactor 1/(2 pi) (src/SU2/SU2FrgCore.cpp:426-430)
  double ts = 0.0, td = 0.0;
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    double x = rs[k], y = rd[k];
    if (k >= FT) {
      x += __shfl_xor(x, 8, 64);
      y += __shfl_xor(y, 8, 64);
    }
    x += __shfl_xor(x, 16, 64);
    y += __shfl_xor(y, 16, 64);
    x += __shfl_xor(x, 32, 64);
    y += __shfl_xor(y, 32, 64);
    if (lane >= 16 * k) {
      ts = x;
      td = y;
    }
  }
  if (lane < L) {
    double2 *out = F.dG + (size_t)item * L + lane;
    const double2 su_sum = *out;
    if (MIXED) {
      const double nan = __builtin_nan("");
      ts += su_sum.x;
      td += su_sum.y;
      if (isinf(ts)) ts = nan;
      if (isinf(td)) td = nan;
      ts = fma(2.0 * F.spin, rpa[0], ts) * (1.0 / kTwoPi);
      td = fma(8.0 * F.spin, rpa[1], td) * (1.0 / kTwoPi);
    } else {
      ts = (fma(2.0 * F.spin, rpa[0], ts) + su_sum.x) * (1.0 / kTwoPi);
      td = (fma(8.0 * F.spin, rpa[1], td) + su_sum.y) * (1.0 / kTwoPi);
    }
    if (scale != 0) {
      ts = ldexp(ts, scale);
      td = ldexp(td, scale);
    }
    *out = make_double2(ts, td);
    if (isnan(ts) || isnan(td)) atomicOr(&F.flags[0], 1);
  }
}

template <int FT, int HT, bool ASYM>
__global__ __launch_bounds__(64 * kRhsWaves, FT + HT == 1 ? 4 : 3) void k_t(const FlowDev *__restrict__ fl, int nflows, long long total) {
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
  int2 *s_off = reinterpret_cast<int2 *>(wl);              // [(point, pair) * 2 + half]
  double2 *s_w = reinterpret_cast<double2 *>(wl + 512);    // [(point, pair) * 2 + half]
  double4 *s_loc = reinterpret_cast<double4 *>(wl + 1536);  // [(point, pair)]
  int *s_fl = reinterpret_cast<int *>(wl + 2560);          // [(point, pair) * 2 + half]
  double *s_c = reinterpret_cast<double *>(wl + 2816);

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 16;
  unsigned sr[NT], sx[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    const int r = k < FT ? 16 * k + (lane & 15) : 16 * FT + (lane & 7);
    sr[k] = r < L ? (unsigned)F.site_rid[r] * 16u : kNoSite;
    sx[k] = ASYM ? (r < L ? (unsigned)F.inv_rid[r] * 16u : kNoSite) : sr[k];
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
      double2 w = make_double2(0.0, 0.0);
      int flag = 0;
      double fs = 0.0, fd = 0.0;
      if (ok) {
        // gathered buffer (the pair's second one: s slot |B|, u slot |A|);
        // lane pj describes the supports of A's index pj
        const Bracket A = pj ? ot : me, B = pj ? me : ot;
        const int ia = A.lo + (pj ? A.step : 0), b0 = B.lo, b1 = B.lo + B.step;
        off.x = ((b0 > ia ? tri(b0, ia) : tri(ia, b0)) * nw + X) * rowbytes;
        off.y = ((b1 > ia ? tri(b1, ia) : tri(ia, b1)) * nw + X) * rowbytes;
        const double wa = pj ? A.b : 1.0 - A.b;
        const double w0 = wa * (1.0 - B.b), w1 = wa * B.b;
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
        double vs = 0.0, vd = 0.0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int is = me.lo + (q ? me.step : 0);
          const double ws = q ? me.b : 1.0 - me.b;
          const int row = ((is > X ? tri(is, X) : tri(X, is)) * nw + ot.lo) * rowbytes;
          const double2 x0 = buf_load<double2>(rG, row), x1 = buf_load<double2>(rG, row + ot.step * rowbytes);
          const double wl0 = ws * (1.0 - ot.b), wl1 = ws * ot.b;
          vs = fma(wl1, x1.x, fma(wl0, x0.x, vs));
          const double d = fma(wl1, x1.y, wl0 * x0.y);
          vd += is < X ? -d : d;
        }
        fs = fma(0.25, vs, -vd);
        fd = -fma(0.75, vs, vd);
      }
      const double fso = pair_swap(fs), fdo = pair_swap(fd);
      wave_lds_fence();
      s_off[lane] = off;
      s_w[lane] = w;
      s_fl[lane] = flag;
      if (pj == 0) {
        // factors of the other pair's bundles: the second buffer B2 and its
        // image B0 (spin equal, density negated):
        // spin (f0 + f1) B2, density (g1 - g0) B2; 2 g0 for the diagonal
        // supports, f0 where the image carries another site exchange; the
        // point's coefficient in pair 0's (bundles of pair 1)
        const double cf = pp == 0 ? (ok ? c : 0.0) : 1.0;
        s_loc[2 * pe + (1 - pp)] = make_double4(cf * (fs + fso), cf * (fdo - fd), cf * 2.0 * fd, cf * fs);
        if (pp == 0) s_c[pe] = ok ? c : 0.0;
      }
      const int en = e0 + kRhsPoints + pe;
      wp_next = en < n ? Wwp[en] : 0.0;
      c_next = en < n ? Wc[en] : 0.0;
      wave_lds_fence();
    }
    for (int eb = 0; eb < nvalid; eb += 8) {
      // gathers one tile of sites, e the lane's point: (c A2, A3) per channel
      auto gather = [&](int k, int e, double (&P)[2], double (&Q)[2]) {
        const unsigned r0 = sr[k], x0 = sx[k];
        const double c = s_c[e];
        double2 v[2][4];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int4 o = reinterpret_cast<const int4 *>(s_off)[2 * e + p];
          const unsigned site = ASYM ? ((s_fl[4 * e + 2 * p] & 1) ? x0 : r0) : r0;
          v[p][0] = buf_load<double2>(rG, o.x + site);
          v[p][1] = buf_load<double2>(rG, o.y + site);
          v[p][2] = buf_load<double2>(rG, o.z + site);
          v[p][3] = buf_load<double2>(rG, o.w + site);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const double2 wa = s_w[4 * e + 2 * p], wb = s_w[4 * e + 2 * p + 1];
          const int2 fl2 = reinterpret_cast<const int2 *>(s_fl)[2 * e + p];
          const double4 lc = s_loc[2 * e + p];
          const Quad q{v[p][0], v[p][1], v[p][2], v[p][3]};
          const double cp = p == 0 ? c : 1.0;
          double S = spin_sum(wa, wb, q), D = density_sum(wa, wb, q);
          if (p == 0) {
            S *= c;
            D *= c;
          }
          settle(S, D);
          rs[k] = fma(lc.x, S, rs[k]);
          rd[k] = fma(lc.y, D, rd[k]);
          settle(rs[k], rd[k]);
          if (__any((fl2.x | fl2.y) & 12)) {
            // supports with equal outer indices keep their sign in the image
            const double dg = ((fl2.x & 4) ? wa.x * q.v0.y : 0.0) + ((fl2.x & 8) ? wa.y * q.v1.y : 0.0) +
                              ((fl2.y & 4) ? wb.x * q.v2.y : 0.0) + ((fl2.y & 8) ? wb.y * q.v3.y : 0.0);
            rd[k] = fma(lc.z, cp * dg, rd[k]);
          }
          if (ASYM) {
            if (fl2.x & 2) {
              // an argument of exactly zero: the image exchanges the sites the other way
              const int4 o = reinterpret_cast<const int4 *>(s_off)[2 * e + p];
              const unsigned si = (fl2.x & 1) ? r0 : x0;
              const Quad g{buf_load<double2>(rG, o.x + si), buf_load<double2>(rG, o.y + si),
                           buf_load<double2>(rG, o.z + si), buf_load<double2>(rG, o.w + si)};
              const double dx = ((fl2.x & 4) ? wa.x * (g.v0.y - q.v0.y) : 0.0) +
                                ((fl2.x & 8) ? wa.y * (g.v1.y - q.v1.y) : 0.0) +
                                ((fl2.y & 4) ? wb.x * (g.v2.y - q.v2.y) : 0.0) +
                                ((fl2.y & 8) ? wb.y * (g.v3.y - q.v3.y) : 0.0);
              rs[k] = fma(lc.w, fma(cp, spin_sum(wa, wb, g), -S), rs[k]);
              rd[k] = fma(0.5 * lc.z, D - cp * density_sum(wa, wb, g), fma(lc.z, cp * dx, rd[k]));
            }
          }
          (p ? Q : P)[0] = S;
          (p ? Q : P)[1] = D;
          __builtin_amdgcn_sched_barrier(0);
        }
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
  t_finish<false, FT, HT>(F, C, rs, rd, wl, item, 0);
}
