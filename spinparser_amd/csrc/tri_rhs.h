// dGamma/dLambda of the TRI core by waves.  Included by tri_flow.hip after the
// flow descriptor TriDev (wave_rhs.h before it).
//
// Structure used, in addition to what su2_rhs.h describes (the U integrals are
// images of the S ones, the bundles of a unit (X, {a, b}) serve two items, the
// buffers of a T pair are images of each other):
//
//  * An access buffer is first interpolated in the stored components (k, l) and
//    sites; support rows read with the outer frequencies exchanged negate the
//    components with l = d, the t / u sign the components with exactly one d.
//    The bundle is that "raw" buffer, or, exchanged, its transpose
//    raw(P l, P k) at the site inv_rid with the spin permutation P of inv_perm.
//    This needs site_rid and site_perm to be identities and inv_rid a
//    permutation, which every lattice of the factory has; other tables, and
//    lattices of more than kMaxTriRhsL sites, run the general kernel.  So do
//    lattices with more than 16 kTriMaxGroups products for each of eight waves
//    (1,280; honeycomb-Kitaev at range 8 and 9, of 23 and 28 sites).
//  * S and U add the 256 products of the components of two bundles, each output's
//    sixteen terms summed first (k_tri_su).  As elements of H (x) H, 4 x 4 real
//    matrices, the bundles would need 64 products, but sums and differences of
//    components mix their sizes: on flowed kagome-DM states the error of the
//    Dzyaloshinskii-Moriya components (1e-5 to 4e-2 of the others) was 1.3 to 2
//    times that of sums over their own terms, and components 1e-8 as large as
//    others had 7e-10 of their size.  The matrices were faster (kagome-DM r5 at
//    cutoff 0.02: k_tri_su 8.2 instead of 9.8 ms).  The U integrals are the S ones with the
//    sign of the l = d components changed in the buffers and in the result.
//  * With s(x, y) = -1 for x a spin and y the density, A(r, m) s(r, m) are 4 x 4
//    matrices whose plain product is the lattice bubble (times s(r, t)), and
//    whose products with one 4 x 4 matrix of the site-local vertex are the
//    chalice and the inverse chalice.  Such products are what the FP64 matrix
//    instruction 4 x 4 x 4 computes, four per instruction, at the vector
//    FP64 rate (measured 73 TFLOP/s; the 16 x 16 x 4 form 38).  They are summed
//    over the points before the overlap lists are applied (k_tri_t).
//
// Kagome with DM exchange, 19 sites, 48 frequencies, against one workgroup per
// item that forms all terms point by point: 12.9 -> 5.5 ms at cutoff 20, 46.3 ->
// 15.0 ms at 0.7, 81.9 -> 25.9 ms at 0.02 (k_tri_su 9.8 ms, its vector instructions
// 70 and its gathers 64 % of the cycles; k_tri_t 15.8 ms, which
// alternates between gathers, 11 ms by themselves, and matrix products, 13 ms by
// themselves: the descriptors of the next points are formed beside the products).
#pragma once

constexpr int kMaxTriRhsL = 32;
// matrix products of k_tri_t: runs of four that share the left factor, four
// runs to a group of four instructions
constexpr int kTriMaxGroups = 10;  // per wave, of at most eight waves

// label of a component in the group the Pauli products follow: d 0, x 1, y 2, z 3
constexpr int pauli_label(int k) { return (k + 1) & 3; }
constexpr int pauli_comp(int label) { return (label + 3) & 3; }
__device__ __forceinline__ double flip(double v, bool neg) { return neg ? -v : v; }
// v with the sign bit changed by bit 31 of s
__device__ __forceinline__ double flip_by(double v, int s) {
  int2 q;
  __builtin_memcpy(&q, &v, 8);
  q.y ^= s & (int)0x80000000;
  __builtin_memcpy(&v, &q, 8);
  return v;
}
// v, or |v| for mask 0x7fffffff
__device__ __forceinline__ double and_sign(double v, int mask) {
  int2 q;
  __builtin_memcpy(&q, &v, 8);
  q.y &= mask;
  __builtin_memcpy(&v, &q, 8);
  return v;
}
// q / d for 0 <= q < 4096 and 8 <= d <= 256 (the error of q * inv stays below 2^20 / d)
__device__ __forceinline__ unsigned div_factor(int d) { return ((1u << 20) + d - 1) / d; }
__device__ __forceinline__ int fast_div(int q, unsigned inv) { return (int)(((unsigned)q * inv) >> 20); }

// s(x, y) and the signs of the site-local vertex in the matrices of the chalice
// (row nu, column t, then the first component ka of the vertex) and of the
// inverse chalice (row r, column ka, then mu): any first (last) index of the
// bundle gives the same ones
constexpr int hat_sign(int x, int y) { return x < 3 && y == 3 ? -1 : 1; }
__host__ __device__ constexpr double tri_hat(int c) { return (c >> 2) < 3 && (c & 3) == 3 ? -1.0 : 1.0; }
constexpr unsigned long long chalice_mask(int r) {
  unsigned long long m = 0;
  for (int n = 0; n < 4; ++n)
    for (int t = 0; t < 4; ++t)
      for (int k = 0; k < 4; ++k) {
        const int l = pauli_comp(pauli_label(n) ^ pauli_label(t) ^ pauli_label(k));
        if (coefficient(2, 4 * r + t, 4 * r + n, 4 * k + l).re * hat_sign(r, t) * hat_sign(r, n) < 0)
          m |= 1ull << ((4 * n + t) * 4 + k);
      }
  return m;
}
constexpr unsigned long long inverse_mask(int t) {
  unsigned long long m = 0;
  for (int r = 0; r < 4; ++r)
    for (int k = 0; k < 4; ++k)
      for (int u = 0; u < 4; ++u) {
        const int n = pauli_comp(pauli_label(r) ^ pauli_label(k) ^ pauli_label(u));
        if (coefficient(3, 4 * r + t, 4 * u + n, 4 * k + t).re * hat_sign(r, t) * hat_sign(k, t) < 0)
          m |= 1ull << ((4 * r + k) * 4 + u);
      }
  return m;
}
constexpr unsigned long long kChaliceMask = chalice_mask(0), kInverseMask = inverse_mask(0);
static_assert(chalice_mask(1) == kChaliceMask && chalice_mask(2) == kChaliceMask && chalice_mask(3) == kChaliceMask,
              "chalice matrix");
static_assert(inverse_mask(1) == kInverseMask && inverse_mask(2) == kInverseMask && inverse_mask(3) == kInverseMask,
              "inverse chalice matrix");

// ---------------------------------------------------------------------------
// S and U channels
// ---------------------------------------------------------------------------
constexpr int kTriRaw = 17;   // stride of a site's 16 components in the raw buffers (doubles; odd: no bank conflicts)
struct TriSuShape {
  int slots, nb, raw;  // points at a time, points per descriptor batch, doubles of one raw buffer
};
__host__ __device__ inline TriSuShape tri_su_shape(int L) {
  TriSuShape s;
  s.slots = 64 / L < kRhsPoints ? 64 / L : kRhsPoints;
  s.nb = s.slots * (kRhsPoints / s.slots);
  s.raw = s.slots * L * kTriRaw;
  return s;
}
__host__ __device__ inline int tri_su_wave_bytes(int L) {
  return 64 * 48 + kRhsPoints * 8 + ((2 * tri_su_shape(L).raw * 8 + 15) & ~15);
}

// A wave evaluates a unit (X, {a, b}).  Gathers: all lanes read rows in order,
// 16 bytes each (eight lanes to a site, whole cache lines: 16.5 cycles of the
// CU per wave load; one lane per site took 141), and leave the raw buffers in
// LDS.  Products: lanes are slots x sites and read both exchange states of a
// buffer from there.
__global__ __launch_bounds__(64 * kRhsWaves, 2) void k_tri_su(TriDev F, long long total) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const long long blk = xcd_position(blockIdx.x, (int)kTriChunk);
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
  unsigned char *wl = lds_raw + ((nw * 8 + 15) & ~15) + wave * tri_su_wave_bytes(L);
  int4 *s_off = reinterpret_cast<int4 *>(wl);
  double2 *s_wa = reinterpret_cast<double2 *>(wl + 64 * 16);
  double2 *s_wb = s_wa + 64;
  double *s_c = reinterpret_cast<double *>(wl + 64 * 48);
  double *s_v = s_c + kRhsPoints;

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 128;
  const TriSuShape sh = tri_su_shape(L);
  const int nch = 8 * L;  // 16-byte pieces of a row
  const unsigned inv = div_factor(nch);
  const int slot0 = lane / L, site = lane - slot0 * L;
  const bool active = slot0 < sh.slots;
  const int slot = active ? slot0 : 0;
  const int isite = F.inv_rid[site];
  const int p0 = F.inv_perm[3 * site], p1 = F.inv_perm[3 * site + 1], p2 = F.inv_perm[3 * site + 2];
  const int base_p = (slot * L + site) * kTriRaw, base_x = (slot * L + isite) * kTriRaw;

  double r1[16], r2[16];  // results (t = b, o = a) and (t = a, o = b)
#pragma unroll
  for (int k = 0; k < 16; ++k) r1[k] = r2[k] = 0.0;

  const int pe = lane >> 2, pp = (lane >> 1) & 1, pj = lane & 1;
  double half;
  {
    const double xm = s_mesh[X], am = s_mesh[un.a], bm = s_mesh[un.b];
    half = 0.5 * (xm + ((pp ^ pj) ? am : -am) + (pj ? -bm : bm));
  }
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;
  const int rule = kind == 1 ? 1 : 0;

  // raw buffers k0 and k0 + 1 of the points eb .. eb + slots; mode 0: for both
  // results, else for result `mode` alone.  A lane always reads the same two
  // components (k, l) and (k, l + 1) of a site, k = pc / 2, l = 2 (pc % 2)
  const int pc = lane & 7;
  const int mask = (pc & 1) ? -1 : 0x7fffffff;  // the sign of the weights is for l = d only
  const int xt = pc >= 6 ? -1 : 0, yt = ((pc & 1) != 0) != (pc >= 6) ? -1 : 0;  // components with the t / u sign
  const int per = sh.slots * nch;
  auto gather = [&](int eb, int k0, int mode) {
    const int tbit = mode == 1 ? 26 : 27;
    for (int q = lane; q < per; q += 64) {
      const int sl = fast_div(q, inv);
      const unsigned o = (q - sl * nch) * 16u;
      const int id = 4 * (eb + sl) + k0;
      double *dst = s_v + (q >> 3) * kTriRaw + 2 * pc;
      double2 v[2][4];
      int fl[2];
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        const int4 d = s_off[id + z];
        fl[z] = d.w;
        v[z][0] = buf_load<double2>(rG, d.x + o);
        v[z][1] = buf_load<double2>(rG, d.x + o + d.z);
        v[z][2] = buf_load<double2>(rG, d.y + o);
        v[z][3] = buf_load<double2>(rG, d.y + o + d.z);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        double2 wa = s_wa[id + z], wb = s_wb[id + z];
        double x = fabs(wa.x) * v[z][0].x;
        x = fma(fabs(wa.y), v[z][1].x, x);
        x = fma(fabs(wb.x), v[z][2].x, x);
        x = fma(fabs(wb.y), v[z][3].x, x);
        if (kind == 2 && mode == 1) {  // the first result's rule on diagonal supports
          if (fl[z] & 4) wa = make_double2(-wa.x, -wa.y);
          if (fl[z] & 8) wb = make_double2(-wb.x, -wb.y);
        }
        double y = and_sign(wa.x, mask) * v[z][0].y;
        y = fma(and_sign(wa.y, mask), v[z][1].y, y);
        y = fma(and_sign(wb.x, mask), v[z][2].y, y);
        y = fma(and_sign(wb.y, mask), v[z][3].y, y);
        const int tu = fl[z] << tbit;
        dst[z * sh.raw] = flip_by(x, tu & xt);
        dst[z * sh.raw + 1] = flip_by(y, tu & yt);
      }
    }
  };
  // a buffer's bundle at the lane's site, times c
  auto bundle = [&](const double *raw, bool ex, double c, double (&m)[16]) {
    // (positions formed here, each time: kept in registers over the loops they
    // would take more than 100)
    int at = ex ? base_x : base_p;
    int q0 = p0, q1 = p1, q2 = p2;
    asm volatile("" : "+v"(at), "+v"(q0), "+v"(q1), "+v"(q2));
    const double *b = raw + at;
    const int A[4] = {ex ? q0 : 0, ex ? q1 : 4, ex ? q2 : 8, ex ? 3 : 12};
    const int B[4] = {ex ? 4 * q0 : 0, ex ? 4 * q1 : 1, ex ? 4 * q2 : 2, ex ? 12 : 3};
#pragma unroll
    for (int k = 0; k < 16; ++k) m[k] = c * b[A[k >> 2] + B[k & 3]];
  };

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
        // arguments (t, o) of the buffer: bits 0, 1 the site exchange, bits 4,
        // 5 the t / u sign in the second and in the first result (of V1, V3 in
        // both); the two differ beyond the exchange at arguments of zero only
        const bool pos = vo > 0, neg = vo < 0, tp = v > 0, tn = v < 0;
        const bool ex2 = pj ? neg : pos, ex1 = pp ? ex2 : (pj ? pos : neg);
        const bool tu2 = pp ? (pj ? tp != neg : tn != pos) : (pj ? tn != neg : tp != pos);
        const bool tu1 = pp ? tu2 : (pj ? tp != pos : tn != neg);
        d = make_int4(b.x, b.y, b.z, b.diag | (ex2 ? 1 : 0) | (ex1 ? 2 : 0) | (tu2 ? 16 : 0) | (tu1 ? 32 : 0));
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
      const int4 f = make_int4(s_off[4 * e].w, s_off[4 * e + 1].w, s_off[4 * e + 2].w, s_off[4 * e + 3].w);
      // results that need buffers of their own are evaluated one after the
      // other: diagonal supports under different rules, t / u signs that differ
      bool apart = (((f.x ^ (f.x >> 1)) | (f.y ^ (f.y >> 1))) & 16) != 0;
      if (kind == 2) apart = apart || ((f.x | f.y | f.z | f.w) & 12) != 0;
      const int m0 = __any(apart) ? 1 : 0, m1 = m0 ? 2 : 0;
      for (int mode = m0; mode <= m1; ++mode) {
        const int want = mode ? outs & mode : outs;
        if (!want) continue;
        const double c = s_c[e];
        double y2[16], y3[16];
        gather(eb, 2, mode);
        wave_lds_fence();
        bundle(s_v, f.z & 1, c, y2);
        bundle(s_v + sh.raw, f.w & 1, c, y3);
        wave_lds_fence();
        gather(eb, 0, mode);
        wave_lds_fence();
        double x[16];
        if (want & 1) {
          bundle(s_v, f.x & 2, 1.0, x);
          add_table<0>(r1, x, y3);
          bundle(s_v + sh.raw, f.y & 2, 1.0, x);
          add_table<0>(r1, x, y2);
        }
        if (want & 2) {
          bundle(s_v, f.x & 1, 1.0, x);
          add_table<0>(r2, x, y2);
          bundle(s_v + sh.raw, f.y & 1, 1.0, x);
          add_table<0>(r2, x, y3);
        }
        wave_lds_fence();
      }
    }
  }

  // sum over the slots, one addition to each value of the
  // item (zeroed before; two additions in all, so their order does not matter)
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (!(outs & (r ? 2 : 1))) continue;
    wave_lds_fence();
    if (active) {
#pragma unroll
      for (int k = 0; k < 16; ++k) s_v[base_p + k] = r ? r2[k] : r1[k];
    }
    wave_lds_fence();
    const bool urule = un.u_rule(r);
    double *out = F.dG + (size_t)un.item(r, nw) * L * 16;
    for (int q = lane; q < 16 * L; q += 64) {
      double v = 0.0;
      for (int z = 0; z < sh.slots; ++z) v += s_v[(z * L + (q >> 4)) * kTriRaw + (q & 15)];
      unsafeAtomicAdd(out + q, (urule && (q & 3) == 3) ? -v : v);
    }
  }
}

// ---------------------------------------------------------------------------
// T channel and the final sum
// ---------------------------------------------------------------------------
// A point contributes, with A0 A1 the pair's bundles and A2 A3 their images
// (A2 = A0 and A3 = A1 up to the sign of the l = d and k = d components, which
// cancels in the product, except on diagonal supports, where it is missing),
//   A0 A1 + A2 A3 = 2 X Y + 2 X' Y'
// per product: X, Y without the stored l = d components of diagonal supports,
// X', Y' those alone, negated.  The chalice and inverse chalice split alike.  A
// point therefore takes one entry of products (X, Y), and where a pair has
// diagonal supports a second one (X', Y'): a full entry, or, where A0 is
// exchanged and A1 is not (the points far from zero frequency, most of them), one of
// which row d of X' and column d of Y' are all there is (kModeEdge).  With an
// argument of exactly zero the exchange of A1 and A3 differs, and the two entries
// are the pairs themselves.
enum { kModeMain = 0, kModeImage = 1, kModeApart = 2, kModeEdge = 3 };
constexpr int kTriTPoints = 8;  // points described at a time, at most
constexpr int kTriEdges = 4;    // matrix instructions per wave for the kModeEdge entries, at most

// Entries lie in pairs, {entry 2 p, entry 2 p + 1} of an element side by side:
// one 16-byte read serves two.  Byte position of element (row, column) of a
// site's matrix: equal rows of all sites together, 64 bytes each, so that four
// sites with different residues (mod 4) lie in different banks (4.4 cycles per
// wave read, 8 to 10 otherwise).  Rows are a multiple of four sites where the
// padding is small, which makes this hold whatever the rows.
__host__ __device__ inline int tri_sites(int L) { return L >= 12 ? (L + 4) & ~3 : L + 1; }
__host__ __device__ inline int tri_el(int L, int site, int row, int col) {
  return ((row * tri_sites(L) + site) * 4 + col) * 16;
}
__host__ __device__ inline int tri_mat(int L) { return tri_sites(L) * 256; }  // bytes of the X (or Y) of a pair of entries

struct TriTLds {
  int dst, off, w, pos, c, loff, lw, lfl, head, loc, area, total;
};
__host__ __device__ inline int tri_t_lanes(int L, int threads) { return (16 * L + threads - 1) / threads * threads; }
__host__ __device__ inline TriTLds tri_t_lds(int nw, int L, int points, int entries, int threads) {
  TriTLds l;
  int o = 0;
  auto take = [&](int bytes) { int r = o; o += (bytes + 15) & ~15; return r; };
  take(nw * 8);
  l.dst = take(4 * 8 * L * 4);
  l.off = take(2 * points * 16);
  l.w = take(2 * points * 32);
  l.pos = take(2 * points * 16);
  l.c = take(2 * points * 8);
  l.loff = take(4 * points * 16);
  l.lw = take(4 * points * 32);
  l.lfl = take(4 * points * 4);
  l.head = take(16);
  l.loc = take(points * 64 * 8);
  const int bun = entries * tri_mat(L);
  const int sums = 4 * threads * 8 + tri_t_lanes(L, threads) * 8;  // a group's products and the sums of the lanes
  l.area = take(bun > sums ? bun : sums);
  l.total = o;
  return l;
}
// groups (of four instructions) per wave that pass through LDS together for the overlap sums
__host__ __device__ inline int tri_t_pass(int L, int entries, int threads) {
  const int g = (entries * tri_mat(L) / 8 - tri_t_lanes(L, threads)) / (4 * threads);
  return g < 1 ? 1 : g;
}

// NG: groups of four matrix instructions (16 products) per wave
template <int NG>
__global__ __launch_bounds__(512, NG <= 5 ? 4 : 2) void k_tri_t(TriDev F) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int nw = F.nw, L = F.L;
  const int nsu = nw * (nw + 1) / 2;
  const long long pos = xcd_position(blockIdx.x, (int)kTriChunk);
  if (pos >= (long long)nsu * nw) return;
  // items t-major: neighbouring workgroups share the mesh slab of their exact t
  const int X = (int)(pos / nsu), su = (int)(pos - (long long)X * nsu);
  const int so = __builtin_amdgcn_readfirstlane(tri_decode(su)), uo = su - so * (so + 1) / 2;
  const size_t item = (size_t)su * nw + X;
  const int nt = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int npt = F.t_points, nent = F.t_entries;
  const TriTLds lay = tri_t_lds(nw, L, npt, nent, nt);
  double *s_mesh = reinterpret_cast<double *>(lds_raw);
  int *s_dst = reinterpret_cast<int *>(lds_raw + lay.dst);
  int4 *s_off = reinterpret_cast<int4 *>(lds_raw + lay.off);         // [(point, pair)]
  double2 *s_w = reinterpret_cast<double2 *>(lds_raw + lay.w);       // [(point, pair)][2], negative: exchanged storage
  int4 *s_pos = reinterpret_cast<int4 *>(lds_raw + lay.pos);         // [(point, pair)] flags, byte positions of the two entries, mode
  double *s_c = reinterpret_cast<double *>(lds_raw + lay.c);         // [(point, pair)] factor
  int4 *s_loff = reinterpret_cast<int4 *>(lds_raw + lay.loff);       // [(point, local)]
  double2 *s_lw = reinterpret_cast<double2 *>(lds_raw + lay.lw);
  int *s_lfl = reinterpret_cast<int *>(lds_raw + lay.lfl);
  int4 *s_head = reinterpret_cast<int4 *>(lds_raw + lay.head);       // points, full entries, edge entries
  double *s_loc = reinterpret_cast<double *>(lds_raw + lay.loc);     // [(point, local)][16]
  unsigned char *area = lds_raw + lay.area;

  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void *)F.G, (short)0, (int)F.g_bytes, 0x00020000);
  const int rowbytes = L * 128;
  const int nch = 8 * L;
  const unsigned inv = div_factor(nch);
  const int mat = tri_mat(L);
  // byte position of full entry e, and of edge entry e (from the end)
  auto full_at = [&](int e) { return (e >> 1) * 2 * mat + (e & 1) * 8; };

  for (int i = tid; i < nw; i += nt) s_mesh[i] = F.mesh[i];
  for (int i = tid; i < 4 * nch; i += nt) s_dst[i] = F.t_dst[i];
  // (the second of a pair may be multiplied by zero before its first use)
  for (int i = tid; i < nent * mat / 16; i += nt) reinterpret_cast<double2 *>(area)[i] = make_double2(0.0, 0.0);
  // operand positions of the lane: left factor | first right factor << 16, second | third << 16, fourth
  int pk[NG][3];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int4 q = F.t_ops[(wave * NG + g) * 64 + lane];
    pk[g][0] = q.x;
    pk[g][1] = q.y;
    pk[g][2] = q.z;
  }
  const int nedge = F.t_edges;
  double C[NG][4], CE[kTriEdges];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) C[g][i] = 0.0;
#pragma unroll
  for (int i = 0; i < kTriEdges; ++i) CE[i] = 0.0;
  __syncthreads();

  // a lane always handles the same two stored components (k, l), (k, l + 1)
  const int pc = tid & 7;
  const bool dens = pc & 1, kd = pc >= 6;
  const int mask = dens ? -1 : 0x7fffffff;
  const int xt = kd ? -1 : 0, yt = kd != dens ? -1 : 0;
  // producer role (first wave): point pe, pair pp, argument pj: A (pj 0) and B
  // of pair 0: A = w1 - w', B = w1p + w'; pair 1: A = w2p - w', B = w2 + w'
  const int pe = lane >> 2, pp = (lane >> 1) & 1, pj = lane & 1;
  const int n = F.Wn[X];
  const double *Wwp = F.Wwp + (size_t)X * F.emax, *Wc = F.Wc + (size_t)X * F.emax;
  // describes the points from e0 on, as many as the entries allow
  auto describe = [&](int e0) {
    const double sm = s_mesh[so], tm = s_mesh[X], um = s_mesh[uo];
    const double half = 0.5 * (sm + (pj ? tm : -tm) + (pp ? -um : um));
    const bool ok = e0 + pe < n;
    const double wp = ok ? Wwp[e0 + pe] : 0.0, c = ok ? Wc[e0 + pe] : 0.0;
    const double v = pj ? half + wp : half - wp;
    const Bracket me = bracket_of(s_mesh, nw, fabs(v), F.geo, F.ga, F.gb);
    Bracket ot;
    ot.lo = pair_swap(me.lo);
    ot.step = pair_swap(me.step);
    ot.b = pair_swap(me.b);
    const double vo = pair_swap(v);
    const Bracket A = pj ? ot : me, B = pj ? me : ot;
    const double av = pj ? vo : v, bv = pj ? v : vo;
    // first buffer of the pair: s slot |A|, u slot |B|; lane pj describes the
    // supports of A's index pj
    const int ia = A.lo + (pj ? A.step : 0), b0 = B.lo, b1 = B.lo + B.step;
    const int2 off = make_int2(((b0 > ia ? tri(b0, ia) : tri(ia, b0)) * nw + X) * rowbytes,
                               ((b1 > ia ? tri(b1, ia) : tri(ia, b1)) * nw + X) * rowbytes);
    const double wa = pj ? A.b : 1.0 - A.b;
    const double w0 = wa * (1.0 - B.b), w1 = wa * B.b;
    const int mydiag = (b0 == ia ? 1 << (2 * pj) : 0) | (b1 == ia ? 2 << (2 * pj) : 0);
    const int diag = mydiag | pair_swap(mydiag);
    // site exchange and t / u sign of the pair's first buffer and of its image
    const bool ex = (av < 0) != (pp ? bv > 0 : bv < 0), exi = (bv < 0) != (pp ? av > 0 : av < 0);
    const bool tu = pp ? bv > 0 : bv < 0, tui = pp ? av > 0 : av < 0;
    // of the point: bit 0 diagonal supports, bit 1 pairs apart, bit 2 not an edge entry
    int any = (diag ? 1 : 0) | (pp && (av == 0.0 || bv == 0.0) ? 2 : 0) | ((diag && ex == (pp != 0)) || !nedge ? 4 : 0);
    any |= __shfl_xor(any, 2, 64);
    any |= __shfl_xor(any, 1, 64);
    const int mode = any & 2 ? kModeApart : (!(any & 1) ? kModeMain : (any & 4 ? kModeImage : kModeEdge));
    // entries before the point's among the batch's, and whether they fit
    const bool twice = mode == kModeImage || mode == kModeApart, mine = pp == 0 && pj == 0 && ok;
    const unsigned long long two = __ballot(mine && twice), edge = __ballot(mine && mode == kModeEdge);
    const unsigned long long before = (1ull << (lane & ~3)) - 1;
    const int f = pe + __popcll(two & before), d = __popcll(edge & before);
    const int f1 = f + (twice ? 2 : 1), d1 = d + (mode == kModeEdge ? 1 : 0);
    const bool fits = ok && pe < npt && ((f1 + 1) & ~1) + d1 <= nent;
    const unsigned long long taken = __ballot(mine && fits);
    if (!fits) return;
    if (lane == 63 - __builtin_clzll(taken)) s_head[0] = make_int4(__popcll(taken), f1, d1, 0);
    reinterpret_cast<int2 *>(s_off)[lane] = off;
    s_w[lane] = make_double2(ia < b0 ? -w0 : w0, ia < b1 ? -w1 : w1);
    if (pj == 0) {
      s_pos[2 * pe + pp] = make_int4((ex ? 1 : 0) | (tu ? 2 : 0) | (exi ? 4 : 0) | (tui ? 8 : 0) | diag << 4,
                                     full_at(f) + pp * mat, full_at(twice ? f + 1 : nent - 1 - d) + pp * mat, mode);
      s_c[2 * pe + pp] = pp ? 1.0 : (mode == kModeApart ? 0.5 * c : c);
    }
    // site-local vertex (u slot exact) with the same brackets: s slot this
    // lane's argument, t slot the other's; pair 1 with (v, -vo, t): l4 (pj
    // 0), l5; pair 0 with (v, -vo, -t): l6, l7
    int lo[4];
    double lw[4];
    int fx = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int is = me.lo + ((q & 1) ? me.step : 0), it = ot.lo + ((q & 2) ? ot.step : 0);
      lo[q] = ((is > X ? tri(is, X) : tri(X, is)) * nw + it) * rowbytes;
      lw[q] = ((q & 1) ? me.b : 1.0 - me.b) * ((q & 2) ? ot.b : 1.0 - ot.b);
      if (is < X) fx |= 4 << q;
    }
    const int l = 4 * pe + (pp ? pj : 2 + pj);
    s_loff[l] = make_int4(lo[0], lo[1], lo[2], lo[3]);
    s_lw[2 * l] = make_double2(lw[0], lw[1]);
    s_lw[2 * l + 1] = make_double2(lw[2], lw[3]);
    const bool lex = pp ? v < 0 : !(v < 0), ltu = pp ? vo > 0 : !(vo > 0);
    s_lfl[l] = fx | (lex ? 1 : 0) | (ltu ? 2 : 0);
  };
  if (wave == 0) describe(0);
  __syncthreads();

  for (int e0 = 0; e0 < n;) {
    const int4 head = s_head[0];
    const int np = __builtin_amdgcn_readfirstlane(head.x);
    const int nfull = __builtin_amdgcn_readfirstlane(head.y), nedges = __builtin_amdgcn_readfirstlane(head.z);
    // site-local vertices and their matrices, two points per wave: 8 lanes to
    // a vertex, two components each; then 16 lanes to a matrix
    for (int p2 = 2 * wave; p2 < np; p2 += nt / 32) {
      const int pt = p2 + (lane >> 5);
      const bool ok = pt < np;
      if (ok) {
        const int l = 4 * pt + ((lane >> 3) & 3), fl = s_lfl[l];
        const int4 o = s_loff[l];
        const double2 v0 = buf_load<double2>(rG, o.x + pc * 16), v1 = buf_load<double2>(rG, o.y + pc * 16);
        const double2 v2 = buf_load<double2>(rG, o.z + pc * 16), v3 = buf_load<double2>(rG, o.w + pc * 16);
        const double2 wa = s_lw[2 * l], wb = s_lw[2 * l + 1];
        // getValueLocal (src/TRI/TRIVertexTwoParticle.hpp:300-309): site 0; the
        // sign of exchanged storage goes by the exchanged components
        const bool ex = fl & 1;
        const int nx = ex && kd ? -1 : 0, ny = (ex ? kd : dens) ? -1 : 0;
        double x = flip_by(wa.x, (fl << 29) & nx) * v0.x, y = flip_by(wa.x, (fl << 29) & ny) * v0.y;
        x = fma(flip_by(wa.y, (fl << 28) & nx), v1.x, x);
        y = fma(flip_by(wa.y, (fl << 28) & ny), v1.y, y);
        x = fma(flip_by(wb.x, (fl << 27) & nx), v2.x, x);
        y = fma(flip_by(wb.x, (fl << 27) & ny), v2.y, y);
        x = fma(flip_by(wb.y, (fl << 26) & nx), v3.x, x);
        y = fma(flip_by(wb.y, (fl << 26) & ny), v3.y, y);
        const int k = pc >> 1, m = 2 * (pc & 1);
        s_loc[l * 16 + (ex ? 4 * m + k : 4 * k + m)] = flip_by(x, (fl << 30) & xt);
        s_loc[l * 16 + (ex ? 4 * (m + 1) + k : 4 * k + m + 1)] = flip_by(y, (fl << 30) & yt);
      }
      wave_lds_fence();
      if (ok) {
        // sides: 1 the chalice of l4, l5 (row i = nu, column j = t) in Y, 0 the
        // inverse chalice of l6, l7 (row r, column ka) in X
        const int side = (lane >> 4) & 1, ij = lane & 15, i = ij >> 2, j = ij & 3;
        const int4 ps = s_pos[2 * pt + side];
        const double *la = s_loc + (4 * pt + (side ? 0 : 2)) * 16, *lb = la + 16;
        const int lab = pauli_label(i) ^ pauli_label(j);
        const int neg = (int)((side ? kChaliceMask : kInverseMask) >> (4 * ij));
        double ka = 0.0, kb = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int o = 4 * k + pauli_comp(lab ^ pauli_label(k));
          ka += flip_by(la[o], neg << (31 - k));
          kb += flip_by(lb[o], neg << (31 - k));
        }
        const double c = s_c[2 * pt + side];
        const double kbd = flip(kb, (side ? i : j) == 3);
        const bool apart = ps.w == kModeApart;  // X carries half the weight there
        unsigned char *M = area + (side ? tri_el(L, L, i, j) : tri_el(L, L, j, i));
        *reinterpret_cast<double *>(M + ps.y) = c * (apart ? 2.0 * ka : ka + kbd);
        if (ps.w != kModeMain) *reinterpret_cast<double *>(M + ps.z) = c * (apart ? 2.0 * kb : kbd - ka);
      }
    }
    // bundles into the entries
    for (int q = tid; q < np * 2 * nch; q += nt) {
      const int id = fast_div(q, inv), ch = q - id * nch;
      const int4 o = s_off[id];
      const int *dst = s_dst + ((id & 1) ? 2 * nch : 0) + ch;
      const double2 v0 = buf_load<double2>(rG, o.x + ch * 16), v1 = buf_load<double2>(rG, o.y + ch * 16);
      const double2 v2 = buf_load<double2>(rG, o.z + ch * 16), v3 = buf_load<double2>(rG, o.w + ch * 16);
      const int4 ps = s_pos[id];
      const int fl = ps.x, mode = ps.w;
      const double2 wa = s_w[2 * id], wb = s_w[2 * id + 1];
      const double c = s_c[id];
      double x = fabs(wa.x) * v0.x;
      x = fma(fabs(wa.y), v1.x, x);
      x = fma(fabs(wb.x), v2.x, x);
      x = fma(fabs(wb.y), v3.x, x);
      double y = and_sign(wa.x, mask) * v0.y;
      y = fma(and_sign(wa.y, mask), v1.y, y);
      y = fma(and_sign(wb.x, mask), v2.y, y);
      y = fma(and_sign(wb.y, mask), v3.y, y);
      x *= c;
      y *= c;
      const int d = dst[(fl & 1) ? nch : 0];
      if (mode == kModeMain) {
        unsigned char *E = area + ps.y;
        *reinterpret_cast<double *>(E + (d & 0x7fff)) = flip_by(x, ((fl << 30) & xt) ^ (d << 16));
        *reinterpret_cast<double *>(E + ((d >> 16) & 0x7fff)) = flip_by(y, ((fl << 30) & yt) ^ d);
      } else {
        double dg = 0.0;  // l = d component of the diagonal supports
        if (dens) {
          dg = fl & 16 ? wa.x * v0.y : 0.0;
          dg = fma(fl & 32 ? wa.y : 0.0, v1.y, dg);
          dg = fma(fl & 64 ? wb.x : 0.0, v2.y, dg);
          dg = fma(fl & 128 ? wb.y : 0.0, v3.y, dg);
          dg *= c;
        }
        unsigned char *E = area + ps.y, *E2 = area + ps.z;
        *reinterpret_cast<double *>(E + (d & 0x7fff)) = flip_by(x, ((fl << 30) & xt) ^ (d << 16));
        *reinterpret_cast<double *>(E + ((d >> 16) & 0x7fff)) =
            flip_by(mode == kModeApart ? y : y - dg, ((fl << 30) & yt) ^ d);
        if (mode == kModeEdge) {
          // row d of X', in the exchanged places, and column d of Y', in the plain ones
          const int de = dst[(id & 1) ? 0 : nch];
          if (dens) *reinterpret_cast<double *>(E2 + ((de >> 16) & 0x7fff)) = flip_by(-dg, ((fl << 30) & yt) ^ de);
        } else {
          const int di = mode == kModeApart ? dst[(fl & 4) ? nch : 0] : d, ti = mode == kModeApart ? fl << 28 : fl << 30;
          const double x2 = mode == kModeApart ? x : 0.0;
          const double y2 = mode == kModeApart ? (dens ? fma(2.0, dg, -y) : y) : -dg;
          *reinterpret_cast<double *>(E2 + (di & 0x7fff)) = flip_by(x2, (ti & xt) ^ (di << 16));
          *reinterpret_cast<double *>(E2 + ((di >> 16) & 0x7fff)) = flip_by(y2, (ti & yt) ^ di);
        }
      }
    }
    // an odd number of entries: nothing from the other half of the last pair
    if (nfull & 1)
      for (int q = tid; q < mat / 16; q += nt) *reinterpret_cast<double *>(area + full_at(nfull) + q * 16) = 0.0;
    __syncthreads();
    e0 += np;
    if (wave == 0 && e0 < n) describe(e0);  // (the products do not read the descriptors)
    for (int p = 0; p < nfull; p += 2) {
      const unsigned char *E = area + p * mat;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // (unpacked here: the compiler would otherwise keep the positions apart)
        asm volatile("" : "+v"(pk[g][0]), "+v"(pk[g][1]), "+v"(pk[g][2]));
        const double2 a = *reinterpret_cast<const double2 *>(E + (pk[g][0] & 0xffff));
        const double2 b0 = *reinterpret_cast<const double2 *>(E + ((unsigned)pk[g][0] >> 16));
        const double2 b1 = *reinterpret_cast<const double2 *>(E + (pk[g][1] & 0xffff));
        const double2 b2 = *reinterpret_cast<const double2 *>(E + ((unsigned)pk[g][1] >> 16));
        const double2 b3 = *reinterpret_cast<const double2 *>(E + pk[g][2]);
        C[g][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b0.x, C[g][0], 0, 0, 0);
        C[g][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b1.x, C[g][1], 0, 0, 0);
        C[g][2] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b2.x, C[g][2], 0, 0, 0);
        C[g][3] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.x, b3.x, C[g][3], 0, 0, 0);
        C[g][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b0.y, C[g][0], 0, 0, 0);
        C[g][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b1.y, C[g][1], 0, 0, 0);
        C[g][2] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b2.y, C[g][2], 0, 0, 0);
        C[g][3] = __builtin_amdgcn_mfma_f64_4x4x4f64(a.y, b3.y, C[g][3], 0, 0, 0);
      }
    }
    if (nedges)
#pragma unroll
      for (int i = 0; i < kTriEdges; ++i) {
        if (i >= nedge) break;
        const unsigned q = F.t_edge_ops[(wave * nedge + i) * 64 + lane];
        for (int e = 0; e < nedges; ++e) {
          const unsigned char *E = area + full_at(nent - 1 - e);
          CE[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(*reinterpret_cast<const double *>(E + (q & 0xffff)),
                                                     *reinterpret_cast<const double *>(E + (q >> 16)), CE[i], 0, 0, 0);
        }
      }
    __syncthreads();
  }

  // overlap lists, S and U values, prefactor 1/(2 pi)
  const int rounds = (16 * L + nt - 1) / nt, lanes = rounds * nt;
  double *s_C = reinterpret_cast<double *>(area), *s_part = s_C + F.t_pass * 4 * nt;
  const int *plan = F.t_plan;
  double *out = F.dG + item * 16 * L;
  double sum[2] = {0.0, 0.0};  // outputs tid and tid + nt (more, on many sites and few waves, are summed in memory)
  for (int g0 = 0; g0 < NG + (nedge ? 1 : 0); g0 = g0 < NG && g0 + F.t_pass >= NG ? NG : g0 + F.t_pass) {
    __syncthreads();
#pragma unroll
    for (int g = 0; g < NG; ++g)
      if (g >= g0 && g < g0 + F.t_pass)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_C[((wave * F.t_pass + g - g0) * 4 + i) * 64 + lane] = C[g][i];
    if (g0 == NG)
#pragma unroll
      for (int i = 0; i < kTriEdges; ++i) s_C[(wave * 4 + i) * 64 + lane] = CE[i];
    const int quads = plan[0], *lane_of = plan + 1, *count = lane_of + 16 * L + 1;
    const uint4 *ent = reinterpret_cast<const uint4 *>(plan + ((2 + 16 * L + lanes + 3) & ~3));
    __syncthreads();
    for (int l = tid; l < lanes; l += nt) s_part[l] = plan_sum(ent + l, lanes, count[l], s_C);
    __syncthreads();
    for (int r = 0; r < rounds; ++r) {
      const int q = r * nt + tid;
      if (q >= 16 * L) break;
      double v = 0.0;
      for (int l = lane_of[q], l1 = lane_of[q + 1]; l < l1; ++l) v += s_part[l];
      if (r == 0) sum[0] += v;
      else if (r == 1) sum[1] += v;
      else out[q] = fma(tri_hat(q & 15), v, out[q]);
    }
    plan = reinterpret_cast<const int *>(ent + (size_t)quads * lanes);
  }
  for (int r = 0; r < rounds; ++r) {
    const int q = r * nt + tid;
    if (q >= 16 * L) break;
    double v = out[q];
    if (r < 2) v = fma(tri_hat(q & 15), r ? sum[1] : sum[0], v);
    v *= 1.0 / kTwoPi;
    out[q] = v;
    if (isnan(v)) atomicOr(&F.flags[0], 1);
  }
}

// ---------------------------------------------------------------------------
// host: tables of k_tri_t
// ---------------------------------------------------------------------------
// Products (left site, right site, Q): rows of the right factor through the
// spin permutation Q = P2 P1^-1 of the overlap entries that refer to it.  Site
// L is the matrix of the site-local vertices.
struct TriPlan {
  int waves = 0, ng = 0, points = 0, entries = 0, pass = 0, edges = 0, lds = 0;
  std::vector<int> dst, plan, edge_ops;
  std::vector<int4> ops;
  bool ok = false;
};
inline bool tri_is_perm(const int *q) { return (1 << q[0] | 1 << q[1] | 1 << q[2]) == 7; }

inline TriPlan build_tri_plan(const sp_tri_problem *p) {
  TriPlan r;
  const int L = p->L;
  if (L > kMaxTriRhsL) return r;
  std::vector<int> source(L, -1);  // source[stored site] = site whose exchanged bundle reads it
  for (int j = 0; j < L; ++j) {
    if (p->site_rid[j] != j || source[p->inv_rid[j]] >= 0 || !tri_is_perm(p->inv_perm + 3 * j)) return r;
    for (int c = 0; c < 3; ++c)
      if (p->site_perm[3 * j + c] != c) return r;
    source[p->inv_rid[j]] = j;
  }
  // positions of two neighbouring stored components in an entry's X and Y,
  // plain and exchanged, bit 15 of each half the sign hat_sign
  r.dst.resize(4 * 8 * (size_t)L);
  for (int side = 0; side < 2; ++side)
    for (int ex = 0; ex < 2; ++ex)
      for (int ch = 0; ch < 8 * L; ++ch) {
        const int stored = ch >> 3, site = ex ? source[stored] : stored;
        int inv[4] = {0, 1, 2, 3};
        if (ex)
          for (int c = 0; c < 3; ++c) inv[p->inv_perm[3 * site + c]] = c;
        unsigned code = 0;
        for (int h = 0; h < 2; ++h) {
          const int k = (ch & 7) >> 1, l = 2 * (ch & 1) + h;
          const int s1 = ex ? inv[l] : k, s2 = ex ? inv[k] : l;
          const unsigned at = side ? tri_el(L, site, s1, s2) : tri_el(L, site, s2, s1);
          code |= (at | (hat_sign(s1, s2) < 0 ? 0x8000u : 0u)) << (16 * h);
        }
        r.dst[(2 * side + ex) * 8 * L + ch] = (int)code;
      }
  // products, by left site
  struct Product {
    int right, q[4];
    int at;  // instruction * 4 + block
  };
  std::vector<std::vector<Product>> left(L + 1);
  auto product = [&](int j1, int j2, const int *q) -> Product & {
    for (Product &x : left[j1])
      if (x.right == j2 && x.q[0] == q[0] && x.q[1] == q[1] && x.q[2] == q[2]) return x;
    left[j1].push_back(Product{j2, {q[0], q[1], q[2], 3}, -1});
    return left[j1].back();
  };
  const int none[3] = {0, 1, 2};
  auto quotient = [&](int i, int (&q)[3]) {
    const int *a = p->ovl_perm1 + 3 * i, *b = p->ovl_perm2 + 3 * i;
    for (int c = 0; c < 3; ++c) q[a[c]] = b[c];
  };
  for (int j = 0; j < L; ++j) {
    product(j, L, none);
    product(L, j, none);
  }
  int q[3];
  for (int i = 0; i < p->ovl_off[L]; ++i) {
    quotient(i, q);
    product(p->ovl_rid1[i], p->ovl_rid2[i], q);
  }
  // runs of four products with a common left factor, by the residue of its
  // site; a group takes four runs of different residues where there are such
  struct Run {
    int left;
    Product *x[4];
  };
  std::vector<Run> by[4];
  int nruns = 0;
  for (int j = 0; j <= L; ++j)
    for (size_t k = 0; k < left[j].size(); k += 4) {
      Run u{j, {nullptr, nullptr, nullptr, nullptr}};
      for (size_t z = 0; z < 4 && k + z < left[j].size(); ++z) u.x[z] = &left[j][k + z];
      by[j & 3].push_back(u);
      ++nruns;
    }
  const int groups = (nruns + 3) / 4;
  int waves = 1;
  // More waves per item shorten the phases between barriers: up to four while a
  // wave has more than three groups (honeycomb r3, 5 sites, at cutoff 0.02: 0.171 ->
  // 0.145 ms, kagome r3, 8 sites: 2.17 -> 2.01 ms; fewer groups gain nothing:
  // kagome r2, 4 sites, 2.14 ms, 2.20 with two waves).  More than five groups do not fit the
  // registers of four waves per SIMD; then eight waves.
  while (waves < 4 && (groups + waves - 1) / waves > 3) waves *= 2;
  while (waves < 8 && (groups + waves - 1) / waves > 5) waves *= 2;
  const int ng = (groups + waves - 1) / waves, nt = 64 * waves;
  if (ng > kTriMaxGroups) return r;
  std::vector<Run> order(4 * (size_t)waves * ng, Run{L, {nullptr, nullptr, nullptr, nullptr}});
  for (int k = 0; k < nruns; ++k) {
    int best = -1;
    for (int c = 0; c < 4; ++c) {
      bool used = false;
      for (int b = k & ~3; b < k; ++b) used = used || (order[b].left & 3) == c;
      if (!by[c].empty() && (best < 0 || (int)by[c].size() - (used ? 4096 : 0) > best))
        best = (int)by[c].size() - (used ? 4096 : 0);
    }
    for (int c = 0; c < 4; ++c) {
      bool used = false;
      for (int b = k & ~3; b < k; ++b) used = used || (order[b].left & 3) == c;
      if (!by[c].empty() && (int)by[c].size() - (used ? 4096 : 0) == best) {
        order[k] = by[c].back();
        by[c].pop_back();
        break;
      }
    }
  }
  // the products of a run in the order that meets the fewest equal banks
  for (size_t g = 0; g < order.size() / 4; ++g)
    for (int b = 1; b < 4; ++b) {
      Run &u = order[4 * g + b];
      int perm[4] = {0, 1, 2, 3}, best[4] = {0, 1, 2, 3}, cost = 1 << 30;
      do {
        int c = 0;
        for (int z = 0; z < 4; ++z)
          for (int o = 0; o < b; ++o) {
            const Product *x = u.x[perm[z]], *y = order[4 * g + o].x[z];
            if (x && y)
              for (int k = 0; k < 4; ++k) {
                const int S = tri_sites(L);
                c += ((x->q[k] * S + x->right) & 3) == ((y->q[k] * S + y->right) & 3);
              }
          }
        if (c < cost) {
          cost = c;
          std::copy(perm, perm + 4, best);
        }
      } while (std::next_permutation(perm, perm + 4));
      const Run was = u;
      for (int z = 0; z < 4; ++z) u.x[z] = was.x[best[z]];
    }
  // operands: group g of wave w is group w ng + g
  r.ops.resize(64 * (size_t)waves * ng);
  const int right0 = tri_mat(L);
  for (int g = 0; g < waves * ng; ++g) {
    for (int b = 0; b < 4; ++b)
      for (int z = 0; z < 4; ++z)
        if (order[4 * g + b].x[z]) order[4 * g + b].x[z]->at = (4 * g + z) * 4 + b;
    for (int lane = 0; lane < 64; ++lane) {
      const int k = lane >> 4, b = (lane >> 2) & 3, i = lane & 3;
      const Run &u = order[4 * g + b];
      int o[4];
      for (int z = 0; z < 4; ++z) o[z] = right0 + (u.x[z] ? tri_el(L, u.x[z]->right, u.x[z]->q[k], i) : tri_el(L, L, k, i));
      r.ops[64 * (size_t)g + lane] = make_int4(tri_el(L, u.left, k, i) | o[0] << 16, o[1] | o[2] << 16, o[3], 0);
    }
  }
  // edge entries: blocks of four left and four right sites, row d of X' and
  // column d of Y' (or the matrices of the site-local vertices)
  struct Block {
    int left, right, q[4];  // fours of sites, -1: site L
  };
  std::vector<Block> blocks;
  auto block = [&](int l, int rt, const int *qq) -> int {
    for (size_t k = 0; k < blocks.size(); ++k)
      if (blocks[k].left == l && blocks[k].right == rt && blocks[k].q[0] == qq[0] && blocks[k].q[1] == qq[1] &&
          blocks[k].q[2] == qq[2])
        return (int)k;
    blocks.push_back(Block{l, rt, {qq[0], qq[1], qq[2], 3}});
    return (int)blocks.size() - 1;
  };
  for (int j = 0; j < L; j += 4) {
    block(j >> 2, -1, none);
    block(-1, j >> 2, none);
  }
  for (int i = 0; i < p->ovl_off[L]; ++i) {
    quotient(i, q);
    block(p->ovl_rid1[i] >> 2, p->ovl_rid2[i] >> 2, q);
  }
  const int edges = ((int)blocks.size() + 4 * waves - 1) / (4 * waves);
  if (edges <= kTriEdges) {
    r.edges = edges;
    r.edge_ops.resize(64 * (size_t)waves * edges);
    for (int z = 0; z < waves * edges; ++z)
      for (int lane = 0; lane < 64; ++lane) {
        const int k = lane >> 4, i = lane & 3;
        const Block x = 4 * z + ((lane >> 2) & 3) < (int)blocks.size() ? blocks[4 * z + ((lane >> 2) & 3)]
                                                                     : Block{-1, -1, {0, 1, 2, 3}};
        const int l = 4 * x.left + i, rt = 4 * x.right + i;
        const int a = x.left < 0 || l >= L ? tri_el(L, L, k, i) : tri_el(L, l, k, 3);
        const int b = x.right < 0 || rt >= L ? tri_el(L, L, x.q[k], i) : tri_el(L, rt, x.q[k], 3);
        r.edge_ops[64 * (size_t)z + lane] = a | (right0 + b) << 16;
      }
  }
  // 16 waves per CU (8 where the sums need more registers)
  const int budget = 160 * 1024 * waves / (ng <= 5 ? 16 : 8);
  r.points = waves >= 4 ? kTriTPoints : kTriTPoints / 2;
  int entries = 2 * r.points;
  while (entries > 4 && tri_t_lds(p->nw, L, r.points, entries, nt).total > budget) entries -= 2;
  r.entries = entries;
  r.pass = tri_t_pass(L, entries, nt);
  if (r.pass > ng) r.pass = ng;
  r.lds = tri_t_lds(p->nw, L, r.points, entries, nt).total;
  r.waves = waves;
  r.ng = ng;
  // sums over the overlap lists, per pass: 4 times the bubble products, the
  // chalice and inverse chalice products once; the element (row, column) of
  // a product is in lane 16 row + 4 block + column of its instruction's result
  const int lanes = tri_t_lanes(L, nt);
  auto append = [&](LanePlan &plan) {
    plan.deal(lanes);
    const size_t head = (2 + 16 * (size_t)L + lanes + 3) & ~(size_t)3, at0 = r.plan.size();
    r.plan.resize(at0 + head + plan.entries());
    int *o = r.plan.data() + at0;
    o[0] = plan.quads();
    std::copy_n(plan.lane_of.begin(), 16 * L + 1, o + 1);
    plan.store(reinterpret_cast<unsigned *>(o + head), o + 2 + 16 * L);
  };
  for (int g0 = 0; g0 < ng; g0 += r.pass) {
    LanePlan plan;
    plan.begin((size_t)waves * r.pass * 256, 16 * L);
    for (int rid = 0; rid < L; ++rid)
      for (int c = 0; c < 16; ++c) {
        auto add = [&](int at, int row, int col, int times) {
          const int g = at >> 4, w = g / ng, gi = g - w * ng;
          if (gi < g0 || gi >= g0 + r.pass) return;
          const unsigned e = ((w * r.pass + gi - g0) * 4 + ((at >> 2) & 3)) * 64 + 16 * row + 4 * (at & 3) + col;
          plan.add(e, times);
        };
        const int s1 = c >> 2, s2 = c & 3;
        add(product(rid, L, none).at, s1, s2, 1);
        add(product(L, rid, none).at, s1, s2, 1);
        for (int i = p->ovl_off[rid]; i < p->ovl_off[rid + 1]; ++i) {
          quotient(i, q);
          add(product(p->ovl_rid1[i], p->ovl_rid2[i], q).at, s1 < 3 ? p->ovl_perm1[3 * i + s1] : 3,
              s2 < 3 ? p->ovl_perm2[3 * i + s2] : 3, 4);
        }
        plan.end_output();
      }
    append(plan);
  }
  if (r.edges) {
    LanePlan plan;
    plan.begin((size_t)waves * 256, 16 * L);
    for (int rid = 0; rid < L; ++rid)
      for (int c = 0; c < 16; ++c) {
        auto add = [&](int b, int row, int col, int times) {
          const int z = b >> 2, w = z / r.edges, zi = z - w * r.edges;
          plan.add((w * 4 + zi) * 64 + 16 * row + 4 * (b & 3) + col, times);
        };
        const int s1 = c >> 2, s2 = c & 3;
        if (s1 == 3) add(block(rid >> 2, -1, none), rid & 3, s2, 1);
        if (s2 == 3) add(block(-1, rid >> 2, none), s1, rid & 3, 1);
        if (c == 15)
          for (int i = p->ovl_off[rid]; i < p->ovl_off[rid + 1]; ++i) {
            quotient(i, q);
            add(block(p->ovl_rid1[i] >> 2, p->ovl_rid2[i] >> 2, q), p->ovl_rid1[i] & 3, p->ovl_rid2[i] & 3, 4);
          }
        plan.end_output();
      }
    append(plan);
  }
  r.ok = true;
  return r;
}
