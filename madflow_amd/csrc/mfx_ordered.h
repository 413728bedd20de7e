// Colour-ordered evaluation of g g > t t~ + n gluons, for processes whose colour flows
// (n! jamps) do not fit the register file next to a Feynman-diagram program.
//
// The jamps are the coefficients of the fundamental-string colour basis
// (T^{a_s1} ... T^{a_sn})_{i_t j_tbar}, the basis of the generated modules'
// jamp lines (madgraph_plugin/PyOut_exporter.py:334-375).  For one ordering s of the
// gluons the jamp is the colour-ordered amplitude, computed by the Berends-Giele
// recursion over consecutive ranges of s (no Feynman diagram is enumerated):
//
//   J(i..j) = 1/P^2 [ GC_10 sum_{i<=k<j} N3(J(i..k), J(k+1..j))
//                     + (-i GC_12) sum_{i<=k<l<j} N4(J(i..k), J(k+1..l), J(l+1..j)) ]
//   O(0) = top,  O(j) = sum_{i<j} FFV1_1(O(i), J(i..j-1))
//   jamp_s = - sum_{i<n} FFV1_0(anti-top, O(i), J(i..n-1))
//
// N3 is the VVV1 Lorentz structure of VVV1P0_1 without its propagator; the colour-
// ordered coefficient of the f^{abc} vertex (-i for the ordered word) cancels its i.
// N4 = 2 V3 (V2.V4) - V2 (V3.V4) - V4 (V2.V3) is the combination VVVV4 - VVVV1 of the
// SM four-gluon Lorentz structures that the word order selects.  The -1 is the
// fermion-flow factor of the generated jamps.  Summed over the Feynman diagrams
// consistent with an ordering, these give exactly the jamp of that ordering.
//
// Kernel 1 (k_ordered_jamps in FP32, k_ordered_mirror in FP64): one event per lane; each
// finished jamp is stored to a workspace [helicity][colour][event] (coalesced), so no lane
// ever holds more than one ordering's currents.
// Kernel 2 (k_colour_mfma): |M|^2 = sum_h Re(J_h^dagger CF J_h) / (CF_DEN * DENOMINATOR)
// as a batched dense contraction on the matrix cores: per helicity, the integer colour
// matrix (NCOLOR x NCOLOR) times a 16-event tile of Re J and Im J (NCOLOR x 16) with
// v_mfma_{f32,f64}_16x16x4, then the column-wise dot product with J.
#pragma once
#include "mfx_smatrix.h"

namespace mfx {

typedef float mfx_f32x4 __attribute__((ext_vector_type(4)));
typedef double mfx_f64x4 __attribute__((ext_vector_type(4)));

// Lorentz structure of VVV1P0_1 without coupling or propagator; V1 slots = V2 + V3.
// With P1 = -(P2 + P3) it reads (V2.V3)(P3 - P2) + V2 (2 V3.P2 + V3.P3) - V3 (V2.P2 + 2 V2.P3).
// Colour-ordered currents of gluons alone are conserved, P.J(i..j) = 0 (external gluons
// on shell and transverse; Berends and Giele, Nucl. Phys. B306 (1988) 759), so the
// V2.P2 and V3.P3 terms vanish and are left out.  d = V2.V3, the dot product the
// structure contains (the four-gluon sums reuse it).
template <class R>
__device__ __forceinline__ void vvv_numerator(const W<R>& V2, const W<R>& V3, W<R>& N, cx<R>& d) {
  R P2[4], P3[4];
  mom_in(V2, P2);
  mom_in(V3, P3);
  N[0] = V2[0] + V3[0];
  N[1] = V2[1] + V3[1];
  const cx<R> TMP2 = mdotp(V3, P2), TMP4 = mdotp(V2, P3);
  const cx<R> TMP5 = mdot(V3, V2);
  const cx<R> c2 = TMP2 + TMP2, c3 = -(TMP4 + TMP4);
#pragma unroll
  for (int mu = 0; mu < 4; ++mu) N[2 + mu] = TMP5 * (P3[mu] - P2[mu]) + V2[2 + mu] * c2 + V3[2 + mu] * c3;
  d = TMP5;
}

// N[2..5] += c V
template <class R>
__device__ __forceinline__ void add_scaled(W<R>& N, const W<R>& V, cx<R> c) {
#pragma unroll
  for (int mu = 2; mu < 6; ++mu) N[mu] += V[mu] * c;
}

template <class R>
__device__ __forceinline__ void add_components(W<R>& acc, const W<R>& t) {
#pragma unroll
  for (int k = 2; k < 6; ++k) acc[k] += t[k];
}

// Colour-ordered currents of one word.  J[i][j] (i <= j) is the gluon current of the
// word positions i..j (J[i][i] = the gluon itself), O[j] the top line carrying the top and
// the first j gluons.  FP32 forms only: P^2 of the gluons at word positions i..j (summed
// where the range's propagator is applied) and rt[j] = P^2 - m_t^2 of the top with the
// first j gluons are sums of the pair invariants pp[a][b] = 2 k_a.k_b (computed in FP64
// per event and rounded once).  Incoming
// momenta enter negated, so these sums can cancel: rt[j] is taken from the shorter of its
// two equal forms, the top with the first j gluons or the anti-top with the others
// (momentum conservation), and of two forms of equal length from the one with the smaller
// sum of magnitudes (summing the top with the first j gluons throughout lost up to 1e-4 of
// |M|^2 in FP32).  All indices are compile-time constants after unrolling, so every
// current lives in registers.
//
// The four-gluon sum of J(i..j) runs over the splits i <= k < l < j into
// V2 = J(i..k), V3 = J(k+1..l), V4 = J(l+1..j).  Two of its three terms only involve dot
// products of adjacent ranges, and summed over one split index those are
// S(a..b) = sum_{a<=m<b} J(a..m).J(m+1..b), the dot products of the three-gluon sum of
// range a..b (kept in S[a][b]):
//   sum_{k<l} V2 (V3.V4) = sum_{i<=k<j-1} J(i..k) S(k+1..j)
//   sum_{k<l} V4 (V2.V3) = sum_{i<l<j}   J(l+1..j) S(i..l)
// so only the 2 V3 (V2.V4) term needs a dot product per split pair.

// J(i..j) (and S(i..j)) for every range ending at j in [J0, J1), shorter ranges first.
template <int NG, int J0, int J1, class R>
__device__ __forceinline__ void ordered_ranges(W<R> (&J)[NG][NG], cx<R> (&S)[NG][NG], const R (&pp)[NG][NG],
                                               const Params<R>& prm) {
  constexpr bool INV = StableForms<R>::value;
  // -i GC_12 multiplies the four-gluon structures (GC_12 = i gs^2: a real gs^2)
  const cx<R> c4 = mul_mi(prm.GC_12);
#pragma unroll
  for (int j = J0; j < J1; ++j) {
#pragma unroll
    for (int i = j - 1; i >= 0; --i) {
      W<R> N3;
      cx<R> sd;
      vvv_numerator(J[i][i], J[i + 1][j], N3, sd);
#pragma unroll
      for (int k = i + 1; k < j; ++k) {
        W<R> t;
        cx<R> d;
        vvv_numerator(J[i][k], J[k + 1][j], t, d);
        add_components(N3, t);
        sd += d;
      }
      S[i][j] = sd;
      W<R> N4;
      N4[0] = N3[0];
      N4[1] = N3[1];
#pragma unroll
      for (int q = 2; q < 6; ++q) N4[q] = cx<R>(R(0), R(0));
#pragma unroll
      for (int k = i; k < j; ++k)
#pragma unroll
        for (int l = k + 1; l < j; ++l) {
          const cx<R> d24 = mdot(J[i][k], J[l + 1][j]);
          add_scaled(N4, J[k + 1][l], d24 + d24);
        }
#pragma unroll
      for (int k = i; k < j - 1; ++k) add_scaled(N4, J[i][k], -S[k + 1][j]);
#pragma unroll
      for (int l = i + 1; l < j; ++l) add_scaled(N4, J[l + 1][j], -S[i][l]);
      // propagator 1/P^2 of the massless gluon
      R den2;
      if constexpr (INV) {
        // P^2 of the gluons at word positions i..j: the sum of their pair invariants
        den2 = R(0);
#pragma unroll
        for (int a = i; a <= j; ++a)
#pragma unroll
          for (int b = a + 1; b <= j; ++b) den2 += pp[a][b];
      } else {
        R P[4];
        mom_out(N3, P);
        den2 = den_from_slots(P, R(0));
      }
      const R rden = recip(den2);
      const cx<R> k3 = prm.GC_10 * rden, k4 = c4 * rden;
      W<R>& o = J[i][j];
      o[0] = N3[0];
      o[1] = N3[1];
#pragma unroll
      for (int q = 2; q < 6; ++q) o[q] = k3 * N3[q] + k4 * N4[q];
    }
  }
}

// O(j) for j in [O0, O1]: O(j) = sum_{i<j} FFV1_1(O(i), J(i..j-1)).  Every term has the
// off-shell momentum of O(j) (top + gluons 0..j-1), so the gamma.J O columns are summed
// and the top propagator is applied once per j.
template <int NG, int O0, int O1, class R>
__device__ __forceinline__ void ordered_top_line(W<R> (&O)[NG], const W<R> (&J)[NG][NG], const R (&rt)[NG],
                                                 const Params<R>& prm) {
#pragma unroll
  for (int j = O0; j <= O1; ++j) {
    VslashF<R> x = vslash_f(O[0], J[0][j - 1]);
#pragma unroll
    for (int i = 1; i < j; ++i) add_col(x, vslash_f(O[i], J[i][j - 1]));
    O[j][0] = O[0][0] + J[0][j - 1][0];
    O[j][1] = O[0][1] + J[0][j - 1][1];
    R P[4];
    mom_out(O[j], P);
    ffv1_1_col(x, prm.GC_11, prm.mdl_MT, prm.mdl_WT, rt[j], P, O[j]);
  }
}

// The closing vertex: jamp = -sum_{i<NG} FFV1_0(anti-top, O(i), J(i..NG-1)).  It is linear
// in the sum of the gamma.J(i..NG-1) O(i) columns, formed once for both anti-top
// helicities (ordered_jamp dots it with each anti-top spinor).
template <int NG, class R>
__device__ __forceinline__ VslashF<R> ordered_close_col(const W<R> (&O)[NG], const W<R> (&J)[NG][NG]) {
  VslashF<R> x = vslash_f(O[0], J[0][NG - 1]);
#pragma unroll
  for (int i = 1; i < NG; ++i) add_col(x, vslash_f(O[i], J[i][NG - 1]));
  return x;
}
template <class R>
__device__ __forceinline__ cx<R> ordered_jamp(const W<R>& atop, const VslashF<R>& x, const Params<R>& prm) {
  return -ffv1_0_col(atop, x, prm.GC_11);
}

// The top line and closing column of a word (REV = false) or of its reversal, from the word's
// currents: a colour-ordered gluon current of m letters is (-1)^(m + 1) times that of the
// letters reversed (Berends and Giele, as above).  The momentum slots of currents of two or
// more letters are not read.
template <class R> __device__ __forceinline__ void sub_col(VslashF<R>& acc, const VslashF<R>& x) {
  acc.c2 -= x.c2;
  acc.c3 -= x.c3;
  acc.c4 -= x.c4;
  acc.c5 -= x.c5;
}
// sum over i of gamma.J(i..last) O(i)
template <bool REV, int NG, class R>
__device__ __forceinline__ VslashF<R> word_col(const W<R> (&O)[NG], const W<R> (&J)[NG][NG], int last) {
  VslashF<R> x = vslash_f(O[last], REV ? J[NG - 1 - last][NG - 1 - last] : J[last][last]);
#pragma unroll
  for (int i = 0; i < last; ++i) {
    const VslashF<R> t = vslash_f(O[i], REV ? J[NG - 1 - last][NG - 1 - i] : J[i][last]);
    if (REV && (last - i) % 2) sub_col(x, t);
    else add_col(x, t);
  }
  return x;
}
// O(1..NG-1), then the closing column
template <bool REV, int NG, class R>
__device__ __forceinline__ VslashF<R> word_top_line(W<R> (&O)[NG], const W<R> (&J)[NG][NG], const Params<R>& prm) {
#pragma unroll
  for (int j = 1; j < NG; ++j) {
    const VslashF<R> x = word_col<REV>(O, J, j - 1);
    const int k = REV ? NG - j : j - 1;
    O[j][0] = O[j - 1][0] + J[k][k][0];
    O[j][1] = O[j - 1][1] + J[k][k][1];
    R P[4];
    mom_out(O[j], P);
    ffv1_1_col(x, prm.GC_11, prm.mdl_MT, prm.mdl_WT, den_from_slots(P, prm.mdl_MT), P, O[j]);
  }
  return word_col<REV>(O, J, NG - 1);
}

// The walk of the FP64 kernel: NC / 2 words in cycles of rotations.  Cycle m starts with the m-th
// permutation (in lexicographic order) whose first letter is 0 and whose second is below its
// last; the next word moves the first letter to the end.  The words and their reversals are
// all orderings.  at[c] and rev[c]: the colour rows (lexicographic numbers) of word c and of
// its reversal.
template <int NG, int NC>
struct MirrorWalk {
  static_assert(NC <= 256, "colour rows are bytes");
  unsigned char at[NC / 2], rev[NC / 2];
};
template <int NG, int NC>
constexpr MirrorWalk<NG, NC> mirror_walk() {
  MirrorWalk<NG, NC> t{};
  int n = 0;
  for (int m = 0; m < NC / NG; ++m) {                 // permutations with first letter 0
    int w[NG] = {}, used[NG] = {}, rem = m, fact = NC / NG;
    used[0] = 1;
    for (int k = 1; k < NG; ++k) {                    // digits of m in the factorial base
      fact /= NG - k;
      int d = rem / fact, x = 1;
      rem %= fact;
      while (used[x] || d-- > 0) ++x;
      w[k] = x;
      used[x] = 1;
    }
    if (w[1] > w[NG - 1]) continue;
    for (int r = 0; r < NG; ++r, ++n)
      for (int way = 0; way < 2; ++way) {
        int rank = 0, f = NC;
        for (int k = 0; k < NG; ++k) {
          const int a = w[(r + (way ? NG - 1 - k : k)) % NG];
          int less = 0;
          for (int l = k + 1; l < NG; ++l) less += w[(r + (way ? NG - 1 - l : l)) % NG] < a;
          f /= NG - k;
          rank += less * f;
        }
        (way ? t.rev : t.at)[n] = (unsigned char)rank;
      }
  }
  return t;
}
template <int NG, int NC>
__constant__ constexpr MirrorWalk<NG, NC> MIRROR_WALK = mirror_walk<NG, NC>();

// the top-line currents O(1..N-1) of both top helicities (empty when unused)
template <class R, int N, bool ON> struct TopPrefix { W<R> o[2][N]; };
template <class R, int N> struct TopPrefix<R, N, false> {};

struct OrderedArgs {
  SmatrixArgs s;
  int64_t ev0;          // first event of this sub-chunk
  int64_t n;            // events in this sub-chunk
  int64_t ld;           // jbuf row stride in events: n rounded up to a 16-event tile, so that
                        // every tile of a colour row is whole 128-byte lines
  int h0, nhel;         // helicity rows h0 .. h0+nhel-1 (or 1 row for an explicit vector)
  int cparts, cper;     // orderings in cparts ranges of cper (even) each, one per block
  void* jbuf;           // [nhel][NCOLOR][n] complex R
};

// Per-lane staging of the FP32 kernel in LDS (lane-major: slot s of lane t at s * BLOCK + t), an
// indexable store: the gluon wavefunctions and the pair invariants are read back in the
// order of each colour ordering (the ordering index is wave-uniform).
template <class T, bool EXPLICIT>
struct OrderedStage {
  static constexpr int NG = T::NG;
  // FP32 runs two waves a SIMD, since one wave alone does not keep its VALU issuing; that takes
  // at most 256 registers a lane, and at most 80 slots here for 8 waves to fit a CU's 160 KB.
  // Four gluons (102 slots in full): COMPACT leaves out what is known to be zero, the
  // polarisations' time component and the imaginary part of their z component (not with an
  // explicit helicity vector, whose BRST polarisation fills all four real parts), the
  // fermions' momenta and one number of the anti-top.  Five gluons: the fermions' spinors, 40
  // slots, go to private memory, read back from cache with a run-time helicity.
  // t t~ g g, 1,048,576 events: 102 slots (6 waves a CU) 35.2 ms, 82 slots (7) 29.9 ms, 80 slots (8)
  // 26.8 ms; spinors in private memory 28.7 ms, and three waves a SIMD with them 29.8 ms (272 B of
  // spills).  t t~ g g g, 50,000 events: one wave a SIMD 33.7 ms, two with 120 slots (5 waves a CU)
  // 32.2 ms, with 80 slots 26.6 ms although 224 B spill.
  // An explicit helicity vector has one row, so one helicity of each fermion (SINGLE): 78 slots
  // (131,072 events, one row: 102 slots 304 us, 78 slots 199 us); five gluons take both calls with
  // the same layout.
  static constexpr bool COMPACT = !EXPLICIT && NG <= 4, SINGLE = EXPLICIT && NG <= 4;
  static constexpr int GW = COMPACT ? 9 : 12;
  static constexpr int NWF = NG * GW;
  // the pair invariants gluon-gluon and top-gluon (pair_index), then anti-top-gluon
  static constexpr int NPI = (NG + 1) * NG / 2, NINV = NPI + NG;
  // the spinor components of the top and the anti-top at both helicities, staged once per event
  static constexpr int FB = NWF + NINV;
  static constexpr bool PRIVATE = NG > 4;           // the spinors in private memory
  static constexpr int NFM = PRIVATE ? 4 : 0;       // momentum slots of a fermion
  static constexpr int NFS = PRIVATE ? 40 : (SINGLE ? 16 : 30);
  static constexpr int NSLOT = NWF + NINV + (PRIVATE ? 0 : NFS);
  static_assert(NSLOT <= 80, "eight waves a CU");
  // slot of component q (its real part; the imaginary part follows) of the top (anti = 0) or
  // the anti-top at helicity bit h
  static constexpr __device__ int fermion(int anti, int h, int q) {
    if (SINGLE) return FB + 8 * anti + 2 * (q - 2);
    return FB + (q < 2 ? 4 * anti + 2 * q : 2 * NFM + 16 * anti + (COMPACT && anti ? 7 : 8) * h + 2 * (q - 2));
  }
  // slot of component q (0, 1: momentum; 2..5: polarisation), part 0 / 1, of a gluon; -1: zero
  static constexpr __device__ int gluon(int q, int part) {
    if (!COMPACT || q < 2) return 2 * q + part;
    return q == 2 ? -1 : (q == 5 ? (part ? -1 : 8) : 4 + 2 * (q - 3) + part);
  }
};

// One block takes 64 events through one set of gluon helicities (its four top / anti-top rows)
// and one range of the orderings: blockIdx.x = the event tile, blockIdx.y = (gluon helicities,
// range).  Nothing is shared between gluon helicity sets but the event's invariants and
// spinors (1-2% of a set's work, computed once more for each), so a call of few events still
// fills the chip, and a large one ends without a half-empty round of long waves.  Against one
// wave walking every set of its 64 events: t t~ g g FP64, 1,000 events, 3,117 -> 103 us; t t~ g g g
// FP32, 257 events, 44.2 -> 0.31 ms, 50,000 events, 42.2 -> 33.7 ms; t t~ g g FP32, 1,048,576
// events, 37.9 -> 35.2 ms (the momenta no longer stay live across the sets: 244 -> 184 VGPRs).
template <class T, int BLOCK, bool EXPLICIT>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) k_ordered_jamps(OrderedArgs a) {
  typedef float R;
  constexpr int NG = T::NG, NE = T::NEXTERNAL, NC = T::NCOLOR;
  using S = OrderedStage<T, EXPLICIT>;
  __shared__ R lds[S::NSLOT * BLOCK];
  const int t = threadIdx.x;
  const int64_t el = (int64_t)blockIdx.x * BLOCK + t;
  if (el >= a.n) return;                 // no block-level synchronisation below
  const int64_t e = a.ev0 + el;
  R p[NE][4];
  load_momenta<T, R>(a.s.all_ps, e, p);
  const Params<R> prm = load_params<R>(a.s, e);
  {
    // 2 k_x.k_y in FP64 for x, y among (gluon slots 0..NG-1, top = slot NG)
    const double* src = a.s.all_ps + e * (NE * 4);
    double k[NG + 1][4];
#pragma unroll
    for (int s = 0; s <= NG; ++s) {
      const int leg = s < NG ? T::gluon_leg(s) : T::TOP_LEG;
      const double sg = T::leg_sign(leg);
#pragma unroll
      for (int c = 0; c < 4; ++c) k[s][c] = sg * src[4 * leg + c];
    }
#pragma unroll
    for (int x = 0; x <= NG; ++x)
#pragma unroll
      for (int y = x + 1; y <= NG; ++y) {
        const double v = 2.0 * (k[x][0] * k[y][0] - k[x][1] * k[y][1] - k[x][2] * k[y][2] - k[x][3] * k[y][3]);
        lds[(S::NWF + T::pair_index(x, y)) * BLOCK + t] = R(v);
      }
    // anti-top with each gluon slot (outgoing anti-top: sign +1)
    const double* ka = src + 4 * T::ATOP_LEG;
#pragma unroll
    for (int x = 0; x < NG; ++x) {
      const double v = 2.0 * (k[x][0] * ka[0] - k[x][1] * ka[1] - k[x][2] * ka[2] - k[x][3] * ka[3]);
      lds[(S::NWF + S::NPI + x) * BLOCK + t] = R(v);
    }
  }
  __attribute__((aligned(16))) R spinor[S::PRIVATE ? 40 : 1];
  R atop_last[2];       // COMPACT: the imaginary part of the anti-top's component 5
  {
    const int* hv = EXPLICIT && a.s.use_helv ? a.s.helv : nullptr;
#pragma unroll
    for (int h = 0; h < (S::SINGLE ? 1 : 2); ++h) {
      W<R> top, atop;
      T::template fermions<R>(p, ((unsigned)h << T::TOP_LEG) | ((unsigned)h << T::ATOP_LEG), hv, prm, top, atop);
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const int ot = S::fermion(0, h, q), oa = S::fermion(1, h, q);
        if constexpr (S::PRIVATE) {
          if (q >= 2 || h == 0) {
            spinor[ot - S::FB] = top[q].re;
            spinor[ot + 1 - S::FB] = top[q].im;
            spinor[oa - S::FB] = atop[q].re;
            spinor[oa + 1 - S::FB] = atop[q].im;
          }
        } else if (q >= 2) {
          lds[ot * BLOCK + t] = top[q].re;
          lds[(ot + 1) * BLOCK + t] = top[q].im;
          lds[oa * BLOCK + t] = atop[q].re;
          if (!S::COMPACT || q < 5) lds[(oa + 1) * BLOCK + t] = atop[q].im;
        }
      }
      atop_last[h] = atop[5].im;
    }
  }
  // spinor of the top (anti = 0) or anti-top (anti = 1) at helicity bit h; from LDS with the top's
  // momentum slots from p, the anti-top's, which are not read, left out
  auto staged_fermion = [&](int anti, int h, W<R>& w) {
    if constexpr (S::PRIVATE) {
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const int o = S::fermion(anti, h, q) - S::FB;
        w[q].re = spinor[o];
        w[q].im = spinor[o + 1];
      }
    } else {
      if (!anti) {
        w[0] = cx<R>(p[T::TOP_LEG][0], p[T::TOP_LEG][3]);
        w[1] = cx<R>(p[T::TOP_LEG][1], p[T::TOP_LEG][2]);
      }
#pragma unroll
      for (int q = 2; q < 6; ++q) {
        const int o = S::fermion(anti, h, q);
        w[q].re = lds[o * BLOCK + t];
        if (!S::COMPACT || q < 5 || !anti) {
          w[q].im = lds[(o + 1) * BLOCK + t];
        } else {
          w[q].im = h ? atop_last[1] : atop_last[0];
          opaque(w[q].im);
        }
      }
    }
  };
  // one real number of the gluon at slot s; a zero is opaque like a loaded value, so that the
  // compiler contracts the products it appears in as it does the others
  auto staged_gluon = [&](int s, int q, int part) -> R {
    if (S::gluon(q, part) >= 0) return lds[(s * S::GW + S::gluon(q, part)) * BLOCK + t];
    R z = R(0);
    opaque(z);
    return z;
  };
  cx<R>* jb = reinterpret_cast<cx<R>*>(a.jbuf);
  // Helicity rows are enumerated here as r = 4 g + 2 ht + ha: g = the gluon helicities
  // (bit s = gluon slot s), ht / ha = the top / anti-top helicity.  The gluon currents of
  // an ordering depend on g alone, so they are computed once for the four rows of g; the
  // top line is linear in the top spinor and is computed once per ht; the closing
  // vertex is linear in the anti-top spinor.  Rows r0 .. r1-1 are this launch's, each
  // stored at slot r - r0.  With an explicit helicity vector there is one row (r = 0),
  // and every helicity comes from the vector.
  static_assert(T::NCOMB == (4 << NG), "every helicity combination is a row");
  const int r0 = a.h0, r1 = a.h0 + a.nhel;
  const int g = (r0 >> 2) + (int)blockIdx.y / a.cparts;
  const int c0 = ((int)blockIdx.y % a.cparts) * a.cper, c1 = c0 + a.cper < NC ? c0 + a.cper : NC;
  constexpr int PRE = NG - 2;
  W<R> J[NG][NG], O[NG];
  cx<R> SD[NG][NG];   // adjacent-range dot sums S(a..b) of the four-gluon terms
  // Five or more gluons: the top-line currents O(1..PRE) of both top helicities, kept from
  // the first ordering of a pair for the second (for four gluons they would cost the second
  // wave per SIMD).
  constexpr bool SHARE_TOP = NG >= 5;
  TopPrefix<R, PRE + 1, SHARE_TOP> OP;
  // The word's pair invariants (gluon-gluon pp, top-gluon tp, anti-top-gluon
  // ap) and the top-line denominators rt (above); pp of the prefix pairs carries over to
  // the second ordering of a pair
  R pp[NG][NG], tp[NG], ap[NG], rt[NG];
  unsigned hbg = 0u;
#pragma unroll
  for (int s = 0; s < NG; ++s) hbg |= ((unsigned)(g >> s) & 1u) << T::gluon_leg(s);
  const int* helv = EXPLICIT && a.s.use_helv ? a.s.helv : nullptr;
#pragma unroll
  for (int s = 0; s < NG; ++s) {
    W<R> gw;
    T::template gluon<R>(p, s, hbg, helv, prm, gw);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      if constexpr (S::COMPACT) {
        if (S::gluon(q, 0) >= 0) lds[(s * S::GW + S::gluon(q, 0)) * BLOCK + t] = gw[q].re;
        if (S::gluon(q, 1) >= 0) lds[(s * S::GW + S::gluon(q, 1)) * BLOCK + t] = gw[q].im;
      } else {
        lds[(s * 12 + 2 * q) * BLOCK + t] = gw[q].re;
        lds[(s * 12 + 2 * q + 1) * BLOCK + t] = gw[q].im;
      }
    }
  }
  // Orderings come in lexicographic order, so orderings 2m and 2m+1 share their first
  // NG-2 gluons: the currents inside that prefix (J(i..j), j < NG-2) are computed once
  // per pair and carried to the second ordering.
#pragma unroll 1
  for (int c = c0; c < c1; ++c) {
    int perm[NG];
#pragma unroll
    for (int k = 0; k < NG; ++k) perm[k] = T::perm(c, k);
    const bool fresh = (c & 1) == 0;
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      if (k < PRE && !fresh) continue;
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        if constexpr (S::COMPACT) {
          J[k][k][q].re = staged_gluon(perm[k], q, 0);
          J[k][k][q].im = staged_gluon(perm[k], q, 1);
        } else {
          J[k][k][q].re = lds[(perm[k] * 12 + 2 * q) * BLOCK + t];
          J[k][k][q].im = lds[(perm[k] * 12 + 2 * q + 1) * BLOCK + t];
        }
      }
    }
    {
      // the word's pair invariants (the prefix pairs of a pair's second ordering are the
      // first's), and rt[j] for the top with the first j gluons from the shorter of its
      // two forms
#pragma unroll
      for (int x = 0; x < NG; ++x) {
        tp[x] = lds[(S::NWF + T::pair_index(perm[x], NG)) * BLOCK + t];
        ap[x] = lds[(S::NWF + S::NPI + perm[x]) * BLOCK + t];
#pragma unroll
        for (int y = x + 1; y < NG; ++y) {
          if (y < PRE && !fresh) continue;
          pp[x][y] = lds[(S::NWF + T::pair_index(perm[x], perm[y])) * BLOCK + t];
        }
      }
#pragma unroll
      for (int j = 1; j < NG; ++j) {
        // direct: the top and gluons 0..j-1; complementary: the anti-top and gluons j..NG-1
        const int nd = j + j * (j - 1) / 2, nc = (NG - j) + (NG - j) * (NG - j - 1) / 2;
        R sd = R(0), md = R(0), sc = R(0), mc = R(0);
#pragma unroll
        for (int a = 0; a < j; ++a) {
          sd += tp[a];
          md += fabs(tp[a]);
#pragma unroll
          for (int b = a + 1; b < j; ++b) {
            sd += pp[a][b];
            md += fabs(pp[a][b]);
          }
        }
#pragma unroll
        for (int a = j; a < NG; ++a) {
          sc += ap[a];
          mc += fabs(ap[a]);
#pragma unroll
          for (int b = a + 1; b < NG; ++b) {
            sc += pp[a][b];
            mc += fabs(pp[a][b]);
          }
        }
        rt[j] = nd < nc ? sd : (nc < nd ? sc : (md <= mc ? sd : sc));
      }
    }
    if (fresh) ordered_ranges<NG, 1, PRE, R>(J, SD, pp, prm);
    ordered_ranges<NG, PRE, NG, R>(J, SD, pp, prm);
    if constexpr (SHARE_TOP) {
      // unrolled: OP is indexed by ht
#pragma unroll
      for (int ht = 0; ht < 2; ++ht) {
        const int rb = 4 * g + 2 * ht;
        if (rb + 1 < r0 || rb >= r1) continue;
        W<R> top, atop;
        staged_fermion(0, ht, top);
        O[0] = top;
        // O(1..PRE) only involve the prefix gluons: computed once per pair of orderings
        if (fresh) {
          ordered_top_line<NG, 1, PRE, R>(O, J, rt, prm);
#pragma unroll
          for (int j = 1; j <= PRE; ++j) OP.o[ht][j] = O[j];
        } else {
#pragma unroll
          for (int j = 1; j <= PRE; ++j) O[j] = OP.o[ht][j];
        }
        ordered_top_line<NG, PRE + 1, NG - 1, R>(O, J, rt, prm);
        const VslashF<R> x = ordered_close_col<NG, R>(O, J);
#pragma unroll 1
        for (int ha = 0; ha < 2; ++ha) {
          const int r = rb + ha;
          if (r < r0 || r >= r1) continue;
          staged_fermion(1, ha, atop);
          jb[((int64_t)(r - r0) * NC + c) * a.ld + el] = ordered_jamp(atop, x, prm);
        }
      }
    } else {
#pragma unroll 1
      for (int ht = 0; ht < 2; ++ht) {
        const int rb = 4 * g + 2 * ht;
        if (rb + 1 < r0 || rb >= r1) continue;
        W<R> top, atop;
        staged_fermion(0, ht, top);
        O[0] = top;
        ordered_top_line<NG, 1, NG - 1, R>(O, J, rt, prm);
        const VslashF<R> x = ordered_close_col<NG, R>(O, J);
#pragma unroll 1
        for (int ha = 0; ha < 2; ++ha) {
          const int r = rb + ha;
          if (r < r0 || r >= r1) continue;
          staged_fermion(1, ha, atop);
          jb[((int64_t)(r - r0) * NC + c) * a.ld + el] = ordered_jamp(atop, x, prm);
        }
      }
    }
  }
}

// The FP64 kernel: blocks as k_ordered_jamps, but each word is evaluated together with its
// reversal, and the words come in cycles of rotations (MirrorWalk): the next word keeps every
// current but those that end in its new last letter, so one current of each length is
// computed for two orderings.  (FP32 keeps the currents of each ordering apart: a current's last
// bits depend on where in the word the compiler contracts it, and FP32 results are held to
// them.)  30,001 events, against every ordering by itself: t t~ g g 1,580 -> 998 us, t t~ g g g 45.9
// -> 42.0 ms (its currents do not fit 512 registers: 1.4 KB of spills a lane).  Momenta of ranges
// are added up again for each word; carried along they made t t~ g g spill and take 1,152 us.
// LDS: the gluons, then the spinor components of the top and the anti-top at both helicities;
// one wave per SIMD (the currents fill the registers), so four blocks a CU may take 40 KB each
// (t t~ g g g, 131,072 events of one explicit row: 46 KB and three blocks 5.85 ms, 38 KB 4.60 ms).
template <class T, bool EXPLICIT>
struct MirrorStage {
  static constexpr int NG = T::NG;
  // a polarisation's time component and the imaginary part of its z component are zero, except
  // with an explicit helicity vector (BRST)
  static constexpr int GW = EXPLICIT ? 12 : 9;
  // one row, so one helicity of each fermion, with an explicit vector
  static constexpr int FB = NG * GW, NH = EXPLICIT ? 1 : 2, NSLOT = FB + 16 * NH;
  static_assert(NSLOT * 64 * 8 <= 40 * 1024, "four blocks a CU");
  static constexpr __device__ int gluon(int q, int part) {
    if (EXPLICIT || q < 2) return 2 * q + part;
    return q == 2 ? -1 : (q == 5 ? (part ? -1 : 8) : 4 + 2 * (q - 3) + part);
  }
};

template <class T, int BLOCK, bool EXPLICIT>
__global__ void __launch_bounds__(BLOCK) k_ordered_mirror(OrderedArgs a) {
  typedef double R;
  constexpr int NG = T::NG, NE = T::NEXTERNAL, NC = T::NCOLOR, NW = NC / 2;
  using S = MirrorStage<T, EXPLICIT>;
  __shared__ R lds[S::NSLOT * BLOCK];
  const int t = threadIdx.x;
  const int64_t el = (int64_t)blockIdx.x * BLOCK + t;
  if (el >= a.n) return;                 // no block-level synchronisation below
  const int64_t e = a.ev0 + el;
  R p[NE][4];
  load_momenta<T, R>(a.s.all_ps, e, p);
  const Params<R> prm = load_params<R>(a.s, e);
  const int* helv = EXPLICIT ? a.s.helv : nullptr;
  const int r0 = a.h0, r1 = a.h0 + a.nhel;
  const int g = (r0 >> 2) + (int)blockIdx.y / a.cparts;
  const int c0 = ((int)blockIdx.y % a.cparts) * a.cper, c1 = c0 + a.cper < NW ? c0 + a.cper : NW;
  unsigned hbg = 0u;
#pragma unroll
  for (int s = 0; s < NG; ++s) hbg |= ((unsigned)(g >> s) & 1u) << T::gluon_leg(s);
#pragma unroll
  for (int s = 0; s < NG; ++s) {
    W<R> gw;
    T::template gluon<R>(p, s, hbg, helv, prm, gw);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      if (S::gluon(q, 0) >= 0) lds[(s * S::GW + S::gluon(q, 0)) * BLOCK + t] = gw[q].re;
      if (S::gluon(q, 1) >= 0) lds[(s * S::GW + S::gluon(q, 1)) * BLOCK + t] = gw[q].im;
    }
  }
#pragma unroll
  for (int h = 0; h < S::NH; ++h) {
    W<R> top, atop;
    T::template fermions<R>(p, ((unsigned)h << T::TOP_LEG) | ((unsigned)h << T::ATOP_LEG), helv, prm, top, atop);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int o = S::FB + 8 * h + 2 * q, oa = o + 8 * S::NH;
      lds[o * BLOCK + t] = top[q + 2].re;
      lds[(o + 1) * BLOCK + t] = top[q + 2].im;
      lds[oa * BLOCK + t] = atop[q + 2].re;
      lds[(oa + 1) * BLOCK + t] = atop[q + 2].im;
    }
  }
  // spinor components of the top (anti = 0) or anti-top (anti = 1) at helicity bit h
  auto spinor = [&](int anti, int h, W<R>& w) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int o = S::FB + 8 * (S::NH * anti + (S::NH > 1 ? h : 0)) + 2 * q;
      w[q + 2] = cx<R>(lds[o * BLOCK + t], lds[(o + 1) * BLOCK + t]);
    }
  };
  cx<R>* jb = reinterpret_cast<cx<R>*>(a.jbuf);
  W<R> J[NG][NG], O[NG];
  cx<R> SD[NG][NG];
  R pp[NG][NG];           // FP32's invariants, not read here
#pragma unroll 1
  for (int c = c0; c < c1; ++c) {
    const int row = MIRROR_WALK<NG, NC>.at[c], rrow = MIRROR_WALK<NG, NC>.rev[c];
    if (c == c0 || c % NG == 0) {
#pragma unroll
      for (int k = 0; k < NG; ++k) {
        const int s = T::perm(row, k);
#pragma unroll
        for (int q = 0; q < 6; ++q) {
          J[k][k][q].re = S::gluon(q, 0) >= 0 ? lds[(s * S::GW + S::gluon(q, 0)) * BLOCK + t] : R(0);
          J[k][k][q].im = S::gluon(q, 1) >= 0 ? lds[(s * S::GW + S::gluon(q, 1)) * BLOCK + t] : R(0);
        }
      }
      ordered_ranges<NG, 1, NG - 1, R>(J, SD, pp, prm);
    } else {
      const W<R> first = J[0][0];
#pragma unroll
      for (int x = 0; x < NG - 1; ++x) J[x][x] = J[x + 1][x + 1];
#pragma unroll
      for (int x = 0; x < NG - 1; ++x) {
#pragma unroll
        for (int y = x + 1; y < NG - 1; ++y) {
#pragma unroll
          for (int q = 2; q < 6; ++q) J[x][y][q] = J[x + 1][y + 1][q];
          SD[x][y] = SD[x + 1][y + 1];
        }
      }
      // momenta are added up again rather than carried in registers, in ordered_ranges' order: a
      // word's bits do not depend on the word its block began with
#pragma unroll
      for (int y = 1; y < NG - 1; ++y) {
#pragma unroll
        for (int x = y - 1; x >= 0; --x) {
          J[x][y][0] = J[x][x][0] + J[x + 1][y][0];
          J[x][y][1] = J[x][x][1] + J[x + 1][y][1];
        }
      }
      J[NG - 1][NG - 1] = first;
    }
    ordered_ranges<NG, NG - 1, NG, R>(J, SD, pp, prm);
#pragma unroll 1
    for (int ht = 0; ht < 2; ++ht) {
      const int rb = 4 * g + 2 * ht;
      if (rb + 1 < r0 || rb >= r1) continue;
      __builtin_amdgcn_sched_barrier(0);
      O[0][0] = cx<R>(p[T::TOP_LEG][0], p[T::TOP_LEG][3]);
      O[0][1] = cx<R>(p[T::TOP_LEG][1], p[T::TOP_LEG][2]);
      spinor(0, ht, O[0]);
      const VslashF<R> x = word_top_line<false, NG, R>(O, J, prm);
      __builtin_amdgcn_sched_barrier(0);
      const VslashF<R> xr = word_top_line<true, NG, R>(O, J, prm);
#pragma unroll 1
      for (int ha = 0; ha < 2; ++ha) {
        const int r = rb + ha;
        if (r < r0 || r >= r1) continue;
        W<R> atop;
        spinor(1, ha, atop);
        cx<R>* out = jb + (int64_t)(r - r0) * NC * a.ld + el;
        out[row * a.ld] = ordered_jamp(atop, x, prm);
        out[rrow * a.ld] = ordered_jamp(atop, xr, prm);
      }
    }
  }
}

// MFMA 16x16x4 on one wave: D += A(16x4) * B(4x16); lane l supplies A[l%16][l/16] and
// B[l/16][l%16] and holds D[drow(l/16, r)][l%16], r = 0..3, where the row is
// 4*(l/16) + r for f32 and (l/16) + 4*r for f64 (measured on gfx950).
__device__ __forceinline__ mfx_f32x4 mfma16x16x4(float a, float b, mfx_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mfx_f64x4 mfma16x16x4(double a, double b, mfx_f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <class R> __device__ __forceinline__ int drow(int lq, int r);
template <> __device__ __forceinline__ int drow<float>(int lq, int r) { return 4 * lq + r; }
template <> __device__ __forceinline__ int drow<double>(int lq, int r) { return lq + 4 * r; }
template <class R> struct Vec4;
template <> struct Vec4<float> { typedef mfx_f32x4 type; };
template <> struct Vec4<double> { typedef mfx_f64x4 type; };

// |M|^2 of the events of one sub-chunk from their jamps: one wave per item, a 16-event tile and a
// range of hper helicity rows, the waves taking items in turn.  Per helicity and tile the matrix cores form D = CF J^T
// (NCP x 16: colour rows, event columns) from the integer colour matrix (A operand, in
// LDS) and the tile's jamps (B operand: lane (i, q) holds J[event i][colour 4 s + q] for
// every k-step s), then each lane dots its D entries with jamps it already holds.  For
// that, the colour of A row drow(q, r) of row tile mt is 4 (4 mt + r) + q: the output the
// lane holds in register r is then the row of the colour of its k-step 4 mt + r, and the
// jamps are read once.  The four lane quarters of each event are summed at the end of a row.
// The rows are added in pairs, the pairs in pairs, and so on (their number is a power of two).
// With more than one range of rows (few events: the rows of one tile are then spread over
// the chip) a wave leaves its 16 sums of a range, a whole branch of that tree each, in place of
// jamps that it alone has read, colour 0 of the range's first row, and k_colour_sum adds the
// branches: an event's bits do not depend on the split, and so not on the size of the call.
template <class T, class R>
__global__ void __launch_bounds__(256) k_colour_mfma(void* jbuf, int64_t n, int64_t ld, int nhel, int hper,
                                                     double scale, int accumulate, double* out) {
  constexpr int NC = T::NCOLOR;
  constexpr int NCP = (NC + 15) / 16 * 16;    // padded colour rows of D
  constexpr int KS = NC / 4;                  // k-steps (NCOLOR is a multiple of 4)
  static_assert(NC % 4 == 0, "NCOLOR must be a multiple of 4");
  constexpr int LEVELS = T::NCOMB <= 64 ? 6 : 7;
  static_assert(T::NCOMB <= 1 << LEVELS, "one branch in wait for each level of the tree");
  typedef typename Vec4<R>::type V4;
  // integer numerators, rows permuted as above: exact in float.  Four columns per load and every
  // load in flight at once: with 120 colours the block reads 61 KB before it starts.
  __shared__ __attribute__((aligned(16))) float cf[NCP * NC];
  // the branches in wait for their right-hand neighbours (12 registers would cost t t~ g g in FP32 two
  // of eight waves a SIMD: 100,000 events 300 us instead of 282)
  __shared__ double branch[LEVELS][4][16];
#pragma unroll
  for (int i0 = 0; i0 < NCP * NC / 4; i0 += 256) {
    const int i = i0 + threadIdx.x;
    if (i < NCP * NC / 4) {
      const int row = i / (NC / 4), k = 4 * (i % (NC / 4));
      const int mt = row / 16, x = row % 16;
      // x = drow(q, r): 4 q + r for f32, q + 4 r for f64
      const int q = drow<R>(1, 0) == 4 ? x / 4 : x % 4, r = drow<R>(1, 0) == 4 ? x % 4 : x / 4;
      const int colour = 4 * (4 * mt + r) + q;
      float4 v = {0.f, 0.f, 0.f, 0.f};
      if (colour < NC)
        v = float4{T::cf(float(), colour, k), T::cf(float(), colour, k + 1), T::cf(float(), colour, k + 2),
                   T::cf(float(), colour, k + 3)};
      *reinterpret_cast<float4*>(cf + row * NC + k) = v;
    }
  }
  __syncthreads();
  const cx<R>* J = reinterpret_cast<const cx<R>*>(jbuf);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lq = lane >> 4;
  // 32 bits hold the items: the jamps of 2^31 of them would take terabytes
  const unsigned ntiles = (unsigned)((n + 15) / 16), parts = (unsigned)((nhel + hper - 1) / hper);
  for (unsigned item = blockIdx.x * 4 + wave; item < ntiles * parts; item += gridDim.x * 4) {
    const int64_t tile = item % ntiles;
    const int h0 = (int)(item / ntiles) * hper, h1 = h0 + hper < nhel ? h0 + hper : nhel;
    const int64_t ea = tile * 16 + lr;          // the event of this lane's B column
    // each helicity's colour terms are summed in R, the helicities in FP64 (an FP32 sum
    // over every helicity and colour would lose digits with the number of rows)
    double acc = 0.0;
    for (int h = h0; h < h1; ++h) {
      const cx<R>* Jh = J + (int64_t)h * NC * ld;
      R are[KS], aim[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const cx<R> v = ea < n ? Jh[(int64_t)(4 * s + lq) * ld + ea] : cx<R>(R(0), R(0));
        are[s] = v.re;
        aim[s] = v.im;
      }
      R part = R(0);
#pragma unroll
      for (int mt = 0; mt < NCP / 16; ++mt) {
        V4 dre = {R(0), R(0), R(0), R(0)}, dim = {R(0), R(0), R(0), R(0)};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const R c = R(cf[(16 * mt + lr) * NC + 4 * s + lq]);
          dre = mfma16x16x4(c, are[s], dre);
          dim = mfma16x16x4(c, aim[s], dim);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * mt + r < KS) part += are[4 * mt + r] * dre[r] + aim[4 * mt + r] * dim[r];
        // one row tile at a time: interleaving the tiles would hold every tile's
        // accumulators at once
        __builtin_amdgcn_sched_barrier(0);
      }
      // sum the four lane quarters that hold the colours of each event
      acc = double(part);
      acc += __shfl_xor(acc, 16, 64);
      acc += __shfl_xor(acc, 32, 64);
      int up = 0;
      for (int k = h - h0; k & 1; k >>= 1) acc += branch[up++][wave][lr];
      if (h + 1 < h1) branch[up][wave][lr] = acc;
    }
    if (lq == 0 && ea < n) {
      if (parts > 1) reinterpret_cast<double*>(static_cast<cx<R>*>(jbuf) + (int64_t)h0 * NC * ld + tile * 16)[lr] = acc;
      else out[ea] = (accumulate ? out[ea] : 0.0) + acc * scale;
    }
  }
}

// The branches of k_colour_mfma, parts (a power of two up to 128) an event; step: jamps (complex R)
// from one range's first row to the next one's.  16 events a block, 16 lanes an event: each adds
// the branch of its neighbouring ranges, then the lanes are added as the tree goes on.
// (One lane an event walking 64 ranges took 17 us, now 3.9 us.)
template <class R>
__global__ void __launch_bounds__(256) k_colour_sum(const void* jbuf, int64_t n, int64_t step, int parts, double scale,
                                                    int accumulate, double* out) {
  constexpr int U = 8;
  const int lane = threadIdx.x & 15, per = parts < 16 ? 1 : parts / 16;
  const int64_t e = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  double v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int p = lane * per + u;
    v[u] = 0.0;
    if (e < n && u < per && p < parts)
      v[u] = reinterpret_cast<const double*>(static_cast<const cx<R>*>(jbuf) + e / 16 * 16 + p * step)[e % 16];
  }
#pragma unroll
  for (int w = 1; w < U; w *= 2)
#pragma unroll
    for (int u = 0; u < U; u += 2 * w) v[u] += v[u + w];
  double acc = v[0];
#pragma unroll
  for (int off = 1; off < 16; off *= 2) acc += __shfl_xor(acc, off, 64);
  if (lane == 0 && e < n) out[e] = (accumulate ? out[e] : 0.0) + acc * scale;
}

// jamps of a single helicity row [NCOLOR][ld] -> (n, NCOLOR, 2) f64
template <class R>
__global__ void k_jamp_transpose(const void* jbuf, int64_t n, int64_t ld, int ncolor, double* jamp_out) {
  const cx<R>* J = reinterpret_cast<const cx<R>*>(jbuf);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * ncolor) return;
  const int64_t e = i / ncolor;
  const int c = (int)(i % ncolor);
  const cx<R> v = J[(int64_t)c * ld + e];
  jamp_out[2 * i] = double(v.re);
  jamp_out[2 * i + 1] = double(v.im);
}

// bytes of jamp workspace per event and helicity row
template <class T>
int64_t ordered_ws_per_row(int precision) {
  return (int64_t)T::NCOLOR * 2 * (precision == 32 ? 4 : 8);
}

// blocks of k_ordered_jamps per SIMD below which the orderings are split too.  One leaves the
// second wave of a SIMD out (t t~ g g g FP32, 1,000 events: 1,056 us against 610 us with two); four
// and eight are within the scatter of the rounds they end in (1,000 events: 652 and 638 us; 2,500
// events: 1,437 and 1,493 us against 1,711 us; 257 events: 296 and 273 us against 267 us).
// FP64 holds one wave a SIMD, but two ranges for each are as often the better split as one: with
// one, two and four, t t~ g g 500 events 30, 35 and 35 us, 1,000 47, 57 and 54, 2,500 125, 109 and 104, 4,000
// 163, 137 and 143, 8,000 254, 282 and 260; t t~ g g g 500 events 720, 876 and 756, 2,500 4,770, 3,830 and
// 3,390, from 4,000 on the same.
constexpr int ORDERED_WAVES = 2;

// (tile, rows) items per wave slot of k_colour_mfma: t t~ g g g FP32, 50,000 events, 27.2 ms a call
// with one round of tiles, 26.0 ms with 4 and with 8 (the colour sum 4.05 -> 3.31 ms)
constexpr int COLOUR_ITEMS = 4;

// Sub-chunks of events and groups of helicity rows sized to the caller's workspace:
// the largest helicity group that still leaves a sub-chunk of min(nev, 65536) events
// (enough waves for every SIMD), then as many events as the workspace holds.
template <class T>
hipError_t launch_ordered(const SmatrixArgs& s, int precision, int per_helicity, void* ws, int64_t ws_bytes,
                          hipStream_t st) {
  if (s.nev <= 0) return hipSuccess;
  const int nrows = per_helicity ? 1 : T::NCOMB;
  const int64_t row = ordered_ws_per_row<T>(precision);
  const int64_t want = s.nev < 65536 ? s.nev : 65536;
  int hg = nrows;
  while (hg > 1 && ws_bytes / (row * hg) < want) hg /= 2;
  // whole 16-event tiles per pass: the row stride (n rounded up to 16) then fits too
  int64_t nsub = ws ? ws_bytes / (row * hg) / 16 * 16 : 0;
  if (nsub < 16) return hipErrorInvalidValue;   // the entry point checks the size first
  // passes of equal size, whole 64-event blocks where the workspace allows
  const int64_t passes = (s.nev + nsub - 1) / nsub;
  const int64_t even = ((s.nev + passes - 1) / passes + 63) / 64 * 64;
  if (even < nsub) nsub = even;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  const double scale = 1.0 / (T::CF_DEN * (per_helicity ? 1.0 : T::DENOMINATOR));
  for (int64_t off = 0; off < s.nev; off += nsub) {
    const int64_t n = s.nev - off < nsub ? s.nev - off : nsub;
    const int64_t tiles = (n + 15) / 16, blocks = (n + 63) / 64;
    for (int h0 = 0; h0 < nrows; h0 += hg) {
      OrderedArgs a;
      a.s = s;
      a.ev0 = off;
      a.n = n;
      a.ld = (n + 15) / 16 * 16;
      a.h0 = h0;
      a.nhel = hg;
      a.jbuf = ws;
      const int ng = ((h0 + hg - 1) >> 2) - (h0 >> 2) + 1;
      // The orderings (FP64: words, for two orderings each) are split over blocks while there are
      // fewer blocks than ORDERED_WAVES per SIMD.  What a block computes for all of them
      // (invariants, spinors) is done once more for each range, and a range starts its first
      // word afresh: FP32 ranges are whole pairs, longer FP64 ranges whole cycles.
      const int unit = precision == 32 ? 2 : 1, count = T::NCOLOR / 2;
      int64_t parts = (4ll * ORDERED_WAVES * cus + blocks * ng - 1) / (blocks * ng);
      parts = parts < 1 ? 1 : (parts > count ? count : parts);
      a.cper = (int)((count + parts - 1) / parts);
      if (precision == 64 && a.cper > T::NG) a.cper = (a.cper + T::NG - 1) / T::NG * T::NG;
      a.cparts = (count + a.cper - 1) / a.cper;
      a.cper *= unit;
      // The colour sum's waves take (tile, range of rows) items in turn, so that a block stages its
      // matrix once: as many blocks as a CU holds (61 KB of matrix each at 120 colours: two), in FP64
      // fewer, as four already read at the rate of the memory (t t~ g g, 100,000 events: 489 us with
      // four, 521 us with eight; 30,000: 169 and 182 us).
      // The rows are split until every wave has COLOUR_ITEMS items, so that few events fill the
      // chip and the last round of many is short.
      const int64_t cslots = (int64_t)cus * (T::NCOLOR > 64 ? 2 : precision == 64 ? 4 : 8);
      int hper = hg;
      while (hper > 1 && tiles * (hg / hper) < COLOUR_ITEMS * 4 * cslots) hper /= 2;
      const int hparts = (hg + hper - 1) / hper;
      int64_t cblk = (tiles * hparts + 3) / 4;
      if (cblk > cslots) cblk = cslots;
      const int acc = h0 > 0;
      const dim3 gj((unsigned)blocks, (unsigned)(ng * a.cparts)), gc((unsigned)cblk);
      const int64_t step = (int64_t)hper * T::NCOLOR * a.ld;
      const dim3 gs((unsigned)tiles);
      if (precision == 32) {
        // five gluons: the layout of both is the same, so one kernel takes both calls
        if constexpr (T::NG > 4) hipLaunchKernelGGL((k_ordered_jamps<T, 64, true>), gj, dim3(64), 0, st, a);
        else if (s.use_helv) hipLaunchKernelGGL((k_ordered_jamps<T, 64, true>), gj, dim3(64), 0, st, a);
        else hipLaunchKernelGGL((k_ordered_jamps<T, 64, false>), gj, dim3(64), 0, st, a);
        hipLaunchKernelGGL((k_colour_mfma<T, float>), gc, dim3(256), 0, st, ws, n, a.ld, hg, hper, scale, acc, s.out + off);
        if (hparts > 1)
          hipLaunchKernelGGL((k_colour_sum<float>), gs, dim3(256), 0, st, (const void*)ws, n, step, hparts, scale, acc,
                             s.out + off);
      } else {
        if (s.use_helv) hipLaunchKernelGGL((k_ordered_mirror<T, 64, true>), gj, dim3(64), 0, st, a);
        else hipLaunchKernelGGL((k_ordered_mirror<T, 64, false>), gj, dim3(64), 0, st, a);
        hipLaunchKernelGGL((k_colour_mfma<T, double>), gc, dim3(256), 0, st, ws, n, a.ld, hg, hper, scale, acc, s.out + off);
        if (hparts > 1)
          hipLaunchKernelGGL((k_colour_sum<double>), gs, dim3(256), 0, st, (const void*)ws, n, step, hparts, scale, acc,
                             s.out + off);
      }
    }
    if (per_helicity && s.jamp_out) {
      const unsigned nb = (unsigned)((n * T::NCOLOR + 255) / 256);
      const int64_t ld = (n + 15) / 16 * 16;
      if (precision == 32)
        hipLaunchKernelGGL((k_jamp_transpose<float>), dim3(nb), dim3(256), 0, st, (const void*)ws, n, ld, T::NCOLOR,
                           s.jamp_out + off * T::NCOLOR * 2);
      else
        hipLaunchKernelGGL((k_jamp_transpose<double>), dim3(nb), dim3(256), 0, st, (const void*)ws, n, ld, T::NCOLOR,
                           s.jamp_out + off * T::NCOLOR * 2);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace mfx

#define MFX_INSTANTIATE_ORDERED(NAME)                                                                   \
  namespace mfx {                                                                                      \
  static const int registered_##NAME = register_process(ProcessEntry{                                  \
      NAME::Traits::PROC_NAME, NAME::Traits::NEXTERNAL, NAME::Traits::NCOMB, NAME::Traits::NCOLOR,      \
      NAME::Traits::NDIAGS, NAME::Traits::NGRAPHS, NAME::Traits::DENOMINATOR, &launch_ordered<NAME::Traits>, \
      &ordered_ws_per_row<NAME::Traits>});                                                           \
  }
