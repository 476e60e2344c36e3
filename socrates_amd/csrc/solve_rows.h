// The column solve over rows of lanes: included by socgpu.hip, whose layer
// inputs and coefficients (LaneCtx, LaneSrc, LayerIn, load_layer,
// layer_coef*) and lane exchanges it uses.
//
// A solve is one (column, g-point) clear or McICA profile: the two-stream
// system of L layers. LN consecutive lanes share one solve, 16 (a DPP row) or, for
// calls of few layers, 4 (kFewL), each lane taking K = ceil(layers / LN) consecutive
// layers in registers, so a wave holds 4 or 16 solves of one column. The layers' coefficients are independent
// and are most of the work; the elimination down the column and the
// back-substitution up it are recurrences, made parallel across the lanes:
//  - each lane composes its layers into one slab (transmission, reflection
//    from above and from below, emitted or scattered flux up and down), by the
//    adding equations;
//  - a prefix scan of the slabs over the row gives every lane the reflectance
//    of the atmosphere above it and the diffuse flux that sends down, from
//    which the lane eliminates its own layers as a single lane would;
//  - back-substitution is affine in the flux at the lane's bottom, so a suffix
//    scan gives every lane that flux.
// Between the sweeps a lane's layers stay in its registers, as far as 256 of them go:
// the builds of up to 24 layers spill none to 39, those of up to 96 none to 27, of up
// to 144 20 to 93, and above 144 layers (512 registers) up to 20. The layers of deep
// cloud, more of them than the LDS holds, are in lane-private memory (240 to 576 B a
// lane). One lane per solve kept the elimination state of all layers there (20 KB a
// lane): the solve then moved 4.6 GB of scratch per 4096 x 90 SW + LW step, waited 63 % of its
// cycles and took 1157 us (FP64). Now it moves 0.5 GB (0.4 mixed) in 559 us (511) and
// is bound by VALU issue: 74 % of the cycles with the two waves per SIMD that 256
// registers a lane allow.
#pragma once

constexpr int kRowLanes = 16;                 // lanes per solve
constexpr int kRows = kWave / kRowLanes;      // solves per wave
constexpr int kLowK = 4;                      // layers per lane of a cloudy part held in LDS
constexpr int kLowQ = 5;                      // doubles per layer there
constexpr int kHotQ = 7;                      // column record slots a wave keeps in LDS
// Builds of the kernel by the call's layers, 6 or 9 per lane (a lane's state is
// in registers; 9 cost the short calls 72 of them), and its optics: power-law
// gases without aerosols; any gas scaling and treatment of scattering; that with
// aerosols. Calls of more layers than kLongL are few: one build for all optics.
constexpr int kShortL = 6 * kRowLanes, kLongL = 9 * kRowLanes;
// Calls of few layers (also three builds by optics): 16 lanes would be idle for the
// most part. Call of 16384 columns in us, FP64 solar, with 16 lanes per solve and with
// 4: 2 layers clear 433 and 285, 5 layers all-sky 752 and 438, 24 all-sky 922 and 704;
// infra-red, 24 all-sky 1125 and 881. (One column of 20 layers 145 and 149.)
constexpr int kFewLanes = 4, kFewL = 6 * kFewLanes;
enum { kOptPlain, kOptGen, kOptAer, kOptAny };

// v of the lane CTRL selects, 0 where there is none; and with 1 there.
template <int CTRL>
__device__ __forceinline__ double dpp_or0(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)lo32(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)hi32(v), CTRL, 0xf, 0xf, true);
  return mk64((unsigned)lo, (unsigned)hi);
}
template <int CTRL>
__device__ __forceinline__ double dpp_or1(double v) { return dpp_f64<CTRL, 0xf>(v, 1.0); }

// row_shr:N (from the lane N below), row_shl:N (N above), row_newbcast:N
constexpr int kShr = 0x110, kShl = 0x100, kBcast = 0x150, kXor1 = 0xB1;

// v of the lane N below or N above in the group of LN lanes, s the lane's place in
// it; 0 (or 1) where there is none; and v of the group's first or last lane.
template <int LN, int N>
__device__ __forceinline__ double below0(double v, int s) {
  const double x = dpp_or0<kShr + N>(v);
  return LN == kRowLanes || s >= N ? x : 0.0;
}
template <int LN, int N>
__device__ __forceinline__ double below1(double v, int s) {
  const double x = dpp_or1<kShr + N>(v);
  return LN == kRowLanes || s >= N ? x : 1.0;
}
template <int LN, int N>
__device__ __forceinline__ double above0(double v, int s) {
  const double x = dpp_or0<kShl + N>(v);
  return LN == kRowLanes || s + N < LN ? x : 0.0;
}
template <int LN>
__device__ __forceinline__ double of_first(double v) {
  return LN == kRowLanes ? dpp_or0<kBcast + 0>(v) : dpp_move<0x00>(v);   // quad_perm [0, 0, 0, 0]
}
template <int LN>
__device__ __forceinline__ double of_last(double v) {
  return LN == kRowLanes ? dpp_or0<kBcast + 15>(v) : dpp_move<0xFF>(v);  // quad_perm [3, 3, 3, 3]
}

// 1 / x of a denominator 1 - R rho: the hardware estimate and two Newton steps
// (within an ulp or two). Of zero or infinity they give NaN where a division gives
// infinity or zero, but x is neither: a layer's reflection is below 1 by about
// sqrt(1 - omega) or more, and where the caller's asymmetry makes it 1 all the same
// (|g| beyond 1e30), its transmission is 0 and the fluxes are NaN either way.
__device__ __forceinline__ double rcp_newton(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}

// A run of layers seen from outside: transmission (the same both ways),
// reflection from above and from below, and its own flux up at the top and
// down at the bottom.
struct Slab {
  double T, Rt, Rb, Su, Sd;
};

// The slab A above the slab B.
__device__ __forceinline__ Slab slab_add(const Slab &A, const Slab &B) {
#pragma clang fp contract(on)
  const double D = rcp_newton(1.0 - A.Rb * B.Rt);
  const double tb = B.T * D, ta = A.T * D;
  Slab S;
  S.Su = A.Su + ta * (B.Su + B.Rt * A.Sd);
  S.Sd = B.Sd + tb * (A.Sd + A.Rb * B.Su);
  S.Rt = A.Rt + ta * B.Rt * A.T;
  S.Rb = B.Rb + tb * A.Rb * B.T;
  S.T = ta * B.T;
  return S;
}

// Only what the slab A above sends on through B: reflection from below and the
// flux down.
__device__ __forceinline__ void slab_below(double Rb, double Sd, const Slab &B, double &rb, double &sd) {
#pragma clang fp contract(on)
  const double tb = B.T * rcp_newton(1.0 - Rb * B.Rt);
  rb = B.Rb + tb * Rb * B.T;
  sd = B.Sd + tb * (Sd + Rb * B.Su);
}

// One step of the prefix scan of slabs: the slab N lanes below in the group
// (zeros where there is none: such a lane's slab already starts at the top of
// the scanned layers, its state is absolute and only Rb and Sd of it are
// used again).
template <int LN, int N>
__device__ __forceinline__ void slab_step(Slab &S, int s) {
  Slab A;
  A.T = below0<LN, N>(S.T, s);
  A.Rt = below0<LN, N>(S.Rt, s);
  A.Rb = below0<LN, N>(S.Rb, s);
  A.Su = below0<LN, N>(S.Su, s);
  A.Sd = below0<LN, N>(S.Sd, s);
  S = slab_add(A, S);
}

// The scan over a group whose consecutive slabs lie NS lanes apart.
template <int LN, int NS>
__device__ __forceinline__ void slab_scan(Slab &S, int s) {
  if (NS == 1) slab_step<LN, 1>(S, s);
  if (LN == kRowLanes) {
    slab_step<LN, 2>(S, s);
    slab_step<LN, 4>(S, s);
  }
  double rb, sd;
  slab_below(below0<LN, LN / 2>(S.Rb, s), below0<LN, LN / 2>(S.Sd, s), S, rb, sd);
  S.Rb = rb;
  S.Sd = sd;
}

template <int LN, int NS>
__device__ __forceinline__ double product_scan(double p, int s) {
  if (NS == 1) p = p * below1<LN, 1>(p, s);
  p = p * below1<LN, 2>(p, s);
  if (LN == kRowLanes) {
    p = p * below1<LN, 4>(p, s);
    p = p * below1<LN, 8>(p, s);
  }
  return p;
}

// Suffix scan of the affine maps x -> A x + C, the last of the group's maps
// being absolute (A unused).
template <int LN, int N>
__device__ __forceinline__ void affine_up_step(double &A, double &C, int s) {
#pragma clang fp contract(on)
  const double A1 = above0<LN, N>(A, s), C1 = above0<LN, N>(C, s);
  C = A * C1 + C;
  A = A * A1;
}
template <int LN, int NS>
__device__ __forceinline__ void affine_up_scan(double A, double &C, int s) {
#pragma clang fp contract(on)
  if (NS == 1) affine_up_step<LN, 1>(A, C, s);
  if (LN == kRowLanes) {
    affine_up_step<LN, 2>(A, C, s);
    affine_up_step<LN, 4>(A, C, s);
  }
  C = A * above0<LN, LN / 2>(C, s) + C;
}

// The same down the group, the first of its maps being absolute.
template <int LN, int N>
__device__ __forceinline__ void affine_down_step(double &A, double &C, int s) {
#pragma clang fp contract(on)
  const double A1 = below0<LN, N>(A, s), C1 = below0<LN, N>(C, s);
  C = A * C1 + C;
  A = A * A1;
}
template <int LN>
__device__ __forceinline__ void affine_down_scan(double A, double &C, int s) {
#pragma clang fp contract(on)
  affine_down_step<LN, 1>(A, C, s);
  if (LN == kRowLanes) {
    affine_down_step<LN, 2>(A, C, s);
    affine_down_step<LN, 4>(A, C, s);
  }
  C = A * below0<LN, LN / 2>(C, s) + C;
}

// Four values per lane summed over the wave's solves, lane by lane of their
// groups: row r gets the sum of value row_value(r) (groups of 4: each of its quads;
// the first adds it to the level sums, leads).
template <int LN>
__device__ __forceinline__ double sum_rows(double v0, double v1, double v2, double v3) {
  double z = swap16_sum(swap32_sum(v0, v1), swap32_sum(v2, v3));
  if (LN != kRowLanes) {
    z = z + dpp_move<0x128>(z);   // row_ror:8
    z = z + dpp_move<0x124>(z);   // row_ror:4
  }
  return z;
}
template <int LN>
__device__ __forceinline__ bool leads(int lane) { return LN == kRowLanes || lane % kRowLanes < LN; }
__device__ __forceinline__ int row_value(int row) { return (row & 1) * 2 + (row >> 1); }

// A wave's level sums in LDS: [up, down, direct][lp], each added to by one
// lane at a time.
__device__ __forceinline__ void acc_add(double *p, double v) {
  (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Two-stream coefficients and sources of one layer. in: the layer is one of
// the solve's (a lane past the last layer carries the identity). f: the direct
// beam at the layer's top, relative to the lane's; moved to its bottom.
template <bool MIXED, bool GEN, bool SOLAR, bool CLR>
__device__ __forceinline__ void row_layer(const LaneCtx &c, const SgTerm &t, const LayerIn &x, bool in, double &f,
                                          double &T, double &R, double &su, double &sd) {
#pragma clang fp contract(on)
  Coef o;
  if (MIXED) layer_coef_mixed<GEN, CLR>(c, t, x, o);
  else layer_coef<GEN, CLR>(c, t, x, o);
  T = in ? o.T : 1.0;
  R = in ? o.R : 0.0;
  if (SOLAR) {
    const double fnew = f * o.T0 * x.q1;
    su = in ? o.s1 * f : 0.0;
    sd = in ? (o.s2 - o.T0) * f + fnew : 0.0;
    f = in ? fnew : f;
  } else {
    su = in ? o.s1 * x.q2 + o.s2 * x.q1 : 0.0;
    sd = in ? -o.s1 * x.q2 + o.s2 * x.q1 : 0.0;
  }
}

// One layer of the elimination: from (rho, dn) at its top to those at its
// bottom; a, b: fu(top) = a fu(bottom) + b.
__device__ __forceinline__ void row_elim(double T, double R, double su, double sd, double &rho, double &dn,
                                         double &a, double &b) {
#pragma clang fp contract(on)
  const double bp = rcp_newton(1.0 - R * rho);
  a = T * bp;
  b = (R * dn + su) * bp;
  const double rho_n = R + T * rho * a;
  dn = T * (rho * b + dn) + sd;
  rho = rho_n;
}

// The layers of a run of n that lane s of its group takes: K on the first lanes,
// K - 1 on the others, from layer i0.
struct RowMap {
  int K, i0;
  bool full;
  __device__ __forceinline__ bool has(int k) const { return k + 1 < K || full; }
};
template <int LN>
__device__ __forceinline__ RowMap row_map(int n, int s) {
  const int K = (n + LN - 1) / LN, rem = n - LN * (K - 1);
  return RowMap{K, s * (K - 1) + min(s, rem), s < rem};
}

// What a lane keeps of its layers between the sweeps. ABS: layers that do not
// scatter, whose reflection (and so rho) is zero.
template <int KMAX, bool ABS>
struct RowState {
  double a[KMAX], b[KMAX], dn[KMAX], rho[ABS ? 1 : KMAX];
};

// General gas optics: the term's absorption in each of the lane's layers,
// ahead of the unrolled layer code (which would hold every scaling K times).
// Look-up terms three layers at a time, so that their loads overlap (one at a
// time, each layer waited for its record and then for its table entries).
// layer(k): the lane's k-th layer; put(k, v): keeps its absorption.
template <bool MIXED, class Layer, class Put>
__device__ __forceinline__ void row_gas(const SgTerm &t, const LaneSrc &src, int K, const Layer &layer,
                                        const Put &put) {
  const bool lut = t.fnc == SG_FNC_LOOKUP;
  if (__any(lut)) {
    const int nt = U(src.spec->n_tmp);
    const double *kl = G(U(src.spec->klut)) + (size_t)(lut ? t.lut : 0) * U(src.spec->n_pre) * nt;
    for (int k0 = 0; k0 < K; k0 += 3) {
      int i[3], o0[3], o1[3];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        i[j] = layer(min(k0 + j, K - 1));
        lut_at(src.grec[(size_t)i[j] * SG_NGQ + SG_G_IDX], nt, o0[j], o1[j]);
      }
      double v[3];
#pragma unroll
      for (int j = 0; j < 3; j++) v[j] = lut_k(kl, o0[j], o1[j], src.grec + (size_t)i[j] * SG_NGQ, src.mmr[i[j]]);
#pragma unroll
      for (int j = 0; j < 3; j++)
        if (k0 + j < K) put(k0 + j, v[j]);
    }
  }
  if (!lut)
    for (int k = 0; k < K; k++) {
      LayerIn x;
      load_layer<MIXED, true, false, true>(src, layer(k), x);
      put(k, x.kx);
    }
}

// The same of a clear run of n layers, into low.
template <bool MIXED>
__device__ __forceinline__ void row_gas_clear(const SgTerm &t, const LaneSrc &src, int n, const RowMap &mp,
                                              double *low, int lane) {
  row_gas<MIXED>(t, src, mp.K, [&](int k) { return max(min(mp.i0 + k, n - 1), 0); },
                 [&](int k, double v) { low[k * kWave + lane] = v; });
}

// Down the first n layers of the column, all clear: eliminates the lane's K
// layers; (rho, dn, fdir) become those at the bottom of the lane's layers
// (the last lane's: at level n). Adds the direct flux at the levels above n, with
// weight W, to acc.
template <bool MIXED, bool GEN, bool SOLAR, int KMAX, int LN>
__device__ __forceinline__ void row_down(const LaneCtx &c, const SgTerm &t, const LaneSrc &src, int n,
                                         const RowMap &mp, int s, double finc, double W,
                                         RowState<KMAX, false> &w, double &rho, double &dn, double &fdir, double *acc,
                                         int lp, double *low, int lane) {
#pragma clang fp contract(on)
  Slab S{1.0, 0.0, 0.0, 0.0, 0.0};
  double f = 1.0, fr[SOLAR ? KMAX : 1];
  if (GEN) row_gas_clear<MIXED>(t, src, n, mp, low, lane);
  // each layer's inputs are loaded while the one before is computed
  LayerIn x, nx;
  load_layer<MIXED, GEN, true>(src, max(min(mp.i0, n - 1), 0), nx);
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < mp.K) {
      x = nx;
      if (GEN) x.kx = low[k * kWave + lane];
      if (k + 1 < KMAX) load_layer<MIXED, GEN, true>(src, min(mp.i0 + k + 1, n - 1), nx);
      if (SOLAR) fr[k] = f;
      row_layer<MIXED, GEN, SOLAR, true>(c, t, x, mp.has(k), f, w.a[k], w.b[k], w.rho[k], w.dn[k]);
      const Slab B{w.a[k], w.b[k], w.b[k], w.rho[k], w.dn[k]};
      S = k == 0 ? B : slab_add(S, B);
    }
  }
  double F = 1.0;
  if (SOLAR) {
    F = finc * below1<LN, 1>(product_scan<LN, 1>(f, s), s);
    S.Su = S.Su * F;
    S.Sd = S.Sd * F;
    const double WF = W * F;
    const int v = row_value(lane / kRowLanes);
#pragma unroll
    for (int k0 = 0; k0 < KMAX; k0 += 4) {
      if (k0 < mp.K) {
        double d[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
          d[j] = (k0 + j < KMAX && k0 + j < mp.K) ? WF * fr[k0 + j < KMAX ? k0 + j : 0] : 0.0;
        const double z = sum_rows<LN>(d[0], d[1], d[2], d[3]);
        const int k = k0 + v;
        if (k < mp.K && mp.has(k) && leads<LN>(lane)) acc_add(acc + 2 * lp + mp.i0 + k, z);
      }
    }
  }
  if (s == 0) S.Sd = S.Sd + S.T * finc;
  slab_scan<LN, 1>(S, s);
  rho = below0<LN, 1>(S.Rb, s);
  dn = below0<LN, 1>(S.Sd, s);
  if (s == 0) dn = finc;
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < mp.K) {
      const double T = w.a[k], R = w.b[k];
      double su = w.rho[k], sd = w.dn[k];
      if (SOLAR) { su = su * F; sd = sd * F; }
      w.rho[k] = rho;
      w.dn[k] = dn;
      row_elim(T, R, su, sd, rho, dn, w.a[k], w.b[k]);
    }
  }
  fdir = SOLAR ? F * f : 0.0;
}

// row_down of infra-red layers that do not scatter, FP64 form: the flux goes
// down them by one affine recurrence, and fu(top) = T fu(bottom) + su.
template <bool GEN, int KMAX, int LN>
__device__ __forceinline__ void row_down_absorb(const LaneCtx &c, const SgTerm &t, const LaneSrc &src, int n,
                                                const RowMap &mp, int s, double finc, RowState<KMAX, true> &w,
                                                double &dn, double *low, int lane) {
#pragma clang fp contract(on)
  if (GEN) row_gas_clear<false>(t, src, n, mp, low, lane);
  LayerIn x, nx;
  load_layer<false, GEN, true>(src, max(min(mp.i0, n - 1), 0), nx);
  double A = 1.0, C = 0.0;
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < mp.K) {
      x = nx;
      if (k + 1 < KMAX) load_layer<false, GEN, true>(src, min(mp.i0 + k + 1, n - 1), nx);
      const double kgas = GEN ? low[k * kWave + lane] : k_term(t, x.lnp, x.lnt, x.mmr);
      double T, s1, s2;
      two_coeff_absorb((x.kgt + kgas) * x.mass, GEN && c.nosc, T, s1, s2);
      const bool in = mp.has(k);
      w.a[k] = in ? T : 1.0;
      w.b[k] = in ? s1 * x.q2 + s2 * x.q1 : 0.0;
      w.dn[k] = in ? -s1 * x.q2 + s2 * x.q1 : 0.0;
      C = w.a[k] * C + w.dn[k];
      A = w.a[k] * A;
    }
  }
  if (s == 0) C = A * finc + C;
  affine_down_scan<LN>(A, C, s);
  dn = below0<LN, 1>(C, s);
  if (s == 0) dn = finc;
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < mp.K) {
      const double sd = w.dn[k];
      w.dn[k] = dn;
      dn = w.a[k] * dn + sd;
    }
  }
}

// Up the same layers: X the (weighted) upward flux at level n, W the weight
// of the sources; adds the weighted upward and downward fluxes of the levels
// above n to acc.
template <int KMAX, bool ABS, int LN>
__device__ __forceinline__ void row_up(const RowMap &mp, int s, int lane, double X, double W,
                                       const RowState<KMAX, ABS> &w, double *acc, int lp) {
#pragma clang fp contract(on)
  double A = 1.0, C = 0.0;
#pragma unroll
  for (int k = KMAX - 1; k >= 0; k--) {
    if (k < mp.K) {
      C = w.a[k] * C + w.b[k];
      A = w.a[k] * A;
    }
  }
  C = C * W;
  if (s == LN - 1) C = A * X + C;
  affine_up_scan<LN, 1>(A, C, s);
  double x = above0<LN, 1>(C, s);
  if (s == LN - 1) x = X;
  const int v = row_value(lane / kRowLanes);
#pragma unroll
  for (int k0 = ((KMAX - 1) / 2) * 2; k0 >= 0; k0 -= 2) {
    if (k0 < mp.K) {
      double up[2] = {0.0, 0.0}, dw[2] = {0.0, 0.0};
#pragma unroll
      for (int j = 1; j >= 0; j--) {
        const int k = k0 + j;
        if (k < KMAX && k < mp.K) {
          x = w.a[k < KMAX ? k : 0] * x + w.b[k < KMAX ? k : 0] * W;
          up[j] = x;
          dw[j] = ABS ? w.dn[k < KMAX ? k : 0] * W : w.rho[ABS ? 0 : (k < KMAX ? k : 0)] * x + w.dn[k < KMAX ? k : 0] * W;
        }
      }
      const double z = sum_rows<LN>(up[0], dw[0], up[1], dw[1]);
      const int k = k0 + (v >> 1);
      if (k < mp.K && mp.has(k) && leads<LN>(lane)) acc_add(acc + (v & 1) * lp + mp.i0 + k, z);
    }
  }
}

// The upward flux at the surface (solver_homogen_direct.F90:93-127).
template <bool SOLAR>
__device__ __forceinline__ double surface_up(double alb_diff, double alb_dir, double sg_lw, double rho, double dn,
                                             double fdir) {
#pragma clang fp contract(on)
  const double sg = SOLAR ? (alb_dir - alb_diff) * fdir : sg_lw;
  return (alb_diff * dn + sg) / (1.0 - alb_diff * rho);
}

// A row's place in its g-point: weights and samples.
struct RowItem {
  int n_clear;      // 1 with a clear solve
  double w_clear;   // its weight
  double w_sub;     // weight of each McICA sample
  int n_s, s0;      // samples, the first one's index
};

// The cloudy part, layers ic..L-1, of each of the row's solves in turn, NS at
// a time (interleaved lanes: lane s works on solve s % NS, position s / NS),
// from the state (rho, dn, fdir) at level ic, which all of them share (every
// layer above ic is clear in every sub-column). Their number per lane varies
// from column to column, so the layers' state is indexed memory: LDS (low, up
// to kLowK layers per lane), or for cloud that reaches higher lane-private
// memory (KPRIV layers per lane). Adds the weighted fluxes of levels ic..L to
// acc; returns the weighted upward flux at level ic.
template <bool MIXED, bool GEN, bool SOLAR, int NS, int KPRIV, int LN>
__device__ __forceinline__ double row_cloudy(const LaneCtx &c, const SgTerm &t, const LaneSrc &src,
                                             const SgSpec *__restrict__ spec, int mode, const RowItem &g, int n_it,
                                             int L, int ic, int s, int lane, double rho_ic, double dn_ic,
                                             double f_ic, double alb_diff, double alb_dir, double sg_lw, double *acc,
                                             int lp, double *low) {
#pragma clang fp contract(on)
  constexpr int NP = LN / NS;   // positions
  const int p = s / NS, q = s % NS, nl = L - ic;
  const int K = (nl + NP - 1) / NP;
  const int v = row_value(lane / kRowLanes);
  const bool first = p == 0, last = p == NP - 1, lead = q == 0 && leads<LN>(lane);
  const int n_clear = g.n_clear;
  double *m = low + lane;
  constexpr int Q = GEN ? kLowQ + 1 : kLowQ;   // the last one the gas absorption
  double priv[KPRIV > 0 ? KPRIV * Q : 1];
#define SG_LOW(k, j) (*(KPRIV > 0 ? &priv[(k) * Q + (j)] : &m[((k) * Q + (j)) * kWave]))
  double xsum = 0.0;
  if (GEN)
    row_gas<MIXED>(t, src, K, [&](int k) { return ic + min(p * K + k, nl - 1); },
                   [&](int k, double v) { SG_LOW(k, kLowQ) = v; });
  for (int it = 0; it < n_it; it++) {
    const int j = it * NS + q, jc = j - n_clear;
    const bool clr = n_clear && j == 0, act = clr || (jc >= 0 && jc < g.n_s);
    LaneSrc sj = src;
    sj.isub = act && !clr ? spec->sub_isub[mode][g.s0 + jc] : 0;
    sj.csub = src.csub + (sj.isub > 0 ? sj.isub - 1 : 0);
    sj.csubf = src.csubf + (sj.isub > 0 ? sj.isub - 1 : 0);
    const double wj = clr ? g.w_clear : (act ? g.w_sub : 0.0);
    Slab S{1.0, 0.0, 0.0, 0.0, 0.0};
    double f = 1.0;
    for (int k = 0; k < K; k++) {
      const int r = p * K + k;
      LayerIn x;
      load_layer<MIXED, GEN>(sj, ic + min(r, nl - 1), x);
      if (GEN) x.kx = SG_LOW(k, kLowQ);
      Slab B;
      if (SOLAR) SG_LOW(k, 4) = f;
      row_layer<MIXED, GEN, SOLAR, false>(c, t, x, r < nl, f, B.T, B.Rt, B.Su, B.Sd);
      B.Rb = B.Rt;
      SG_LOW(k, 0) = B.T;
      SG_LOW(k, 1) = B.Rt;
      SG_LOW(k, 2) = B.Su;
      SG_LOW(k, 3) = B.Sd;
      S = slab_add(S, B);
    }
    double F = 1.0;
    if (SOLAR) {
      const double e = below1<LN, NS>(product_scan<LN, NS>(f, s), s);
      F = f_ic * e;
      S.Su = S.Su * F;
      S.Sd = S.Sd * F;
    }
    {
      double rb, sd;
      slab_below(rho_ic, dn_ic, S, rb, sd);
      S.Rb = first ? rb : S.Rb;
      S.Sd = first ? sd : S.Sd;
    }
    slab_scan<LN, NS>(S, s);
    double rho = below0<LN, NS>(S.Rb, s), dn = below0<LN, NS>(S.Sd, s);
    if (first) { rho = rho_ic; dn = dn_ic; }
    double A = 1.0, C = 0.0;   // fu(top of the lane) = A fu(bottom) + C
    for (int k = 0; k < K; k++) {
      const double T = SG_LOW(k, 0), R = SG_LOW(k, 1);
      double su = SG_LOW(k, 2), sd = SG_LOW(k, 3);
      if (SOLAR) { su = su * F; sd = sd * F; }
      SG_LOW(k, 2) = rho;
      SG_LOW(k, 3) = dn;
      double a, b;
      row_elim(T, R, su, sd, rho, dn, a, b);
      SG_LOW(k, 0) = a;
      SG_LOW(k, 1) = b;
      C = C + A * b;
      A = A * a;
    }
    const double fdir = SOLAR ? F * f : 0.0;
    const double fus = surface_up<SOLAR>(alb_diff, alb_dir, sg_lw, rho, dn, fdir);
    {
      // level L, from the last position's lanes
      const double wl = last ? wj : 0.0;
      double z = sum_rows<LN>(wl * fus, wl * (rho * fus + dn), wl * fdir, 0.0);
      if (NS == 2) z = z + dpp_move<kXor1>(z);
      if (last && lead && v < (SOLAR ? 3 : 2)) acc_add(acc + v * lp + L, z);
    }
    if (last) C = A * fus + C;
    affine_up_scan<LN, NS>(A, C, s);
    double fu = above0<LN, NS>(C, s);
    if (last) fu = fus;
    for (int k = K - 1; k >= 0; k--) {
      fu = SG_LOW(k, 0) * fu + SG_LOW(k, 1);
      const double fd = SG_LOW(k, 2) * fu + SG_LOW(k, 3);
      const double fb = SOLAR ? F * SG_LOW(k, 4) : 0.0;
      double z = sum_rows<LN>(wj * fu, wj * fd, wj * fb, 0.0);
      if (NS == 2) z = z + dpp_move<kXor1>(z);
      const int r = p * K + k;
      if (r < nl && lead && v < (SOLAR ? 3 : 2)) acc_add(acc + v * lp + ic + r, z);
    }
    if (first) xsum = xsum + wj * fu;
  }
#undef SG_LOW
  if (NS == 2) xsum = xsum + dpp_move<kXor1>(xsum);
  return of_first<LN>(xsum);
}

// The solves of one group of a column: some of its rounds of 4 (or 16) g-points.
// (mcica_sample.F90:453-930; monochromatic_radiance.F90:429-691;
// mcica_column.F90:255-622; solver_homogen_direct.F90:93-127.)
//
// In a column with McICA cloud every layer above the first cloudy one (ic) is
// clear in every sample, so a row goes down those layers once per g-point,
// then through the layers from ic down once per solve (the clear one and each
// sample), and back up the shared layers once for all of them together: they
// share fu(i) = a(i) fu(i+1) + b(i), so the weighted sum X(i) obeys X(i) =
// a(i) X(i+1) + b(i) W with W the sum of the weights. (mcica_column.F90:266-298
// recomputes those layers for every sample.)
//
// Output: partial[wave][up, down, direct][L+1] of the group's weighted sums
// (direct: solar calls only); fold: of the wave's groups 0 to group.
template <bool MIXED, int OPT, bool SOLAR, int KMAX, int LN>
__device__ __forceinline__ void solve_rows(const CallDims &d, const SgSpec *__restrict__ spec, int l_rayleigh,
                                           const double *__restrict__ colrec, const double *__restrict__ grec,
                                           const double *__restrict__ colscal, const double *__restrict__ bandrec,
                                           const double *__restrict__ bandscal, const double *__restrict__ c_sub,
                                           const double *__restrict__ cldopt, const double *__restrict__ aerrec,
                                           double *__restrict__ partial, int wave, bool fold, int group, int lane,
                                           double *acc, int lp, double *low, double *hot) {
#pragma clang fp contract(on)
  constexpr bool GEN = OPT != kOptPlain;
  const int L = d.L, NB = d.NB, G = spec->n_g;
  constexpr int kSolves = kWave / LN;
  const int col = fold ? wave : wave / d.nw, part = fold ? group : wave - col * d.nw;
  const int s = lane % LN;
  const double *cs = colscal + (size_t)col * SG_NS;
  const double fc = d.mcica ? cs[SG_S_FC] : 0.0;
  const bool cloudy = d.mcica && fc > 0.0;
  const int ic = cloudy ? min(max((int)cs[SG_S_CT], 0), L) : L;
  for (int i = lane; i < 3 * lp; i += kWave) acc[i] = 0.0;
  // the column's ln p, ln T, mass and mixing ratios, read by every round
  static_assert(SG_Q_LNP == 0 && SG_Q_LNT == 1 && SG_Q_MASS == 2 && SG_Q_MMR == 3, "the record's first kHotQ slots");
  for (int i = lane; i < L; i += kWave) {
    const double *r = colrec + ((size_t)col * L + i) * SG_NQ;
#pragma unroll
    for (int j = 0; j < kHotQ; j++) hot[j * lp + i] = r[j];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  const int n_round = (G + kSolves - 1) / kSolves;
  const int r1 = min(n_round, (part + 1) * d.rpw);
  for (int rd = part * d.rpw; rd < r1; rd++) {
    const int item = rd * kSolves + lane / LN;
    const bool act = item < G;
    const int gi = act ? item : 0;
    const SgTerm t = spec->g[gi];
    const int b = t.band;
    RowItem g;
    g.n_s = (act && cloudy) ? spec->g_n_sub[d.mode][gi] : 0;
    g.s0 = g.n_s > 0 ? spec->g_sub0[d.mode][gi] : 0;
    g.n_clear = act && fc < 1.0;
    g.w_clear = g.n_clear ? t.w * (1.0 - fc) : 0.0;
    g.w_sub = g.n_s > 0 ? t.w * (fc * spec->sub_inv_s[d.mode][g.s0]) : 0.0;
    const double *br = bandrec + ((size_t)col * NB + b) * L * SG_NBQ;
    const double *bs = bandscal + ((size_t)col * NB + b) * SG_NBQ;
    LaneCtx c;
    c.solar = SOLAR;
    c.sec0 = cs[SG_S_SEC0];
    c.ksc_clear = (SOLAR && l_rayleigh) ? spec->band[b].rayleigh : 0.0;
    c.ice = d.ice && !MIXED;
    c.nosc = GEN && !SOLAR ? term_nosc(d.scat, t.iscat) : 0;
    c.aer = OPT == kOptAer || (OPT == kOptAny && aerrec != nullptr);
    LaneSrc src;
    src.aer = c.aer ? aerrec + ((size_t)col * NB + b) * L * 4 : nullptr;
    src.rec = colrec + (size_t)col * L * SG_NQ;
    src.br = br;
    src.cop = d.mcica ? cldopt + ((size_t)col * NB + b) * L * d.co_stride : nullptr;
    src.co_stride = d.co_stride;
    src.ice = d.ice && !MIXED;
    src.ksc_clear = c.ksc_clear;
    src.copf = d.mcica ? (const float *)cldopt + ((size_t)col * NB + b) * L * 4 : nullptr;
    src.csub = c_sub + (size_t)col * L * SG_MAXSUBCOL;
    src.csubf = (const float *)c_sub + (size_t)col * L * SG_MAXSUBCOL;
    src.hot = hot;
    src.hp = lp;
    src.mmr = hot + (3 + t.gas) * lp;
    src.isub = 0;
    src.fnc = t.fnc;
    src.term = spec->g + gi;
    src.spec = spec;
    src.grec = grec ? grec + (size_t)col * L * SG_NGQ : nullptr;
    const double alb_diff = bs[2], alb_dir = bs[3];
    const double finc = SOLAR ? bs[0] / c.sec0 : -bs[0];   // flux_inc_down, flux_inc_direct
    const double sg_lw = SOLAR ? 0.0 : (1.0 - alb_diff) * (bs[1] - br[(L - 1) * SG_NBQ + 3]);
    // the group's solves, and the most any group of the wave has
    const int n_clear = g.n_clear;
    int n_solve = n_clear + g.n_s;
#pragma unroll
    for (int o = LN; o < kWave; o *= 2) n_solve = max(n_solve, __shfl_xor(n_solve, o, kWave));
    n_solve = __builtin_amdgcn_readfirstlane(n_solve);
    const int nl = L - ic;
    const RowMap mp = row_map<LN>(ic, s);
    const double W = g.w_clear + g.n_s * g.w_sub;
    // the layers from ic down: the surface, or the cloudy part first
    const auto below = [&](double rho, double dn, double fdir) -> double {
      if (nl == 0) {
        const double fus = surface_up<SOLAR>(alb_diff, alb_dir, sg_lw, rho, dn, fdir);
        const double X = W * fus;
        const double z = sum_rows<LN>(X, W * (rho * fus + dn), W * fdir, 0.0);
        const int v = row_value(lane / kRowLanes);
        if (s == 0 && leads<LN>(lane) && v < (SOLAR ? 3 : 2)) acc_add(acc + v * lp + L, z);
        return X;
      }
      // two solves side by side where the cloudy layers fit half of the group's lanes
      if (nl <= LN / 2 * kLowK)
        return row_cloudy<MIXED, GEN, SOLAR, 2, 0, LN>(c, t, src, spec, d.mode, g, (n_solve + 1) / 2, L, ic, s, lane,
                                                       rho, dn, fdir, alb_diff, alb_dir, sg_lw, acc, lp, low);
      return row_cloudy<MIXED, GEN, SOLAR, 1, KMAX, LN>(c, t, src, spec, d.mode, g, n_solve, L, ic, s, lane, rho, dn,
                                                        fdir, alb_diff, alb_dir, sg_lw, acc, lp, low);
    };
    double rho, dn, fdir;
    if (!MIXED && !SOLAR && !c.aer) {
      // infra-red clear air without aerosols does not scatter
      RowState<KMAX, true> w;
      row_down_absorb<GEN, KMAX, LN>(c, t, src, ic, mp, s, finc, w, dn, low, lane);
      const double X = below(0.0, of_last<LN>(dn), 0.0);
      row_up<KMAX, true, LN>(mp, s, lane, X, W, w, acc, lp);
    } else {
      RowState<KMAX, false> w;
      row_down<MIXED, GEN, SOLAR, KMAX, LN>(c, t, src, ic, mp, s, finc, W, w, rho, dn, fdir, acc, lp, low, lane);
      rho = of_last<LN>(rho);
      dn = of_last<LN>(dn);
      if (SOLAR) fdir = of_last<LN>(fdir);
      const double X = below(rho, dn, fdir);
      row_up<KMAX, false, LN>(mp, s, lane, X, W, w, acc, lp);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  double *out = partial + (size_t)wave * 3 * (L + 1);
  const bool add = fold && group > 0;
  for (int i = lane; i <= L; i += kWave)
#pragma unroll
    for (int v = 0; v < (SOLAR ? 3 : 2); v++) {
      double *o = out + v * (L + 1) + i;
      *o = add ? *o + acc[v * lp + i] : acc[v * lp + i];
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
}

// LDS of one wave: the cloudy part's layers, the level sums and the column.
// (general gas optics keep a cloudy layer's absorption beside its state)
__host__ __device__ constexpr int solve_low(int opt) {
  return kLowK * (opt == kOptPlain ? kLowQ : kLowQ + 1) * kWave;
}
template <int KMAX, int OPT, int LN>
__host__ __device__ constexpr int solve_lds_doubles() {
  return solve_low(OPT) + (3 + kHotQ) * (KMAX * LN + 1);
}

// Waves (64 threads each) of the calls of one build: W the work space. Where FOLD is
// set, a wave of a folding call takes a column's groups in turn, and sums them in the
// order in which the output kernel sums those of a wave each. (A loop over the groups
// in every build took 0.5 to 2 % of a step.)
template <bool MIXED, int OPT, int KMAX, int LN, int W>
__global__ __launch_bounds__(256, KMAX <= 9 ? 2 : 1) void b_solve_kernel(const BatchHdr *h, const ReqDesc *rq) {
  extern __shared__ double lds[];
  constexpr int lp = KMAX * LN + 1;
  constexpr bool FOLD = W == W_SOLVE_FOLD || LN == kFewLanes;
  const long long tot = h->tot[W];
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  double *low = lds + wv * solve_lds_doubles<KMAX, OPT, LN>(), *acc = low + solve_low(OPT), *hot = acc + 3 * lp;
  const long long nw = (long long)gridDim.x * (blockDim.x / kWave);
  for (long long w0 = (blockIdx.x * (long long)blockDim.x + threadIdx.x) / kWave; w0 < tot; w0 += nw) {
    const int w = __builtin_amdgcn_readfirstlane((int)w0);
    const int r = find_req(h, rq, W, w);
    const ReqDesc &q = rq[r];
    const int wave = w - (int)q.s[W];
    const bool fold = FOLD && q.d.fold;
    const int n = fold ? q.d.nw : 1;
    for (int g = 0; g < n; g++) {
      if (q.d.isolir == SOCGPU_SOURCE_SOLAR)
        solve_rows<MIXED, OPT, true, KMAX, LN>(q.d, G(q.spec), q.l_rayleigh, G(q.colrec), G(q.grec), G(q.colscal),
                                               G(q.bandrec), G(q.bandscal), G(q.csub), G(q.cldopt), G(q.aerrec),
                                               G(q.partial), wave, fold, g, lane, acc, lp, low, hot);
      else
        solve_rows<MIXED, OPT, false, KMAX, LN>(q.d, G(q.spec), q.l_rayleigh, G(q.colrec), G(q.grec), G(q.colscal),
                                                G(q.bandrec), G(q.bandscal), G(q.csub), G(q.cldopt), G(q.aerrec),
                                                G(q.partial), wave, fold, g, lane, acc, lp, low, hot);
    }
  }
}
