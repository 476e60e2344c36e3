// The triple-column solve: included by socgpu.hip, whose coefficients
// (two_coeff*, k_term*, k_scaled) and lane exchanges it uses.
//
// One solve is one (column, major k-term) of three regions (clear, stratiform and
// convective cloud) coupled by the overlap coefficients of each level
// (triple_column.F90:255-569). One block takes a column, each wave 21 of its
// k-terms, three lanes each:
//  - in and below the call's cloud top each lane takes a region, layer by layer:
//    the direct beam down (solar), the elimination of the regions' albedos and
//    sources up (solver_triple_hogan.F90:207-312), the substitution down. The
//    regions are mixed by exchanges between the three lanes;
//  - above it there is one region, and the lanes take three layers at a time:
//    their coefficients side by side, the elimination (downward, like the column
//    solve's) one after the other. The two halves meet at the cloud top.
// A lane's elimination state, 4 doubles per layer, goes through the workspace; the
// column's record, its overlap coefficients and the level sums are in LDS. The
// solar direct beam has a sweep of its own that forms its transmission again
// (keeping all coefficients of that sweep for the elimination moved 28 % more
// bytes and took 1578 us instead of 1516 in a 4096 x 90 FP64 step, SW + LW).
// What bounds it: the workspace (2.0 GB read and 1.5 GB written in that step's two
// solves of 1165 us together) beside FP64 arithmetic (VALU busy in 57 % of the
// cycles). One lane per k-term (all regions in turn, 64 k-terms a wave) took 1605 us
// there, waiting 74 % of its cycles on the column's records and the workspace with
// 2.7 waves per SIMD.
#pragma once

constexpr int kTriTerms = kWave / 3;      // k-terms per wave
constexpr int kTriWaves = 3;              // most waves per block (column)
constexpr int kTriQ = 4;                  // state per layer and lane
constexpr int kTriHot = 12;               // column record slots in LDS: lnp, lnt, mass, four gases,
                                          // cloud fraction, the two types' fractions, their reciprocals

__host__ __device__ inline int tri_chunks(int n_g) { return (n_g + kTriTerms - 1) / kTriTerms; }
// Doubles per layer and state of a column's workspace, which starts on a line: whole
// 128-byte lines for each wave (rows of 3 n_g, whose lines two waves write in part, had
// the 4096 x 90 step at 2515 us instead of 1578; whole lines of a workspace that began
// within one 1506 instead of 1489), but never more than the 64 lanes per 64 k-terms and
// three regions that callers' workspaces have held: 64 k-terms, whose padded row would
// be longer, take rows of 3 n_g.
__host__ __device__ inline int tri_row(int n_g) {
  const int full = n_g / kTriTerms, last = 3 * (n_g - full * kTriTerms);
  const int row = kWave * full + (last + 15) / 16 * 16, most = 3 * kWave * ((n_g + kWave - 1) / kWave);
  return row <= most ? row : 3 * n_g;
}
inline size_t tri_lds_doubles(int L, int waves) { return (size_t)(L + 1) * (kTriHot + kOv + 3 * waves); }

// The value of the lane at byte address 4 * lane.
__device__ __forceinline__ double lane_at(int addr, double v) {
  return mk64((unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)lo32(v)),
              (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)hi32(v)));
}

// Two-stream coefficients of one region of one layer for one lane: single
// scattering and delta-rescaling (single_scattering_all.F90,
// rescale_tau_omega.F90:73-80) of the region's grey optics kg (extinction,
// with the equivalent extinction), ks (scattering), g (rescaled asymmetry),
// fw (forward scattering) plus the lane's gas absorption kgas, then
// two_coeff (FP64) or two_coeff_f32 (mixed form, with the absorption formed
// in FP64 before rounding, as in layer_coef_mixed).
template <bool MIXED>
__device__ __forceinline__ void region_coef(const LaneCtx &c, double kgas, double mass, double kg, double ks,
                                            double g, double fw, Coef &o) {
#pragma clang fp contract(on)
  if (!MIXED) {
    double ktot = kg + kgas;
    double tau = ktot * mass;
    double om = fmin(ks / (ktot + kTiny), 1.0 - 32.0 * kEps);
    tau = tau * (1.0 - om * fw);
    om = om * (1.0 - fw) / (1.0 - om * fw);
    two_coeff(c.solar, tau, om, g, c.sec0, o);
  } else {
    const float ktot = (float)(kg + kgas);
    const float kab = (float)((kg - ks) + kgas);
    const float omc_min = (float)(32.0 * kEps);
    float tau = ktot * (float)mass;
    float omc = ktot > 0.0f ? fmaxf(SG_FDIV(kab, ktot), omc_min) : 1.0f;
    float om = 1.0f - omc;
    const float sc = 1.0f - om * (float)fw;
    tau = tau * sc;
    omc = SG_FDIV(omc, sc);
    om = 1.0f - omc;
    CoefF f;
    two_coeff_f32(c.solar, tau, om, omc, (float)g, (float)c.sec0, f);
    coef_from_f32(f, o);
  }
}

// The k-term's absorption in one layer: h the layer's record in LDS, r and g
// its records in memory (general gas optics only).
template <bool MIXED, bool GEN>
__device__ __forceinline__ double tri_kgas(const SgTerm &t, const SgSpec *spec, const double *h, const double *r,
                                           const double *g) {
  if (GEN && t.fnc != SG_FNC_POWER_LAW) {
    const double k = k_scaled(t, spec, h[0], r[SG_Q_P], r[SG_Q_T], g, h[3 + t.gas]);
    return MIXED ? (double)(float)k : k;
  }
  if (MIXED) return (double)k_term_f32(t, (float)h[0], (float)h[1], (float)h[3 + t.gas]);
  return k_term(t, h[0], h[1], h[3 + t.gas]);
}

// One layer's inputs of a lane's region, loaded a layer ahead.
struct TriIn {
  double kg, ks, g, fw;   // extinction, scattering, asymmetry, forward scattering
  double q1, q2;          // solar: adjustment of the direct beam; infra-red: Planck terms
};

struct TriLane {
  const double *br, *cop, *ab;   // band, cloud optics and aerosol records of the k-term's band
  double ksc;                    // Rayleigh scattering
};

// Region k's optics of layer i.
template <bool SOLAR, bool GEN>
__device__ __forceinline__ TriIn tri_in(const TriLane &x, int k, int i) {
  TriIn o;
  const double *bq = x.br + (size_t)i * SG_NBQ;
  const double *p = k > 0 ? x.cop + (size_t)i * 8 + 4 * (k - 1) : bq;
  o.q1 = bq[1];
  o.q2 = SOLAR ? 0.0 : bq[2];
  o.kg = p[0]; o.ks = p[1]; o.g = p[2]; o.fw = p[3];
  if (k == 0) { o.ks = x.ksc; o.g = 0.0; o.fw = 0.0; }
  if (GEN && x.ab && k == 0) {
#pragma clang fp contract(off)
    // clear region with aerosols: moments over the scattering, the phase
    // function delta-rescaled (grey_opt_prop.F90:1360-1440,
    // rescale_phase_fnc.F90:116-124)
    const double *ar = x.ab + (size_t)i * 4;
    double ks = ar[0], pf = ar[1], fw = ar[2];
    if (ks > kTiny) {
      const double inv = 1.0 / ks;
      fw = fw * inv;
      pf = pf * inv;
    }
    pf = (pf - fw) / (1.0 - fw);
    o.ks = ks; o.g = pf; o.fw = fw;
  }
  return o;
}

// Region coefficients in cloudy layers, weighted as two_coeff_region.F90:200-445
// forms them: the type's coefficients times its fraction f, summed from zero,
// times the reciprocal inv of the region fraction (the same fraction here; 1 for
// the clear region); zero where the type is absent.
template <bool MIXED>
__device__ __forceinline__ void tri_coef(const LaneCtx &c, double kgas, double mass, const TriIn &x, double f,
                                         double inv, Coef &o) {
  if (f > kTiny) {
    region_coef<MIXED>(c, kgas, mass, x.kg, x.ks, x.g, x.fw, o);
    o.T = (0.0 + f * o.T) * inv;
    o.R = (0.0 + f * o.R) * inv;
    o.T0 = (0.0 + f * o.T0) * inv;
    o.s1 = (0.0 + f * o.s1) * inv;
    o.s2 = (0.0 + f * o.s2) * inv;
  } else {
    o.T = 0.0; o.R = 0.0; o.T0 = 0.0; o.s1 = 0.0; o.s2 = 0.0;
  }
}

// The solve of 21 k-terms of one column. hot, ov: the column's record and overlap
// coefficients, acc: the wave's level sums [up, down, direct][L + 1], ws: the
// column's workspace [layer][kTriQ][tri_row].
template <bool MIXED, bool GEN, bool SOLAR>
__device__ __forceinline__ void tri_rows(const CallDims &d, const SgSpec *__restrict__ spec, int l_rayleigh, int col,
                                         int chunk, int lane, const double *__restrict__ colrec,
                                         const double *__restrict__ grec, const double *__restrict__ colscal,
                                         const double *__restrict__ bandrec, const double *__restrict__ bandscal,
                                         const double *__restrict__ cldopt, const double *__restrict__ aerrec,
                                         int nct, const double *hot, const double *ov, double *acc,
                                         double *__restrict__ ws) {
#pragma clang fp contract(on)
  const int L = d.L, NB = d.NB, lp = L + 1, n = nct - 1;   // n clear layers
  // the last lane and the lanes past the last k-term repeat a lane before them
  // without weight: they store what it stores (a store or load under a branch would
  // be counted as none, and the next wait for a load then wait for the stores too)
  const int n_g = U(spec->n_g), left = n_g - chunk * kTriTerms;
  const int l3 = min(lane, 3 * min(left, kTriTerms) - 1 - (2 - min(lane, 3 * kTriTerms - 1) % 3)), k = l3 % 3;
  const int item = chunk * kTriTerms + l3 / 3;
  const SgTerm t = spec->g[item];
  const double wgt = l3 == lane ? t.w : 0.0;
  const int a0 = 4 * (l3 - k), a1 = a0 + 4, a2 = a0 + 8;     // addresses of the three lanes
  const double *rec = colrec + (size_t)col * L * SG_NQ;
  const double *gr = GEN && grec ? grec + (size_t)col * L * SG_NGQ : nullptr;
  const double *bs = bandscal + ((size_t)col * NB + t.band) * SG_NBQ;
  LaneCtx c;
  c.solar = SOLAR;
  c.sec0 = colscal[(size_t)col * SG_NS + SG_S_SEC0];
  c.ice = false;
  c.nosc = 0;
  c.aer = false;
  TriLane x;
  x.br = bandrec + ((size_t)col * NB + t.band) * L * SG_NBQ;
  x.cop = cldopt + ((size_t)col * NB + t.band) * L * 8;
  x.ab = GEN && aerrec ? aerrec + ((size_t)col * NB + t.band) * L * 4 : nullptr;
  x.ksc = SOLAR && l_rayleigh ? spec->band[t.band].rayleigh : 0.0;
  const double alb_diff = bs[2], alb_dir = bs[3], bs0 = bs[0], bs1 = bs[1];
  const double finc = SOLAR ? bs0 / c.sec0 : -bs0;   // flux_inc_down (= flux_inc_direct)
  // workspace of layer i (of a clear layer's group of three: of the first)
  const int row = tri_row(n_g), nl = 3 * min(left, kTriTerms);
  double *const wl = ws + (row == 3 * n_g ? chunk * 3 * kTriTerms + l3
                                          : chunk * kWave + (lane < (nl + 15) / 16 * 16 ? lane : l3));
  auto wc = [&](int i, int q) -> double & { return wl[(i * kTriQ + q) * row]; };
  auto kgas = [&](int i) {
    return tri_kgas<MIXED, GEN>(t, spec, hot + i * kTriHot, rec + (size_t)i * SG_NQ,
                                GEN && gr ? gr + (size_t)i * SG_NGQ : nullptr);
  };

  // --- clear layers, down: (rho, dn, F) the reflectance of the layers above, the
  // diffuse flux they send down and the direct flux
  double rho = 0.0, dn = finc, F = finc;
  for (int i0 = 0; i0 < n; i0 += 3) {
    const bool in = i0 + k < n;
    const int i = min(i0 + k, n - 1);
    const TriIn y = tri_in<SOLAR, GEN>(x, 0, i);
    Coef o;
    region_coef<MIXED>(c, kgas(i), hot[i * kTriHot + 2], y.kg, y.ks, y.g, y.fw, o);
    const double T = in ? o.T : 1.0, R = in ? o.R : 0.0;
    double su, sd;
    if (SOLAR) {
      const double tr = o.T0 * y.q1, p = in ? tr : 1.0;
      const double f1 = F * lane_at(a0, p), f2 = f1 * lane_at(a1, p);
      const double top = k == 0 ? F : (k == 1 ? f1 : f2);
      F = f2 * lane_at(a2, p);
      su = in ? o.s1 * top : 0.0;
      sd = in ? (o.s2 - o.T0) * top + top * tr : 0.0;
      const double z = in ? wgt * top : 0.0;
      double v[8] = {k == 0 ? z : 0.0, k == 1 ? z : 0.0, k == 2 ? z : 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      reduce8(v, lane);
      const int m = lane >> 3;
      if ((lane & 7) == 0 && m < 3 && i0 + m < n) acc[2 * lp + i0 + m] += v[0];
    } else {
      su = in ? o.s1 * y.q2 + o.s2 * y.q1 : 0.0;
      sd = in ? -o.s1 * y.q2 + o.s2 * y.q1 : 0.0;
    }
    double a = 0.0, b = 0.0, rk = 0.0, dk = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const int am = m == 0 ? a0 : (m == 1 ? a1 : a2);
      const double Tm = lane_at(am, T), Rm = lane_at(am, R), um = lane_at(am, su), dm = lane_at(am, sd);
      if (k == m) { rk = rho; dk = dn; }
      double ea, eb;
      row_elim(Tm, Rm, um, dm, rho, dn, ea, eb);
      if (k == m) { a = ea; b = eb; }
    }
    wc(i0, 0) = a;
    wc(i0, 1) = b;
    wc(i0, 2) = rk;
    wc(i0, 3) = dk;
  }

  // coefficients of the lane's region in layer i; the gas absorption of three
  // layers at a time, one per lane (the first of them when j is 0, in steps of dir)
  double kg3 = 0.0;
  auto coef = [&](int i, int j, int dir, const TriIn &y, Coef &o) {
    if (j == 0) kg3 = kgas(max(min(i + dir * k, L - 1), n));
    const double *h = hot + i * kTriHot;
    tri_coef<MIXED>(c, lane_at(a0 + 4 * j, kg3), h[2], y, k == 0 ? 1.0 : h[7 + k], k == 0 ? 1.0 : h[9 + k], o);
  };

  // --- cloudy layers, solar: the direct flux entering each
  // region of each layer (triple_solar_source.F90:180-412)
  double base = k == 0 ? F : 0.0;    // leaving the region of the layer above
  if (SOLAR) {
    double v[8];
    TriIn nx = tri_in<SOLAR, GEN>(x, k, n);
    auto put = [&](int i) {          // direct flux at level i, summed 8 levels at a time
      const int m = (i - n) & 7;
      const double z = wgt * base;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (j == m) v[j] = z;
        else if (j > m && i == L) v[j] = 0.0;
      }
      if (m == 7 || i == L) {
        reduce8(v, lane);
        const int lev = i - m + (lane >> 3);
        if ((lane & 7) == 0 && lev <= L) acc[2 * lp + lev] += v[0];
      }
    };
    for (int i = n, j = 0; i < L; i++, j = j == 2 ? 0 : j + 1) {
      const TriIn y = nx;
      nx = tri_in<SOLAR, GEN>(x, k, min(i + 1, L - 1));
      put(i);
      const double *u = ov + i * kOv + 3 * k;   // interface at the layer's top
      Coef o;
      coef(i, j, 1, y, o);
      const double top = u[0] * lane_at(a0, base) + u[1] * lane_at(a1, base) + u[2] * lane_at(a2, base);
      base = top * o.T0 * y.q1;
      wc(i, 0) = top;
    }
    put(L);
  }

  // --- cloudy layers, upward elimination (solver_triple_hogan.F90:207-312)
  double a = alb_diff, g;
  if (SOLAR) {
    g = (alb_dir - alb_diff) * base;
  } else {
    const double dps = bs1 - x.br[(size_t)(L - 1) * SG_NBQ + 3];
    g = ov[L * kOv + 9 + 3 * k] * (1.0 - alb_diff) * dps;
  }
  {
    TriIn nx;
    double ntop = 0.0;
    auto load = [&](int i) {
      nx = tri_in<SOLAR, GEN>(x, k, i);
      if (SOLAR) ntop = wc(i, 0);
    };
    load(L - 1);
    for (int i = L - 1, j = 0; i >= n; i--, j = j == 2 ? 0 : j + 1) {
      const TriIn y = nx;
      const double top = ntop;
      load(max(i - 1, n));
      Coef o;
      coef(i, j, -1, y, o);
      const double T = o.T, R = o.R;
      double su, sd;
      if (SOLAR) {
        su = o.s1 * top;
        sd = (o.s2 - o.T0) * top + top * o.T0 * y.q1;
      } else {
        const double *h = hot + i * kTriHot;
        const double w = h[7], wk = k == 0 ? 1.0 - w : w * h[7 + k];   // area of the region
        su = wk * (o.s1 * y.q2 + o.s2 * y.q1);
        sd = wk * (-o.s1 * y.q2 + o.s2 * y.q1);
      }
      const double *vb = ov + (i + 1) * kOv + k, *ut = ov + i * kOv + 9 + 3 * k;
      const double th = lane_at(a0, a) * vb[0] + lane_at(a1, a) * vb[3] + lane_at(a2, a) * vb[6];
      const double binv = rcp_newton(1.0 - th * R);
      const double c1 = th * T * binv;
      const double c2 = (g + th * sd) * binv;
      const double lsrc = su + T * c2;
      a = R + T * c1;
      // fu(bottom) = c1 fd + c2, fd(bottom) = e1 fd + e2
      wc(i, 0) = c1;
      wc(i, 1) = c2;
      wc(i, 2) = T + R * c1;
      wc(i, 3) = R * c2 + sd;
      g = ut[0] * lane_at(a0, lsrc) + ut[1] * lane_at(a1, lsrc) + ut[2] * lane_at(a2, lsrc);
    }
  }

  // --- where the halves meet: the fluxes at the cloud top (level n); from a
  // cloud top in the last layer the clear region's albedo alone is carried up
  double fu, fd;
  {
    const double *vb = ov + n * kOv;
    const double b0 = lane_at(a0, a), g0 = lane_at(a0, g);
    const double mix = b0 * vb[0] + lane_at(a1, a) * vb[3] + lane_at(a2, a) * vb[6];
    const double th = n > 0 && nct == L ? b0 : mix;
    fd = (rho * g0 + dn) * rcp_newton(1.0 - rho * th);
    fu = th * fd + g0;
  }

  // --- cloudy layers, downward substitution: the fluxes at every level, summed
  // over the wave 4 levels at a time
  {
    double v[8];
    auto put = [&](int lev, double u, double w) {
      const int m = (lev - n) & 3;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (j == m) { v[2 * j] = u; v[2 * j + 1] = w; }
        else if (j > m && lev == L) { v[2 * j] = 0.0; v[2 * j + 1] = 0.0; }
      }
      if (m == 3 || lev == L) {
        reduce8(v, lane);
        const int j = lane >> 3, lv = lev - m + (j >> 1);
        if ((lane & 7) == 0 && lv <= L) acc[(j & 1) * lp + lv] += v[0];
      }
    };
    double dk = k == 0 ? fd : 0.0;
    put(n, k == 0 ? wgt * fu : 0.0, wgt * dk);
    double nw[kTriQ] = {};
    auto load = [&](int i) {
#pragma unroll
      for (int q = 0; q < kTriQ; q++) nw[q] = wc(i, q);
    };
    load(n);
    for (int i = n; i < L; i++) {
      double w[kTriQ];
#pragma unroll
      for (int q = 0; q < kTriQ; q++) w[q] = nw[q];
      load(min(i + 1, L - 1));
      const double *vt = ov + i * kOv + 3 * k;
      const double top = vt[0] * lane_at(a0, dk) + vt[1] * lane_at(a1, dk) + vt[2] * lane_at(a2, dk);
      dk = w[2] * top + w[3];
      put(i + 1, wgt * (w[0] * top + w[1]), wgt * dk);
    }
  }

  // --- clear layers, up
  for (int i0 = (n - 1) / 3 * 3; i0 >= 0 && n > 0; i0 -= 3) {
    const bool in = i0 + k < n;
    const double ak = wc(i0, 0), bk = wc(i0, 1), rk = wc(i0, 2), dk = wc(i0, 3);
    double xk = 0.0;
#pragma unroll
    for (int m = 2; m >= 0; m--) {
      const int am = m == 0 ? a0 : (m == 1 ? a1 : a2);
      fu = lane_at(am, ak) * fu + lane_at(am, bk);
      if (k == m) xk = fu;
    }
    const double zu = in ? wgt * xk : 0.0, zd = in ? wgt * (rk * xk + dk) : 0.0;
    double v[8] = {k == 0 ? zu : 0.0, k == 0 ? zd : 0.0, k == 1 ? zu : 0.0, k == 1 ? zd : 0.0,
                   k == 2 ? zu : 0.0, k == 2 ? zd : 0.0, 0.0, 0.0};
    reduce8(v, lane);
    const int m = lane >> 4, f = (lane >> 3) & 1;
    if ((lane & 7) == 0 && m < 3 && i0 + m < n) acc[f * lp + i0 + m] += v[0];
  }
}

template <bool MIXED, bool GEN>
__global__ __launch_bounds__(kTriWaves * kWave, 3) void b_tsolve_kernel(const BatchHdr *h, const ReqDesc *rq,
                                                                       int space) {
  extern __shared__ double lds[];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int nwv = blockDim.x / kWave;
  const long long tot = h->tot[space];
  for (long long w = blockIdx.x; w < tot; w += gridDim.x) {
    const ReqDesc &q = rq[find_req(h, rq, space, w)];
    const CallDims d = U_struct(q.d);
    const int col = (int)(w - U(q.s[space])), L = d.L, lp = L + 1;
    const SgSpec *spec = G(U(q.spec));
    const double *colrec = G(U(q.colrec)) + (size_t)col * L * SG_NQ;
    const double *ovl = G(U(q.ovl)) + (size_t)col * lp * kOv;
    double *hot = lds, *ov = hot + L * kTriHot, *acc = ov + lp * kOv;
    for (int e = threadIdx.x; e < L * kTriHot; e += blockDim.x) {
      const int i = e / kTriHot, s = e - i * kTriHot;
      const double z = colrec[(size_t)i * SG_NQ + (s < 8 ? s : ((s & 1) == 0 ? SG_Q_FRAC1 : SG_Q_FRAC2))];
      hot[e] = s < 10 ? z : 1.0 / z;
    }
    for (int e = threadIdx.x; e < lp * kOv; e += blockDim.x) ov[e] = ovl[e];
    for (int e = threadIdx.x; e < 3 * lp * nwv; e += blockDim.x) acc[e] = 0.0;
    __syncthreads();
    const int n_g = U(spec->n_g), nch = tri_chunks(n_g);
    double *ws = G(U(q.tws)) + (size_t)col * L * kTriQ * tri_row(n_g);
    const int nct = min(*G(U(q.krange)), L);   // 1-based cloud top of the call
    for (int ch = wv; ch < nch; ch += nwv) {
      if (d.isolir == SOCGPU_SOURCE_SOLAR)
        tri_rows<MIXED, GEN, true>(d, spec, U(q.l_rayleigh), col, ch, lane, G(U(q.colrec)), G(U(q.grec)),
                                   G(U(q.colscal)), G(U(q.bandrec)), G(U(q.bandscal)), G(U(q.cldopt)),
                                   G(U(q.aerrec)), nct, hot, ov, acc + wv * 3 * lp, ws);
      else
        tri_rows<MIXED, GEN, false>(d, spec, U(q.l_rayleigh), col, ch, lane, G(U(q.colrec)), G(U(q.grec)),
                                    G(U(q.colscal)), G(U(q.bandrec)), G(U(q.bandscal)), G(U(q.cldopt)),
                                    G(U(q.aerrec)), nct, hot, ov, acc + wv * 3 * lp, ws);
    }
    __syncthreads();
    double *out = G(U(q.partial)) + (size_t)col * 3 * lp;
    for (int e = threadIdx.x; e < 3 * lp; e += blockDim.x) {
      double z = acc[e];
      for (int j = 1; j < nwv; j++) z += acc[j * 3 * lp + e];
      out[e] = z;
    }
    __syncthreads();
  }
}
