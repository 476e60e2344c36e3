// The band kernel: included by socgpu.hip after solve_rows.h, whose row
// operations it uses.
//
// Per (column, band): the equivalent extinction of the band's minor gases
// (solve_band_k_eqv_scl.F90:572-1047), then the band's per-layer records. The
// band's gases and their k-terms in turn:
//  - solar: each term's direct-beam transmission down the column (:654-739);
//    k_eqv = sum_k k T_k(surface) / sum_k T_k(surface) per gas (:826-846), and
//    adjust_solar_ke from the per-layer ratios of the summed transmissions
//    (:848-891);
//  - infra-red: each term's non-scattering fluxes (monochromatic_gas_flux.F90:
//    115-196, diffusivity 1.66), two affine recurrences; k_eqv = sum k |F| /
//    sum |F| over the layer's two levels (:995-1019);
//  - where the weighting flux vanishes, the smallest k of the gas's terms.
//
// A block takes 4 columns and its waves the bands in turn; in a wave a row of 16
// lanes takes one column, 16 consecutive layers at a time, all of a column's in
// registers; the recurrences down and up it are scans over the rows. The columns'
// records are brought into LDS once for all bands, and the tables are read by
// scalar loads (U). (One wave per column and band, a layer
// per lane, waited two thirds of its cycles: on the records, on six-step scans of
// 64 lanes per 64 layers, on the LDS-routed reversal of the upward scan; and left
// 38 of 128 lanes idle at 90 layers. 4096 x 90 SW + LW: 457 us then, 257 now, where
// VALU instructions issue in 61 % of the cycles.)
#pragma once

// Waves per block: 4 share the staging of 4 columns well while two blocks fit a CU
// (two waves per SIMD; at three, 168 registers, the kernel spills). A launch of few
// blocks gives every band a wave of its own, in 3 blocks per 4 columns (64 x 60
// LW: 23 us with all 9 bands in a block of 8 waves).
constexpr int kBandWaves = 4, kBandFew = 128, kBandFewWaves = 3, kBandFewBlocks = 3;
constexpr int kBandQ = 9;       // staged per layer: ln p, ln T, mass, H2O, CO2, O3, T, level T,
                                // cloud (type fraction, or the total for the triple column)

__host__ __device__ inline int band_quads(const CallDims &d) { return (d.P + kRows - 1) / kRows; }

// LDS doubles of a block of n waves: the staged columns, and per wave three values
// per lane and layer.
__host__ __device__ constexpr int band_lds_doubles(int kmax, int n) {
  return kBandQ * kRows * (kmax * kRowLanes + 1) + n * 3 * kmax * kWave;
}

struct BandSrc {
  const double *st;   // the row's column in LDS: quantity q of layer i at st[q lp + i]
  int lp;
  __device__ __forceinline__ double operator()(int q, int i) const { return st[q * lp + i]; }
};

// Droplet (and ice) optics at unit condensate scaling of one layer of a McICA
// column (they depend on the band, not on the k-term; the solve scales them by
// each sub-column's c_sub), written only where the layer has cloud: the solve
// uses them only in cloudy layers of a sub-column.
__device__ __forceinline__ void band_cloud(const CallDims &d, const SgSpec *__restrict__ spec, const double *r,
                                           double *__restrict__ cldopt, size_t at, int b) {
  double kext, kscat, phf, fwd;
  drop_optics(spec->drop[d.drop], b, r[SG_Q_LWC], r[SG_Q_RE], kext, kscat, phf, fwd);
  double ie = 0.0, is = 0.0, ip = 0.0, iff = 0.0;
  if (d.ice) ice_optics(spec->ice[d.ice_t], b, r[SG_Q_IWC], r[SG_Q_DE], r[SG_Q_T], ie, is, ip, iff);
  if (d.f32) {
    // mixed form: droplets and ice together, (kext, kext - kscat, phf, fwd) in
    // FP32, the absorption formed here in FP64
    kext = kext + ie; kscat = kscat + is; phf = phf + ip; fwd = fwd + iff;
    ((float4 *)cldopt)[at] = make_float4((float)kext, (float)(kext - kscat), (float)phf, (float)fwd);
  } else {
    double *co = cldopt + at * d.co_stride;
    co[0] = kext; co[1] = kscat; co[2] = phf; co[3] = fwd;
    if (d.ice) { co[4] = ie; co[5] = is; co[6] = ip; co[7] = iff; }
  }
}

// Triple column: grey optics of each cloud type (grey_opt_prop.F90:975-1000,
// 1185-1230: the clear-air totals (kclr = kaer + kcont, ksc, pfa, fwa), then the
// type's droplets and its ice component, at layers from the call's cloud top
// where the column has cloud), the equivalent extinction
// (solve_band_k_eqv_scl.F90:1038-1045), moments normalised by the scattering
// (grey_opt_prop.F90:1474-1500) and the delta-rescaled phase function
// (rescale_phase_fnc.F90).
__device__ __forceinline__ void band_regions(const CallDims &d, const SgSpec *__restrict__ spec, const double *r,
                                             double *__restrict__ co, int b, bool cloudy, double kclr, double ksc_clr,
                                             double pfa, double fwa, double keq, double kgrey) {
  for (int k = 0; k < 2; k++) {
    double kgt = kclr + ksc_clr, ksc = ksc_clr, phf = pfa, fwd = fwa;
    if (cloudy) {
      double ct, cs, cp, cf;
      drop_optics(spec->drop[k == 0 ? d.drop : d.drop2], b, r[k == 0 ? SG_Q_LWC : SG_Q_LWC2],
                  r[k == 0 ? SG_Q_RE : SG_Q_RE2], ct, cs, cp, cf);
      kgt = kgt + ct;
      ksc = ksc + cs;
      phf = phf + cp;
      fwd = fwd + cf;
      // the type's ice component
      ct = 0.0; cs = 0.0; cp = 0.0; cf = 0.0;
      if (d.ice)
        ice_optics(spec->ice[k == 0 ? d.ice_t : d.ice_t2], b, r[k == 0 ? SG_Q_IWC : SG_Q_IWC2],
                   r[k == 0 ? SG_Q_DE : SG_Q_DE2], r[SG_Q_T], ct, cs, cp, cf);
      kgt = kgt + ct;
      ksc = ksc + cs;
      phf = phf + cp;
      fwd = fwd + cf;
    }
    kgt = kgt + keq + kgrey;
    if (ksc > kTiny) {
      const double inv = 1.0 / ksc;
      fwd = fwd * inv;
      phf = phf * inv;
    }
    phf = (phf - fwd) / (1.0 - fwd);
    co[4 * k + 0] = kgt;
    co[4 * k + 1] = ksc;
    co[4 * k + 2] = phf;
    co[4 * k + 3] = fwd;
  }
}

// The scans of a column's recurrences. Layer i = 16 c + s is lane s's c-th; each
// run of 16 layers is scanned over the row, and the runs are joined in groups of
// four: the second takes the first's total, the third and the fourth (after
// taking the third's total) the first two's. The order of every product and sum
// is fixed by the layer alone, so a layer's equivalent extinction does not depend
// on the split (the optical depths it enters are amplified by the reference's
// ill-conditioned source terms, where a last-bit change moves heating rates by
// 1e-7).
struct Affine {
  double A, C;
};
__device__ __forceinline__ Affine after(const Affine &x, const Affine &y) {   // y, then x
  return Affine{x.A * y.A, x.A * y.C + x.C};
}
template <int CTRL>
__device__ __forceinline__ void affine_fold(Affine &x) {
  const double A0 = dpp_or1<CTRL>(x.A), C0 = dpp_f64<CTRL, 0xf>(x.C, 0.0);
  x.C = x.A * C0 + x.C;
  x.A = x.A * A0;
}
template <int CTRL>
__device__ __forceinline__ Affine affine_bcast(const Affine &x) {
  return Affine{dpp_or0<CTRL>(x.A), dpp_or0<CTRL>(x.C)};
}

// One band of the wave's 4 columns, the row's column (col, clamped into the
// call; live: it is one of the call's).
template <int KMAX, bool GEN, bool SOLAR>
__device__ __forceinline__ void band_rows(const ReqDesc &q, const CallDims &d, const BandSrc &x, int col, bool live,
                                          int b, int s, int lane, double *buf) {
  const SgSpec *__restrict__ spec = G(U(q.spec));
  const int L = d.L, NB = d.NB, K = (L + kRowLanes - 1) / kRowLanes;
  const SgBand &B = spec->band[b];
  const int n_gas = U(B.n_minor_gas), minor0 = U(B.minor0), grey1 = d.grey1;
  const double *rec = G(U(q.colrec)) + (size_t)col * L * SG_NQ;
  const double *colscal = G(U(q.colscal)) + (size_t)col * SG_NS;
  const double *grec = U(q.grec) ? G(U(q.grec)) + (size_t)col * L * SG_NGQ : nullptr;
  double *bs = G(U(q.bandscal)) + ((size_t)col * NB + b) * SG_NBQ;
  const double sec0 = colscal[SG_S_SEC0], alb = bs[2];
  const bool first = s == 0, last = s == kRowLanes - 1;
  const auto has = [&](int c) { return c * kRowLanes + s < L; };
  const auto layer = [&](int c) { return min(c * kRowLanes + s, L - 1); };
  PlanckBand pb;
  double db[SOLAR ? 1 : KMAX], b_top = 0.0, b_bot = 0.0, bg = 0.0;   // Planck difference of each layer; the ends
  if (!SOLAR) {
    pb = planck_coef(spec, B);
#pragma unroll
    for (int c = 0; c < KMAX; c++)
      db[c] = planck_band(pb, x(7, layer(c) + 1)) - planck_band(pb, x(7, layer(c)));
    b_top = planck_band(pb, x(7, 0));
    b_bot = planck_band(pb, x(7, L));
    bg = colscal[SG_S_LFG] != 0.0 ? bs[1] : planck_band(pb, colscal[SG_S_TGROUND]);
  }
  double keq[KMAX], adj[SOLAR ? KMAX : 1];
#pragma unroll
  for (int c = 0; c < KMAX; c++) {
    keq[c] = 0.0;
    if (SOLAR) adj[c] = 1.0;
  }
  const double sqe = 1.4901161193847656e-08;
  // the absorption of a term in layer i. Further gases (general gas optics): the
  // call's field, clamped at 0, else its well-mixed ratio
  // (socrates_set_atm.F90:535-622)
  const auto amount = [&](const SgTerm &t, int i) -> double {
    if (GEN && t.gas >= SG_GAS_WM0) {
      const double *fld = G(U(q.a.gas_field[t.gas - SG_GAS_WM0]));
      return fld ? fmax(fld[(size_t)i * d.P + col], 0.0) : U(q.a.gas_mix_ratio[t.gas - SG_GAS_WM0]);
    }
    return t.gas == SG_GAS_ZERO ? 0.0 : x(3 + t.gas, i);
  };
  const auto absorb = [&](const SgTerm &t, int i) -> double {
    const double mmr = amount(t, i);
    if (GEN && t.fnc != SG_FNC_POWER_LAW)
      return k_scaled(t, spec, x(0, i), rec[(size_t)i * SG_NQ + SG_Q_P], x(6, i),
                      grec ? grec + (size_t)i * SG_NGQ : nullptr, mmr);
    return k_term(t, x(0, i), x(1, i), mmr);
  };
  const int nt = GEN ? U(spec->n_tmp) : 0;
  int t0 = minor0;
  for (int j = 0; j < n_gas; j++) {
    const int nk = U(B.minor_nk[j]);
    if (grey1 && nk == 1) {   // joins the grey extinction as it is (below)
      t0 += nk;
      continue;
    }
    // (the loops over a lane's layers run to KMAX without a branch, the missing layers
    // being identities, so that the scans of a term overlap)
    double num[KMAX], den[KMAX];
#pragma unroll
    for (int c = 0; c < KMAX; c++) { num[c] = 0.0; den[c] = 0.0; }
    double sflux = 0.0;
    for (int qt = 0; qt < nk; qt++) {
      const SgTerm t = U_term(spec->minor[t0 + qt]);
      double kk[KMAX];
      if (GEN && t.fnc == SG_FNC_LOOKUP) {
        // (unrolled, so that the layers' table entries are read together: one at a
        // time, each layer waited for its record and then for its entries, and the
        // kernel took 220 us of a 1024 x 70 infra-red segment with look-up tables)
        const double *kl = G(U(spec->klut)) + (size_t)t.lut * U(spec->n_pre) * nt;
        int o0[KMAX], o1[KMAX];
#pragma unroll
        for (int c = 0; c < KMAX; c++) lut_at(grec[(size_t)layer(c) * SG_NGQ + SG_G_IDX], nt, o0[c], o1[c]);
#pragma unroll
        for (int c = 0; c < KMAX; c++) {
          const double v = lut_k(kl, o0[c], o1[c], grec + (size_t)layer(c) * SG_NGQ, amount(t, layer(c)));
          kk[c] = has(c) ? v : 0.0;
        }
      } else {
        if (GEN)
          for (int c = 0; c < K; c++) buf[c * kWave + lane] = absorb(t, layer(c));
#pragma unroll
        for (int c = 0; c < KMAX; c++) {
          const double v = GEN ? (c < K ? buf[c * kWave + lane] : 0.0) : absorb(t, layer(c));
          kk[c] = has(c) ? v : 0.0;
        }
      }
      if (SOLAR) {
        // direct-beam transmission: f = w prod exp(-k m sec0) down to the bottom
        // of each layer; den accumulates f (summed over terms, fg)
        double fdt = t.w, f[KMAX], t02 = 1.0, p31 = 1.0;
#pragma unroll
        for (int c = 0; c < KMAX; c++) {
          {
            const double e = exp(-kk[c] * x(2, layer(c)) * sec0);
            double p = product_scan<kRowLanes, 1>(has(c) ? e : 1.0, s);
            const double tot = dpp_or0<kBcast + 15>(p);
            if (c % 4 == 1 || c % 4 == 3) p = p * t02;
            if (c % 4 >= 2) p = p * p31;
            if (c % 4 == 1) p31 = dpp_or0<kBcast + 15>(p);
            t02 = tot;
            f[c] = fdt * p;
            if (c % 4 == 3 || c == KMAX - 1) fdt = dpp_or0<kBcast + 15>(f[c]);
          }
        }
        const double fs = fdt;   // the transmission to the surface
#pragma unroll
        for (int c = 0; c < KMAX; c++) {
          {
            num[c] = num[c] + kk[c] * fs;
            den[c] = den[c] + f[c];
          }
        }
        sflux = sflux + fs;
      } else {
        // downward differential flux at the top of each layer
        double tr[KMAX], su[KMAX], fd[KMAX], F = -b_top, above = F;
        Affine t02{1.0, 0.0}, p31{1.0, 0.0};
#pragma unroll
        for (int c = 0; c < KMAX; c++) {
          {
            const double tau = kk[c] * x(2, layer(c));
            tr[c] = exp(-kDiffMinor * tau);
            su[c] = (1.0 - tr[c] + sqe) * db[c] / (kDiffMinor * tau + sqe);
            if (!has(c)) { tr[c] = 1.0; su[c] = 0.0; }
            Affine m{tr[c], -su[c]};
            affine_fold<kShr + 1>(m);
            affine_fold<kShr + 2>(m);
            affine_fold<kShr + 4>(m);
            affine_fold<kShr + 8>(m);
            const Affine tot = affine_bcast<kBcast + 15>(m);
            if (c % 4 == 1 || c % 4 == 3) m = after(m, t02);
            if (c % 4 >= 2) m = after(m, p31);
            if (c % 4 == 1) p31 = affine_bcast<kBcast + 15>(m);
            t02 = tot;
            const double below = m.A * F + m.C;
            fd[c] = dpp_or0<kShr + 1>(below);
            if (first) fd[c] = above;
            above = dpp_or0<kBcast + 15>(below);
            if (c % 4 == 3) F = above;
          }
        }
        // the upward flux at the surface, and at the bottom of each layer
        double Us = (bg - b_bot) + alb * above, under = Us;
        Affine t31{1.0, 0.0}, p32{1.0, 0.0};
#pragma unroll
        for (int c = KMAX - 1; c >= 0; c--) {
          {
            if (c % 4 == 3 || c == KMAX - 1) { t31 = Affine{1.0, 0.0}; p32 = t31; }
            Affine m{tr[c], su[c]};
            affine_fold<kShl + 1>(m);
            affine_fold<kShl + 2>(m);
            affine_fold<kShl + 4>(m);
            affine_fold<kShl + 8>(m);
            const Affine tot = affine_bcast<kBcast + 0>(m);
            if (c % 4 == 2 || c % 4 == 0) m = after(m, t31);
            if (c % 4 <= 1) m = after(m, p32);
            if (c % 4 == 2) p32 = affine_bcast<kBcast + 0>(m);
            t31 = tot;
            const double up = m.A * Us + m.C;   // at the top of the layer
            double u = dpp_or0<kShl + 1>(up);
            if (last) u = under;
            under = dpp_or0<kBcast + 0>(up);
            if (c % 4 == 0) Us = under;
            const double a = t.w * fabs(fd[c]), bb = t.w * fabs(u);
            num[c] = num[c] + (kk[c] * a + kk[c] * bb);
            den[c] = den[c] + (a + bb);
          }
        }
      }
    }
    // where no flux is left to weight with, the smallest k of the gas's terms
    bool none = SOLAR && !(sflux > 0.0);
    if (!SOLAR) {
#pragma unroll
      for (int c = 0; c < KMAX; c++)
        if (c < K) none = none || (has(c) && !(den[c] > 0.0));
    }
    if (__any(none))
      for (int c = 0; c < K; c++) {
        double kmin = DBL_MAX;
        for (int qt = 0; qt < nk; qt++) kmin = fmin(kmin, absorb(U_term(spec->minor[t0 + qt]), layer(c)));
        buf[c * kWave + lane] = kmin;
      }
    // this gas's equivalent extinction and (solar) direct-beam adjustment. fgp:
    // the summed transmission one layer up (1 above the first layer)
    double carry = 1.0;
#pragma unroll
    for (int c = 0; c < KMAX; c++) {
      if (c < K) {
        const double wt = SOLAR ? sflux : den[c];
        const double kq = wt > 0.0 ? num[c] / wt : buf[c * kWave + lane];
        if (SOLAR) {
          double fgp = dpp_or0<kShr + 1>(den[c]);
          if (first) fgp = carry;
          carry = dpp_or0<kBcast + 15>(den[c]);
          if (has(c) && fgp > 0.0) adj[c] = adj[c] * den[c] / fgp;
        }
        keq[c] = keq[c] + kq;
      }
    }
    t0 += nk;
  }

  // the band's records
  const size_t base = ((size_t)col * NB + b) * L;
  double *bandrec = G(U(q.bandrec)), *cldopt = G(U(q.cldopt));
  const double *aerrec = G(U(q.aerrec));
  const double ray = (SOLAR && U(q.l_rayleigh)) ? U(B.rayleigh) : 0.0;
  const bool mcica = d.mcica, triple = d.triple, ir_lin = d.ir_lin, aer = d.n_aer > 0;
  // clear-air continuum absorption (grey_opt_prop.F90:801-835) of the general gas
  // optics, and minor gases with a single k-term under l_grey_single, whose
  // absorption joins the grey extinction as it is (solve_band_k_eqv_scl.F90:
  // 941-951)
  const int n_cont = GEN && !d.no_cont ? U(B.n_cont) : 0;
  double *bc = buf + lane, *bg1 = bc + KMAX * kWave;
  if (n_cont > 0 || grey1)
    for (int c = 0; c < K; c++) {
      const int i = layer(c);
      bc[c * kWave] = n_cont > 0 ? continuum_k(B, rec[(size_t)i * SG_NQ + SG_Q_P], x(6, i),
                                               grec[(size_t)i * SG_NGQ + SG_G_RHO], x(3 + SG_GAS_H2O, i))
                                 : 0.0;
      double kgrey = 0.0;
      if (grey1)
        for (int j = 0, t1 = minor0; j < n_gas; t1 += U(B.minor_nk[j]), j++)
          if (U(B.minor_nk[j]) == 1) kgrey = kgrey + absorb(U_term(spec->minor[t1]), i);
      bg1[c * kWave] = kgrey;
    }
#pragma unroll
  for (int c = 0; c < KMAX; c++) {
    if (c < K && has(c) && live) {
      const int i = c * kRowLanes + s;
      // clear-air grey extinction: modal aerosols' absorption, continua, Rayleigh
      // scattering and the aerosols' (the sums over the modes are formed by the
      // pack kernel, aer_sums), then the equivalent extinction
      double kaer = 0.0, ksc = ray;
      if (aer) {
        const double *ar = aerrec + (base + i) * 4;
        ksc = ar[0];
        kaer = ar[3];
      }
      const double kcont = n_cont > 0 ? bc[c * kWave] : 0.0, kgrey = grey1 ? bg1[c * kWave] : 0.0;
      double4 br;
      br.x = ((kaer + kcont) + ksc) + keq[c] + kgrey;
      if (SOLAR) {
        // direct-beam adjustment with the exponential of the equivalent optical
        // depth (solve_band_k_eqv_scl.F90:848-891)
        const double temp_max = 36.043653389117154;  // log(1/DBL_EPSILON)
        br.y = adj[c] * exp(fmin(keq[c] * x(2, i) * sec0, temp_max));
        br.z = 0.0;
        br.w = 0.0;
      } else {
        // Planck terms (diff_planck_source_mod.F90:100-134); diff_2 zero for a
        // linear source, whose sources (ir_source.F90:52-59) are the quadratic
        // ones without it
        const double b0 = planck_band(pb, x(7, i)), b1 = planck_band(pb, x(7, i + 1));
        const double bt = planck_band(pb, x(6, i));
        br.y = ir_lin ? 0.0 : 2.0 * (b1 + b0 - 2.0 * bt);
        br.z = b1 - b0;   // diff
        br.w = b1;        // planck at the bottom of the layer
      }
      *(double4 *)(bandrec + (base + i) * SG_NBQ) = br;
    }
  }
  if (first && live) {
    if (SOLAR) {
      bs[0] = colscal[SG_S_SOL] * U(B.solar_flux);
      bs[1] = 0.0;
    } else {
      bs[0] = b_top;
      // (a given surface emission was stored by the pack kernel)
      if (colscal[SG_S_LFG] == 0.0) bs[1] = bg;
    }
  }
  if (mcica) {
    if (live)
      for (int i = s; i < L; i += kRowLanes)
        if (x(8, i) > 0.0) band_cloud(d, spec, rec + (size_t)i * SG_NQ, cldopt, base + i, b);
  } else if (triple) {
    double *bk = bg1 + KMAX * kWave;
#pragma unroll
    for (int c = 0; c < KMAX; c++)
      if (c < K) bk[c * kWave] = keq[c];
    const int nct = min(G(U(q.krange))[0], L);
    for (int c = 0; c < K; c++) {
      if (!has(c) || !live) continue;
      const int i = c * kRowLanes + s;
      double kaer = 0.0, ksc = ray, pfa = 0.0, fwa = 0.0;
      if (aer) {
        const double *ar = aerrec + (base + i) * 4;
        ksc = ar[0]; pfa = ar[1]; fwa = ar[2]; kaer = ar[3];
      }
      const double kcont = n_cont > 0 ? bc[c * kWave] : 0.0, kgrey = grey1 ? bg1[c * kWave] : 0.0;
      band_regions(d, spec, rec + (size_t)i * SG_NQ, cldopt + (base + i) * 8, b, i + 1 >= nct && x(8, i) > 0.0,
                   kaer + kcont, ksc, pfa, fwa, bk[c * kWave], kgrey);
    }
  }
}

template <int KMAX, bool GEN, int W>
__global__ __launch_bounds__(kWave * kBandWaves, KMAX == 6 ? 2 : 1) void b_band_kernel(
    const BatchHdr *h, const ReqDesc *rq) {
  extern __shared__ double lds[];
  constexpr int lp = KMAX * kRowLanes + 1;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int nwv = blockDim.x / kWave * gridDim.y, wv0 = blockIdx.y * (blockDim.x / kWave) + wv;
  const int row = lane / kRowLanes, s = lane % kRowLanes;
  double *buf = lds + kBandQ * kRows * lp + wv * 3 * KMAX * kWave;
  const long long tot = h->tot[W];
  for (long long w = blockIdx.x; w < tot; w += gridDim.x) {
    const ReqDesc &q = rq[find_req(h, rq, W, w)];
    const CallDims d = U_struct(q.d);
    const int c0 = (int)(w - U(q.s[W])) * kRows, P = d.P, L = d.L;
    const double *colrec = G(U(q.colrec)), *tlev = G(U(q.tlev));
    for (int e = threadIdx.x; e < kRows * (L + 1); e += blockDim.x) {
      const int c = e / (L + 1), i = e - c * (L + 1), col = min(c0 + c, P - 1);
      double *o = lds + c * kBandQ * lp + i;
      o[7 * lp] = tlev[(size_t)col * (L + 1) + i];
      if (i < L) {
        const double *r = colrec + ((size_t)col * L + i) * SG_NQ;
        o[0] = r[SG_Q_LNP];
        o[lp] = r[SG_Q_LNT];
        o[2 * lp] = r[SG_Q_MASS];
        o[3 * lp] = r[SG_Q_MMR + SG_GAS_H2O];
        o[4 * lp] = r[SG_Q_MMR + SG_GAS_CO2];
        o[5 * lp] = r[SG_Q_MMR + SG_GAS_O3];
        o[6 * lp] = r[SG_Q_T];
        o[8 * lp] = d.triple ? r[SG_Q_WCLD] : r[SG_Q_FRAC1];
      }
    }
    __syncthreads();
    const BandSrc x{lds + row * kBandQ * lp, lp};
    for (int b = wv0; b < d.NB; b += nwv) {
      if (d.isolir == SOCGPU_SOURCE_SOLAR)
        band_rows<KMAX, GEN, true>(q, d, x, min(c0 + row, P - 1), c0 + row < P, b, s, lane, buf);
      else
        band_rows<KMAX, GEN, false>(q, d, x, min(c0 + row, P - 1), c0 + row < P, b, s, lane, buf);
    }
    __syncthreads();
  }
}
