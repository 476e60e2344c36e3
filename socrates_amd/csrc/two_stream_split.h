// The kernel-level two-stream solve on prescribed optical properties: included
// by socgpu.hip after solve_rows.h, whose slab composition it uses.
#pragma once

// Arrays [term][layer][profile] (optical properties, outputs [term][level]
// [profile]) and [layer][profile] / [profile] for the rest.
struct TwoStreamArgs {
  int P, L, G, isolir, l_scale_solar, l_quad;
  const double *tau, *omega, *asym, *sec0, *finc_down, *finc_dir, *alb_diff, *alb_dir;
  const double *dpl, *dpl2, *dsurf, *adjust;
  double *fdir, *fup, *fdown;
  long long first;   // the launch's first solve
};

// One lane per (term, profile), profile fastest, so every per-layer read and
// per-level write is coalesced; the layers of COLS such solves are split over
// GROUPS groups of a block's lanes (a wave each, or half of one), at most KMAX
// consecutive ones each, whose state stays in registers (128 a lane, which four waves
// per SIMD allow: the solar builds of 9 layers spill 16 to 48 of them, 68 to 84 B a
// lane, those of 12 80 to 110, up to 228 B, the infra-red ones of 12 40 to 48, up to
// 84 B). Each group composes its layers into one slab; the slabs pass through LDS,
// every group eliminates down those above its own to find the state at its top, and
// after the local elimination the affine maps of the groups below pass the upward
// flux back the same way. What bounds it: its loads, which each layer waits for
// (4096 x 90 x 16 solar solves: 97 us of kernel for 0.30 GB, VALU busy in 61 % of the
// cycles with 3.9 waves per SIMD). With the whole column in one lane the elimination
// state went through lane-private memory (64 B a layer beside the 48 B the solve has
// to move) and a small call was one chain of all its layers.
// (two_coeff, ir_source.F90:93-120, solar_source.F90:104-162, the surface source
// of column_solver.F90:160-185, solver_homogen_direct.F90:93-127.)
template <bool MIXED, bool SOLAR, int KMAX, int COLS, int GROUPS>
__global__ __launch_bounds__(GROUPS *COLS, 4) void two_stream_kernel(TwoStreamArgs a) {
#pragma clang fp contract(on)
  constexpr int kQ = 6;
  __shared__ double sh[GROUPS][kQ][COLS];
  const int lane = threadIdx.x % COLS;
  const int wv = COLS == kWave ? __builtin_amdgcn_readfirstlane(threadIdx.x / COLS) : threadIdx.x / COLS;
  const int P = a.P, L = a.L;
  const long long n = (long long)P * a.G, idx = a.first + (long long)blockIdx.x * COLS + lane;
  const bool act = idx < n;
  // lanes past the last solve repeat it and store nothing
  const long long id = act ? idx : n - 1;
  const int g = (int)(id / P), l = (int)(id - (long long)g * P);
  const int K = (L + GROUPS - 1) / GROUPS, i0 = wv * K, nk = max(0, min(K, L - i0));
  const int n_wave = (L + K - 1) / K;   // waves with layers
  const double sec0 = SOLAR ? a.sec0[l] : 1.0;
  const size_t t0 = (size_t)g * L * P + l, o0 = (size_t)g * (L + 1) * P + l;
  const double finc_down = a.finc_down[l], finc_dir = SOLAR ? a.finc_dir[l] : 0.0;

  double w0[KMAX], w1[KMAX], w2[KMAX], w3[KMAX], wf[SOLAR ? KMAX : 1];
  Slab S{1.0, 0.0, 0.0, 0.0, 0.0};
  double f = 1.0;   // the direct beam relative to the wave's top
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < nk) {
      const size_t kk = t0 + (size_t)(i0 + k) * P, kl = (size_t)(i0 + k) * P + l;
      const double tau = a.tau[kk], om = a.omega[kk], asym = a.asym[kk];
      Coef o;
      if (MIXED) {
        CoefF c;
        two_coeff_f32(SOLAR, (float)tau, (float)om, (float)fmax(1.0 - om, 32.0 * kEps), (float)asym, (float)sec0, c);
        coef_from_f32(c, o);
      } else {
        two_coeff(SOLAR, tau, om, asym, sec0, o);
      }
      double su, sd;
      if (SOLAR) {
        wf[k] = f;
        su = o.s1 * f;
        if (a.l_scale_solar) {
          const double fnew = f * o.T0 * a.adjust[kl];
          sd = (o.s2 - o.T0) * f + fnew;
          f = fnew;
        } else {
          sd = o.s2 * f;
          f = f * o.T0;
        }
      } else if (a.l_quad) {
        su = o.s1 * a.dpl[kl] + o.s2 * a.dpl2[kl];
        sd = -o.s1 * a.dpl[kl] + o.s2 * a.dpl2[kl];
      } else {
        su = o.s1 * a.dpl[kl];
        sd = -su;
      }
      w0[k] = o.T;
      w1[k] = o.R;
      w2[k] = su;
      w3[k] = sd;
      const Slab B{o.T, o.R, o.R, su, sd};
      if (GROUPS > 1) S = k == 0 ? B : slab_add(S, B);
    }
  }
  sh[wv][0][lane] = S.T;
  sh[wv][1][lane] = S.Rt;
  sh[wv][2][lane] = S.Rb;
  sh[wv][3][lane] = S.Su;
  sh[wv][4][lane] = S.Sd;
  if (SOLAR) sh[wv][5][lane] = f;
  __syncthreads();
  // down the slabs above
  double rho = 0.0, dn = finc_down, F = finc_dir;
  for (int u = 0; u < wv && u < n_wave; u++) {
    Slab B{sh[u][0][lane], sh[u][1][lane], sh[u][2][lane], sh[u][3][lane], sh[u][4][lane]};
    if (SOLAR) { B.Su = B.Su * F; B.Sd = B.Sd * F; }
    double rb, sd;
    slab_below(rho, dn, B, rb, sd);
    rho = rb;
    dn = sd;
    if (SOLAR) F = F * sh[u][5][lane];
  }
  __syncthreads();
  double A = 1.0, C = 0.0;   // fu(top of the wave) = A fu(bottom) + C
#pragma unroll
  for (int k = 0; k < KMAX; k++) {
    if (k < nk) {
      const double T = w0[k], R = w1[k];
      double su = w2[k], sd = w3[k];
      if (SOLAR) {
        su = su * F;
        sd = sd * F;
        if (act && a.fdir) a.fdir[o0 + (size_t)(i0 + k) * P] = wf[k] * F;
      }
      w2[k] = rho;
      w3[k] = dn;
      row_elim(T, R, su, sd, rho, dn, w0[k], w1[k]);
      C = C + A * w1[k];
      A = A * w0[k];
    }
  }
  const bool bottom = wv == n_wave - 1;
  sh[wv][0][lane] = A;
  sh[wv][1][lane] = C;
  if (bottom) {
    const double ad = a.alb_diff[l], fd = F * f;
    const double sg = SOLAR ? (a.alb_dir[l] - ad) * fd : (1.0 - ad) * a.dsurf[l];
    const double fu = (ad * dn + sg) / (1.0 - ad * rho);
    sh[wv][2][lane] = fu;
    if (act) {
      a.fup[o0 + (size_t)L * P] = fu;
      a.fdown[o0 + (size_t)L * P] = rho * fu + dn;
      if (SOLAR && a.fdir) a.fdir[o0 + (size_t)L * P] = fd;
    }
  }
  __syncthreads();
  // up from the surface through the waves below
  double fu = sh[n_wave - 1][2][lane];
  for (int u = n_wave - 1; u > wv; u--) fu = sh[u][0][lane] * fu + sh[u][1][lane];
#pragma unroll
  for (int k = KMAX - 1; k >= 0; k--) {
    if (k < nk) {
      fu = w0[k] * fu + w1[k];
      if (act) {
        a.fup[o0 + (size_t)(i0 + k) * P] = fu;
        a.fdown[o0 + (size_t)(i0 + k) * P] = w2[k] * fu + w3[k];
      }
    }
  }
}

// A launch's work-items, up to 16 per solve, have to be fewer than 2^32, and the entry
// point takes up to 2^31 solves: 2^27 of them (2^31 work-items) a launch.
constexpr long long kTsPerLaunch = 1LL << 27;

// Columns per block: 64, a wave per group of layers; 32, two groups per wave, where
// that still gives every CU (256) at most one block, so that twice as many of them
// work. FP64, a call in us with 64 and with 32 columns: solar 2997 solves of 137
// layers 55 and 51, 8000 of 90 48 and 44, but 12288 of 60 43 and 45, where some CUs
// have two blocks; infra-red 2997 of 137 50 and 44 (mixed 47 and 42); 65536 of 90
// solar 119 and 121.
constexpr long long kTsFew = 256 * 32;

template <bool MIXED, bool SOLAR, int KMAX, int COLS, int GROUPS = 16>
static void two_stream_run(TwoStreamArgs a, hipStream_t s) {
  const long long n = (long long)a.P * a.G;
  for (a.first = 0; a.first < n; a.first += kTsPerLaunch) {
    const int blocks = (int)((std::min(n - a.first, kTsPerLaunch) + COLS - 1) / COLS);
    two_stream_kernel<MIXED, SOLAR, KMAX, COLS, GROUPS><<<blocks, GROUPS * COLS, 0, s>>>(a);
  }
}
template <bool MIXED, bool SOLAR, int COLS>
static void two_stream_cols(const TwoStreamArgs &a, hipStream_t s) {
  if (a.L <= 48) two_stream_run<MIXED, SOLAR, 3, COLS>(a, s);
  else if (a.L <= 96) two_stream_run<MIXED, SOLAR, 6, COLS>(a, s);
  else if (a.L <= 144) two_stream_run<MIXED, SOLAR, 9, COLS>(a, s);
  else two_stream_run<MIXED, SOLAR, 12, COLS>(a, s);
}

// Few layers: one lane per solve up to 3, 4 groups up to 12, since 16 groups would be
// idle for the most part. FP64, a call in us with 16 groups and so: solar 65536 x 16
// solves of 2 layers 186 and 51, of 5 264 and 109, of 10 379 and 174; infra-red 113,
// 146, 222 and 48, 80, 132; 4096 x 16 solar solves of 12 layers 48 and 39.
template <bool MIXED, bool SOLAR>
static void two_stream_launch(const TwoStreamArgs &a, hipStream_t s) {
  if (a.L <= 3) two_stream_run<MIXED, SOLAR, 3, kWave, 1>(a, s);
  else if (a.L <= 12) two_stream_run<MIXED, SOLAR, 3, kWave, 4>(a, s);
  else if ((long long)a.P * a.G <= kTsFew) two_stream_cols<MIXED, SOLAR, 32>(a, s);
  else two_stream_cols<MIXED, SOLAR, kWave>(a, s);
}
