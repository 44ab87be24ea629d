// nlm_mix_rows.hip -- standalone transforms and pump rows through the mixed-radix
// transform of nlm_mix.hpp: nlm_fft, the linear pump (src/_NonlinearMedium.cpp:225-250)
// and Chi3::runPumpSimulation (solvers/Chi3.cpp:25-54).
#include "nlm_mix.hpp"

template <int R>
__global__ void __launch_bounds__(MIX_MAX_THREADS) k_mix_fft(MixRows r, MixPlan p) {
  const cplx* tab = mix::load_table(p, mix_lds);
  const mix::Place a = mix::place(p);
  mix::Fft<R> f(p, mix_lds + p.N + (size_t)a.slot * p.bufElems, tab, a.j);
  const int row = blockIdx.x * p.FPB + a.slot;
  const bool act = f.on && row < r.count;
  cplx v[R];
  mix::get_row(f, v, r.in + (size_t)(act ? row : 0) * p.N);
  if (r.inverse) {
    f.template run<true>(v);
    mix::put_scaled(f, r.out + (size_t)row * p.N, v, act);
  } else {
    f.template run<false>(v);
    mix::put_row(f, r.out + (size_t)row * p.N, v, act);
  }
}

// Row i: freq = F0 exp(i (i dzp) D_p), time = IFFT(freq), row 0's time row the
// envelope itself; both times strength[i].
template <int R>
__global__ void __launch_bounds__(MIX_MAX_THREADS) k_mix_pump_linear(MixRows r, MixPlan p) {
  const cplx* tab = mix::load_table(p, mix_lds);
  const mix::Place a = mix::place(p);
  mix::Fft<R> f(p, mix_lds + p.N + (size_t)a.slot * p.bufElems, tab, a.j);
  const int row = blockIdx.x * p.FPB + a.slot;
  const bool act = f.on && row < r.nZP;
  const int i = act ? row : 0;
  const double zi = (double)i * r.dzp, s = r.strength ? r.strength[i] : 1.0;
  cplx v[R], t[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int at = f.on ? f.at(k) : 0;
    v[k] = r.F0[at];
    if (i > 0) {
      double sn, cs;
      sincos_reduced(zi * r.Dp[at], &sn, &cs);
      v[k] = v[k] * mk(cs, sn);
    }
    t[k] = v[k];
  }
  f.template run<true>(t);
#pragma unroll
  for (int k = 0; k < R; k++) {
    t[k] = i == 0 ? r.env[f.on ? f.at(k) : 0] : t[k] * p.invN;
    if (r.strength) {
      v[k] = v[k] * s;
      t[k] = t[k] * s;
    }
  }
  mix::put_row(f, r.pumpF + (size_t)i * p.N, v, act);
  mix::put_row(f, r.pumpT + (size_t)i * p.N, t, act);
}

// The nonlinear pump, serial over its 2nZ-1 rows in one workgroup.
template <int R>
__global__ void __launch_bounds__(MIX_MAX_THREADS) k_mix_pump_chi3(MixRows r, MixPlan p) {
  const cplx* tab = mix::load_table(p, mix_lds);
  const mix::Place a = mix::place(p);
  mix::Fft<R> f(p, mix_lds + p.N + (size_t)a.slot * p.bufElems, tab, a.j);
  const bool act = f.on && a.slot == 0;
  cplx v[R], dsp[R];
  mix::get_row(f, v, r.env);
  mix::get_row(f, dsp, r.dstepP);
  f.template run<false>(v);
#pragma unroll
  for (int k = 0; k < R; k++) {
    double s, c;
    sincos((0.5 * r.dzp) * r.Dp[f.on ? f.at(k) : 0], &s, &c);
    v[k] = v[k] * mk(c, s);
  }
  mix::put_row(f, r.pumpF, v, act);
  f.template run<true>(v);
  mix::scale_row(f, v);
  mix::put_row(f, r.pumpT, v, act);
  for (int i = 1; i < r.nZP; i++) {
    const cplx q = r.relI[i - 1];
    self_phase<R>(v, q);
    f.template run<false>(v);
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = v[k] * dsp[k];
    if (i == r.nZP - 1) {
#pragma unroll
      for (int k = 0; k < R; k++) {
        double s, c;
        sincos((-0.5 * r.dzp) * r.Dp[f.on ? f.at(k) : 0], &s, &c);
        v[k] = v[k] * mk(c, s);
      }
    }
    mix::put_row(f, r.pumpF + (size_t)i * p.N, v, act);
    f.template run<true>(v);
    mix::scale_row(f, v);
    mix::put_row(f, r.pumpT + (size_t)i * p.N, v, act);
  }
}

namespace {
template <int R>
void launch(int kind, const MixRows& r, const MixPlan& p, hipStream_t s) {
  const int items = kind == MIX_ROWS_FFT ? r.count : kind == MIX_ROWS_LINEAR ? r.nZP : 1;
  const dim3 grid((items + p.FPB - 1) / p.FPB), block(p.threads);
  if (kind == MIX_ROWS_FFT) hipLaunchKernelGGL((k_mix_fft<R>), grid, block, p.ldsBytes, s, r, p);
  else if (kind == MIX_ROWS_LINEAR) hipLaunchKernelGGL((k_mix_pump_linear<R>), grid, block, p.ldsBytes, s, r, p);
  else hipLaunchKernelGGL((k_mix_pump_chi3<R>), grid, block, p.ldsBytes, s, r, p);
}
}  // namespace

bool nlm_mix_rows(int kind, const MixRows& r, const MixPlan& p, hipStream_t s) {
  switch (p.R) {
    case 2: launch<2>(kind, r, p, s); return true;
    case 3: launch<3>(kind, r, p, s); return true;
    case 4: launch<4>(kind, r, p, s); return true;
    case 5: launch<5>(kind, r, p, s); return true;
    case 6: launch<6>(kind, r, p, s); return true;
    case 8: launch<8>(kind, r, p, s); return true;
    case 9: launch<9>(kind, r, p, s); return true;
    case 10: launch<10>(kind, r, p, s); return true;
  }
  return false;
}
