// nlm_quad.hpp -- the step-table propagation with four points per lane, for launches that
// leave most of the chip idle.
//
// With few fields (one signal, a Green's function of a small grid) every wave has a SIMD to
// itself and a step takes as long as one wave's chain of instructions and LDS exchanges.
// Four points per lane instead of eight halve the arithmetic of that chain and use twice the
// waves; a transform of N = 2^L takes radix 4 stages and one of radix 2 if L is odd, at most
// one exchange more.  A field is at most one wave (N <= 256), so the exchanges are ordered
// within the wave; with barriers between several waves the form loses (one field, 199 steps: N = 512
// 415 -> 450 us, 1024 531 -> 594; Chi3 pump N = 512 2.25 -> 2.32 us per row).  Calls of 200 steps, us (eight points -> four): signal N = 32
// 256 -> 194, 64 275 -> 203, 256 370 -> 262; Green's N = 16 261 -> 151, 32 238 -> 193, 64 283 ->
// 226, 256 504 -> 470 (of which the rows fetched two steps ahead instead of one: 5 %, 20 % at 256).
#pragma once
#include "nlm_tab.hpp"

namespace quad {

template <int L>
struct Shape {
  static constexpr int N = 1 << L, T = N / 4, S = (L + 1) / 2;
  static constexpr int radix(int s) { return s == S - 1 && (L & 1) ? 2 : 4; }
  static constexpr int before(int s) { return 1 << (2 * s); }
  static constexpr int FPB = 64 / T;         // fields per workgroup of one wave
  static constexpr int ELEMS = N + N / 4;    // LDS of a field: one slot after every four
};
__device__ __forceinline__ int pad(int x) { return x + (x >> 2); }

template <int L>
struct Twiddles {
  cplx w[Shape<L>::S][4];
  __device__ __forceinline__ void init(const cplx* __restrict__ table, int t) {
#pragma unroll
    for (int s = 0; s < Shape<L>::S - 1; s++) {
      const int P = Shape<L>::before(s), M = Shape<L>::N / P / 4;
#pragma unroll
      for (int c = 1; c < 4; c++) w[s][c] = table[((t % M) * c * P) & (Shape<L>::N - 1)];
    }
  }
};

// Stages from s on; the twiddled radix-4 outputs of stage s - 1 are in buf.
template <int L, bool INV, int s>
__device__ __forceinline__ void stages(cplx (&v)[4], cplx* __restrict__ buf, int t, const Twiddles<L>& tw) {
  using F = Shape<L>;
  constexpr int R = F::radix(s), P = F::before(s), Mp = F::N / P, M = Mp / R, NB = 4 / R;
  exchange_sync<true>();
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const int beta = t + F::T * j, b = beta % M, g = beta / M;
#pragma unroll
    for (int a = 0; a < R; a++) v[j * R + a] = buf[pad(g * Mp + a * M + b)];
  }
#pragma unroll
  for (int j = 0; j < NB; j++) dft_small<R, INV>(v + j * R);
  if constexpr (s == F::S - 1) {
    if constexpr (NB == 2) {  // back to the stride layout
      const cplx x = v[1];
      v[1] = v[2];
      v[2] = x;
    }
  } else {
    exchange_sync<true>();
    const int b = t % M, g = t / M;
#pragma unroll
    for (int c = 0; c < 4; c++) buf[pad((g + P * c) * M + b)] = c == 0 ? v[0] : twmul<INV>(v[c], tw.w[s][c]);
    stages<L, INV, s + 1>(v, buf, t, tw);
  }
}

// Transform of a field in stride layout: lane t holds x[t + T m], m = 0..3.
template <int L, bool INV>
__device__ __forceinline__ void fft(cplx (&v)[4], cplx* __restrict__ buf, int t, const Twiddles<L>& tw) {
  dft_small<4, INV>(v);
  exchange_sync<true>();
#pragma unroll
  for (int c = 0; c < 4; c++) buf[pad(c * Shape<L>::T + t)] = c == 0 ? v[0] : twmul<INV>(v[c], tw.w[0][c]);
  stages<L, INV, 1>(v, buf, t, tw);
}

template <int L>
__device__ __forceinline__ void load(cplx (&v)[4], const cplx* __restrict__ row, int t) {
#pragma unroll
  for (int m = 0; m < 4; m++) v[m] = row[t + Shape<L>::T * m];
}
template <int L>
__device__ __forceinline__ void mul(cplx (&v)[4], const cplx* __restrict__ row, int t) {
#pragma unroll
  for (int m = 0; m < 4; m++) v[m] = v[m] * row[t + Shape<L>::T * m];
}
template <int L>
__device__ __forceinline__ void store(cplx* __restrict__ row, const cplx (&v)[4], int t, bool active, double s = 1.0) {
  if (active) {
#pragma unroll
    for (int m = 0; m < 4; m++) row[t + Shape<L>::T * m] = v[m] * s;
  }
}
template <int L>
__device__ __forceinline__ void load_step(cplx (&al)[4], cplx (&be)[4], const cplx* __restrict__ row, int t) {
#pragma unroll
  for (int m = 0; m < 4; m++) {
    al[m] = row[(t + Shape<L>::T * m) * 2];
    be[m] = row[(t + Shape<L>::T * m) * 2 + 1];
  }
}

// The propagation of tab_field: Green's, batch and grid kinds, checkpoints.
template <int L>
__global__ void __launch_bounds__(64) k_prop_quad(KParams kp) {
  using F = Shape<L>;
  constexpr int N = F::N, T = F::T;
  constexpr double inv = 1.0 / N;
  __shared__ cplx lds[F::FPB * F::ELEMS];
  const int lf = threadIdx.x / T, t = threadIdx.x % T, field = blockIdx.x * F::FPB + lf;
  const bool active = field < kp.nFields, grids = kp.kind == KIND_GRID;
  cplx* buf = lds + lf * F::ELEMS;
  Twiddles<L> tw;
  tw.init(kp.tw, t);
  cplx v[4], ds[4], al[4], be[4], al2[4], be2[4];
  load<L>(ds, kp.dstep, t);
#pragma unroll
  for (int m = 0; m < 4; m++) v[m] = mk(0.0, 0.0);
  if (active) {
    if (kp.kind == KIND_GREENS) {  // impulse e_i (even fields) or i e_i (odd) in the one mode
      const int pos = (field >> 1) % N;
#pragma unroll
      for (int m = 0; m < 4; m++)
        if (t + T * m == pos) v[m] = field & 1 ? mk(0.0, 1.0) : mk(1.0, 0.0);
    } else if (kp.inPos[0] >= 0) {
      load<L>(v, kp.in + (size_t)field * kp.inCols + (size_t)kp.inPos[0] * N, t);
    }
  }
  if (kp.inTime) fft<L, false>(v, buf, t, tw);
  mul<L>(v, kp.halfIn, t);
  if (grids) store<L>(grid_row(kp, kp.gridF, field, 1, 0, 0, N), v, t, active);
  if (kp.nZ > 1) {
    fft<L, true>(v, buf, t, tw);  // unscaled: the table holds the 1/N
    if (grids) store<L>(grid_row(kp, kp.gridT, field, 1, 0, 0, N), v, t, active, inv);
    if (kp.ckpt) store<L>(kp.ckpt + (size_t)field * kp.nSeg * N, v, t, active, inv);
    load_step<L>(al, be, kp.tab + (size_t)N * 2, t);
    if (kp.nZ > 2) load_step<L>(al2, be2, kp.tab + (size_t)N * 4, t);
  }
  // one step from the rows in (al, be), which are then fetched for step i + 2: a row comes from
  // HBM or the Infinity Cache and would take longer than the rest of a step
  const auto step = [&](int i, cplx (&al)[4], cplx (&be)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const cplx x = v[m];
      v[m] = mk(al[m].re * x.re + al[m].im * x.im, be[m].re * x.re + be[m].im * x.im);
    }
    if (i + 2 < kp.nZ) load_step<L>(al, be, kp.tab + (size_t)(i + 2) * N * 2, t);
    fft<L, false>(v, buf, t, tw);
#pragma unroll
    for (int m = 0; m < 4; m++) v[m] = v[m] * ds[m];
    if (i < kp.nZ - 1) {
      if (grids) store<L>(grid_row(kp, kp.gridF, field, 1, 0, i, N), v, t, active);
      fft<L, true>(v, buf, t, tw);
      if (grids) store<L>(grid_row(kp, kp.gridT, field, 1, 0, i, N), v, t, active, inv);
      if (kp.ckpt && i % kp.ckptEvery == 0)
        store<L>(kp.ckpt + ((size_t)field * kp.nSeg + i / kp.ckptEvery) * N, v, t, active, inv);
    }
  };
  for (int i = 1; i < kp.nZ; i += 2) {
    step(i, al, be);
    if (i + 1 < kp.nZ) step(i + 1, al2, be2);
  }
  mul<L>(v, kp.halfOut, t);
  if (grids) store<L>(grid_row(kp, kp.gridF, field, 1, 0, kp.nZ - 1, N), v, t, active);
  if (grids || kp.outTime) fft<L, true>(v, buf, t, tw);
  const double s = grids || kp.outTime ? inv : 1.0;
  if (grids) store<L>(grid_row(kp, kp.gridT, field, 1, 0, kp.nZ - 1, N), v, t, active, s);
  else if (kp.outPos[0] >= 0) store<L>(kp.out + (size_t)field * kp.nOut * N + (size_t)kp.outPos[0] * N, v, t, active, s);
}

// The nonlinear pump of Chi3 (solvers/Chi3.cpp:25-54), one field serial over its 2nZ-1 rows:
// always a single wave's chain.  Per row, us, eight points -> four: N = 64 1.59 -> 1.13, N = 256
// 2.08 -> 1.47.
template <int L>
__global__ void __launch_bounds__(Shape<L>::T)
    k_pump_chi3(const cplx* __restrict__ env, const double* __restrict__ Dp, double dzp,
                const cplx* __restrict__ dstepP, const cplx* __restrict__ relI, int nZP, cplx* __restrict__ pumpF,
                cplx* __restrict__ pumpT, const cplx* __restrict__ twt) {
  using F = Shape<L>;
  constexpr int N = F::N, T = F::T;
  constexpr double inv = 1.0 / N;
  __shared__ cplx buf[F::ELEMS];
  const int t = threadIdx.x;
  Twiddles<L> tw;
  tw.init(twt, t);
  cplx v[4], dsp[4];
  load<L>(v, env, t);
  load<L>(dsp, dstepP, t);
  const auto half = [&](double dz) __attribute__((always_inline)) {  // exp(i dz/2 D_p)
#pragma unroll
    for (int m = 0; m < 4; m++) {
      double s, c;
      sincos((0.5 * dz) * Dp[t + T * m], &s, &c);
      v[m] = v[m] * mk(c, s);
    }
  };
  cplx next = relI[0];
  for (int i = 0; i < nZP; i++) {
    if (i > 0) {
      const cplx r = next;
      next = relI[i];  // nZP entries; the last is not used
      self_phase<4>(v, r);
    }
    fft<L, false>(v, buf, t, tw);
    if (i == 0) {
      half(dzp);
    } else {
#pragma unroll
      for (int m = 0; m < 4; m++) v[m] = v[m] * dsp[m];
      if (i == nZP - 1) half(-dzp);
    }
    store<L>(pumpF + (size_t)i * N, v, t, true);
    fft<L, true>(v, buf, t, tw);
#pragma unroll
    for (int m = 0; m < 4; m++) v[m] = v[m] * inv;
    store<L>(pumpT + (size_t)i * N, v, t, true);
  }
}

template <int L>
void launch(const KParams& kp, int, hipStream_t s) {
  const int grid = (kp.nFields + Shape<L>::FPB - 1) / Shape<L>::FPB;
  hipLaunchKernelGGL(k_prop_quad<L>, dim3(grid), dim3(64), 0, s, kp);
}

}  // namespace quad
