// nlm_tab.hpp -- a propagation with a precomputed RK4 step propagator (see
// nlm_prop_tab.hip), shared by the step-table kernel and the heterogeneous batches.
#pragma once
#include "nlm_prop.hpp"

// The RK4 step of a one-mode, one-pump model applied to x.
template <class M>
__device__ __forceinline__ cplx rk4_step(const cplx* c, const cplx* cc, cplx x, cplx P0, cplx P1, cplx P2) {
  constexpr int NC = M::NC;
  cplx xs[1] = {x}, y[1], k1[1], k2[1], k3[1], k4[1], p0[1] = {P0}, p1[1] = {P1}, p2[1] = {P2};
  M::template f<0>(c, cc, xs, p0, k1);
  y[0] = x + 0.5 * k1[0];
  M::template f<1>(c + NC, cc, y, p1, k2);
  y[0] = x + 0.5 * k2[0];
  M::template f<2>(c + NC, cc, y, p1, k3);
  y[0] = x + k3[0];
  M::template f<3>(c + 2 * NC, cc, y, p2, k4);
  return x + (((k1[0] + 2.0 * k2[0]) + 2.0 * k3[0]) + k4[0]) * (1. / 6.);
}

// The RK4 step as a real 2 x 2 matrix on (Re x, Im x), times s: columns R(1) and R(i),
// row p = (Re R(1), Re R(i)), row q = (Im R(1), Im R(i)).
template <class M>
struct StepMatrix {
  static __device__ __forceinline__ void eval(const cplx* c, const cplx* cc, cplx P0, cplx P1, cplx P2, double s,
                                              cplx& p, cplx& q) {
    const cplx a = rk4_step<M>(c, cc, mk(1.0, 0.0), P0, P1, P2);
    const cplx b = rk4_step<M>(c, cc, mk(0.0, 1.0), P0, P1, P2);
    p = mk(s * a.re, s * b.re);
    q = mk(s * a.im, s * b.im);
  }
};

// Chi2PDC: k(x) = m conj(x) with m1, m2, m3 = c P at the three positions, so the RK4
// stages expand to x' = alpha x + beta conj(x),
//   alpha = 1 + (m2 conj(m1) + |m2|^2 + m3 conj(q)) / 6,
//   beta = (m1 + 2 m2 + 2 q + (1 + |m2|^2 / 2) m3) / 6,   q = m2 + |m2|^2 m1 / 4:
// ~45 FP64 operations instead of two RK4 steps' ~120.
template <>
struct StepMatrix<MChi2PDC> {
  static __device__ __forceinline__ void eval(const cplx* c, const cplx*, cplx P0, cplx P1, cplx P2, double s, cplx& p,
                                              cplx& q) {
    const cplx m1 = c[0] * P0, m2 = c[1] * P1, m3 = c[2] * P2;
    const double n = abs2(m2);
    const cplx r = m2 + (0.25 * n) * m1;
    const cplx u = m2 * conj(m1) + m3 * conj(r);
    const cplx be = (m1 + 2.0 * (m2 + r) + (1.0 + 0.5 * n) * m3) * (1. / 6.);
    const double ar = 1.0 + (u.re + n) * (1. / 6.), ai = u.im * (1. / 6.);
    p = mk(s * (ar + be.re), s * (be.im - ai));
    q = mk(s * (ai + be.im), s * (ar - be.re));
  }
};

template <int L>
__device__ __forceinline__ void load_prop_row(cplx (&al)[8], cplx (&be)[8], const cplx* __restrict__ row, int t) {
  constexpr int T = FftShape<L>::T;
#pragma unroll
  for (int m = 0; m < 8; m++) {
    al[m] = row[(size_t)(t + T * m) * 2];
    be[m] = row[(size_t)(t + T * m) * 2 + 1];
  }
}

// Where the step's rows live, per size and launch.  MANY: more fields than one wave
// per SIMD.
//  Up to N = 512 (one wave per field): the propagator rows are fetched after the
//    forward transform; at N = 512 the dispersion row is read from L1/L2 where it is
//    used (held across a step both spilled to AGPRs: 92 register moves per step, 3 %).
//  N = 1024, 2048 with few fields: one wave per SIMD with all its registers; N = 1024
//    fetches the propagator rows after the forward transform (7 %), N = 2048 before it.
//  N = 1024, 2048 with MANY fields, and N = 4096 (HOOK): the dispersion row and the
//    propagator rows are fetched before the last exchange of the transform that
//    precedes their use, so they are live for one stage only and the loop with its
//    twiddles fits 256 registers: two waves share a SIMD, one's LDS accesses under
//    the other's arithmetic.  Green's launches, ms: N = 1024, nZ = 200 2.35 -> 1.79;
//    N = 2048, nZ = 50 2.81 -> 1.87; N = 4096, nZ = 16 4.67 -> 3.59 (one field 0.161 ->
//    0.126).  With few fields it is slower at N = 1024 (one field 0.49 -> 0.53, 512
//    fields, whose waves then pair up on half of the SIMDs, 0.61 -> 0.82).
//  N = 8192 (1024 lanes, 128 registers): twiddles from the table, rows at use.
template <int L, bool MANY>
struct TabPolicy {
  static constexpr int LOG = FftShape<L>::LOG;
  static constexpr bool HOOK = LOG == 12 || (MANY && (LOG == 10 || LOG == 11));
  static constexpr bool LATE = LOG == 9 || LOG == 10;
  static constexpr bool DS_MEM = LOG == 9 || LOG > 12;
  using TW = typename std::conditional<HOOK, RegTwiddles<L>, typename PropTw<L>::type>::type;
  static constexpr bool TW_LDS = !HOOK && PropTw<L>::IN_LDS;
  static constexpr int TW_ELEMS = TW_LDS ? PropTw<L>::LDS_ELEMS : 1;
};

// One propagation of field `field` on the T lanes that hold it: the same contract as
// prop_field (Green's, batch and grid kinds, checkpoints) for a medium with one
// signal mode and a step propagator table kp.tab.
template <int L, bool MANY>
__device__ __forceinline__ void tab_field(const KParams& kp, int field, bool active, int t, cplx* buf,
                                          const cplx* twl) {
  using F = FftShape<L>;
  constexpr int N = F::N, T = F::T;
  using Policy = TabPolicy<L, MANY>;
  constexpr bool HOOK = Policy::HOOK, LATE = Policy::LATE, DS_MEM = Policy::DS_MEM;
  typename Policy::TW tw;
  init_twiddles<L>(tw, kp.tw, twl, t);
  cplx ds[HOOK || !DS_MEM ? 8 : 1];
  if constexpr (!HOOK && !DS_MEM) load_pump<L>(ds, kp.dstep, t);

  cplx a[1][8];
  load_inputs<L, 1>(a, kp, field, t, active);
  prologue<L, 1>(a, kp, buf, t, tw, field, active);
  cplx al[8], be[8];
  if (kp.nZ > 1) {
    fft_field1<L, true, kWaveFft<L>>(a[0], buf, t, tw);  // unscaled: the table holds the 1/N
    if (kp.kind == KIND_GRID) store_scaled<L>(grid_row(kp, kp.gridT, field, 1, 0, 0, N), a[0], t, active);
    if (kp.ckpt) store_scaled<L>(kp.ckpt + (size_t)field * kp.nSeg * N, a[0], t, active);
    load_prop_row<L>(al, be, kp.tab + (size_t)N * 2, t);
  }

  const int t0 = t;
#ifdef NLM_TAB_SMALL
  // two steps per iteration let the scheduler overlap one step's last exchange
  // and stores with the next step's first loads (N = 512: 1.88 against 1.97 ms per
  // launch, same box; four steps 2.01 ms; from N = 1024 no change)
#pragma unroll 2
#endif
  for (int i = 1; i < kp.nZ; i++) {
    // HOOK: LDS and memory offsets formed inside the step, not held across it
    const int t = HOOK ? opaque_lane(t0) : t0;
    // --- RK4 nonlinear step as its R-linear propagator (a real 2 x 2 matrix)
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const cplx x = a[0][m];
      a[0][m] = mk(al[m].re * x.re + al[m].im * x.im, be[m].re * x.re + be[m].im * x.im);
    }
    if (!HOOK && !LATE && i + 1 < kp.nZ) load_prop_row<L>(al, be, kp.tab + (size_t)(i + 1) * N * 2, t);

    // --- dispersion step (src/_NonlinearMedium.hpp:212-215)
    if constexpr (HOOK)
      fft_field1<L, false, kWaveFft<L>>(a[0], buf, t, tw,
                                        [&]() __attribute__((always_inline)) { load_pump<L>(ds, kp.dstep, t); });
    else
      fft_field1<L, false, kWaveFft<L>>(a[0], buf, t, tw);
#pragma unroll
    for (int m = 0; m < 8; m++) a[0][m] = a[0][m] * (HOOK || !DS_MEM ? ds[HOOK || !DS_MEM ? m : 0] : kp.dstep[t + T * m]);
    if (!HOOK && LATE && i + 1 < kp.nZ) load_prop_row<L>(al, be, kp.tab + (size_t)(i + 1) * N * 2, t);
    if (i < kp.nZ - 1) {
      if (kp.kind == KIND_GRID) store_row<L>(grid_row(kp, kp.gridF, field, 1, 0, i, N), a[0], t, active);
      if constexpr (HOOK)
        fft_field1<L, true, kWaveFft<L>>(a[0], buf, t, tw, [&]() __attribute__((always_inline)) {
          load_prop_row<L>(al, be, kp.tab + (size_t)(i + 1) * N * 2, t);
        });
      else
        fft_field1<L, true, kWaveFft<L>>(a[0], buf, t, tw);
      if (kp.kind == KIND_GRID) store_scaled<L>(grid_row(kp, kp.gridT, field, 1, 0, i, N), a[0], t, active);
      if (kp.ckpt && i % kp.ckptEvery == 0)
        store_scaled<L>(kp.ckpt + ((size_t)field * kp.nSeg + i / kp.ckptEvery) * N, a[0], t, active);
    }
  }
  epilogue<L, 1>(a, kp, buf, t, tw, field, active);
}
