// nlm_modes.hpp -- the split step with one group of lanes per signal mode.
//
// A propagation of a medium with NS >= 2 signal modes runs on NS groups of lanes,
// group g holding mode g in the stride layout of its transform F (the power-of-two
// transform of nlm_fft.hpp through Pow2 below, or the mixed-radix one of
// nlm_mix.hpp), so the modes' transforms run side by side on different waves
// instead of one after another in the same ones.  For the RK4 step, which couples
// the modes at every time point, the groups exchange their points through LDS and
// each group evaluates the step for a share of the points.
//
// What bounds it: a wave's FP64 instructions (4 cycles each), its 16-byte LDS accesses
// (~30 cycles each for one wave per SIMD) and the barriers add up, since every wave of
// a workgroup is in the same phase.  Against all modes in the same lanes (k_prop,
// still used where the groups exceed 1024 lanes or their buffers the LDS) this halves
// a wave's work and its registers, so that two to four waves share a SIMD instead of
// one, and it removes the spills of k_prop at N = 4096 and of the four-mode media.
// Measured, kernel ms of 59 steps, k_prop -> this, for 1 / 100 / 2048 rows:
//   Chi2SHG N = 256     0.267 -> 0.155   0.272 -> 0.159   0.364 -> 0.343
//   Chi2SHG N = 1024    0.382 -> 0.283   0.396 -> 0.292   1.95 -> 1.62
//   Chi2SHG N = 2048    0.464 -> 0.435   0.482 -> 0.455   4.15 -> 4.01
//   Chi2SHG N = 4096    1.28 -> 0.87     1.33 -> 0.92     (512 rows) 2.86 -> 2.05
//   Chi2PDCII N = 256   0.299 -> 0.176   0.302 -> 0.182   0.388 -> 0.372
//   Chi2PDCII N = 4096  2.06 -> 0.93     2.52 -> 0.98     (512 rows) 5.94 -> 2.18
//   Chi2DSFG N = 512    0.571 -> 0.197   0.585 -> 0.206   1.82 -> 1.04
//   Chi2SFGII N = 512   1.70 -> 0.22     1.76 -> 0.23     7.97 -> 1.57
#pragma once
#include "nlm_prop.hpp"

namespace modes {

__device__ __forceinline__ void sync_if(bool wave) {
  if (wave) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  else lds_barrier();
}

template <class F>
__device__ __forceinline__ void put_row(const F& f, cplx* __restrict__ dst, const cplx (&v)[F::R], bool act) {
  if (act)
#pragma unroll
    for (int k = 0; k < F::R; k++) dst[f.at(k)] = v[k];
}
template <class F>
__device__ __forceinline__ void put_scaled(const F& f, cplx* __restrict__ dst, const cplx (&v)[F::R], bool act) {
  const double s = f.invN();
  if (act)
#pragma unroll
    for (int k = 0; k < F::R; k++) dst[f.at(k)] = v[k] * s;
}
template <class F>
__device__ __forceinline__ void get_row(const F& f, cplx (&v)[F::R], const cplx* __restrict__ src) {
#pragma unroll
  for (int k = 0; k < F::R; k++) v[k] = src[f.on ? f.at(k) : 0];
}
template <class F>
__device__ __forceinline__ void mul_row(const F& f, cplx (&v)[F::R], const cplx* __restrict__ tab) {
#pragma unroll
  for (int k = 0; k < F::R; k++) v[k] = v[k] * tab[f.on ? f.at(k) : 0];
}
template <class F>
__device__ __forceinline__ void scale_row(const F& f, cplx (&v)[F::R]) {
#pragma unroll
  for (int k = 0; k < F::R; k++) v[k] = v[k] * f.invN();
}

template <int NS>
__device__ __forceinline__ int of_mode(const int (&a)[4], int g) {
  int r = a[0];
#pragma unroll
  for (int q = 1; q < NS; q++) r = g == q ? a[q] : r;
  return r;
}

// Input of mode g and the half dispersion step in (src/_NonlinearMedium.hpp:164-198,
// src/_NonlinearMedium.cpp:329-340); leaves the spectrum.
template <int NS, class F>
__device__ __forceinline__ void enter(const KParams& kp, F& f, int field, int g, bool act, cplx (&v)[F::R]) {
  const int N = f.n();
#pragma unroll
  for (int k = 0; k < F::R; k++) v[k] = mk(0.0, 0.0);
  if (act) {
    if (kp.kind == KIND_GREENS) {
      const int i = field >> 1, w = field & 1, src = i / N, pos = i - src * N;
      const cplx val = w ? mk(0.0, 1.0) : mk(1.0, 0.0);
      if (kp.inputs[src] == g)
#pragma unroll
        for (int k = 0; k < F::R; k++)
          if (f.at(k) == pos) v[k] = val;
    } else {
      const int ch = of_mode<NS>(kp.inPos, g);
      if (ch >= 0) {
        const cplx* row = kp.in + (size_t)field * kp.inCols + (size_t)ch * N;
#pragma unroll
        for (int k = 0; k < F::R; k++) v[k] = row[f.at(k)];
      }
    }
  }
  if (kp.inTime) f.template run<false>(v);
  mul_row(f, v, kp.halfIn + (size_t)g * N);
  if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridF, field, NS, g, 0, N), v, act);
}

// Half step out and outputs (src/_NonlinearMedium.hpp:235-238, src/_NonlinearMedium.cpp:333-345, 428-431).
template <int NS, class F>
__device__ __forceinline__ void leave(const KParams& kp, F& f, int field, int g, bool act, cplx (&v)[F::R]) {
  const int N = f.n(), last = kp.nZ - 1;
  mul_row(f, v, kp.halfOut + (size_t)g * N);
  if (kp.kind == KIND_GRID) {
    put_row(f, grid_row(kp, kp.gridF, field, NS, g, last, N), v, act);
    f.template run<true>(v);
    put_scaled(f, grid_row(kp, kp.gridT, field, NS, g, last, N), v, act);
  } else {
    if (kp.outTime) {
      f.template run<true>(v);
      scale_row(f, v);
    }
    const int op = of_mode<NS>(kp.outPos, g);
    if (op >= 0) put_row(f, kp.out + (size_t)field * kp.nOut * N + (size_t)op * N, v, act);
  }
}

// The RK4 step (DiffEq and update, src/_NonlinearMedium.hpp:207-210) of one time point.
template <class M>
__device__ __forceinline__ void rk4_point(const cplx* c, const cplx* cc, cplx (&x)[M::NS],
                                          const cplx (&P0)[M::NP > 0 ? M::NP : 1],
                                          const cplx (&P1)[M::NP > 0 ? M::NP : 1],
                                          const cplx (&P2)[M::NP > 0 ? M::NP : 1]) {
  constexpr int NS = M::NS, NC = M::NC;
  cplx y[NS], k1[NS], k2[NS], k3[NS], k4[NS];
  M::template f<0>(c, cc, x, P0, k1);
#pragma unroll
  for (int q = 0; q < NS; q++) y[q] = x[q] + 0.5 * k1[q];
  M::template f<1>(c + NC, cc, y, P1, k2);
#pragma unroll
  for (int q = 0; q < NS; q++) y[q] = x[q] + 0.5 * k2[q];
  M::template f<2>(c + NC, cc, y, P1, k3);
#pragma unroll
  for (int q = 0; q < NS; q++) y[q] = x[q] + k3[q];
  M::template f<3>(c + 2 * NC, cc, y, P2, k4);
#pragma unroll
  for (int q = 0; q < NS; q++) x[q] = x[q] + (((k1[q] + 2.0 * k2[q]) + 2.0 * k3[q]) + k4[q]) * (1. / 6.);
}

// One mode (group g) of a propagation of a pointwise model with NS >= 2 modes.
template <class M, class F>
__device__ __forceinline__ void modes_field(const KParams& kp, F& f, cplx* fieldBuf, int field, int g, bool act) {
  constexpr int NS = M::NS, NP = M::NP, NC = M::NC, NPP = NP > 0 ? NP : 1;
  constexpr int KS = (F::R + NS - 1) / NS;  // points of this group's share: k = kk NS + g
  const int N = f.n();
  cplx v[F::R];
  enter<NS>(kp, f, field, g, act, v);
  if (kp.nZ > 1) {
    f.template run<true>(v);
    scale_row(f, v);
    if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridT, field, NS, g, 0, N), v, act);
  }
  // the share's pump rows 2i-2 (pp), 2i-1 (pi), 2i (pc) of step i
  cplx pp[NPP][KS], pi[NPP][KS], pc[NPP][KS];
  const cplx* pumps[2] = {kp.pump0, kp.pump1};
  auto pump = [&](cplx (&dst)[KS], const cplx* row) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      const int k = kk * NS + g;
      dst[kk] = row[f.on && k < F::R ? f.at(k) : 0];
    }
  };
#pragma unroll
  for (int r = 0; r < NP; r++) {
    pump(pp[r], pumps[r]);
    if (kp.nZ > 1) {
      pump(pi[r], pumps[r] + N);
      pump(pc[r], pumps[r] + (size_t)2 * N);
    }
  }
  constexpr int NCC = M::NCC > 0 ? M::NCC : 1;
  cplx cc[NCC];
  {
    const uniform_cplx* ccq = to_uniform(kp.cconst);
#pragma unroll
    for (int k = 0; k < M::NCC; k++) cc[k] = mk(ccq[k].re, ccq[k].im);
  }
  for (int i = 1; i < kp.nZ; i++) {
    cplx c[3 * NC];
    {
      const uniform_cplx* cq = to_uniform(kp.coef + (size_t)i * 3 * NC);
#pragma unroll
      for (int k = 0; k < 3 * NC; k++) c[k] = mk(cq[k].re, cq[k].im);
    }
    // --- RK4 step: every group offers its mode's points, takes all modes of its
    // share, and returns them
    f.sync();  // the transform's readers of this group's buffer are done
    if (f.on)
#pragma unroll
      for (int k = 0; k < F::R; k++) f.buf[f.at(k)] = v[k];
    f.syncAll();
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
      const int k = kk * NS + g;
      if (f.on && k < F::R) {
        const int at = f.at(k);
        cplx x[NS], P0[NPP], P1[NPP], P2[NPP];
#pragma unroll
        for (int r = 0; r < NPP; r++) {
          P0[r] = NP ? pp[r][kk] : mk(0, 0);
          P1[r] = NP ? pi[r][kk] : mk(0, 0);
          P2[r] = NP ? pc[r][kk] : mk(0, 0);
        }
#pragma unroll
        for (int q = 0; q < NS; q++) x[q] = fieldBuf[q * f.bufElems() + at];
        rk4_point<M>(c, cc, x, P0, P1, P2);
#pragma unroll
        for (int q = 0; q < NS; q++) fieldBuf[q * f.bufElems() + at] = x[q];
      }
    }
    f.syncAll();
    if (f.on)
#pragma unroll
      for (int k = 0; k < F::R; k++) v[k] = f.buf[f.at(k)];
    // --- dispersion step (src/_NonlinearMedium.hpp:212-215)
    f.template run<false>(v);
    mul_row(f, v, kp.dstep + (size_t)g * N);
    if (i < kp.nZ - 1) {
      if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridF, field, NS, g, i, N), v, act);
      f.template run<true>(v, [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < NP; r++) {
#pragma unroll
          for (int kk = 0; kk < KS; kk++) pp[r][kk] = pc[r][kk];
          pump(pi[r], pumps[r] + (size_t)(2 * i + 1) * N);
          pump(pc[r], pumps[r] + (size_t)(2 * i + 2) * N);
        }
      });
      scale_row(f, v);
      if (kp.kind == KIND_GRID) put_row(f, grid_row(kp, kp.gridT, field, NS, g, i, N), v, act);
    }
  }
  leave<NS>(kp, f, field, g, act, v);
}

// The power-of-two transform of one group: T = N/8 lanes, eight points each.  ONE: a
// workgroup holds one field however few its lanes.
template <int L, int NS, bool ONE = false>
struct Pow2 {
  using S = FftShape<L>;
  static constexpr int R = 8, T = S::T;
  static constexpr int ALL = NS * T;                         // lanes per field
  static constexpr int FPB = ONE || ALL >= 64 ? 1 : 64 / ALL;  // fields per workgroup
  static constexpr int THREADS = ONE && ALL < 64 ? ALL : (FPB * ALL + 63) / 64 * 64;
  static constexpr int SLOTS = (THREADS + ALL - 1) / ALL;    // the spare lanes have buffers too
  static constexpr bool WAVE = T <= 64 && 64 % T == 0;       // a group lies in one wave
  static constexpr bool WAVE_ALL = THREADS <= 64;
  // Beyond 512 lanes a wave has 128 registers: all but the first stage's twiddles come
  // from LDS, and the padding is one slot per 32 elements so that both fit.
  static constexpr bool LEAN = THREADS > 512;
  static constexpr int CODE = LEAN && S::PAD != 5 ? L + 32 : L;
  using SC = FftShape<CODE>;
  static constexpr int BUF = SC::lds_elems;
  static constexpr int TABLE = LEAN ? StageTwiddles<CODE>::ELEMS : 0;
  static constexpr size_t LDS_BYTES = ((size_t)SLOTS * NS * BUF + TABLE) * sizeof(cplx);
  static constexpr bool OK = THREADS <= 1024 && LDS_BYTES <= 160 * 1024;
  using TW = typename std::conditional<LEAN, StageTwiddles<CODE>, RegTwiddles<CODE>>::type;

  cplx* buf;
  int j;
  static constexpr bool on = true;
  TW tw;
  static __device__ __forceinline__ constexpr int n() { return S::N; }
  static __device__ __forceinline__ constexpr double invN() { return 1.0 / S::N; }
  static __device__ __forceinline__ constexpr int bufElems() { return BUF; }
  __device__ __forceinline__ int at(int k) const { return j + T * k; }
  __device__ __forceinline__ void sync() const { exchange_sync<WAVE>(); }
  __device__ __forceinline__ void syncAll() const { exchange_sync<WAVE_ALL>(); }
  template <bool INV, class Fetch>
  __device__ __forceinline__ void run(cplx (&v)[8], const Fetch& fetch) {
    j = opaque_lane(j);
    if constexpr (LEAN) tw.t = j;
    fft_field1<CODE, INV, WAVE>(v, buf, j, tw, fetch);
  }
  template <bool INV>
  __device__ __forceinline__ void run(cplx (&v)[8]) {
    run<INV>(v, NoFetch());
  }
};

// Field slot, group and lane of this thread, the twiddles and the LDS buffers of F
// (lds: SLOTS * NS * BUF elements, then the twiddles of LEAN); returns the field's buffers.
template <int L, int NS, bool ONE>
__device__ __forceinline__ cplx* place(Pow2<L, NS, ONE>& f, cplx* lds, const cplx* tw, int* slot, int* g) {
  using F = Pow2<L, NS, ONE>;
  int s = threadIdx.x / F::ALL;
  const int r = threadIdx.x - s * F::ALL;
  int gg = r / F::T;
  f.j = r - gg * F::T;
  if constexpr (F::T >= 64) gg = __builtin_amdgcn_readfirstlane(gg);
  *slot = s;
  *g = gg;
  cplx* fieldBuf = lds + (size_t)s * NS * F::BUF;
  f.buf = fieldBuf + gg * F::BUF;
  if constexpr (F::LEAN) {
    f.tw.init(lds + (size_t)F::SLOTS * NS * F::BUF, tw, f.j);
    __syncthreads();
  } else {
    fft_load_twiddles<F::CODE>(f.tw.w, tw, f.j);
  }
  return fieldBuf;
}

// Waves per SIMD asked of the compiler (registers per lane): four (128) where the
// lanes have no more, and for media without a pump up to N = 512, which need only ~150
// and fill the chip better so (Chi2SHG N = 512, 2048 rows, 59 steps: 0.67 against
// 0.77 ms; few rows 2 % slower); otherwise two (256): with 128, Chi2SHG N = 1024 is 15 %
// slower and the pumped media, which hold pump rows, spill.
template <class M, int L>
struct ModesWaves {
  static constexpr int N = Pow2<L, M::NS>::LEAN || (M::NP == 0 && L <= 9) ? 4 : 2;
};

template <class M, int L>
__global__ void __launch_bounds__((Pow2<L, M::NS>::THREADS), (ModesWaves<M, L>::N)) k_prop_modes(KParams kp) {
  using F = Pow2<L, M::NS>;
  __shared__ cplx lds[F::LDS_BYTES / sizeof(cplx)];
  F f;
  int slot, g;
  cplx* fieldBuf = place(f, lds, kp.tw, &slot, &g);
  const int field = blockIdx.x * F::FPB + slot;
  modes_field<M>(kp, f, fieldBuf, field, g, slot < F::FPB && field < kp.nFields);
}

template <class M, int L>
void launch_prop_modes(const KParams& kp, int, hipStream_t s) {
  using F = Pow2<L, M::NS>;
  hipLaunchKernelGGL((k_prop_modes<M, L>), dim3((kp.nFields + F::FPB - 1) / F::FPB), dim3(F::THREADS), 0, s, kp);
}

}  // namespace modes
