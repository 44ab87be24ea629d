// nlm_multi_stage.hip -- pump rows and step tables of a heterogeneous batch, formed
// before its propagations (see nlm_multi.hpp).
//
// A propagation advances one step after another, but its pump rows, and for a one-mode
// medium the step's propagator made of them, depend on nothing but the step number:
// all steps of all instances are formed at once, chip wide, and the serial chains
// are left with the signal's own two transforms per step.  One lane group per chunk of
// MULTI_CHUNK steps; the pump phase exp(i r dzp D_p) is exact at the chunk's first row
// and advanced by products over the 2 MULTI_CHUNK rows after it.
// What bounds it: the FP64 work of two transforms and, for a table, two RK4 steps per
// point, and the write of 32 bytes per point and step.
#include "nlm_multi.hpp"

namespace {

template <int L, bool TAB, class M>
__global__ void __launch_bounds__((Launch<L>::THREADS), 2)
    k_multi_stage(const MultiInst* __restrict__ inst, const int* __restrict__ chunks, int n,
                  const cplx* __restrict__ twt) {
  using F = FftShape<L>;
  constexpr int N = F::N, T = F::T, FPB = Launch<L>::FPB;
  __shared__ cplx lds[FPB * F::lds_elems];
  // beside the rows held per lane the twiddles of the larger transforms spilled: all
  // but the first stage's come from LDS there
  constexpr bool COMPACT = L >= 9;
  __shared__ cplx twl[COMPACT ? StageTwiddles<L>::ELEMS : 1];
  const int lf = threadIdx.x / T, t0 = threadIdx.x % T;
  const int ch = blockIdx.x * FPB + lf;
  if (ch >= n) return;  // only where chunks share a wave, which then has no barriers
  cplx* buf = lds + lf * F::lds_elems;
  const MultiInst& I = inst[chunks[2 * ch]];
  const int i0 = chunks[2 * ch + 1];
  const int i1 = i0 + MULTI_CHUNK < I.nZ ? i0 + MULTI_CHUNK : I.nZ;
  cplx* rows = const_cast<cplx*>(I.pump0);
  typename std::conditional<COMPACT, StageTwiddles<L>, RegTwiddles<L>>::type tw;
  if constexpr (COMPACT) {
    tw.init(twl, twt, t0);
    __syncthreads();
  } else {
    init_twiddles<L>(tw, twt, nullptr, t0);
  }
  // p0: row r0 = 2 i0 - 2 (the envelope itself for r0 = 0); cur: the spectrum of row
  // `at`, max(r0, 1) to begin with
  const int r0 = 2 * i0 - 2;
  cplx cur[8], e1[8], p0[8];
#pragma unroll
  for (int m = 0; m < 8; m++) {
    cur[m] = I.env[t0 + T * m];
    p0[m] = cur[m] * (I.strength ? I.strength[0] : 1.0);
  }
  fft_field1<L, false, kWaveFft<L>>(cur, buf, t0, tw);
#pragma unroll
  for (int m = 0; m < 8; m++) {
    const double d = I.Dp[t0 + T * m];
    double sn, cs;
    sincos_reduced((double)(r0 > 0 ? r0 : 1) * I.dzp * d, &sn, &cs);
    cur[m] = cur[m] * mk(cs, sn);
    sincos_reduced(I.dzp * d, &sn, &cs);
    e1[m] = mk(cs, sn);
  }
  int at = r0 > 0 ? r0 : 1;  // the row whose spectrum cur is
  const auto row = [&](int r, cplx (&out)[8]) __attribute__((always_inline)) {
    const int t = opaque_lane(t0);
    if constexpr (COMPACT) tw.t = t;
    if (r > at) {
#pragma unroll
      for (int m = 0; m < 8; m++) cur[m] = cur[m] * e1[m];
      at = r;
    }
#pragma unroll
    for (int m = 0; m < 8; m++) out[m] = cur[m];
    fft_field1<L, true, kWaveFft<L>>(out, buf, t, tw);
    const double sc = (I.strength ? I.strength[r] : 1.0) * (1.0 / N);
#pragma unroll
    for (int m = 0; m < 8; m++) out[m] = out[m] * sc;
  };
  if (r0 > 0) row(r0, p0);
  if (!TAB && i0 == 1) store_row<L>(rows, p0, t0, true);
  for (int i = i0; i < i1; i++) {
    cplx p1[8], p2[8];
    row(2 * i - 1, p1);
    row(2 * i, p2);
    const int t = opaque_lane(t0);
    if constexpr (TAB) {
      cplx c[3 * M::NC];
      const uniform_cplx* cq = to_uniform(I.coef + (size_t)i * 3 * M::NC);
#pragma unroll
      for (int k = 0; k < 3 * M::NC; k++) c[k] = mk(cq[k].re, cq[k].im);
      constexpr double s = 1.0 / N;
      cplx* dst = I.tab + (size_t)i * N * 2;
#pragma unroll
      for (int m = 0; m < 8; m++) {
        cplx p, q;
        StepMatrix<M>::eval(c, nullptr, p0[m], p1[m], p2[m], s, p, q);
        dst[(size_t)(t + T * m) * 2] = p;
        dst[(size_t)(t + T * m) * 2 + 1] = q;
        p0[m] = p2[m];
      }
    } else {
      store_row<L>(rows + (size_t)(2 * i - 1) * N, p1, t, true);
      store_row<L>(rows + (size_t)(2 * i) * N, p2, t, true);
    }
  }
}

// Step tables from the media's pump grids: one workgroup per chunk.
template <class M>
__global__ void __launch_bounds__(256)
    k_multi_grid_tab(const MultiInst* __restrict__ inst, const int* __restrict__ chunks, int N) {
  const MultiInst& I = inst[chunks[2 * blockIdx.x]];
  const int i0 = chunks[2 * blockIdx.x + 1];
  const int i1 = i0 + MULTI_CHUNK < I.nZ ? i0 + MULTI_CHUNK : I.nZ;
  const double s = 1.0 / N;
  for (int i = i0; i < i1; i++) {
    const cplx* c = I.coef + (size_t)i * 3 * M::NC;
    for (int k = threadIdx.x; k < N; k += blockDim.x) {
      const cplx P0 = I.pump0[(size_t)(2 * i - 2) * N + k], P1 = I.pump0[(size_t)(2 * i - 1) * N + k],
                 P2 = I.pump0[(size_t)(2 * i) * N + k];
      cplx p, q;
      StepMatrix<M>::eval(c, I.cconst, P0, P1, P2, s, p, q);
      I.tab[((size_t)i * N + k) * 2] = p;
      I.tab[((size_t)i * N + k) * 2 + 1] = q;
    }
  }
}

template <int L>
void launch(int kind, const MultiInst* inst, const int* chunks, int n, const cplx* tw, hipStream_t s) {
  const dim3 grid((n + Launch<L>::FPB - 1) / Launch<L>::FPB), block(Launch<L>::THREADS);
  if (kind == STAGE_TAB)
    hipLaunchKernelGGL((k_multi_stage<L, true, MChi2PDC>), grid, block, 0, s, inst, chunks, n, tw);
  else
    hipLaunchKernelGGL((k_multi_stage<L, false, MChi2PDC>), grid, block, 0, s, inst, chunks, n, tw);
}

}  // namespace

void nlm_multi_stage(int kind, int model, int L, const MultiInst* inst, const int* chunks, int n, const cplx* tw,
                     hipStream_t s) {
  if (n <= 0 || kind == STAGE_NONE) return;
  if (kind == STAGE_TAB_GRID) {
    if (model == NLM_CHI3)
      hipLaunchKernelGGL(k_multi_grid_tab<MChi3>, dim3(n), dim3(256), 0, s, inst, chunks, 1 << L);
    else
      hipLaunchKernelGGL(k_multi_grid_tab<MChi2PDC>, dim3(n), dim3(256), 0, s, inst, chunks, 1 << L);
    return;
  }
  switch (L) {
    case 5: launch<5>(kind, inst, chunks, n, tw, s); break;
    case 6: launch<6>(kind, inst, chunks, n, tw, s); break;
    case 7: launch<7>(kind, inst, chunks, n, tw, s); break;
    case 8: launch<8>(kind, inst, chunks, n, tw, s); break;
    case 9: launch<9>(kind, inst, chunks, n, tw, s); break;
    case 10: launch<10>(kind, inst, chunks, n, tw, s); break;
    case 11: launch<11>(kind, inst, chunks, n, tw, s); break;
    case 12: launch<12>(kind, inst, chunks, n, tw, s); break;
  }
}
