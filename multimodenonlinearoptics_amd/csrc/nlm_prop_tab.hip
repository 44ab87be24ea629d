// nlm_prop_tab.hip -- split step with a precomputed RK4 step propagator for the
// single-signal-mode undepleted media (Chi3, Chi2PDC).
//
// With the pump grid fixed, the DiffEq of these media is R-linear in the
// signal: Chi2PDC (solvers/Chi2PDC.cpp:27-47) has k = (c P) conj(x), Chi3
// (solvers/Chi3.cpp:57-69) has k = i nl (2|P|^2 x + P^2 conj(x)).  Every RK4
// stage (src/_NonlinearMedium.hpp:207-210) is then R-linear too, and one
// whole RK4 step at time sample k of step i is
//     x -> alpha[i][k] x + beta[i][k] conj(x),
// with alpha = (R(1) - i R(i)) / 2 and beta = (R(1) + i R(i)) / 2 for R the
// RK4 step applied to the inputs 1 and i; as a real 2 x 2 matrix acting on
// (Re x, Im x) its columns are R(1) and R(i).  k_step_table evaluates R with the
// model's own DiffEq functor once per (step, sample) for all fields and stores
// the matrix; the propagation kernel then spends 4 FP64 operations per point on
// the nonlinear step instead of four DiffEq evaluations, for every one of the 2N
// Green's impulses or batch rows.  The propagator also absorbs the inverse
// transform's 1/N (an exact power of two), so the field between steps is kept
// unscaled.
#include "nlm_quad.hpp"

// tab[(i*N + k)*2 + {0,1}] = {(Re R(1), Re R(i)), (Im R(1), Im R(i))} * scale for
// steps i = 1..nZ-1: Re x' = p.re Re x + p.im Im x, Im x' = q.re Re x + q.im Im x.
template <class M>
__global__ void k_step_table(const cplx* __restrict__ coef, const cplx* __restrict__ cconst,
                             const cplx* __restrict__ pump, int N, int nZ, double scale, cplx* __restrict__ tab) {
  static_assert(M::NS == 1 && M::NP == 1, "single signal mode, single pump");
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(nZ - 1) * N;
  if (idx >= total) return;
  const int i = 1 + (int)(idx / N), k = (int)(idx % N);
  const cplx* c = coef + (size_t)i * 3 * M::NC;
  const cplx P0 = pump[(size_t)(2 * i - 2) * N + k];
  const cplx P1 = pump[(size_t)(2 * i - 1) * N + k];
  const cplx P2 = pump[(size_t)(2 * i) * N + k];
  const cplx r1 = rk4_step<M>(c, cconst, mk(1.0, 0.0), P0, P1, P2);
  const cplx ri = rk4_step<M>(c, cconst, mk(0.0, 1.0), P0, P1, P2);
  tab[((size_t)i * N + k) * 2] = mk(scale * r1.re, scale * ri.re);
  tab[((size_t)i * N + k) * 2 + 1] = mk(scale * r1.im, scale * ri.im);
}

// WAVES: waves per SIMD asked of the compiler (0: none asked).
template <int L, bool MANY, int WAVES>
__global__ void __launch_bounds__((Launch<L>::THREADS), (WAVES)) k_prop_tab(KParams kp) {
  using F = FftShape<L>;
  constexpr int T = F::T, FPB = Launch<L>::FPB;
  __shared__ cplx lds[FPB * F::lds_elems];
  __shared__ cplx twl[TabPolicy<L, MANY>::TW_ELEMS];
  if constexpr (TabPolicy<L, MANY>::TW_LDS) fill_twiddle_lds<L>(twl, kp.tw);
  const int lf = threadIdx.x / T, t = threadIdx.x % T;
  const int field = blockIdx.x * FPB + lf;
  tab_field<L, MANY>(kp, field, field < kp.nFields, t, lds + lf * F::lds_elems, twl);
}

template <int L, bool MANY, int WAVES>
static void launch_tab(const KParams& kp, int grid, hipStream_t s) {
  hipLaunchKernelGGL((k_prop_tab<L, MANY, WAVES>), dim3(grid), dim3(Launch<L>::THREADS), 0, s, kp);
}

// The form of a launch (TabPolicy): the two-waves form where it exists and the
// launch's waves exceed one per SIMD.  Asking for one wave per SIMD where a launch of
// few fields leaves the chip idle changes nothing (199 steps of 1, 8, 64, 200 fields, ms:
// N = 1024 0.479 / 0.484 / 0.487 / 0.499 with it, 0.479 / 0.484 / 0.487 / 0.498 without;
// N = 2048 0.718 / 0.735 / 0.729 / 0.737 and 0.718 / 0.731 / 0.729 / 0.737).
template <int L>
static void launch_prop_tab(const KParams& kp, int grid, hipStream_t s) {
  if constexpr (TabPolicy<L, false>::HOOK) {
    launch_tab<L, false, 2>(kp, grid, s);
  } else if constexpr (TabPolicy<L, true>::HOOK) {
    if ((long)grid * (Launch<L>::THREADS / 64) > 4 * device_cus()) launch_tab<L, true, 2>(kp, grid, s);
    else launch_tab<L, false, 0>(kp, grid, s);
  } else {
    launch_tab<L, false, 0>(kp, grid, s);
  }
}

// This file is compiled once per schedule variant NLM_TAB_VARIANT (see FftShape);
// variants other than 0 exist for nFreqs 512..8192, where the autotuner chooses.
#ifndef NLM_TAB_VARIANT
#define NLM_TAB_VARIANT 0
#endif
#define NLM_CAT2(a, b) a##b
#define NLM_CAT(a, b) NLM_CAT2(a, b)

#ifdef NLM_TAB_SMALL
// The single-wave sizes (nFreqs 8..512, schedule 0) are compiled in a translation
// unit of their own, with LLVM's memory-clause machine scheduler: at one wave per
// SIMD nothing hides the row loads and LDS exchanges, and its order was 4 % faster
// at N = 512 (1.95 against 2.03 ms per Green's launch, same box), while from
// N = 1024 (two or more waves per SIMD) it was 1-5 % slower.
prop_fn nlm_pick_prop_tab_small(int L) {
  switch (L) {
    case 3: return &launch_prop_tab<3>;
    case 4: return &launch_prop_tab<4>;
    case 5: return &launch_prop_tab<5>;
    case 6: return &launch_prop_tab<6>;
    case 7: return &launch_prop_tab<7>;
    case 8: return &launch_prop_tab<8>;
    case 9: return &launch_prop_tab<9>;
  }
  return nullptr;
}

// Four points per lane, nFreqs 8..256.
prop_fn nlm_pick_prop_quad(int L) {
  switch (L) {
    case 3: return &quad::launch<3>;
    case 4: return &quad::launch<4>;
    case 5: return &quad::launch<5>;
    case 6: return &quad::launch<6>;
    case 7: return &quad::launch<7>;
    case 8: return &quad::launch<8>;
  }
  return nullptr;
}
#else
prop_fn nlm_pick_prop_tab_small(int L);

prop_fn NLM_CAT(nlm_pick_prop_tab_var, NLM_TAB_VARIANT)(int L) {
  constexpr int V = NLM_TAB_VARIANT, C = 32 * V;
  // bit 1 (small radix last) only differs from the default when log2 N is not a multiple of 3
  if (V != 0 && (L < 9 || L > 13 || ((V & 2) && L % 3 == 0))) return nullptr;
  switch (L) {
#if NLM_TAB_VARIANT == 0
    case 3:
    case 4:
    case 5:
    case 6:
    case 7:
    case 8:
    case 9: return nlm_pick_prop_tab_small(L);
    case 12: return &launch_prop_tab<12>;
#elif (NLM_TAB_VARIANT & 2) == 0
    case 9: return &launch_prop_tab<9 + C>;
    case 12: return &launch_prop_tab<12 + C>;
#endif
    case 10: return &launch_prop_tab<10 + C>;
    case 11: return &launch_prop_tab<11 + C>;
    case 13: return &launch_prop_tab<13 + C>;
  }
  return nullptr;
}

#if NLM_TAB_VARIANT == 0
prop_fn nlm_pick_prop_tab_var1(int L);
prop_fn nlm_pick_prop_tab_var2(int L);
prop_fn nlm_pick_prop_tab_var3(int L);

prop_fn nlm_pick_prop_tab(int L) { return nlm_pick_prop_tab_var0(L); }

prop_fn nlm_pick_prop_tab_variant(int L, int variant) {
  switch (variant) {
    case 0: return nlm_pick_prop_tab_var0(L);
    case 1: return nlm_pick_prop_tab_var1(L);
    case 2: return nlm_pick_prop_tab_var2(L);
    case 3: return nlm_pick_prop_tab_var3(L);
  }
  return nullptr;
}

// Build the step propagator table of `model` (NLM_CHI3 or NLM_CHI2PDC) into tab
// ([nZ][N][2] complex; row 0 unused).  Returns false for other models.
bool nlm_launch_step_table(int model, const cplx* coef, const cplx* cconst, const cplx* pump, int N, int nZ,
                           cplx* tab, hipStream_t s) {
  const long total = (long)(nZ - 1) * N;
  if (total <= 0) return true;
  const dim3 grid((unsigned)((total + 255) / 256)), block(256);
  const double scale = 1.0 / N;
  if (model == NLM_CHI2PDC)
    hipLaunchKernelGGL(k_step_table<MChi2PDC>, grid, block, 0, s, coef, cconst, pump, N, nZ, scale, tab);
  else if (model == NLM_CHI3)
    hipLaunchKernelGGL(k_step_table<MChi3>, grid, block, 0, s, coef, cconst, pump, N, nZ, scale, tab);
  else
    return false;
  return true;
}
#endif  // NLM_TAB_VARIANT == 0
#endif  // NLM_TAB_SMALL
