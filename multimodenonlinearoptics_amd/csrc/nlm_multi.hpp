// nlm_multi.hpp -- the persistent queue kernel of heterogeneous batches
// (nlm_multi.hip), instantiated per model in nlm_multi_inst.hip.
#pragma once
#include <type_traits>

#include "nlm_modes.hpp"
#include "nlm_tab.hpp"

struct MultiInst {
  const cplx* dstep;
  const cplx* halfIn;
  const cplx* halfOut;
  const cplx* coef;
  const cplx* cconst;
  const cplx* in;
  cplx* out;
  const cplx* env;     // generated linear pump: envelope, D_p, beam-profile factors, dzp
  const double* Dp;
  const double* strength;
  double dzp;
  const cplx* pump0;   // otherwise the medium's device pump grids, or the staged rows
  const cplx* pump1;
  cplx* tab;           // staged step table of a one-mode medium [nZ][N][2]
  const cplx* raman;   // Chi3GNLSE
  const cplx* filt;
  int nZ, inTime, inCols, nOut;
  int inPos[4], outPos[4];
};

// How a class's kernel runs one instance per workgroup.
enum {
  MULTI_FIELD = NLM_MULTI_FIELD,    // all modes in the same lanes, pump rows from a grid
  MULTI_INLINE = NLM_MULTI_INLINE,  // the same, the pump rows generated in the kernel
  MULTI_MODES = NLM_MULTI_MODES,    // one lane group per mode (nlm_modes.hpp), pump rows from a grid
  MULTI_TAB = NLM_MULTI_TABLE,      // one mode with a step table
};

template <class M, int L, int FORM>
struct MultiLaunch {
  using P = modes::Pow2<L, M::NS, true>;
  static constexpr int T = FftShape<L>::T;
  static constexpr int THREADS = FORM == MULTI_MODES ? P::THREADS : T;
  static constexpr int WAVES = FORM == MULTI_MODES ? (P::LEAN ? 4 : 2) : FORM == MULTI_TAB && L == 12 ? 2 : 0;
  static constexpr int LDS = FORM == MULTI_MODES ? (int)(P::LDS_BYTES / sizeof(cplx)) : FftShape<L>::lds_elems;
  static constexpr bool TW_LDS = FORM == MULTI_TAB ? TabPolicy<L, false>::TW_LDS
                                                   : FORM != MULTI_MODES && !std::is_same<M, MChi3GNLSE>::value;
  static constexpr int TW = TW_LDS ? PropTw<L>::LDS_ELEMS : 1;
};

// Workgroups take instances from the class's queue (one atomic counter) until it is
// empty.
template <class M, int L, int FORM>
__global__ void __launch_bounds__((MultiLaunch<M, L, FORM>::THREADS), (MultiLaunch<M, L, FORM>::WAVES))
    k_prop_multi(const MultiInst* __restrict__ inst, const int* __restrict__ order, int n, int* counter,
                 const cplx* tw) {
  using ML = MultiLaunch<M, L, FORM>;
  __shared__ cplx lds[ML::LDS];
  __shared__ cplx twl[ML::TW];
  __shared__ int item;
  const int t = threadIdx.x;
  if constexpr (ML::TW_LDS) fill_twiddle_lds<L>(twl, tw);
  for (;;) {
    __syncthreads();  // the previous instance's readers of `item` are done
    if (t == 0) item = atomicAdd(counter, 1);
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(item);
    if (w >= n) break;  // uniform: every workgroup leaves once the queue is empty
    const MultiInst& I = inst[order[w]];
    KParams kp{};
    kp.nZ = I.nZ;
    kp.kind = KIND_BATCH;
    kp.nFields = 1;
    kp.inTime = I.inTime;
    kp.outTime = I.inTime;
    kp.inCols = I.inCols;
    kp.nOut = I.nOut;
    for (int q = 0; q < 4; q++) {
      kp.inPos[q] = I.inPos[q];
      kp.outPos[q] = I.outPos[q];
    }
    kp.in = I.in;
    kp.out = I.out;
    kp.tw = tw;
    kp.dstep = I.dstep;
    kp.halfIn = I.halfIn;
    kp.halfOut = I.halfOut;
    kp.coef = I.coef;
    kp.cconst = I.cconst;
    kp.env = I.env;
    kp.Dp = I.Dp;
    kp.strength = I.strength;
    kp.dzp = I.dzp;
    kp.pump0 = I.pump0;
    kp.pump1 = I.pump1;
    kp.raman = I.raman;
    kp.filt = I.filt;
    kp.tab = I.tab;
    if constexpr (FORM == MULTI_MODES) {
      modes::Pow2<L, M::NS, true> f;
      int slot, g;
      cplx* fieldBuf = modes::place(f, lds, tw, &slot, &g);
      modes::modes_field<M>(kp, f, fieldBuf, 0, g, slot == 0);
    } else if constexpr (FORM == MULTI_TAB) {
      tab_field<L, false>(kp, 0, true, t, lds, twl);
    } else if constexpr (std::is_same<M, MChi3GNLSE>::value) {
      gnlse_field<L>(kp, 0, true, t, lds);
    } else {
      prop_field<M, L, FORM == MULTI_INLINE>(kp, 0, true, t, lds, twl);
    }
  }
}

typedef void (*multi_fn)(const MultiInst*, const int*, int, int*, const cplx*, int grid, hipStream_t);

template <class M, int L, int FORM>
void launch_multi(const MultiInst* inst, const int* order, int n, int* counter, const cplx* tw, int grid,
                  hipStream_t s) {
  hipLaunchKernelGGL((k_prop_multi<M, L, FORM>), dim3(grid), dim3(MultiLaunch<M, L, FORM>::THREADS), 0, s, inst,
                     order, n, counter, tw);
}

// Per-model launchers (nlm_multi_inst.hip), log2 N = 5..12; nullptr where the model
// has no kernel of that form.
multi_fn nlm_pick_multi_0(int L, int form), nlm_pick_multi_1(int L, int form), nlm_pick_multi_2(int L, int form),
    nlm_pick_multi_4(int L, int form), nlm_pick_multi_5(int L, int form), nlm_pick_multi_6(int L, int form),
    nlm_pick_multi_7(int L, int form), nlm_pick_multi_8(int L, int form), nlm_pick_multi_9(int L, int form),
    nlm_pick_multi_10(int L, int form), nlm_pick_multi_11(int L, int form), nlm_pick_multi_12(int L, int form),
    nlm_pick_multi_14(int L, int form);

// Staging (nlm_multi_stage.hip): before a class's propagations, one launch forms, in
// chunks of MULTI_CHUNK steps (chunks[2b] = instance, chunks[2b+1] = first step),
// either the step tables of a one-mode class (from generated pump rows, or from the
// media's pump grids) or the pump rows of a multi-mode class with a generated pump.
constexpr int MULTI_CHUNK = 16;
enum { STAGE_NONE = 0, STAGE_TAB = 1, STAGE_TAB_GRID = 2, STAGE_ROWS = 3 };
void nlm_multi_stage(int kind, int model, int L, const MultiInst* inst, const int* chunks, int n, const cplx* tw,
                     hipStream_t s);
