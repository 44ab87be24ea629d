// nlm_multi_inst.hip -- heterogeneous-batch kernels of one model for nFreqs
// 32..4096.  Compiled once per model with -DNLM_INST_MODEL=<id>.
#include "nlm_multi.hpp"

#ifndef NLM_INST_MODEL
#error "NLM_INST_MODEL must be defined"
#endif

#define NLM_CAT2(a, b) a##b
#define NLM_CAT(a, b) NLM_CAT2(a, b)

namespace {
using MM = typename ModelOf<NLM_INST_MODEL>::type;
constexpr bool GNLSE = NLM_INST_MODEL == NLM_CHI3GNLSE;
// the pump rows can be generated in the kernel for a single linear pump
// (_NonlinearMedium::runPumpSimulation); Chi3's pump is nonlinear (solvers/Chi3.cpp:25-54)
constexpr bool LINEAR = MM::NP == 1 && NLM_INST_MODEL != NLM_CHI3;
// media with a step table (R-linear, one mode): Chi3 and Chi2PDC
constexpr bool TABLE = MM::NS == 1 && MM::NP == 1;

template <int L, int FORM>
constexpr bool has() {
  if constexpr (FORM == MULTI_MODES) return MM::NS > 1 && modes::Pow2<L, MM::NS, true>::OK;
  else if constexpr (FORM == MULTI_TAB) return TABLE;
  else if constexpr (FORM == MULTI_INLINE) return LINEAR;
  // lanes shared by all modes: media without a generated pump where the mode groups
  // do not fit, and one-mode media whose table was not staged
  else return GNLSE || TABLE || (MM::NS > 1 && !modes::Pow2<L, MM::NS, true>::OK);
}

template <int L, int FORM>
multi_fn one() {
  if constexpr (has<L, FORM>()) return &launch_multi<MM, L, FORM>;
  else return nullptr;
}

template <int FORM>
multi_fn pick(int L) {
  switch (L) {
    case 5: return one<5, FORM>();
    case 6: return one<6, FORM>();
    case 7: return one<7, FORM>();
    case 8: return one<8, FORM>();
    case 9: return one<9, FORM>();
    case 10: return one<10, FORM>();
    case 11: return one<11, FORM>();
    case 12: return one<12, FORM>();
  }
  return nullptr;
}
}  // namespace

multi_fn NLM_CAT(nlm_pick_multi_, NLM_INST_MODEL)(int L, int form) {
  switch (form) {
    case MULTI_FIELD: return pick<MULTI_FIELD>(L);
    case MULTI_INLINE: return pick<MULTI_INLINE>(L);
    case MULTI_MODES: return pick<MULTI_MODES>(L);
    case MULTI_TAB: return pick<MULTI_TAB>(L);
  }
  return nullptr;
}
