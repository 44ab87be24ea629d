// nlm_mix_inst.hip -- the mixed-radix split step (nlm_mix.hpp) of one model for every
// first radix.  Compiled once per model with -DNLM_INST_MODEL=<id>; id 1 is the
// step-table kernel of the one-mode media (Chi3, Chi2PDC).
#include "nlm_mix.hpp"

#ifndef NLM_INST_MODEL
#error "NLM_INST_MODEL must be defined"
#endif

#define NLM_CAT2(a, b) a##b
#define NLM_CAT(a, b) NLM_CAT2(a, b)

template <int MODEL>
struct MixModel {
  using type = typename ModelOf<MODEL>::type;
};
template <>
struct MixModel<NLM_CHI2PDC> {
  using type = mix::Table;
};
using MM = typename MixModel<NLM_INST_MODEL>::type;

mix_fn NLM_CAT(nlm_pick_mix_, NLM_INST_MODEL)(int R) {
  switch (R) {
    case 2: return &launch_mix_prop<MM, 2>;
    case 3: return &launch_mix_prop<MM, 3>;
    case 4: return &launch_mix_prop<MM, 4>;
    case 5: return &launch_mix_prop<MM, 5>;
    case 6: return &launch_mix_prop<MM, 6>;
    case 8: return &launch_mix_prop<MM, 8>;
#if NLM_INST_MODEL != 14  // Chi3GNLSE, whose four register arrays leave room for R <= 8
    case 9: return &launch_mix_prop<MM, 9>;
    case 10: return &launch_mix_prop<MM, 10>;
#endif
  }
  return nullptr;
}
