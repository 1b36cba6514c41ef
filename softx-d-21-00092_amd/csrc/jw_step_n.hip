// jw_step_n.hip -- the fused step of one lattice size and storage type, compiled once
// for each (JW_STEP_N, JW_STEP_C given by the Makefile).
#include "jw_engine.hpp"

namespace jw {

template hipError_t step_fused_layout<JW_STEP_N, JW_STEP_C>(jw_ctx*, JW_STEP_C*, JW_STEP_C*, JW_STEP_C*, JW_STEP_C*,
                                                            JW_STEP_C*, const StepArgs&, const int*);

}  // namespace jw
