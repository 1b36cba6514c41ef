// jw_step_multi.hip -- one launch per kernel class over every size group of a batch, compiled once
// for each storage type (JW_STEP_F32 given by the Makefile).
#include "jw_engine.hpp"

namespace jw {

#if JW_STEP_F32
hipError_t step_multi_f32(hipStream_t st, const GroupArgs* g, int ng, const StepArgs& a) {
    return step_multi_from<cplxf>(st, g, ng, a);
}
#else
hipError_t step_multi(hipStream_t st, const GroupArgs* g, int ng, const StepArgs& a) {
    return step_multi_from<cplx>(st, g, ng, a);
}
#endif

}  // namespace jw
