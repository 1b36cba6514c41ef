// jw_step_large.hip -- the large-lattice step (N = 4096, 8192), compiled once
// for each storage type (JW_STEP_F32 given by the Makefile).
#include "jw_packed.hpp"

namespace jw {

#if JW_STEP_F32
hipError_t step_large_f32(jw_ctx* c, cplxf* U, cplxf* Xi, cplxf* Vv, cplxf* ZA, cplxf* ZB, const StepArgs& a) {
    return step_large_t(c, U, Xi, Vv, ZA, ZB, a);
}
#else
hipError_t step_large(jw_ctx* c, cplx* U, cplx* Xi, cplx* Vv, cplx* ZA, cplx* ZB, const StepArgs& a) {
    return step_large_t(c, U, Xi, Vv, ZA, ZB, a);
}
#endif

}  // namespace jw
