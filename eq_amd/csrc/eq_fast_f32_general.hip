// eq_fast_f32_general.hip -- the fast solver's transform kernels: single precision, varying rows.
#include "eq_fast_launch.h"

namespace eqk {
template int fast_allow_lds<float, true>(const FastSolver*);
template void fast_forward<float, true>(eq_batch*, int, bool);
template void fast_backward<float, true>(eq_batch*, int);
} // namespace eqk
