// eq_fast_f32.hip -- the fast solver's transform kernels: single precision, constant rows.
#include "eq_fast_launch.h"

namespace eqk {
template int fast_allow_lds<float, false>(const FastSolver*);
template void fast_forward<float, false>(eq_batch*, int, bool);
template void fast_backward<float, false>(eq_batch*, int);
} // namespace eqk
