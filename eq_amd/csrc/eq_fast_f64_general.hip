// eq_fast_f64_general.hip -- the fast solver's transform kernels: double precision, varying rows.
#include "eq_fast_launch.h"

namespace eqk {
template int fast_allow_lds<double, true>(const FastSolver*);
template void fast_forward<double, true>(eq_batch*, int, bool);
template void fast_backward<double, true>(eq_batch*, int);
} // namespace eqk
