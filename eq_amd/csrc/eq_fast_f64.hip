// eq_fast_f64.hip -- the fast solver's transform kernels: double precision, constant rows.
#include "eq_fast_launch.h"

namespace eqk {
template int fast_allow_lds<double, false>(const FastSolver*);
template void fast_forward<double, false>(eq_batch*, int, bool);
template void fast_backward<double, false>(eq_batch*, int);
} // namespace eqk
