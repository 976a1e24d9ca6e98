// The two-kernel 3D Navier-Stokes/Euler stepper (psg_split.hpp) in FP64.
#include "psg_split.hpp"

namespace psg {
template int split_run<double>(Ctx *, cpx<double> *, int, bool, bool);
}  // namespace psg
