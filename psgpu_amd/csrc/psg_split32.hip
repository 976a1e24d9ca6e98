// The two-kernel 3D Navier-Stokes/Euler stepper (psg_split.hpp) in FP32 passes.
#include "psg_split.hpp"

namespace psg {
template int split_run<float>(Ctx *, cpx<float> *, int, bool, bool);
}  // namespace psg
