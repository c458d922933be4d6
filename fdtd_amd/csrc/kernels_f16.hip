// kernels_f16.hip -- the half-step kernels of FP16 storage, two cells per
// thread (pair_sweep.h).
#include "pair_sweep.h"

namespace fdtd {

template hipError_t launch_pair_t<_Float16>(bool, int, const KArgs &, int, hipStream_t, bool);

}  // namespace fdtd
