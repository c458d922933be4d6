// kernels_bf16.hip -- the half-step kernels of BF16 storage, two cells per
// thread (pair_sweep.h).
#include "pair_sweep.h"

namespace fdtd {

template hipError_t launch_pair_t<bf16_t>(bool, int, const KArgs &, int, hipStream_t, bool);

}  // namespace fdtd
