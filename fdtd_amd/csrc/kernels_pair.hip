// kernels_pair.hip -- half-steps of 16-bit storage: the storage form's kernels
// (pair_sweep.h).
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "internal.h"

namespace fdtd {

template <class T>
hipError_t launch_pair_t(bool efield, int mode, const KArgs &a, int m, hipStream_t s, bool gen_cells);

// storage: 1 FP16, 2 BF16, 3 block-scaled int16.
hipError_t launch_pair_half_step(bool efield, int storage, int mode, const KArgs &a, int m, hipStream_t s,
                                 bool gen_cells)
{
    switch (storage) {
    case 1: return launch_pair_t<_Float16>(efield, mode, a, m, s, gen_cells);
    case 2: return launch_pair_t<bf16_t>(efield, mode, a, m, s, gen_cells);
    case 3: return launch_pair_t<bq16_t>(efield, mode, a, m, s, gen_cells);
    default: return hipErrorInvalidValue;
    }
}

int pair_tile_cols() { return 2 * TX; }

}  // namespace fdtd
