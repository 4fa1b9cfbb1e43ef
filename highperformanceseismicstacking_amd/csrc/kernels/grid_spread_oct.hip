// Spread grid search: instantiations for HSS_OCT (see grid_spread.hpp).
#include "grid_spread.hpp"

namespace hss {
bool launch_spread_oct(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                       hipStream_t stream, int *status) {
    return launch_grid_spread<HSS_OCT>(a, n_slots, variant, storage, tl, stream, status);
}
}  // namespace hss
