// Spread grid search: instantiations for HSS_CMP (see grid_spread.hpp).
#include "grid_spread.hpp"

namespace hss {
bool launch_spread_cmp(const GridArgs &a, int n_slots, int variant, int storage, int tl,
                       hipStream_t stream, int *status) {
    return launch_grid_spread<HSS_CMP>(a, n_slots, variant, storage, tl, stream, status);
}
}  // namespace hss
