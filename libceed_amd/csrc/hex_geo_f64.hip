// FP64 instantiations of the line kernel that recomputes trilinear geometric factors.
#include "hex_plan.hpp"

namespace mi355 {
GeoLinesFn pick_geo_f64(int P, int Q, int num_comp, int qf) { return pick_geo<double>(P, Q, num_comp, qf); }
}  // namespace mi355
