// ik_gather_rules_2d.hip -- tile-gather instantiations for 2 x 2 output
// tensors with fixed rules other than the Octic 5-node one, bond entries in
// double (one translation unit per form, compiled in parallel).
#include "ik_gather_launch.hpp"

namespace pgt {

void launch_tile_rules_2d(const LaunchCtx &c, unsigned fields, int cg) { launch_tile_rules<2>(c, fields, cg); }

}  // namespace pgt
