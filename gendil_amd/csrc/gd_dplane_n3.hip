// Diffusion plane kernel instances with 3 nodes per dimension.
#include "gd_dplane.hpp"
#include "gd_dplane_api.hpp"

namespace gd {
namespace pl {

#define GD_DPLANE(Q) DEntry{3, Q, &launch_diff<double, 3, Q>, &launch_diff<float, 3, Q>}

static const DEntry kEntries[] = {GD_DPLANE(3), GD_DPLANE(4), GD_DPLANE(5)};

DList diff_instances_n3() { return DList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
