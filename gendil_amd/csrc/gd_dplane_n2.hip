// Diffusion plane kernel instances with 2 nodes per dimension.
#include "gd_dplane.hpp"
#include "gd_dplane_api.hpp"

namespace gd {
namespace pl {

#define GD_DPLANE(Q) DEntry{2, Q, &launch_diff<double, 2, Q>, &launch_diff<float, 2, Q>}

static const DEntry kEntries[] = {GD_DPLANE(3), GD_DPLANE(4)};

DList diff_instances_n2() { return DList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
