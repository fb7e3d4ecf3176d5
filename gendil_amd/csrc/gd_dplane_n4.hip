// Diffusion plane kernel instances with 4 nodes per dimension.
#include "gd_dplane.hpp"
#include "gd_dplane_api.hpp"

namespace gd {
namespace pl {

#define GD_DPLANE(Q) DEntry{4, Q, &launch_diff<double, 4, Q>, &launch_diff<float, 4, Q>}

static const DEntry kEntries[] = {GD_DPLANE(4), GD_DPLANE(5), GD_DPLANE(6)};

DList diff_instances_n4() { return DList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
