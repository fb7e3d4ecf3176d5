// Plane kernel instances with 2 nodes per dimension.
#include "gd_plane_inst.hpp"

namespace gd {
namespace pl {

static const Entry kEntries[] = {GD_PLANE(2, 2), GD_PLANE(2, 3), GD_PLANE(2, 4)};

List instances_n2() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
