// Plane kernel instances with 3 nodes per dimension.
#include "gd_plane_inst.hpp"

namespace gd {
namespace pl {

static const Entry kEntries[] = {GD_PLANE(3, 3), GD_PLANE(3, 4), GD_PLANE(3, 5)};

List instances_n3() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
