// Plane kernel instances with 4 nodes per dimension.
#include "gd_plane_inst.hpp"

namespace gd {
namespace pl {

static const Entry kEntries[] = {GD_PLANE(4, 4), GD_PLANE(4, 5), GD_PLANE(4, 6)};

List instances_n4() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
