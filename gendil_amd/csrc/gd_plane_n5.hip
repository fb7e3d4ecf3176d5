// Plane kernel instances with 5 nodes per dimension.
#include "gd_plane_inst.hpp"

namespace gd {
namespace pl {

static const Entry kEntries[] = {GD_PLANE(5, 5), GD_PLANE(5, 6)};

List instances_n5() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
