// Kronecker kernel instances for 4D meshes.
#include "gd_kron.hpp"
#include "gd_kron_api.hpp"

namespace gd {
namespace kron {

#define GD_KRON(N) Entry{N, &launch_any<double, 4, N>, &launch_any<float, 4, N>}

static const Entry kEntries[] = {GD_KRON(2), GD_KRON(3), GD_KRON(4), GD_KRON(5)};

List instances_d4() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace kron
}  // namespace gd
