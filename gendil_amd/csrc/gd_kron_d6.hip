// Kronecker kernel instances for 6D meshes.
#include "gd_kron.hpp"
#include "gd_kron_api.hpp"

namespace gd {
namespace kron {

#define GD_KRON(N) Entry{N, &launch_any<double, 6, N>, &launch_any<float, 6, N>}

static const Entry kEntries[] = {GD_KRON(2), GD_KRON(3), GD_KRON(4)};

List instances_d6() { return List{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace kron
}  // namespace gd
