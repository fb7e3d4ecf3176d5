// Adjoint plane kernel instances with 3 nodes per dimension.
#include "gd_padj.hpp"
#include "gd_padj_api.hpp"

namespace gd {
namespace pl {

static const AdjEntry kEntries[] = {{3, 3, &launch_adj<3, 3>}, {3, 4, &launch_adj<3, 4>}, {3, 5, &launch_adj<3, 5>}};

AdjList adjoint_instances_n3() { return AdjList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
