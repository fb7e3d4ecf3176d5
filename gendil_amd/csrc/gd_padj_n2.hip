// Adjoint plane kernel instances with 2 nodes per dimension.
#include "gd_padj.hpp"
#include "gd_padj_api.hpp"

namespace gd {
namespace pl {

static const AdjEntry kEntries[] = {{2, 2, &launch_adj<2, 2>}, {2, 3, &launch_adj<2, 3>}, {2, 4, &launch_adj<2, 4>}};

AdjList adjoint_instances_n2() { return AdjList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
