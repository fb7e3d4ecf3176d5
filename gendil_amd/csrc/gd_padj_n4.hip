// Adjoint plane kernel instances with 4 nodes per dimension.
#include "gd_padj.hpp"
#include "gd_padj_api.hpp"

namespace gd {
namespace pl {

static const AdjEntry kEntries[] = {{4, 4, &launch_adj<4, 4>}, {4, 5, &launch_adj<4, 5>}, {4, 6, &launch_adj<4, 6>}};

AdjList adjoint_instances_n4() { return AdjList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
