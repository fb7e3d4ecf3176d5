// Adjoint plane kernel instances with 5 nodes per dimension.
#include "gd_padj.hpp"
#include "gd_padj_api.hpp"

namespace gd {
namespace pl {

static const AdjEntry kEntries[] = {{5, 5, &launch_adj<5, 5>}, {5, 6, &launch_adj<5, 6>}};

AdjList adjoint_instances_n5() { return AdjList{kEntries, (int)(sizeof(kEntries) / sizeof(kEntries[0]))}; }

}  // namespace pl
}  // namespace gd
