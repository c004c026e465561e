// Symmetric-contraction weight gradients over pair sums, input lmax 3, target lmax 1, correlation 3.
#include "sc_table.h"
namespace ictc {
namespace sc {
ICTC_SC_TAB_DEFINE_DW(3, 1, 3)
}  // namespace sc
}  // namespace ictc
