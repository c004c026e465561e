// Symmetric-contraction weight gradients over pair sums, input lmax 2, target lmax 2, correlation 3.
#include "sc_table.h"
namespace ictc {
namespace sc {
ICTC_SC_TAB_DEFINE_DW(2, 2, 3)
}  // namespace sc
}  // namespace ictc
