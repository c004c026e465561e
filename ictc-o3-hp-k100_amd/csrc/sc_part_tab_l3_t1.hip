// Symmetric-contraction launchers over coefficient tables, input lmax 3, target lmax 1, correlation 3.
#include "sc_table.h"
namespace ictc {
namespace sc {
ICTC_SC_TAB_DEFINE(3, 1, 3)
}  // namespace sc
}  // namespace ictc
