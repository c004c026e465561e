// Symmetric-contraction launchers over coefficient tables, input lmax 2, target lmax 2, correlation 3.
#include "sc_table.h"
namespace ictc {
namespace sc {
ICTC_SC_TAB_DEFINE(2, 2, 3)
}  // namespace sc
}  // namespace ictc
