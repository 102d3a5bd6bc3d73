// bottom_cell.hip -- bottom-solve kernels of the cell-centred and EB hierarchies.
#include "eb_kernels.h"
#include "mac_kernels.h"

namespace mgx {
MGX_BOTTOM_INSTANCE(, MacRows<float>, float);
MGX_BOTTOM_INSTANCE(, MacRows<double>, double);
MGX_BOTTOM_INSTANCE(, EBRows, double);
}  // namespace mgx
