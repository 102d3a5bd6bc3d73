// bottom_nodal.hip -- bottom-solve kernels of the nodal hierarchies.
#include "bottom_kernels.h"

namespace mgx {
MGX_BOTTOM_INSTANCE(, NodalRows<float>, float);
MGX_BOTTOM_INSTANCE(, NodalRows<double>, double);
}  // namespace mgx
