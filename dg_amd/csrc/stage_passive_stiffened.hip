// Tile kernel (stage.cuh): the passive-scalar and stiffened-gas instances.
#include "stage.cuh"

namespace dgx {

DGX_STAGE_PHYS(2)
DGX_STAGE_PHYS(3)

}  // namespace dgx
