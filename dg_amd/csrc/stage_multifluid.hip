// Tile kernel (stage.cuh): the two-fluid instances.
#include "stage.cuh"

namespace dgx {

DGX_STAGE_PHYS(1)

}  // namespace dgx
