// FP32 element kernels of the RHS between FP64 arrays, periodic meshes.
#include "elem_registry.hpp"

TRIXI_REG_DEFAULTS(float, false, trixi_hip::ELEM_RHS64)
TRIXI_REG_ALT_TILES_RHS64()
