// FP32 element kernels of the RHS between FP64 arrays, meshes with boundaries or
// mortars (default tiles only).
#include "elem_registry.hpp"

TRIXI_REG_DEFAULTS(float, true, trixi_hip::ELEM_RHS64)
