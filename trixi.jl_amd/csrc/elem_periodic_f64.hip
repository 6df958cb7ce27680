// FP64 element kernels for periodic meshes (no boundary states).
#include "elem_registry.hpp"

TRIXI_REG_DEFAULTS(double, false, trixi_hip::ELEM_RHS)
