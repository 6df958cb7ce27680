// F32 element kernels that apply the 2N stage update (default tiles, bounded meshes).
#include "elem_registry.hpp"

TRIXI_REG_DEFAULTS(float, true, trixi_hip::ELEM_STAGE)
