// Stage kernels for elements of any shape.
#include "dg_rk_stage.hpp"

NSEM_RK_SHAPE(0, 0, 0)
