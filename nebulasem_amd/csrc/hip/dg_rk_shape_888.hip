// Stage kernels for elements of 8 x 8 x 8 nodes.
#include "dg_rk_stage.hpp"

NSEM_RK_SHAPE(8, 8, 8)
