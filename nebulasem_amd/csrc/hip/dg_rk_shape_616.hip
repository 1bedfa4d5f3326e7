// Stage kernels for elements of 6 x 1 x 6 nodes.
#include "dg_rk_stage.hpp"

NSEM_RK_SHAPE(6, 1, 6)
