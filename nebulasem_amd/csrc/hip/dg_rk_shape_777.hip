// Stage kernels for elements of 7 x 7 x 7 nodes.
#include "dg_rk_stage.hpp"

NSEM_RK_SHAPE(7, 7, 7)
