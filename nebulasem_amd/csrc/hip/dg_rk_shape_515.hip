// Stage kernels for elements of 5 x 1 x 5 nodes.
#include "dg_rk_stage.hpp"

NSEM_RK_SHAPE(5, 1, 5)
