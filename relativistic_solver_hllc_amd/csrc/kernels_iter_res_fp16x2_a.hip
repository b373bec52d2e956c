// Grouped split iteration, resident-panel plans of 1 to 14 K-steps (1 to 448 directions), form fp16x2.
#include "split_iter_res.hpp"

RSH_ITER_RES_RANGE(1, 2, 1, 14)
