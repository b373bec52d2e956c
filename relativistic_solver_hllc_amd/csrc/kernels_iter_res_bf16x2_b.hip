// Grouped split iteration, resident-panel plans of 15 to 25 K-steps (449 to 800 directions), form bf16x2.
#include "split_iter_res.hpp"

RSH_ITER_RES_RANGE(0, 2, 15, 25)
