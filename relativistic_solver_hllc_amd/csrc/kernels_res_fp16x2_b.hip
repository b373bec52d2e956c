// Single-problem split contraction: the unrolled plans of 15 to 25 K-steps, fp16x2.
#include "split_single_res.hpp"

RSH_SINGLE_RES_RANGE(1, 2, 15, 25)
