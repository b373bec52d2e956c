// Single-problem split contraction: the unrolled plans of 1 to 14 K-steps, fp16x2.
#include "split_single_res.hpp"

RSH_SINGLE_RES_RANGE(1, 2, 1, 14)
