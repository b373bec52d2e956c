// Single-problem split contraction: the unrolled plans of 1 to 14 K-steps, bf16x3.
#include "split_single_res.hpp"

RSH_SINGLE_RES_RANGE(0, 3, 1, 14)
