// Single-problem split contraction: the unrolled plans of 15 to 25 K-steps, bf16x2.
#include "split_single_res.hpp"

RSH_SINGLE_RES_RANGE(0, 2, 15, 25)
