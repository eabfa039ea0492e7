// gemm_group_s.hip -- grouped launches of FP32 problems
#include "gemm_group.h"

extern "C" int bx_launch_group_s(const bxh_problem_t *probs, int nprob, const bxh_seg_t *segs, int total,
                                 int grid, const int *counts, void *stream)
{
    return launch_group<float>(probs, nprob, segs, total, grid, counts, (hipStream_t)stream);
}
