// gemm_group_z.hip -- grouped launches of complex128 problems
#include "gemm_group.h"

extern "C" int bx_launch_group_z(const bxh_problem_t *probs, int nprob, const bxh_seg_t *segs, int total,
                                 int grid, const int *counts, void *stream)
{
    return launch_group<cplx>(probs, nprob, segs, total, grid, counts, (hipStream_t)stream);
}
