// Grouped FP32 GETT on the BF16 MFMAs.
#include "gett_group.hpp"

// FP32 results through the split (tccg_gett_f32_split's contract per problem).
extern "C" int tccg_gett_group_f32_split(int tile, const tccg_group_operand* ops, int nops,
                                         const tccg_group_job* jobs, int njobs, const tccg_group_problem* problems,
                                         int nproblems, const tccg_batch_work* work, int nwork, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  if (workspace_bytes < 256 + tccg::kPackedTailBytes)
    return tccg_lib::fail(1, "workspace smaller than the guard header and the prefetch tail pad");
  return tccg_lib::run_group<tccg::F32X3>(tile, ops, nops, jobs, njobs, problems, nproblems, work, nwork, workspace,
                                           workspace_bytes, stream);
}
