// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_gdn_qkvz: (20,16,16) -> (16,32,32), rank 8, bf16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_BF16, 1, 2, 0, 20, 16, 16, 16, 32, 32, 8};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 192, 2, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1473, 1536)  // ring3_join_w8<120,192,2,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 2, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 2195, 2304)  // ring3_join_w8<120,192,2,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 2, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 2823, 3072)  // ring3_join_w8<120,192,2,8,16,1,1,1>
};

}  // namespace

int join_register_gen_bf16_20x16x16_16x32x32_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
