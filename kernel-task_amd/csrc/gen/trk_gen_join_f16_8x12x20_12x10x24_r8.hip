// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// r8: (8,12,20) -> (12,10,24), rank 8, f16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined, for cores that trk_plan_admit finds even.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_F16, 1, 2, 0, 8, 12, 20, 12, 10, 24, 8};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 48, 1, 2, 12, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 86, 96)  // ring3_join_w8<120,48,1,2,12,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 2, 12, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 97, 128)  // ring3_join_w8<120,64,1,2,12,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 4, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 171, 256)  // ring3_join_w8<120,64,1,4,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 4, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 262, 512)  // ring3_join_w8<120,128,1,4,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 2, 4, 12, 1, 2, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 513, 768)  // ring3_join_w8<120,96,2,4,12,1,2,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 8, 12, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 769, 1024)  // ring3_join_w8<120,128,1,8,12,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 2, 8, 12, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1025, 1536)  // ring3_join_w8<120,96,2,8,12,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 2, 8, 12, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1537, 2048)  // ring3_join_w8<120,128,2,8,12,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 2, 8, 12, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 2049, 3072)  // ring3_join_w8<120,192,2,8,12,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 2, 8, 12, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 3073, 1073741824)  // ring3_join_w8<120,128,2,8,12,1,1,1>
};

}  // namespace

int join_register_gen_f16_8x12x20_12x10x24_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
