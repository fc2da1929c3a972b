// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// r8_fp32: (8,12,20) -> (12,10,24), rank 8, f32, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_F32, 1, 2, 0, 8, 12, 20, 12, 10, 24, 8};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 1, 12, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 33, 64)  // ring3_join_w8<120,64,1,1,12,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 1, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 65, 96)  // ring3_join<120,96,1,1,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 112, 1, 1, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 97, 112)  // ring3_join<120,112,1,1,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 113, 128)  // ring3_join<120,64,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 80, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 129, 160)  // ring3_join<120,80,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 2, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 161, 192)  // ring3_join_w8<120,96,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 112, 1, 2, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 193, 224)  // ring3_join_w8<120,112,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 225, 256)  // ring3_join<120,128,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 80, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 257, 320)  // ring3_join<120,80,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 2, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 321, 384)  // ring3_join_w8<120,96,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 112, 1, 2, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 385, 448)  // ring3_join_w8<120,112,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 449, 512)  // ring3_join<120,128,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 112, 1, 2, 12, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 513, 640)  // ring3_join_w8<120,112,1,2,12,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 2, 12, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 641, 1073741824)  // ring3_join<120,128,1,2,12,1,4,1>
};

}  // namespace

int join_register_gen_f32_8x12x20_12x10x24_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
