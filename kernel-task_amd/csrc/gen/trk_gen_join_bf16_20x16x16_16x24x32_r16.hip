// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_attn_q_gate: (20,16,16) -> (16,24,32), rank 16, bf16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_BF16, 1, 2, 0, 20, 16, 16, 16, 24, 32, 16};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 32, 3, 1, 16, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 17, 32)  // ring3_join<120,32,3,1,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 48, 3, 1, 16, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 33, 48)  // ring3_join<120,48,3,1,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 3, 1, 16, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 49, 64)  // ring3_join<120,64,3,1,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 4, 16, 1, 2, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 65, 96)  // ring3_join_w8<120,96,1,4,16,1,2,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 4, 16, 1, 2, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 97, 128)  // ring3_join_w8<120,128,1,4,16,1,2,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 1, 4, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 129, 192)  // ring3_join<120,192,1,4,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 193, 256)  // ring3_join_w8<120,128,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 1, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 257, 384)  // ring3_join_w8<120,192,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 224, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 385, 448)  // ring3_join<120,224,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 449, 512)  // ring3_join<120,256,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 513, 640)  // ring3_join_w8<120,128,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 1, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 641, 896)  // ring3_join_w8<120,192,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 224, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 897, 1024)  // ring3_join<120,224,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1025, 1280)  // ring3_join<120,256,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 1, 8, 16, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1281, 1536)  // ring3_join_w8<120,192,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 224, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1537, 1792)  // ring3_join<120,224,1,8,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 1, 8, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1793, 1073741824)  // ring3_join<120,256,1,8,16,1,1,1>
};

}  // namespace

int join_register_gen_bf16_20x16x16_16x24x32_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
