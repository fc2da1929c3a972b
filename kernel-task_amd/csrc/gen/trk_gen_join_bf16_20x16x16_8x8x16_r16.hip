// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_attn_kv: (20,16,16) -> (8,8,16), rank 16, bf16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_BF16, 1, 2, 0, 20, 16, 16, 8, 8, 16, 16};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 48, 1, 1, 8, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 65, 96)  // ring3_join_w8<120,48,1,1,8,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 1, 8, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 97, 128)  // ring3_join_w8<120,64,1,1,8,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 80, 1, 1, 8, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 129, 160)  // ring3_join_w8<120,80,1,1,8,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 1, 8, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 161, 192)  // ring3_join_w8<120,96,1,1,8,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 2, 1, 8, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 193, 256)  // ring3_join<120,64,2,1,8,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 2, 8, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 257, 384)  // ring3_join_w8<120,96,1,2,8,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 2, 8, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 385, 512)  // ring3_join_w8<120,128,1,2,8,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 4, 8, 1, 2, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 513, 1024)  // ring3_join_w8<120,128,1,4,8,1,2,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 2, 8, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1025, 1152)  // ring3_join_w8<120,96,1,2,8,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 8, 8, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 1153, 2048)  // ring3_join_w8<120,128,1,8,8,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 192, 1, 8, 8, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 2049, 3072)  // ring3_join_w8<120,192,1,8,8,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 8, 8, 1, 1, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 3073, 1073741824)  // ring3_join_w8<120,128,1,8,8,1,1,1>
};

}  // namespace

int join_register_gen_bf16_20x16x16_8x8x16_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
