// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// llama_up: (16,16,16) -> (16,28,32), rank 8, bf16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_BF16, 1, 2, 0, 16, 16, 16, 16, 28, 32, 8};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN_PAIR(tile(kShape120, 160, 1, 8, 16, 1, 1, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 257, 320)  // ring3_join<120,160,1,8,16,1,1,2>
    TRK_ENTRY_JOIN_PAIR(tile(kShape120, 128, 1, 8, 16, 1, 1, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 449, 512)  // ring3_join<120,128,1,8,16,1,1,2>
    TRK_ENTRY_JOIN_PAIR(tile(kShape120, 160, 1, 8, 16, 1, 1, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 513, 640)  // ring3_join<120,160,1,8,16,1,1,2>
    TRK_ENTRY_JOIN_PAIR(tile(kShape120, 160, 1, 8, 16, 1, 1, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1025, 1280)  // ring3_join<120,160,1,8,16,1,1,2>
    TRK_ENTRY_JOIN_PAIR(tile(kShape120, 128, 1, 8, 16, 1, 1, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1537, 1073741824)  // ring3_join<120,128,1,8,16,1,1,2>
};

}  // namespace

int join_register_gen_bf16_16x16x16_16x28x32_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
