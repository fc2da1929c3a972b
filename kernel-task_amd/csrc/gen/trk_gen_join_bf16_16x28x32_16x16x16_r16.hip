// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// llama_down: (16,28,32) -> (16,16,16), rank 16, bf16, chain order (1,2,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py --joined.
#include "trk_join_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape120{TRK_DTYPE_BF16, 1, 2, 0, 16, 28, 32, 16, 16, 16, 16};

const Entry kEntries[] = {
    TRK_ENTRY_JOIN(tile(kShape120, 48, 1, 1, 16, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 33, 48)  // ring3_join_w8<120,48,1,1,16,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 1, 1, 16, 1, 4, 2, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 49, 64)  // ring3_join<120,64,1,1,16,1,4,2>
    TRK_ENTRY_JOIN(tile(kShape120, 80, 1, 1, 16, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 65, 80)  // ring3_join_w8<120,80,1,1,16,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 1, 1, 16, 1, 8, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 81, 96)  // ring3_join_w8<120,96,1,1,16,1,8,1>
    TRK_ENTRY_JOIN(tile(kShape120, 64, 2, 1, 16, 1, 4, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 97, 128)  // ring3_join<120,64,2,1,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 96, 2, 1, 16, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 129, 192)  // ring3_join_w8<120,96,2,1,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 2, 16, 1, 4, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 193, 256)  // ring3_join_w8<120,128,1,2,16,1,4,1>
    TRK_ENTRY_JOIN(tile(kShape120, 128, 1, 4, 16, 1, 2, 1, 0, 16, 8, 0, 0, 0, 0, 0, 0, 1), 257, 512)  // ring3_join_w8<120,128,1,4,16,1,2,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 1, 4, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 513, 1024)  // ring3_join<120,256,1,4,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 2, 4, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 1025, 2048)  // ring3_join<120,256,2,4,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 1, 4, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 2049, 2560)  // ring3_join<120,256,1,4,16,1,1,1>
    TRK_ENTRY_JOIN(tile(kShape120, 256, 2, 4, 16, 1, 1, 1, 0, 16, 4, 0, 0, 0, 0, 0, 0, 1), 2561, 1073741824)  // ring3_join<120,256,2,4,16,1,1,1>
};

}  // namespace

int join_register_gen_bf16_16x28x32_16x16x16_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
