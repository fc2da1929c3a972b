// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_mlp_gate_up: (20,16,16) -> (16,34,32), rank 8, bf16, chain order (0,1,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 20, 16, 16, 16, 34, 32, 8};

const Entry kEntries[] = {
    TRK_ENTRY_PAIR(tile(kShape012, 1, 1, 5, 32, 8, 2, 2), 1, 2)  // mid_1of8_k2
    TRK_ENTRY_PAIR(tile(kShape012, 1, 1, 17, 32, 8, 2, 1, 8, 32, 8), 3, 8)  // wide8x32w8_t1k2n1_ic8
    TRK_ENTRY_PAIR(tile(kShape012, 1, 2, 17, 32, 8, 1, 2, 8, 32, 8), 9, 16)  // wide8x32w8_f2k1n2_ic8
    TRK_ENTRY_PAIR(tile(kShape012, 1, 2, 17, 32, 4, 1, 2, 4, 32, 4), 17, 160)  // wide4x32_f2k1n2_ic4
};

}  // namespace

int mfma_register_gen_bf16_20x16x16_16x34x32_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
