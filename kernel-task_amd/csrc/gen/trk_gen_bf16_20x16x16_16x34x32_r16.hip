// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_mlp_gate_up: (20,16,16) -> (16,34,32), rank 16, bf16, chain order (0,2,1); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape021{TRK_DTYPE_BF16, 0, 2, 1, 20, 16, 16, 16, 34, 32, 16};

const Entry kEntries[] = {
    TRK_ENTRY_PAIR(tile(kShape021, 1, 1, 4, 17, 2, 8, 1, 0, 16, 8), 1, 1)  // t1_l17_s4_w8_k8
    TRK_ENTRY_PAIR(tile(kShape021, 1, 1, 16, 34, 2, 2, 1, 8, 32, 8, 1), 2, 8)  // wide8x32w8_t1k2n1_ic2_p
    TRK_ENTRY_PAIR(tile(kShape021, 1, 2, 16, 34, 2, 1, 2, 8, 32, 8), 9, 16)  // wide8x32w8_f2k1n2_ic2
    TRK_ENTRY_PAIR(tile(kShape021, 4, 1, 16, 34, 1, 1, 2, 8, 32, 8, 1), 17, 32)  // wide8x32w8_t4k1n2_p
};

}  // namespace

int mfma_register_gen_bf16_20x16x16_16x34x32_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
