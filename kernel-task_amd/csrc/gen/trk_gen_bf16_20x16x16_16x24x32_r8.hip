// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_attn_q_gate: (20,16,16) -> (16,24,32), rank 8, bf16, chain order (0,1,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 20, 16, 16, 16, 24, 32, 8};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape012, 1, 1, 4, 16, 16, 8, 1, 0, 16, 8), 1, 1)  // t1_l16_s4_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 6, 32, 8, 2, 2), 2, 4)  // mid_1of4_k2
    TRK_ENTRY(tile(kShape012, 1, 1, 24, 32, 8, 2, 1, 8, 32, 8), 5, 8)  // wide8x32w8_t1k2n1_ic8
    TRK_ENTRY(tile(kShape012, 1, 1, 24, 32, 8, 1, 2, 8, 32, 8), 9, 16)  // wide8x32w8_t1k1n2_ic8
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 8, 1, 2, 8, 32, 8), 17, 32)  // wide8x32w8_f2k1n2_ic8
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 4, 1, 2, 4, 32, 4), 33, 476)  // wide4x32_f2k1n2_ic4
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 4, 1, 2, 4, 32, 4), 513, 536)  // wide4x32_f2k1n2_ic4
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 4, 1, 2, 4, 32, 4), 769, 928)  // wide4x32_f2k1n2_ic4
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 4, 1, 2, 4, 32, 4), 1537, 1568)  // wide4x32_f2k1n2_ic4
    TRK_ENTRY(tile(kShape012, 1, 2, 24, 32, 4, 1, 2, 4, 32, 4), 2049, 2179)  // wide4x32_f2k1n2_ic4
};

}  // namespace

int mfma_register_gen_bf16_20x16x16_16x24x32_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
