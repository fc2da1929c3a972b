// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_mlp_down: (34,32,16) -> (16,16,20), rank 8, bf16, chain order (0,1,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 34, 32, 16, 16, 16, 20, 8};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape012, 1, 1, 2, 10, 8, 8, 1, 0, 16, 8), 1, 1)  // t1_l10_s2_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 4, 10, 8, 8, 1, 0, 16, 8), 2, 2)  // t1_l10_s4_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 16, 20, 4, 2, 1, 8, 32, 8, 1), 3, 8)  // wide8x32w8_t1k2n1_ic4_p
    TRK_ENTRY(tile(kShape012, 1, 1, 16, 20, 4, 1, 2, 8, 32, 8), 9, 16)  // wide8x32w8_t1k1n2_ic4
    TRK_ENTRY(tile(kShape012, 1, 2, 16, 20, 4, 1, 2, 8, 32, 8, 1), 17, 288)  // wide8x32w8_f2k1n2_ic4_p
};

}  // namespace

int mfma_register_gen_bf16_34x32x16_16x16x20_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
