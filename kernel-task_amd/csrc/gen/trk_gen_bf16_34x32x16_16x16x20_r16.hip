// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_mlp_down: (34,32,16) -> (16,16,20), rank 16, bf16, chain orders (0,1,2), (1,0,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 34, 32, 16, 16, 16, 20, 16};
constexpr Shape kShape102{TRK_DTYPE_BF16, 1, 0, 2, 34, 32, 16, 16, 16, 20, 16};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape012, 1, 1, 2, 10, 2, 8, 1, 0, 16, 8), 1, 1)  // t1_l10_s2_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 4, 10, 1, 8, 1, 0, 16, 8, 1), 2, 2)  // t1_l10_s4_w8_k8_p
    TRK_ENTRY(tile(kShape102, 1, 1, 4, 20, 1, 2, 2), 3, 8)  // mid_1of4_k2@102
};

}  // namespace

int mfma_register_gen_bf16_34x32x16_16x16x20_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
