// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// llama_down: (16,28,32) -> (16,16,16), rank 16, bf16, chain order (2,1,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape210{TRK_DTYPE_BF16, 2, 1, 0, 16, 28, 32, 16, 16, 16, 16};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape210, 1, 1, 1, 16, 2, 4, 1, 0, 16, 8, 1), 1, 1)  // t1_s1_w8_k4_p
    TRK_ENTRY(tile(kShape210, 1, 1, 2, 16, 2, 4, 1, 0, 16, 8, 1), 2, 2)  // t1_s2_w8_k4_p
    TRK_ENTRY(tile(kShape210, 1, 1, 8, 16, 4, 8, 1, 8, 32, 8, 0, 0, 0, 0, 1), 3, 8)  // ring3_mfma_wide8x32w8_sl<210,1,1,8,16,4,8,1>
    TRK_ENTRY(tile(kShape210, 1, 1, 16, 16, 2, 2, 1, 8, 32, 8, 1, 2), 9, 16)  // ring3_mfma_wide8x32w8p_s2<210,1,1,16,16,2,2,1>
    TRK_ENTRY(tile(kShape210, 1, 2, 16, 16, 2, 2, 1, 8, 32, 8, 1, 4, 0, 0, 1), 17, 32)  // ring3_mfma_wide8x32w8p_s4_sl<210,1,2,16,16,2,2,1>
};

}  // namespace

int mfma_register_gen_bf16_16x28x32_16x16x16_r16(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
