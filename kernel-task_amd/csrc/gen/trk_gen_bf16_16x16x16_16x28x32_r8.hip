// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// llama_up: (16,16,16) -> (16,28,32), rank 8, bf16, chain orders (0,1,2), (1,0,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 16, 16, 16, 16, 28, 32, 8};
constexpr Shape kShape102{TRK_DTYPE_BF16, 1, 0, 2, 16, 16, 16, 16, 28, 32, 8};

const Entry kEntries[] = {
    TRK_ENTRY_PAIR(tile(kShape012, 1, 1, 4, 16, 16, 4, 1, 0, 16, 4, 0, 0, 0, 0, 1), 1, 1)  // t1_l16_s4_k4_sl
    TRK_ENTRY_PAIR(tile(kShape102, 1, 1, 8, 32, 8, 1, 2, 0, 16, 4, 1), 2, 4)  // mid_half_p@102
    TRK_ENTRY_PAIR(tile(kShape012, 1, 1, 28, 32, 4, 1, 2, 8, 32, 8, 2, 4, 0, 0, 1), 5, 16)  // ring3_mfma_wide8x32w8p2_s4_sl<012,1,1,28,32,4,1,2>
    TRK_ENTRY_PAIR(tile(kShape012, 1, 2, 28, 32, 4, 1, 2, 8, 32, 8, 1, 4), 17, 32)  // ring3_mfma_wide8x32w8p_s4<012,1,2,28,32,4,1,2>
    TRK_ENTRY_PAIR(tile(kShape012, 1, 2, 28, 32, 4, 2, 1, 8, 32, 8, 0, 4), 33, 64)  // ring3_mfma_wide8x32w8_s4<012,1,2,28,32,4,2,1>
    TRK_ENTRY_PAIR(tile(kShape012, 1, 8, 28, 32, 2, 2, 1, 8, 32, 8, 1), 65, 128)  // wide8x32w8_f8sc28k2n1_ic2_p
    TRK_ENTRY_PAIR(tile(kShape012, 1, 8, 28, 32, 2, 2, 1, 8, 32, 8, 1), 193, 384)  // wide8x32w8_f8sc28k2n1_ic2_p
    TRK_ENTRY_PAIR(tile(kShape012, 1, 8, 28, 32, 2, 2, 1, 8, 32, 8, 1), 1537, 1664)  // wide8x32w8_f8sc28k2n1_ic2_p
    TRK_ENTRY_PAIR(tile(kShape012, 1, 8, 28, 32, 2, 2, 1, 8, 32, 8, 1), 2177, 2432)  // wide8x32w8_f8sc28k2n1_ic2_p
};

}  // namespace

int mfma_register_gen_bf16_16x16x16_16x28x32_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
