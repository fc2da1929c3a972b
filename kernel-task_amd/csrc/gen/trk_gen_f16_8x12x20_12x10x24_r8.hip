// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// r8: (8,12,20) -> (12,10,24), rank 8, f16, chain order (2,1,0); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape210{TRK_DTYPE_F16, 2, 1, 0, 8, 12, 20, 12, 10, 24, 8};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape210, 1, 1, 2, 12, 8, 4, 1, 0, 16, 4, 0, 0, 4), 1, 1)  // t1_s2_x4
    TRK_ENTRY(tile(kShape210, 1, 1, 2, 12, 8, 4, 1), 2, 2)  // t1_s2
    TRK_ENTRY(tile(kShape210, 1, 1, 10, 12, 8, 2, 1, 8, 32, 8), 3, 8)  // wide8x32w8_t1k2n1_ic8
    TRK_ENTRY(tile(kShape210, 1, 1, 10, 12, 4, 2, 1, 4, 32, 4, 0, 0, 0, 0, 1), 9, 32)  // wide4x32_t1k2n1_ic4_sl
    TRK_ENTRY(tile(kShape210, 1, 2, 10, 12, 4, 2, 1, 4, 32, 4, 0, 0, 0, 0, 1), 33, 64)  // ring3_mfma_wide4x32_sl<210,1,2,10,12,4,2,1>
    TRK_ENTRY(tile(kShape210, 1, 8, 10, 12, 2, 1, 2, 4, 32, 8, 1), 65, 1073741824)  // ring3_mfma_wide4x32w8p<210,1,8,10,12,2,1,2>
    TRK_ENTRY(tile(kShape210, 1, 1, 10, 12, 8, 4, 1, 0, 16, 8, 0, 0, 1), 0, 0)  // t1_all_w8_xl
    TRK_ENTRY(tile(kShape210, 3, 1, 10, 12, 4, 2, 1, 4, 32, 4), 0, 0)  // cover_t3_w4
    TRK_ENTRY(tile(kShape210, 2, 3, 10, 12, 2, 2, 1, 4, 32, 4), 0, 0)  // cover_t2f3_w4
};

}  // namespace

int mfma_register_gen_f16_8x12x20_12x10x24_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
