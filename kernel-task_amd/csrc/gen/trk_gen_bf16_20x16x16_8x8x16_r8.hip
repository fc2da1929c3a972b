// Generated by kernel-task_amd/factorized_inference/tilegen.py; do not edit.
// qwen_attn_kv: (20,16,16) -> (8,8,16), rank 8, bf16, chain order (0,1,2); token ranges measured by kernel-task_amd/benchmarks/autotune.py.
#include "trk_mfma_kernel.h"

namespace trk {
namespace {

constexpr Shape kShape012{TRK_DTYPE_BF16, 0, 1, 2, 20, 16, 16, 8, 8, 16, 8};

const Entry kEntries[] = {
    TRK_ENTRY(tile(kShape012, 1, 1, 2, 8, 16, 8, 1, 0, 16, 8), 1, 1)  // t1_l8_s2_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 1, 8, 16, 8, 1, 0, 16, 8), 2, 2)  // t1_l8_s1_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 2, 8, 16, 8, 1, 0, 16, 8), 3, 4)  // t1_l8_s2_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 4, 8, 16, 8, 1, 0, 16, 8), 5, 8)  // t1_l8_s4_w8_k8
    TRK_ENTRY(tile(kShape012, 1, 1, 8, 16, 8, 2, 1, 4, 32, 8, 1), 9, 32)  // wide4x32w8_t1k2n1_ic8_p
    TRK_ENTRY(tile(kShape012, 1, 2, 8, 16, 8, 1, 2, 4, 32, 8, 2), 33, 64)  // wide4x32w8_f2k1n2_ic8_p2
    TRK_ENTRY(tile(kShape012, 1, 2, 8, 16, 4, 1, 2, 4, 32, 8, 1), 65, 128)  // wide4x32w8_f2k1n2_ic4_p
    TRK_ENTRY(tile(kShape012, 1, 2, 8, 16, 4, 1, 2, 4, 32, 4), 129, 384)  // wide4x32_f2k1n2_ic4
};

}  // namespace

int mfma_register_gen_bf16_20x16x16_8x8x16_r8(Plan *plan) {
    return register_entries(plan, kEntries, int(sizeof(kEntries) / sizeof(kEntries[0])));
}

}  // namespace trk
