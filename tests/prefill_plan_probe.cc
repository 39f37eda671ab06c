// Test-only view of the prefill launch plan
// (infinicore_amd/csrc/infiniop/ops/paged_attention_prefill/amd/prefill_plan.h): compiled with the host compiler by
// tests/test_prefill_plan.py, no GPU and no HIP needed.
#include "infiniop/ops/paged_attention_prefill/amd/prefill_plan.h"

namespace {

using op::paged_attention_prefill::PagedAttentionPrefillInfo;
using op::paged_attention_prefill::amd::Plan;

// in: {num_seqs, total_q_tokens, num_heads, num_kv_heads, value_size, block_size, max_blocks_per_seq, compute_units,
//      has_alibi, head_size}
Plan planOf(const long long *in, float scale) {
    PagedAttentionPrefillInfo info{};
    info.dtype = INFINI_DTYPE_BF16;
    info.index_dtype = INFINI_DTYPE_I64;
    info.scale = scale;
    info.num_seqs = in[0];
    info.total_q_tokens = in[1];
    info.num_heads = in[2];
    info.num_kv_heads = in[3];
    info.head_size = in[9];
    info.value_size = in[4];
    info.page_block_size = in[5];
    info.max_num_blocks_per_seq = in[6];
    info.num_blocks = 1 << 20;
    info.has_alibi = in[8] != 0;
    // packed tensors
    info.q_head_stride = in[9];
    info.q_stride = in[2] * in[9];
    info.o_head_stride = in[4];
    info.o_stride = in[2] * in[4];
    info.k_row_stride = in[9];
    info.k_head_stride = in[5] * in[9];
    info.k_batch_stride = in[3] * in[5] * in[9];
    info.v_row_stride = in[4];
    info.v_head_stride = in[5] * in[4];
    info.v_batch_stride = in[3] * in[5] * in[4];
    info.block_table_batch_stride = in[6];
    return op::paged_attention_prefill::amd::makePlan(info, device::amd::DeviceInfo{static_cast<int>(in[7]), 64, false});
}

} // namespace

// Keys of 576 (the first nine of `in`). Returns 64-row groups per workgroup, 0 if the element-wise kernel runs.
extern "C" int latentPrefillProbe(const long long *in, float scale) {
    long long all[10];
    for (int i = 0; i < 9; ++i) {
        all[i] = in[i];
    }
    all[9] = 576;
    const Plan plan = planOf(all, scale);
    return plan.tiled ? plan.groups_per_wave : 0;
}

// out: {tiled, max_parts, merge_workgroups, split_from, workspace bytes, bytes of accumulators, of pairs, of flags}; returns
// what a part costs in tokens
extern "C" float splitPrefillProbe(const long long *in, long long *out) {
    const Plan plan = planOf(in, 0.1f);
    out[0] = plan.tiled;
    out[1] = plan.max_parts;
    out[2] = plan.merge_workgroups;
    out[3] = plan.split_from;
    out[4] = static_cast<long long>(plan.workspaceBytes());
    out[5] = static_cast<long long>(plan.part_acc_bytes);
    out[6] = static_cast<long long>(plan.part_ml_bytes);
    out[7] = static_cast<long long>(plan.part_flags_bytes);
    return plan.part_cost;
}
