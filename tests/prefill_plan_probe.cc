// Test-only view of the prefill launch plan
// (infinicore_amd/csrc/infiniop/ops/paged_attention_prefill/amd/prefill_plan.h): compiled with the host compiler by
// tests/test_prefill_plan.py, no GPU and no HIP needed.
#include "infiniop/ops/paged_attention_prefill/amd/prefill_plan.h"

// in: {num_seqs, total_q_tokens, num_heads, num_kv_heads, value_size, block_size, max_blocks_per_seq, compute_units,
//      has_alibi}; keys of 576. Returns 64-row groups per workgroup, 0 if the element-wise kernel runs.
extern "C" int latentPrefillProbe(const long long *in, float scale) {
    using namespace op::paged_attention_prefill;
    PagedAttentionPrefillInfo info{};
    info.dtype = INFINI_DTYPE_BF16;
    info.index_dtype = INFINI_DTYPE_I64;
    info.scale = scale;
    info.num_seqs = in[0];
    info.total_q_tokens = in[1];
    info.num_heads = in[2];
    info.num_kv_heads = in[3];
    info.head_size = 576;
    info.value_size = in[4];
    info.page_block_size = in[5];
    info.max_num_blocks_per_seq = in[6];
    info.num_blocks = 1 << 20;
    info.has_alibi = in[8] != 0;
    // packed tensors
    info.q_head_stride = 576;
    info.q_stride = in[2] * 576;
    info.o_head_stride = in[4];
    info.o_stride = in[2] * in[4];
    info.k_row_stride = 576;
    info.k_head_stride = in[5] * 576;
    info.k_batch_stride = in[3] * in[5] * 576;
    info.v_row_stride = in[4];
    info.v_head_stride = in[5] * in[4];
    info.v_batch_stride = in[3] * in[5] * in[4];
    info.block_table_batch_stride = in[6];
    const device::amd::DeviceInfo dev{static_cast<int>(in[7]), 64, false};
    const amd::Plan plan = amd::makePlan(info, dev);
    return plan.tiled ? plan.groups_per_wave : 0;
}
