// paged_attention_prefill on AMD Instinct MI355X: descriptor, kernel choice and launches.
// Takes the place of the reference's nvidia backend host code
// (src/infiniop/ops/paged_attention_prefill/nvidia/paged_attention_prefill_nvidia.cu:1572-1886)
// for the AMD device.
#include "paged_attention_prefill_amd.h"
#include "../../../handle.h"
#include "../../../../utils/check.h"
#include "../../../devices/amd/amd_device.h"
#include "prefill_common.h"
#include "prefill_generic.h"
#include "prefill_latent.h"
#include "prefill_plan.h"
#include "prefill_tiled.h"

namespace op::paged_attention_prefill::amd {

namespace {

using op::paged_attention::amd::BFloat16;
using op::paged_attention::amd::Half;
using op::paged_attention::amd::IndexI32;
using op::paged_attention::amd::IndexI64;
using op::paged_attention::amd::IndexU32;

template <typename T, typename Tindex>
void launchGeneric(const PrefillArgs &a, const Plan &plan, hipStream_t stream) {
    const dim3 grid(a.total_q_tokens, a.num_heads);
    switch (plan.dims_per_lane) {
    case 1: prefillGenericKernel<T, Tindex, 1><<<grid, 64, 0, stream>>>(a); break;
    case 2: prefillGenericKernel<T, Tindex, 2><<<grid, 64, 0, stream>>>(a); break;
    case 3: prefillGenericKernel<T, Tindex, 3><<<grid, 64, 0, stream>>>(a); break;
    case 4: prefillGenericKernel<T, Tindex, 4><<<grid, 64, 0, stream>>>(a); break;
    default: prefillGenericKernel<T, Tindex, 9><<<grid, 64, 0, stream>>>(a); break;
    }
}

template <typename T, typename Tindex, int KHEAD, int VHEAD, bool PLAIN>
void launchTiledHead(const PrefillArgs &args, const Plan &plan, hipStream_t stream) {
    PrefillArgs a = args;
    // sum over sequences of ceil(rows / block_rows) is at most floor(total rows / block_rows) + num_seqs
    const long long rows = static_cast<long long>(a.total_q_tokens) * a.group;
    const int groups = KHEAD == 576 && !PLAIN ? 1 : plan.groups_per_wave; // slopes handed over unannounced
    const int block_rows = prefillBlockRows(groups);
    static_assert(prefillBlockRows(2) == kLatentRows);
    const dim3 grid(static_cast<unsigned>((rows / block_rows + a.num_seqs) * a.num_kv_heads));
    const int resident = groups == 2 ? prefillWorkgroupsPerUnit<KHEAD, 2>() : prefillWorkgroupsPerUnit<KHEAD, 1>();
    const unsigned slots = static_cast<unsigned>(plan.compute_units * resident);
    a.longest_first = longestFirst<KHEAD>(grid.x, slots) ? 1 : 0;
    a.slots = slots;
    if constexpr (KHEAD == VHEAD && KHEAD <= 256) {
        if (groups == 2) {
            prefillTiledKernel<T, Tindex, KHEAD, VHEAD, 2, PLAIN><<<grid, kPrefillThreads, 0, stream>>>(a);
            return;
        }
    }
    if constexpr (KHEAD == 576 && VHEAD == 512 && PLAIN) {
        if (groups == 2) {
            prefillLatentKernel<T, Tindex><<<grid, kLatentThreads, 0, stream>>>(a);
            return;
        }
    }
    if (a.max_parts > 1) {
        a.row_blocks = static_cast<int32_t>(grid.x / static_cast<unsigned>(a.num_kv_heads));
        a.part_workgroups = grid.x * static_cast<unsigned>(a.max_parts);
        const dim3 all(a.part_workgroups + grid.x * static_cast<unsigned>(a.merge_workgroups));
        prefillTiledKernel<T, Tindex, KHEAD, VHEAD, 1, PLAIN, true><<<all, kPrefillThreads, 0, stream>>>(a);
        return;
    }
    prefillTiledKernel<T, Tindex, KHEAD, VHEAD, 1, PLAIN><<<grid, kPrefillThreads, 0, stream>>>(a);
}

template <typename T, typename Tindex, bool PLAIN>
void launchTiledPlain(const PrefillArgs &a, const Plan &plan, hipStream_t stream) {
    switch (a.head_size) {
    case 64: launchTiledHead<T, Tindex, 64, 64, PLAIN>(a, plan, stream); break;
    case 128: launchTiledHead<T, Tindex, 128, 128, PLAIN>(a, plan, stream); break;
    case 192: launchTiledHead<T, Tindex, 192, 192, PLAIN>(a, plan, stream); break;
    case 256: launchTiledHead<T, Tindex, 256, 256, PLAIN>(a, plan, stream); break;
    default:
        if (a.value_size == 576) {
            launchTiledHead<T, Tindex, 576, 576, PLAIN>(a, plan, stream);
        } else {
            launchTiledHead<T, Tindex, 576, 512, PLAIN>(a, plan, stream);
        }
        break;
    }
}

template <typename T, typename Tindex>
void launchTiled(const PrefillArgs &a, const Plan &plan, hipStream_t stream) {
    if (a.alibi_slopes == nullptr && a.scale_log2 > 0.0f) {
        launchTiledPlain<T, Tindex, true>(a, plan, stream);
    } else {
        launchTiledPlain<T, Tindex, false>(a, plan, stream);
    }
}

template <typename T>
infiniStatus_t launchByIndex(infiniDtype_t index_dtype, const PrefillArgs &a, const Plan &plan, bool tiled,
                             hipStream_t stream) {
    switch (index_dtype) {
    case INFINI_DTYPE_I64:
        tiled ? launchTiled<T, IndexI64>(a, plan, stream) : launchGeneric<typename T::Base, IndexI64>(a, plan, stream);
        break;
    case INFINI_DTYPE_I32:
        tiled ? launchTiled<T, IndexI32>(a, plan, stream) : launchGeneric<typename T::Base, IndexI32>(a, plan, stream);
        break;
    case INFINI_DTYPE_U32:
        tiled ? launchTiled<T, IndexU32>(a, plan, stream) : launchGeneric<typename T::Base, IndexU32>(a, plan, stream);
        break;
    default: return INFINI_STATUS_BAD_TENSOR_DTYPE;
    }
    return INFINI_STATUS_SUCCESS;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

} // namespace

struct Descriptor::Opaque {
    Plan plan;
};

Descriptor::~Descriptor() { delete _opaque; }

infiniStatus_t Descriptor::create(infiniopHandle_t handle, Descriptor **desc_ptr, infiniopTensorDescriptor_t out_desc,
                                  infiniopTensorDescriptor_t q_desc, infiniopTensorDescriptor_t k_cache_desc,
                                  infiniopTensorDescriptor_t v_cache_desc, infiniopTensorDescriptor_t block_tables_desc,
                                  infiniopTensorDescriptor_t seq_lens_desc, infiniopTensorDescriptor_t cum_seq_lens_q_desc,
                                  infiniopTensorDescriptor_t alibi_slopes_desc, float scale) {
    auto info = PagedAttentionPrefillInfo::create(out_desc, q_desc, k_cache_desc, v_cache_desc, block_tables_desc,
                                                  seq_lens_desc, cum_seq_lens_q_desc, alibi_slopes_desc, scale);
    CHECK_RESULT(info);
    const PagedAttentionPrefillInfo in = info.take();
    const Plan plan = makePlan(in, device::amd::deviceInfo(handle->device_id));
    // Scratch for the partial results of split row blocks, with 256 spare bytes to align it; 0 where none are split: a row
    // block then keeps its softmax state in registers from the first to the last K/V token.
    *desc_ptr = new Descriptor(new Opaque{plan}, in, plan.workspaceBytes(), handle->device, handle->device_id);
    return INFINI_STATUS_SUCCESS;
}

infiniStatus_t Descriptor::calculate(void *workspace, size_t workspace_size, void *out, const void *q,
                                     const void *k_cache, const void *v_cache, const void *block_tables,
                                     const void *seq_lens, const void *cum_seq_lens_q, const void *alibi_slopes,
                                     void *stream_) const {
    const PagedAttentionPrefillInfo &in = _info;
    const Plan &plan = _opaque->plan;
    if (in.num_seqs == 0 || in.num_heads == 0 || in.total_q_tokens == 0) {
        return INFINI_STATUS_SUCCESS;
    }
    if (out == nullptr || q == nullptr || k_cache == nullptr || v_cache == nullptr || block_tables == nullptr
        || seq_lens == nullptr || cum_seq_lens_q == nullptr) {
        return INFINI_STATUS_NULL_POINTER;
    }
    if (in.has_alibi && alibi_slopes == nullptr) {
        return INFINI_STATUS_NULL_POINTER;
    }
    if (in.max_num_blocks_per_seq == 0 || in.num_blocks == 0 || in.page_block_size == 0) {
        return INFINI_STATUS_SUCCESS; // no sequence can hold a token
    }
    if (in.total_q_tokens > 0x7fffffff || in.num_seqs > 0x7fffffff || in.num_heads > 65535) {
        return INFINI_STATUS_BAD_TENSOR_SHAPE;
    }

    PrefillArgs a{};
    a.out = out;
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.block_tables = block_tables;
    a.kv_lens = seq_lens;
    a.cu_seqlens_q = cum_seq_lens_q;
    a.alibi_slopes = static_cast<const float *>(alibi_slopes);
    a.scale_log2 = in.scale * kLog2e;
    a.num_seqs = static_cast<int32_t>(in.num_seqs);
    a.total_q_tokens = static_cast<int32_t>(in.total_q_tokens);
    a.num_heads = static_cast<int32_t>(in.num_heads);
    a.num_kv_heads = static_cast<int32_t>(in.num_kv_heads);
    a.group = static_cast<int32_t>(in.num_heads / in.num_kv_heads);
    a.head_size = static_cast<int32_t>(in.head_size);
    a.value_size = static_cast<int32_t>(in.value_size);
    a.block_size = static_cast<int32_t>(in.page_block_size);
    a.block_shift = -1;
    if ((in.page_block_size & (in.page_block_size - 1)) == 0) {
        a.block_shift = __builtin_ctzll(in.page_block_size);
    }
    a.num_blocks = static_cast<int32_t>(in.num_blocks > 0x7fffffff ? 0x7fffffff : in.num_blocks);
    a.max_blocks_per_seq = static_cast<int32_t>(in.max_num_blocks_per_seq > 0x7fffffff ? 0x7fffffff : in.max_num_blocks_per_seq);
    a.q_stride = in.q_stride;
    a.q_head_stride = in.q_head_stride;
    a.o_stride = in.o_stride;
    a.o_head_stride = in.o_head_stride;
    a.k_batch_stride = in.k_batch_stride;
    a.k_head_stride = in.k_head_stride;
    a.k_row_stride = in.k_row_stride;
    a.v_batch_stride = in.v_batch_stride;
    a.v_head_stride = in.v_head_stride;
    a.v_row_stride = in.v_row_stride;
    a.block_table_batch_stride = in.block_table_batch_stride;

    // The tiled kernel moves 16 bytes per lane; base addresses that are not 16-byte aligned take
    // the element-wise kernel instead.
    a.max_parts = 1;
    if (plan.max_parts > 1 && workspace != nullptr && workspace_size >= _workspace_size) {
        const size_t left_marks = static_cast<size_t>(plan.row_block_grid) * kMergeWavefronts; // behind the tokens
        char *ws = reinterpret_cast<char *>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~static_cast<uintptr_t>(255));
        a.part_acc = reinterpret_cast<float *>(ws);
        a.part_ml = reinterpret_cast<float2 *>(ws + plan.part_acc_bytes);
        a.part_flags = reinterpret_cast<unsigned long long *>(ws + plan.part_acc_bytes + plan.part_ml_bytes);
        a.part_left = a.part_flags + (plan.part_flags_bytes / sizeof(unsigned long long) - left_marks);
        a.token = device::amd::nextToken();
        a.max_parts = plan.max_parts;
        a.merge_workgroups = plan.merge_workgroups;
        a.merge_polls = plan.merge_polls;
        a.split_from = plan.split_from;
        a.part_cost = plan.part_cost;
    } // without the workspace it asks for, the call runs unsplit
    const bool tiled = plan.tiled && aligned16(out) && aligned16(q) && aligned16(k_cache) && aligned16(v_cache);
    auto stream = static_cast<hipStream_t>(stream_);

    infiniStatus_t status;
    if (in.dtype == INFINI_DTYPE_F16) {
        status = launchByIndex<TileF16>(in.index_dtype, a, plan, tiled, stream);
    } else {
        status = launchByIndex<TileBF16>(in.index_dtype, a, plan, tiled, stream);
    }
    if (status != INFINI_STATUS_SUCCESS) {
        return status;
    }
    return hipGetLastError() == hipSuccess ? INFINI_STATUS_SUCCESS : INFINI_STATUS_INTERNAL_ERROR;
}

} // namespace op::paged_attention_prefill::amd
