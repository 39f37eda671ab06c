// Prefill calls too small to fill the device: the tokens of a row block split over several workgroups.
//
// A few new tokens over a long history are few row blocks (one per 64 rows), and a workgroup takes its steps one after
// the other: one sequence of 3 new tokens over 5 800 with 8 heads is eight workgroups of 91 steps on 256 compute units. So
// max_parts workgroups share a block (prefillTiledKernel, SPLIT), each from its first step to its last as if the others did
// not exist, and leave their accumulators, reference points and denominators in the workspace in fp32; the kernel here
// merges them as the decode kernels do:
//   M = max_p m_p,  out = sum_p acc_p * 2^(m_p - M) / (sum_p l_p * 2^(m_p - M) + 1e-6)
// Blocks with fewer than two parts' worth of tokens are finished by the first kernel.
// A part pays a workgroup's start (three dependent round trips) and its rows (32 KiB at head 128, if all 64 exist), so no
// part but the last is below 128 tokens: one sequence of 3 tokens over 600, 13.2 us with at least 256, 11.1 with 128.
// The walk of a part is bound by one workgroup's dependent steps as before (~0.9 us per 64 tokens at head 128, alone on its
// unit); how many parts, and what that measured, is at splitParts in prefill_plan.h.
#ifndef INFINICORE_AMD_PA_PREFILL_SPLIT_H
#define INFINICORE_AMD_PA_PREFILL_SPLIT_H

#include "../../paged_attention/amd/decode_reduce.h"
#include "prefill_tiled.h"

namespace op::paged_attention_prefill::amd {

constexpr int kMergeThreads = 256;
constexpr int kMergeRows = kMergeThreads / 64; // rows of a workgroup, a wavefront each

// Grid: row blocks x KV heads as in prefillTiledKernel, then 64 / kMergeRows. A wavefront reads a part's row with one
// instruction per 64 columns; the weights are formed by the lanes, a part each (max_parts <= 64).
template <typename T, typename Tindex, int KHEAD, int VHEAD>
__global__ void __launch_bounds__(kMergeThreads) prefillMergeKernel(PrefillArgs a) {
    using S = typename T::storage;
    using op::paged_attention::amd::mergeWeight;
    using op::paged_attention::amd::waveMax;
    using op::paged_attention::amd::waveSum;
    constexpr int BM = prefillBlockRows(1);
    constexpr int BN = prefillStepTokens<KHEAD, 1>();
    constexpr int kCols = VHEAD / 64;

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kv_head = blockIdx.x % a.num_kv_heads;
    const int block_index = blockIdx.x / a.num_kv_heads;
    int seq = 0, block = 0;
    SeqSpan span;
    if (!findRowBlock<Tindex>(a, lane, BM, block_index, seq, block, span)) {
        return;
    }
    const int total_rows = span.q_len * a.group;
    const int block_row0 = block * BM;
    const int last_row = min(block_row0 + BM, total_rows) - 1;
    const int block_visible = visibleTokens(span, last_row / a.group);
    const int local_row = blockIdx.y * kMergeRows + w;
    const int row = block_row0 + local_row;
    if (block_visible <= 0 || row > last_row) {
        return;
    }
    const int parts = splitSteps((block_visible + BN - 1) / BN, BN, a.max_parts).used;
    const int token = row / a.group;
    if (parts <= 1 || visibleTokens(span, token) <= 0) {
        return;
    }
    const int64_t part0 = (static_cast<int64_t>(block_index) * a.num_kv_heads + kv_head) * a.max_parts;
    float2 ml = make_float2(-INFINITY, 0.0f);
    if (lane < parts) {
        ml = a.part_ml[(part0 + lane) * BM + local_row];
    }
    const float weight = mergeWeight(ml.x, waveMax(ml.x));
    const float l = waveSum(ml.y * weight);
    float sum[kCols];
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        sum[i] = 0.0f;
    }
    const float *acc = a.part_acc + (part0 * BM + local_row) * VHEAD + lane;
    constexpr int kInFlight = 4; // parts; divides kMaxSplitParts, so that lanes past the last part exist and weigh nothing
    for (int p = 0; p < parts; p += kInFlight) {
        float x[kInFlight][kCols];
#pragma unroll
        for (int n = 0; n < kInFlight; ++n) {
#pragma unroll
            for (int i = 0; i < kCols; ++i) {
                x[n][i] = acc[static_cast<int64_t>(min(p + n, parts - 1)) * BM * VHEAD + 64 * i];
            }
        }
#pragma unroll
        for (int n = 0; n < kInFlight; ++n) {
            const float f = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), p + n));
#pragma unroll
            for (int i = 0; i < kCols; ++i) {
                sum[i] += f == 0.0f ? 0.0f : x[n][i] * f; // a part the row sees nothing of: V may hold anything there
            }
        }
    }
    const float inv_l = 1.0f / (l + 1e-6f);
    const int head = kv_head * a.group + (row - token * a.group);
    unsigned short *o_ptr = reinterpret_cast<unsigned short *>(static_cast<S *>(a.out) + (span.q_start + token) * a.o_stride + head * a.o_head_stride) + lane;
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        o_ptr[64 * i] = static_cast<unsigned short>(T::pack2(sum[i] * inv_l, 0.0f));
    }
}

} // namespace op::paged_attention_prefill::amd

#endif
