// Prefill calls too small to fill the device: the tokens of a row block split over several workgroups.
//
// A few new tokens over a long history are few row blocks (one per 64 rows), and a workgroup takes its steps one after
// the other: one sequence of 3 new tokens over 5 800 with 8 heads is eight workgroups of 91 steps on 256 compute units. So
// up to max_parts workgroups share a block (prefillTiledKernel, SPLIT), each from its first step to its last as if the others
// did not exist, and leave their accumulators, reference points and denominators in the workspace in fp32; further
// workgroups of the same launch merge them as the decode kernels do:
//   M = max_p m_p,  out = sum_p acc_p * 2^(m_p - M) / (sum_p l_p * 2^(m_p - M) + 1e-6)
// How many parts a block really gets is settled in the kernel, from the tokens it sees: the host only knows what the block
// table can hold, and a server hands over tables of its longest possible sequence. A block that is not worth a split is
// finished by its first workgroup, the workgroups of its other parts and of its merge leave at once, and there is no second
// launch to wait for. (A merge kernel costs 3 - 6 us more on every call whose table might hold a long sequence, prefill_plan.h;
// merging by the part that arrives last would spare the workgroups that merge, but leaves a block's rows to one of them.)
//
// Parts and merge meet as pieces and reader of the decode kernel do (decode_common.h has the accesses): a part's wavefront
// writes its rows through to memory, waits for that, and stores the call's token beside each row; the wavefront that merges
// a row polls the tokens of its parts, reads past the caches, and clears the tokens, so that a replay of the call starts
// clean. Every row that a part flags is merged, and only flagged rows are waited for: both sides
// go by partRowExists.
// Merging workgroups come last in the grid and parts wait for nobody, so alone on the device they always get their rows. Beside
// another such call, on another stream, they may not: each die takes the workgroups of its queues in its own order, and
// merging workgroups of one call can hold the places that the other's parts need on one die, and the other way round on another.
// So a merging wavefront waits for merge_polls at most. Then it marks its rows as left (part_left), looks once more, and
// goes; a part's wavefront looks for such marks after its tokens are in memory, and merges the rows that are complete. Whichever
// of the two came second sees the other's word, so every row is merged: by either, or by both from the same rows to the same
// bits. Nothing waits without bound and no row depends on who waited.
#ifndef INFINICORE_AMD_PA_PREFILL_SPLIT_H
#define INFINICORE_AMD_PA_PREFILL_SPLIT_H

#include "../../paged_attention/amd/decode_reduce.h"
#include "prefill_common.h"
#include "prefill_plan.h"

namespace op::paged_attention_prefill::amd {

constexpr int kPartRows = 64;       // rows of a split block
constexpr int kSplitTokens = 128;   // a block has a part per that many tokens, at most

// The steps of one row block as its parts take them: `per` each, `used` parts in all.
struct SplitSteps {
    int per, used;
};
// (wave-uniform; `visible`: the tokens that the block sees, in n_steps steps)
__device__ __forceinline__ SplitSteps splitSteps(const PrefillArgs &a, int visible, int n_steps) {
    int parts = 1;
    if (visible >= a.split_from) { // (the same comparison that says whether a batch has any block to split)
        // P parts take a P-th of the walk and cost P times part_cost tokens of it: least at P = sqrt(visible / part_cost)
        const float best = __builtin_amdgcn_sqrtf(static_cast<float>(visible) * a.part_cost); // tokens per part
        const int each = max(static_cast<int>(best), kSplitTokens);
        parts = __builtin_amdgcn_readfirstlane(min(min(a.max_parts, n_steps), (visible + each - 1) / each));
    }
    SplitSteps s;
    s.per = (n_steps + parts - 1) / parts;
    s.used = (n_steps + s.per - 1) / s.per;
    return s;
}

// Rows that parts leave and a merge reads.
__device__ __forceinline__ bool partRowExists(int row, int last_row, int visible) { return row <= last_row && visible > 0; }

// First row of a part of a row block, of all parts in the workspace.
__device__ __forceinline__ int64_t partFirstRow(const PrefillArgs &a, int block_index, int kv_head, int part) {
    return ((static_cast<int64_t>(block_index) * a.num_kv_heads + kv_head) * a.max_parts + part) * kPartRows;
}

// One wavefront's 16 rows (from `row0` of the block on) of a part go to the workspace. Lane (g, c): o[e][rr] and l[rr] of
// row 4 g + rr, column 16 e + c; m (log2) of row c, which exists where `exists`. Accumulators of four column blocks go out
// together: chunk 16 h + c of a row holds those of blocks 4 h .. 4 h + 3 (columns 64 h + c, + 16, + 32, + 48).
template <int VHEAD, typename Acc>
__device__ __forceinline__ void publishPart(const PrefillArgs &a, int64_t row0, const Acc *o, const Acc &l, float m, bool exists, int lane) {
    using namespace op::paged_attention::amd;
    const int c = lane & 15, g = lane >> 4;
    const unsigned long long wanted = __builtin_amdgcn_ballot_w64(exists); // bit c: row c
    const auto rows = agentBuffer(a.part_acc + row0 * VHEAD, 16 * VHEAD * 4);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        if ((wanted >> (4 * g + rr)) & 1) {
#pragma unroll
            for (int h = 0; h < VHEAD / 64; ++h) {
                storeAgent16(rows, ((4 * g + rr) * VHEAD + 64 * h + 4 * c) * 4, o[4 * h][rr], o[4 * h + 1][rr], o[4 * h + 2][rr],
                             o[4 * h + 3][rr]);
            }
        }
    }
    float l_row = 0.0f; // of row c: lanes of group c / 4 have it
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const float x = __shfl(l[rr], 16 * (c >> 2), 64);
        l_row = (c & 3) == rr ? x : l_row;
    }
    const bool mine = g == 0 && exists;
    if (mine) {
        storeAgent8(agentBuffer(a.part_ml + row0, 16 * 8), 8 * c, m, l_row);
    }
    waitVectorMemory(); // the rows are in memory
    if (mine) {
        storeAgent(a.part_flags + row0 + c, a.token);
    }
}

__device__ __forceinline__ unsigned long long *leftMarks(const PrefillArgs &a, int block_index, int kv_head) {
    return a.part_left + (static_cast<int64_t>(block_index) * a.num_kv_heads + kv_head) * kMergeWavefronts;
}

// One wavefront merges its rows of a split block: wave, wave + waves, .. of all that exist, two at a time. With WAITS it is
// that wavefront of the merging workgroups; else a part's in its place, which takes the rows that are complete. A part's row is
// VHEAD / 4 chunks of 16 bytes; up to head 128 several parts' rows fit the lanes of one load. The code is kept short: it
// runs once or a few times per launch, out of a cold instruction cache (all rows of a wavefront unrolled: twice as long).
template <typename T, int VHEAD, bool WAITS>
__device__ __forceinline__ void mergeParts(const PrefillArgs &a, const SeqSpan &span, int block_index, int kv_head, int block_row0,
                                           int last_row, int wave, int waves, SplitSteps split, int step_tokens, int lane) {
    using namespace op::paged_attention::amd;
    using S = typename T::storage;
    constexpr int N = 2; // rows at once
    constexpr int kChunks = VHEAD / 4;
    constexpr int kSide = kChunks <= 32 ? 64 / kChunks : 1; // parts beside one another in a load: 4, 2 or 1
    constexpr int kMine = (kChunks + 63) / 64;              // chunks of a lane
    constexpr int kInFlight = kMine == 1 ? 8 / (kSide > 2 ? 2 : 1) : (kMine == 2 ? 4 : 2); // loads per row and chunk
    const int64_t part0 = partFirstRow(a, block_index, kv_head, 0);
    unsigned long long *const flags = a.part_flags + part0; // of part p and row r of the block: [64 p + r]
    const auto pairs = agentBuffer(a.part_ml + part0, split.used * kPartRows * 8);
    const auto sums = agentBuffer(a.part_acc + part0 * VHEAD, split.used * kPartRows * VHEAD * 4);
    const int side = kSide > 1 ? lane / kChunks : 0;
    const int chunk = kSide > 1 ? lane % kChunks : lane;
    const int part_tokens = split.per * step_tokens;
    unsigned long long *const mark = leftMarks(a, block_index, kv_head) + wave;
    bool left = !WAITS; // the rows may be merged by somebody else as well
    if (WAITS && lane == 0) {
        storeAgent(mark, 0); // (a replay that left rows)
    }

    for (int first_row = wave; first_row < kPartRows; first_row += N * waves) {
        int token[N], head[N], seen[N]; // seen: parts that the row sees any token of
        bool exists[N], any = false;
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const int row = block_row0 + first_row + n * waves;
            token[n] = row / a.group;
            head[n] = kv_head * a.group + (row - token[n] * a.group);
            const int visible = visibleTokens(span, token[n]);
            exists[n] = first_row + n * waves < kPartRows && partRowExists(row, last_row, visible);
            seen[n] = min(split.used, (visible + part_tokens - 1) / part_tokens);
            any |= exists[n];
        }
        if (!any) {
            return; // nor any row behind
        }
        bool complete = false;
        for (int polls = 0;; ++polls) {
            bool here = true;
#pragma unroll
            for (int n = 0; n < N; ++n) {
                if (exists[n] && lane < split.used) {
                    here = here && loadAgent(flags + kPartRows * lane + first_row + n * waves) == a.token;
                }
            }
            complete = __builtin_amdgcn_ballot_w64(!here) == 0;
            if (complete || left) {
                break;
            }
            if (polls >= a.merge_polls) {
                left = true;
                if (lane == 0) {
                    storeAgent(mark, a.token);
                }
                waitVectorMemory(); // the mark is in memory before the last look
            } else {
                __builtin_amdgcn_s_sleep(1);
            }
        }
        if (!complete) {
            continue; // the part that completes them finds the mark; or somebody has merged them
        }
        compilerMemoryBarrier(); // the loads below stay below the flag loads above
        float2 ml[N];
        float4 sum[N][kMine];
#pragma unroll
        for (int n = 0; n < N; ++n) {
            ml[n] = loadAgent8(pairs, (kPartRows * lane + first_row + n * waves) * 8); // lane p: part p
#pragma unroll
            for (int k = 0; k < kMine; ++k) {
                sum[n][k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
        float weight[N], l[N];
        for (int p0 = 0; p0 < split.used; p0 += kInFlight * kSide) {
            float4 x[N][kInFlight][kMine];
#pragma unroll
            for (int n = 0; n < N; ++n) {
#pragma unroll
                for (int i = 0; i < kInFlight; ++i) {
#pragma unroll
                    for (int k = 0; k < kMine; ++k) {
                        // (past the last part, or past the row's chunks: beyond the buffer, or not used)
                        const int p = p0 + i * kSide + side;
                        x[n][i][k] = loadAgent16(sums, ((kPartRows * p + first_row + n * waves) * kChunks + chunk + 64 * k) * 16);
                    }
                }
            }
            if (p0 == 0) {
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    const float m = lane < seen[n] ? ml[n].x : -INFINITY;
                    weight[n] = mergeWeight(m, laneMax(m));
                    l[n] = laneSum(lane < seen[n] ? ml[n].y * weight[n] : 0.0f);
                }
            }
#pragma unroll
            for (int n = 0; n < N; ++n) {
#pragma unroll
                for (int i = 0; i < kInFlight; ++i) {
                    const int p = p0 + i * kSide + side;
                    float f = laneOf(weight[n], p0 + i * kSide);
#pragma unroll
                    for (int other = 1; other < kSide; ++other) {
                        f = side == other ? laneOf(weight[n], p0 + i * kSide + other) : f;
                    }
                    // Parts that the row sees nothing of are left out, whatever they hold (0 times an infinity in V is
                    // NaN); in the others a weight of 0 counts, as in a block that is not split.
                    const bool counts = p < seen[n];
#pragma unroll
                    for (int k = 0; k < kMine; ++k) {
                        sum[n][k].x += counts ? x[n][i][k].x * f : 0.0f;
                        sum[n][k].y += counts ? x[n][i][k].y * f : 0.0f;
                        sum[n][k].z += counts ? x[n][i][k].z * f : 0.0f;
                        sum[n][k].w += counts ? x[n][i][k].w * f : 0.0f;
                    }
                }
            }
        }
#pragma unroll
        for (int n = 0; n < N; ++n) {
            if constexpr (kSide > 1) {
#pragma unroll
                for (int off = kChunks; off < 64; off <<= 1) {
                    sum[n][0].x += __shfl_xor(sum[n][0].x, off, 64);
                    sum[n][0].y += __shfl_xor(sum[n][0].y, off, 64);
                    sum[n][0].z += __shfl_xor(sum[n][0].z, off, 64);
                    sum[n][0].w += __shfl_xor(sum[n][0].w, off, 64);
                }
            }
            if (!exists[n]) {
                continue;
            }
            const float inv_l = 1.0f / (l[n] + 1e-6f);
            unsigned short *o_ptr = reinterpret_cast<unsigned short *>(static_cast<S *>(a.out) + (span.q_start + token[n]) * a.o_stride + head[n] * a.o_head_stride);
#pragma unroll
            for (int k = 0; k < kMine; ++k) {
                const int q = chunk + 64 * k; // columns 64 (q / 16) + q % 16, + 16, + 32, + 48
                if (side == 0 && q < kChunks) {
                    unsigned short *o = o_ptr + 64 * (q >> 4) + (q & 15);
                    o[0] = static_cast<unsigned short>(T::packProducts(sum[n][k].x, 0.0f, inv_l));
                    o[16] = static_cast<unsigned short>(T::packProducts(sum[n][k].y, 0.0f, inv_l));
                    o[32] = static_cast<unsigned short>(T::packProducts(sum[n][k].z, 0.0f, inv_l));
                    o[48] = static_cast<unsigned short>(T::packProducts(sum[n][k].w, 0.0f, inv_l));
                }
            }
            if (lane < split.used) { // consumed: a replay of this call (same token) starts clean
                storeAgent(flags + kPartRows * lane + first_row + n * waves, 0);
            }
        }
    }
}

// A part's wavefront, its rows published: the rows that merging wavefronts of this block have left.
template <typename T, int VHEAD>
__device__ __forceinline__ void mergeLeftRows(const PrefillArgs &a, const SeqSpan &span, int block_index, int kv_head, int block_row0,
                                              int last_row, SplitSteps split, int step_tokens, int lane) {
    using namespace op::paged_attention::amd;
    const int waves = 4 * a.merge_workgroups;
    waitVectorMemory(); // this wavefront's tokens are in memory before it looks for marks
    unsigned long long marked = __builtin_amdgcn_ballot_w64(lane < waves && loadAgent(leftMarks(a, block_index, kv_head) + lane) == a.token);
    while (marked != 0) {
        const int wave = __builtin_ctzll(marked);
        marked &= marked - 1;
        mergeParts<T, VHEAD, false>(a, span, block_index, kv_head, block_row0, last_row, wave, waves, split, step_tokens, lane);
    }
}

} // namespace op::paged_attention_prefill::amd

#endif
