// Launch plan of the paged-attention prefill on AMD Instinct MI355X: which kernel runs, with how many rows per
// workgroup. Host-only code without any HIP dependency, so that the arithmetic can be exercised on a machine
// without a GPU.
#ifndef INFINICORE_AMD_PA_PREFILL_PLAN_H
#define INFINICORE_AMD_PA_PREFILL_PLAN_H

#include "../../../devices/amd/amd_device.h"
#include "../info.h"
#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace op::paged_attention_prefill::amd {

// Decided once, at descriptor creation, from shapes and the device alone (sequence lengths live in
// device memory and are never read on the host).
struct Plan {
    bool tiled;          // matrix-core kernel (head 64 / 128 / 192 / 256 or keys 576 with values 512 / 576, power-of-two pages >= 8, 16-byte aligned strides)
    int groups_per_wave; // tiled: R = 1 or 2 -> 64 R rows per workgroup (R column groups of each of four wavefronts; latent attention with R = 2: one of each of eight)
    int compute_units;
    int max_parts;       // tiled, 64 rows: workgroups that may share a row block (prefill_split.h); 1 = none is split
    int merge_workgroups; // of a row block: 1, 2, 4 or 8
    long long row_block_grid; // row blocks x KV heads that the batch can have
    int merge_polls;     // of a wavefront that merges, before it leaves its rows to the parts (prefill_split.h)
    int split_from;      // tokens from which a row block is split, and what a further part costs in tokens (PrefillArgs)
    float part_cost;
    size_t part_acc_bytes, part_ml_bytes, part_flags_bytes; // workspace of the parts, each a multiple of 256 bytes
    size_t workspaceBytes() const { return max_parts > 1 ? part_acc_bytes + part_ml_bytes + part_flags_bytes + 256 : 0; }
    int dims_per_lane;   // element-wise kernel: ceil(max(head_size, value_size) / 64)
};

inline bool multipleOf8(ptrdiff_t x) { return (x % 8) == 0; }

// Latent attention (keys of 576): 64 or 128 rows per workgroup, as 1 or 2. One workgroup per compute unit with either
// kernel, and one of 128 rows (prefill_latent.h) takes 1.4 x as long as one of 64 over the same tokens. So 128 rows where
// they save more than a third of the rounds of workgroups. Measured with the longest blocks first (prefill_tiled.h), us with
// 64 rows / with 128, by 64-row blocks (16 heads, bf16, 256 compute units):
//   * three rounds against two: 640 blocks over 2 000 tokens of history 317 / 295, 740 303 / 292; 64 sequences of 40
//     without history 36 / 37; 16 of 60 - 260 without history 44.6 / 43.4, over 500 - 4 000 311 / 268; six of 200 - 750 over up
//     to 3 000 234 / 206. The line was drawn where blocks started as the sequences come (312 / 320 and 330 / 340 then); in this
//     order 128 rows would be the better ones for most of these
//   * four against two: 1 000 over 2 000 409 / 310, over 500 150 / 119; 16 sequences of 200 without history 58 / 48, four
//     of 900 114 / 90, 16 of 100 - 380 over 500 - 4 000 435 / 350; five against three: 100 sequences of 50 75 / 63, 40 of 30 -
//     190 over up to 3 000 357 / 291
//   * two rounds against one: the second round is short where a block's tokens grow along the sequence (the longest blocks
//     start first, the last ones fit behind the shortest of the first round) or where sequences differ in length, and
//     then 128 rows only make the longest block longer. One sequence without history, 275 blocks 60 / 85, 500 112 / 141; two
//     of 900 59 / 72; four of 128 - 512 over 1 024 - 8 192 423 / 502. With much history and equal lengths it is a whole
//     round: four of 500 over 2 000 221 / 178. The lengths of several sequences are not known here: 64 rows. For one
//     sequence the table says how much history there can be, and its blocks are dealt in order: block 256 + j starts when
//     block 256 - j ends, after 2 history + 2 n (1 - 256 / blocks) tokens of n new ones in all, against 1.4 (history + n).
//     1 600 over 1 200: 180 / 191, over 3 000 334 / 300; 2 000 over 1 000 199 / 202, over 2 000 283 / 265. (A table wider
//     than the sequence looks like history.)
inline int latentRowGroups(const PagedAttentionPrefillInfo &in, const device::amd::DeviceInfo &dev, long long rows_per_seq) {
    const long long units = dev.compute_units > 0 ? dev.compute_units : 1;
    const long long seqs = in.num_seqs > 0 ? static_cast<long long>(in.num_seqs) : 1;
    const long long streams = seqs * static_cast<long long>(in.num_kv_heads);
    const long long blocks = streams * ((rows_per_seq + 63) / 64);
    const long long rounds64 = (blocks + units - 1) / units;
    const long long rounds128 = (streams * ((rows_per_seq + 127) / 128) + units - 1) / units;
    if (rounds64 == 2 && rounds128 == 1) {
        const double n = static_cast<double>(in.total_q_tokens);
        const double history = std::max(0.0, static_cast<double>(in.max_num_blocks_per_seq) * in.page_block_size - n);
        return seqs == 1 && 2 * history + 2 * n * (blocks - units) / blocks > 1.4 * (history + n) ? 2 : 1;
    }
    return 2 * rounds64 > 3 * rounds128 ? 2 : 1;
}

constexpr int kMergeWavefronts = 32; // that merge a block, at most: eight workgroups of four
// ~1 us each, 2 ms in all: far beyond the time between the parts of a call that has the device for itself (a walk of
// 16 384 tokens in two parts takes 0.1 ms, latent 0.35)
constexpr int kMergePolls = 2000;
constexpr int kMaxSplitParts = 64; // the merge forms the weights of a row with a lane per part
constexpr long long kSplitTableTokens = 128; // a part per that many tokens at most (kSplitTokens of prefill_split.h)

// How many workgroups may share the tokens of a row block of 64 rows, and what the kernel needs to settle how many do.
// Unsplit, a call that leaves compute units idle takes as long as its longest block: `walk` microseconds for the tokens it
// sees (measured with one block per KV head over 5 800 tokens). P parts take a P-th of that (1.4 times that where two of
// them share a unit), 2.9 us to meet, and 0.3 us per MB of rows that they leave and that are read back. The host knows what
// the table can hold, not the lengths: it picks the P of the longest walk (among those the device holds beside one another)
// if that takes a fifth off it, and hands on the tokens from which a block gains at all and what a part costs, so that
// the kernel leaves short blocks whole and cuts middling ones into fewer parts (splitSteps).
// Measured, us (bf16; 32 / 8 heads of 128 unless said otherwise), never split / on a table as wide as the sequence / on one
// of 32 768 tokens; in brackets the latter two with a merge kernel of its own, which was launched wherever the table was wide:
//   * one sequence, 3 tokens over 2 000: 33.5 / 10.0 / 9.9 (12.0, 11.8); 100 over 2 000: 37.1 / 18.4 / 18.2 (20.0, 17.8); four
//     of 64 over 5 000: 83 / 42 / 42 (42, 41); 16 of 5 over 2 000: 34.9 / 29.7 / 29.5 (28.5, 28.1)
//   * 16 heads of 64, four of 64 over 2 000: 31.3 / 17.9 / 17.6 (19.6, 18.5); 28 / 4 heads of 256, one of 100 over 2 000:
//     50.6 / 27.3 / 26.8 (28.6, 25.0); 16 latent heads, one of 3 over 2 000: 90 / 19.8 / 19.5 (20.1, 20.1), 16 of 5: 97 / 30.7 / 30.3
//   * round the length that it pays from, one of 100 over 400: 12.8 / 12.9 / 14.3, over 500 14.5 / 14.7 / 14.8 (14.7, 14.5),
//     over 600 15.7 / 15.6 / 14.2, over 700 17.5 / 14.6 / 15.0; four of 64 over 700 17.0 / 17.0 / 18.6, over 1 000 21.8 / 21.8 / 22.6; latent, one of 20 over 100
//     15.7 / 15.7 / 17.2, over 200 20.0 / 20.0 / 18.2, over 400 28.2 / 18.5 / 18.4
//   * without history, where nothing is split and the table alone says that it might be: one of 3 tokens 5.9 / 6.0 / 6.5
//     (6.2, 9.7), one of 100 7.5 / 7.4 / 8.1 (7.5, 10.9), four of 64 6.5 / 6.6 / 7.2 (6.8, 12.9), 16 of 5 6.2 / 6.4 / 7.0 (6.5, 11.5)
// What such a call still pays, 0.6 - 1.5 us, is workgroups that look the batch up and leave.
inline void planSplit(const PagedAttentionPrefillInfo &in, const device::amd::DeviceInfo &dev, long long rows_per_seq, Plan &plan) {
    const long long seqs = in.num_seqs > 0 ? static_cast<long long>(in.num_seqs) : 1;
    const long long kv_heads = static_cast<long long>(in.num_kv_heads);
    // Row blocks: of equal sequences, or half a block more for each than its rows if that is more. (Two of 137 and 92 rows are
    // five blocks, not twice the two of 114.5: with parts for four, some wait for a second round, 28.6 us instead of 24.9
    // over 5 531 and 3 798 at 8 heads; 16 latent heads, 33 and 30 tokens over 6 920 and 4 337, 51.5 instead of 46.4.)
    const long long ragged = seqs == 1 || rows_per_seq % 64 == 0 ? 0 : (rows_per_seq * seqs + 32 * seqs + 63) / 64;
    const long long blocks = kv_heads * std::max(seqs * ((rows_per_seq + 63) / 64), ragged);
    const long long tokens = static_cast<long long>(in.max_num_blocks_per_seq) * static_cast<long long>(in.page_block_size);
    const long long slots = static_cast<long long>(dev.compute_units) * (in.head_size <= 192 ? 2 : 1);
    plan.max_parts = 1;
    if (blocks <= 0) {
        return;
    }
    const int most = static_cast<int>(std::min(std::min(slots / blocks, (tokens + kSplitTableTokens - 1) / kSplitTableTokens),
                                               static_cast<long long>(kMaxSplitParts)));
    const double us_per_token = 1e-3 * (in.head_size == 64 ? 11 : in.head_size == 128 ? 14 : in.head_size == 192 ? 22
                                      : in.head_size == 256 ? 20 : 41);
    const double row_bytes = static_cast<double>(rows_per_seq) * seqs * kv_heads * in.value_size * sizeof(float);
    const double meet_cost = 2.9, part_cost = 0.3e-6 * row_bytes;
    // time of the best split of a walk of `t` tokens
    auto split = [&](double t, int &best) {
        double least = 1e30;
        for (int p = 2; p <= most && (p - 1) * kSplitTableTokens < t; ++p) {
            const double shared = blocks * p > dev.compute_units && in.head_size <= 192 ? 1.4 : 1.0;
            const double us = shared * us_per_token * t / p + meet_cost + part_cost * p;
            if (us < least) {
                best = p, least = us;
            }
        }
        return least;
    };
    int best = 1, any = 1;
    if (split(static_cast<double>(tokens), best) >= 0.8 * us_per_token * static_cast<double>(tokens)) {
        return;
    }
    plan.max_parts = best;
    long long from = kSplitTableTokens;
    while (from < tokens && split(static_cast<double>(from), any) >= us_per_token * static_cast<double>(from)) {
        from += 32;
    }
    plan.split_from = static_cast<int>(from);
    plan.part_cost = static_cast<float>(part_cost / us_per_token);
}

inline Plan makePlan(const PagedAttentionPrefillInfo &in, const device::amd::DeviceInfo &dev) {
    Plan plan{};
    const long long bs = static_cast<long long>(in.page_block_size);
    const bool pow2_page = bs >= 8 && (bs & (bs - 1)) == 0;
    const long long group = static_cast<long long>(in.num_heads / in.num_kv_heads);
    const long long rows = static_cast<long long>(in.total_q_tokens) * group; // per KV head
    const bool equal_sizes = in.value_size == in.head_size
                          && (in.head_size == 64 || in.head_size == 128 || in.head_size == 192 || in.head_size == 256);
    // keys 576 with values 512 (latent attention) or 576 (a shape of the reference's decode tests,
    // test/infiniop/paged_attention.py:106, taken here as well so that prompt and decode run the same class of kernel)
    const bool latent = in.head_size == 576 && (in.value_size == 512 || in.value_size == 576);
    plan.tiled = (equal_sizes || latent) && pow2_page
              && multipleOf8(in.q_stride) && multipleOf8(in.q_head_stride) && multipleOf8(in.o_stride)
              && multipleOf8(in.o_head_stride) && multipleOf8(in.k_batch_stride) && multipleOf8(in.k_head_stride)
              && multipleOf8(in.k_row_stride) && multipleOf8(in.v_batch_stride) && multipleOf8(in.v_head_stride)
              && multipleOf8(in.v_row_stride) && in.num_blocks > 0 && in.num_blocks <= 0x7fffffff
              && rows < (1LL << 30) && (rows / 64 + static_cast<long long>(in.num_seqs)) * static_cast<long long>(in.num_kv_heads) < (1LL << 31)
              // lane offsets inside a tile (15 rows + one row of bytes) are kept in 32 bits
              && in.k_row_stride > 0 && in.k_row_stride < (1 << 26) && in.v_row_stride > 0 && in.v_row_stride < (1 << 26)
              && static_cast<long long>(in.max_num_blocks_per_seq) * bs < (1LL << 30);
    if (const char *env = std::getenv("INFINIOP_AMD_PREFILL_KERNEL")) {
        if (std::strcmp(env, "generic") == 0) {
            plan.tiled = false;
        }
    }
    // Rows per workgroup: 128 (two column groups per wavefront: every K / V operand read from LDS then feeds two
    // matrix instructions) unless the average sequence fills no more than 64, or the batch is too small to give
    // every compute unit as many workgroups of 128 as it holds at a time: two up to head 128, one above (there the
    // accumulators of 128 rows need more than half the register file).
    const long long seqs = in.num_seqs > 0 ? static_cast<long long>(in.num_seqs) : 1;
    const long long rows_per_seq = rows / seqs;
    const long long resident = in.head_size <= 128 ? 2 : 1;
    int r = 2;
    if (rows_per_seq <= 64 || rows / 128 * static_cast<long long>(in.num_kv_heads) < resident * dev.compute_units) {
        r = 1;
    }
    if (latent && plan.tiled) {
        r = latentRowGroups(in, dev, rows_per_seq);
    }
    if (const char *env = std::getenv("INFINIOP_AMD_PREFILL_GROUPS")) {
        const int forced = std::atoi(env);
        if (forced == 1 || forced == 2) {
            r = forced;
        }
    }
    if (latent && (in.value_size != 512 || in.has_alibi || !(in.scale > 0.0f))) {
        // 128 rows have a kernel of their own (prefill_latent.h) for values of 512 without ALiBi only, whatever the
        // knob says (grid and kernel must agree on the rows per workgroup)
        r = 1;
    }
    plan.groups_per_wave = r;
    plan.compute_units = dev.compute_units;
    // (a forced number of rows asks for those kernels as they are)
    const bool rows_forced = std::getenv("INFINIOP_AMD_PREFILL_GROUPS") != nullptr;
    plan.max_parts = 1;
    if (plan.tiled && r == 1 && !rows_forced) {
        planSplit(in, dev, rows_per_seq, plan);
    }
    if (const char *env = std::getenv("INFINIOP_AMD_PREFILL_PARTS")) {
        const int forced = std::atoi(env);
        if (plan.tiled && r == 1 && forced >= 1 && forced <= kMaxSplitParts) {
            plan.max_parts = forced;
            plan.split_from = 0;
            plan.part_cost = 0.0f;
        }
    }
    if (plan.max_parts > 1) {
        const size_t part_rows = static_cast<size_t>(rows / 64 + seqs) * in.num_kv_heads * static_cast<size_t>(plan.max_parts) * 64;
        if (part_rows >= (size_t{1} << 31)) { // a knob's doing: more workgroups than a launch has
            plan.max_parts = 1;
        }
        // Workgroups that merge a block, up to eight (two rows per wavefront), while all of them are one and a half rounds of
        // the device: us with 1 / 2 / 4 / 8 at 64 blocks (one sequence of 100 tokens over 1 900, eight parts)
        // 33.7 / 24.7 / 19.9 / 17.4, at 160 (four of 64, four parts) 41.1 / 31.3 / 26.8 / 28.7
        const long long grid = (rows / 64 + seqs) * static_cast<long long>(in.num_kv_heads);
        const long long room = 3 * dev.compute_units * (in.head_size <= 192 ? 2 : 1) / 2 / grid;
        plan.merge_workgroups = room >= 8 ? 8 : (room >= 4 ? 4 : (room >= 2 ? 2 : 1));
        plan.part_acc_bytes = part_rows * in.value_size * sizeof(float);
        plan.part_ml_bytes = part_rows * 2 * sizeof(float);
        plan.row_block_grid = grid;
        plan.part_flags_bytes = (part_rows + static_cast<size_t>(grid) * kMergeWavefronts) * sizeof(unsigned long long);
        plan.merge_polls = kMergePolls;
        if (const char *env = std::getenv("INFINIOP_AMD_PREFILL_MERGE_POLLS")) {
            plan.merge_polls = std::max(0, std::atoi(env));
        }
    }
    const size_t widest = in.head_size > in.value_size ? in.head_size : in.value_size;
    plan.dims_per_lane = static_cast<int>((widest + 63) / 64);
    return plan;
}

} // namespace op::paged_attention_prefill::amd

#endif
