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
    int max_parts;       // tiled, 64 rows: workgroups that may share a row block (prefill_split.h); 1 = not split
    size_t part_acc_bytes, part_ml_bytes; // workspace of the parts, either a multiple of 256 bytes
    size_t workspaceBytes() const { return max_parts > 1 ? part_acc_bytes + part_ml_bytes + 256 : 0; }
    int dims_per_lane;   // element-wise kernel: ceil(max(head_size, value_size) / 64)
};

inline bool multipleOf8(ptrdiff_t x) { return (x % 8) == 0; }

// Latent attention (keys of 576): 64 or 128 rows per workgroup, as 1 or 2. One workgroup per compute unit with either
// kernel, and one of 128 rows (prefill_latent.h) takes 1.4 x as long as one of 64 over the same tokens. So 128 rows where
// they save more than a third of the rounds of workgroups. Measured, us with 64 rows / with 128, by 64-row blocks (16
// heads, bf16, 256 compute units):
//   * three rounds against two: 640 blocks over 2 000 tokens of history 312 / 320, 740 330 / 340; 64 sequences of 40
//     without history 41 / 43
//   * four against two: 1 000 over 2 000 452 / 385, over 500 212 / 197; 16 sequences of 200 without history 57 / 56, four
//     of 900 113.5 / 114.5; five against three: 100 sequences of 50 75 / 70
//   * two rounds against one: the second round is short where a block's tokens grow along the sequence (the longest blocks
//     start first, the last ones fit behind the shortest of the first round) or where sequences differ in length, and
//     then 128 rows only make the longest block longer. One sequence without history, 275 blocks 64 / 90, 500 111 / 142; two
//     of 900 60 / 74; four of 128 - 512 over 1 024 - 8 192 419 / 501. With much history and equal lengths it is a whole
//     round: four of 500 over 2 000 219 / 176. The lengths of several sequences are not known here: 64 rows. For one
//     sequence the table says how much history there can be, and its blocks are dealt in order: block 256 + j starts when
//     block 256 - j ends, after 2 history + 2 n (1 - 256 / blocks) tokens of n new ones in all, against 1.4 (history + n).
//     1 600 over 1 200: 177 / 189, over 3 000 327 / 299; 2 000 over 1 000 194 / 205, over 2 000 276 / 267. (A table wider
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

constexpr int kMaxSplitParts = 64; // the merge forms the weights of a row with a lane per part
constexpr long long kSplitTableTokens = 128; // the shortest part (kSplitTokens of prefill_tiled.h)

// How many workgroups share the tokens of a row block of 64 rows. Unsplit, a call that leaves compute units idle takes as
// long as its longest block: `walk` microseconds for the tokens the table can hold (measured with one block per KV head
// over 5 800 tokens). P parts take a P-th of that (1.4 times that where two of them share a unit), write and read their
// rows back (0.9 us per MB of them) and need the merge kernel (3 us): P where the sum is smallest, among those the device
// holds beside one another, if it takes a fifth off the walk. Measured, us unsplit / with the P this chooses / with
// the best of 2 .. 32 (bf16; 32 / 8 heads of 128 unless said otherwise):
//   * one sequence, 3 tokens over 600 / 5 800: 14.0 / 11.1 / 10.8, 87.7 / 14.0 / 14.2; 128 over 8 000: 130 / 34.5 / 34.5
//   * four of 64 over 4 000: 68.8 / 36.7 / 36.2, over 500: 14.4 unsplit / 18.8; 16 of 5 over 2 000: 35.3 / 28.8 / 28.8
//   * 16 heads of 64, 16 of 5 over 2 000 (a block per unit): 28.3 unsplit / 28.9; 28 / 4 heads of 256, one of 128 over
//     8 000: 175 / 60.7 / 61.2; 16 latent heads, one of 3 over 5 800: 243 / 28.1 / 26.8, 16 of 5 over 2 000: 93 / 33 / 31
inline int splitParts(const PagedAttentionPrefillInfo &in, const device::amd::DeviceInfo &dev, long long rows_per_seq) {
    const long long seqs = in.num_seqs > 0 ? static_cast<long long>(in.num_seqs) : 1;
    const long long kv_heads = static_cast<long long>(in.num_kv_heads);
    const long long blocks = seqs * ((rows_per_seq + 63) / 64) * kv_heads;
    const long long tokens = static_cast<long long>(in.max_num_blocks_per_seq) * static_cast<long long>(in.page_block_size);
    const long long slots = static_cast<long long>(dev.compute_units) * (in.head_size <= 192 ? 2 : 1);
    if (blocks <= 0) {
        return 1;
    }
    const long long most = std::min(std::min(slots / blocks, (tokens + kSplitTableTokens - 1) / kSplitTableTokens),
                                    static_cast<long long>(kMaxSplitParts));
    const double us_per_1000 = in.head_size == 64 ? 11 : in.head_size == 128 ? 14 : in.head_size == 192 ? 22
                             : in.head_size == 256 ? 20 : 41;
    const double walk = us_per_1000 * 1e-3 * static_cast<double>(tokens);
    const double row_bytes = static_cast<double>(rows_per_seq) * seqs * kv_heads * in.value_size * sizeof(float);
    const double row_cost = 0.9e-6 * row_bytes, merge_cost = 3.0;
    int best = 1;
    double least = 0.8 * walk;
    for (int p = 2; p <= most; ++p) {
        const double shared = blocks * p > dev.compute_units && in.head_size <= 192 ? 1.4 : 1.0;
        const double t = shared * walk / p + row_cost * p + merge_cost;
        if (t < least) {
            best = p, least = t;
        }
    }
    return best;
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
    plan.max_parts = plan.tiled && r == 1 && !rows_forced ? splitParts(in, dev, rows_per_seq) : 1;
    if (const char *env = std::getenv("INFINIOP_AMD_PREFILL_PARTS")) {
        const int forced = std::atoi(env);
        if (plan.tiled && r == 1 && forced >= 1 && forced <= kMaxSplitParts) {
            plan.max_parts = forced;
        }
    }
    if (plan.max_parts > 1) {
        const size_t part_rows = static_cast<size_t>(rows / 64 + seqs) * in.num_kv_heads * static_cast<size_t>(plan.max_parts) * 64;
        if (part_rows >= (size_t{1} << 31)) { // a knob's doing: more workgroups than a launch has
            plan.max_parts = 1;
        }
        plan.part_acc_bytes = part_rows * in.value_size * sizeof(float);
        plan.part_ml_bytes = part_rows * 2 * sizeof(float);
    }
    const size_t widest = in.head_size > in.value_size ? in.head_size : in.value_size;
    plan.dims_per_lane = static_cast<int>((widest + 63) / 64);
    return plan;
}

} // namespace op::paged_attention_prefill::amd

#endif
