// Prefill kernel for latent attention (keys of 576, values of 512 elements), 128 rows per workgroup, on gfx950.
//
// What the four-wavefront kernel of prefill_tiled.h pays at these sizes: a wavefront there owns 16 rows, so every K
// and V operand read from LDS feeds one matrix instruction, and all four wavefronts read all of both tiles: 272 KiB
// of LDS reads (2 176 clocks at 128 bytes per clock) against 1 104 clocks of matrix instructions per step of 32 tokens
// and 64 rows; a compute unit takes one direct load of 1 KiB every ~15 ns, 68 of them per step; and its registers
// leave one wavefront per SIMD, with nothing to run beside it (matrix units busy 30 % of their clocks, LDS 44 %, a vector
// instruction beside 0.3 % of the matrix clocks).
//
// Here one workgroup of eight wavefronts (two per SIMD) takes 128 rows, which halves the loads per row, and splits
// the two products differently:
//   * K.Q^T by rows: wavefront w owns rows 16 w .. 16 w + 15, their query in registers and their softmax state, and
//     reads the whole K tile.
//   * P.V by rows and columns: wavefront w takes the 64 rows of its half (w / 4) and 128 of the 512 columns (w % 4), so
//     an operand of V feeds four matrix instructions. The probabilities pass through LDS (8 KiB per step) in the
//     register layout they are computed and used in, the rescaling factors of a step beside them.
// Per step of 32 tokens and 128 rows: 288 KiB of K, 64 KiB of V and 32 KiB of probabilities out of LDS (3 072 clocks),
// 2 208 clocks of matrix instructions per SIMD. 128 accumulator and 72 query registers per lane leave room for two
// wavefronts per SIMD, and 56 for everything else: nothing of the loop is in scratch memory (a reload there waits for the
// direct loads in flight too: with one query operand reloaded behind them the case below took 1 287 us).
// Measured (16 sequences, 16 heads, 128 - 512 new tokens over 1 024 - 8 192 of history, bf16; the kernels in turn on
// one GPU): 1 265 -> 961 us (647 -> 852 TFLOP/s); 1 308 -> 995 on another. Neither pipe bounds it: matrix units and LDS are
// each busy 37 % of their clocks, a vector instruction beside 16 % of the matrix clocks, 1.66 of the two wavefronts of a
// SIMD present on average (the last round of workgroups). All eight wavefronts pass two barriers per step in the same
// phase, so that K.Q^T (LDS), the softmax and P.V (matrix) follow one another.
// Everything else (block search, page ids, layout of V in LDS, masks, lazy reference point) is as in prefill_tiled.h.
#ifndef INFINICORE_AMD_PA_PREFILL_LATENT_H
#define INFINICORE_AMD_PA_PREFILL_LATENT_H

#include "prefill_tiled.h"

namespace op::paged_attention_prefill::amd {

constexpr int kLatentThreads = 512;
constexpr int kLatentRows = 128;

// No ALiBi and scale > 0 (PLAIN of prefillTiledKernel): the ALiBi distances would cost registers that are not there.
template <typename T, typename Tindex>
__global__ void __launch_bounds__(kLatentThreads, 2) prefillLatentKernel(PrefillArgs a) {
    using S = typename T::storage;
    constexpr int KHEAD = 576, VHEAD = 512;
    using G = PrefillGeometry<KHEAD, VHEAD>;
    constexpr int BN = 32;
    constexpr int kTileChunksK = kTileTokens * G::kChunksPerRowK, kTileChunksV = kTileTokens * G::kChunksPerRowV;
    constexpr int kWaves = kLatentThreads / 64;
    constexpr int kCols = G::kColsV / 4; // blocks of 16 value columns of a wavefront
    constexpr int kAdds = 0, kRescales = 1, kUnseen = 2;
    struct Shared {
        // K of a 16-token tile: columns 0..511 of the 16 rows, then columns 512..575 of the 16 rows; a row's 16-byte chunks
        // XOR-swizzled by the row (sixteen at a time; the last eight by half the row), so that 16 lanes that read one
        // chunk of the 16 rows touch all 64 banks once. One load instruction brings the first 64 chunks of one row, or
        // the last eight of eight rows, and its lane offsets cost one exclusive-or. (In one run of 72 chunks as in
        // prefillTiledKernel, only eight of them swizzled and a load across two rows: 1 270 against 1 034 us. Bank conflicts
        // are not the reason: the counter reads the same with both kernels, the two-byte stores of the epilogue.)
        uint4 k[2][2 * kTileChunksK];
        uint4 v[2][2 * kTileChunksV]; // layout as in prefillTiledKernel
        uint4 p[kWaves][64];        // probabilities of 16 rows x 32 tokens, as the lanes of P.V take them
        float4 alpha[kWaves][4];    // factors by which the accumulators of the 16 rows are rescaled this step
        int4 update[kWaves / 4];    // ... and what the step does to them, per group of 16 rows: kAdds, kRescales or kUnseen
        float4 denominator[kWaves][4];
    };
    __shared__ Shared lds;
    static_assert(__builtin_offsetof(Shared, v) == sizeof(uint4) * 4 * kTileChunksK, "V follows K (pend_dst)");

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15;
    const int g = lane >> 4;
    const int kv_head = blockIdx.x % a.num_kv_heads;
    const int block_index = blockIdx.x / a.num_kv_heads;

    int seq = 0, block = 0;
    SeqSpan span;
    if (!findRowBlock<Tindex>(a, lane, kLatentRows, block_index, seq, block, span)) {
        return;
    }
    const int total_rows = span.q_len * a.group; // > 0 here
    const int block_row0 = block * kLatentRows;
    const int last_row = min(block_row0 + kLatentRows, total_rows) - 1;
    const int block_visible = __builtin_amdgcn_readfirstlane(visibleTokens(span, last_row / a.group));
    if (block_visible <= 0) {
        return;
    }
    const int kv_len = __builtin_amdgcn_readfirstlane(max(span.kv_len, block_visible));
    const int n_steps = (block_visible + BN - 1) / BN;

    // ---- this lane's row of K.Q^T ----
    uint4 q_reg[G::kLoadsK];
    int visible;
    {
        const int row = block_row0 + w * 16 + c;
        const bool valid = row < total_rows;
        const int token = valid ? row / a.group : 0;
        const int head = kv_head * a.group + (valid ? row - token * a.group : 0);
        visible = valid ? visibleTokens(span, token) : 0;
        const S *q_ptr = static_cast<const S *>(a.q) + (span.q_start + token) * a.q_stride + head * a.q_head_stride;
#pragma unroll
        for (int kk = 0; kk < G::kLoadsK; ++kk) {
            q_reg[kk] = valid ? *reinterpret_cast<const uint4 *>(q_ptr + 32 * kk + 8 * g) : make_uint4(0, 0, 0, 0);
        }
    }

    // ---- copy side: wavefronts 0..3 bring K, 4..7 V, each half of the load instructions of one 16-token tile ----
    const bool copies_k = w < 4;
    const int copy_tile = (w >> 1) & 1, copy_half = w & 1;
    constexpr int kHalfK = G::kLoadsK / 2, kHalfV = G::kLoadsV / 2;
    static_assert(G::kLoadsK % 2 == 0 && G::kLoadsV % 2 == 0 && kHalfK >= kHalfV, "two wavefronts share a tile's loads");
    const char *k_head = reinterpret_cast<const char *>(static_cast<const S *>(a.k_cache) + kv_head * a.k_head_stride);
    const char *v_head = reinterpret_cast<const char *>(static_cast<const S *>(a.v_cache) + kv_head * a.v_head_stride);
    const int64_t table_row = seq * a.block_table_batch_stride;
    const int block_mask = a.block_size - 1;
    const bool small_pages = a.block_size < 16;
    const int last_entry = (kv_len - 1) >> a.block_shift;

    auto loadIdBatch = [&](int batch) {
        const int entry = batch * 64 + lane;
        int id = 0;
        if (entry <= last_entry) {
            id = static_cast<int>(loadIndex<Tindex>(a.block_tables, table_row + entry));
        }
        return id;
    };
    int id_batch = 0;
    int ids_cur = loadIdBatch(0), ids_next = loadIdBatch(1);
    auto pageOfEntry = [&](int entry) {
        const int e = min(entry, last_entry);
        const int raw = (e >> 6) == id_batch ? __builtin_amdgcn_readlane(ids_cur, e & 63)
                                             : __builtin_amdgcn_readlane(ids_next, e & 63);
        return clampPage(raw, a.num_blocks);
    };
    auto vRowOfSlot = [](int slot) { return 8 * (slot / (8 * G::kChunksPerRowV)) + (slot % 16) / 2; };
    auto vChunkOfSlot = [](int slot) { return 2 * ((slot % (8 * G::kChunksPerRowV)) / 16) + slot % 2; };

    // A wavefront brings eight rows of its tile. K: instruction i < 8 the chunks 0..63 of row i, instruction 8 the chunks
    // 64..71 of all eight rows. V: instruction i four blocks of 16 columns of the eight rows, 128 bytes on from i - 1.
    static_assert(G::kChunksPerRowK == 72 && kHalfK == 9 && kHalfV == 8 && 64 * kHalfV == 8 * G::kChunksPerRowV);
    const uint32_t first_off = copies_k ? 16 * static_cast<uint32_t>(lane ^ (8 * copy_half))
                                        : vRowOfSlot(lane) * static_cast<uint32_t>(a.v_row_stride) * sizeof(S) + 16 * vChunkOfSlot(lane);
    const uint32_t last_off = (lane >> 3) * static_cast<uint32_t>(a.k_row_stride) * sizeof(S) + 16 * (64 + ((lane & 7) ^ (4 * copy_half + (lane >> 4))));
    // row strides are below 2^26 elements (plan): seven of them fit 32 bits
    const uint32_t step_bytes = __builtin_amdgcn_readfirstlane(copies_k ? static_cast<uint32_t>(a.k_row_stride) * sizeof(S) : 128u);
    const uint32_t xor_mask = copies_k ? 0x70 : 0, k_only = copies_k ? ~0u : 0u;
    const int64_t half_rows = 8 * copy_half; // the rows of the tile that this wavefront brings begin here
    // The instructions of a stage are issued one at a time between the matrix instructions of the step before it, as in
    // prefillTiledKernel: loadStage records where they read and write, issueSlot(i) issues the i-th.
    // All of it is the same in all lanes; said once more where it is used, it stays in scalar registers.
    const char *pend_src = k_head;
    uint32_t pend_dst = 0; // slot of the wavefront's first 64 chunks, counted from lds.k
    uint32_t pend_live = 0; // all lanes or none
    auto issueSlot = [&](int i) {
        const uint64_t address = reinterpret_cast<uint64_t>(pend_src);
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address >> 32));
        const char *src = reinterpret_cast<const char *>(static_cast<uint64_t>(hi) << 32 | lo);
        const uint32_t dst = __builtin_amdgcn_readfirstlane(pend_dst);
        const uint32_t live = __builtin_amdgcn_readfirstlane(i < 8 ? pend_live : (pend_live & k_only));
        const unsigned long long lanes = static_cast<unsigned long long>(live) << 32 | live;
        uint4 *const first = &lds.k[0][0];
        if (i < 8) {
            uint32_t off = first_off;
            asm volatile("" : "+v"(off)); // eight hoisted offsets would be spilled
            loadLane16ToLdsMasked(src + i * step_bytes, off ^ ((16 * i) & xor_mask), first + dst + 64 * i, lanes);
        } else { // from slot 64 * 8 * copy_half of the tile on to slot 64 * (16 + copy_half)
            loadLane16ToLdsMasked(src, last_off, first + dst + 64 * (16 - 7 * copy_half), lanes);
        }
    };
    auto loadStage = [&](int step) {
        pend_live = 0;
        int own = lane; // what the rare path derives from the lane is formed there: hoisted, it would cost registers
        asm volatile("" : "+v"(own));
        const int t = step * BN + kTileTokens * copy_tile;
        const int e0 = t >> a.block_shift;
        if ((min(e0, last_entry) >> 6) > id_batch) {
            ids_cur = ids_next;
            ++id_batch;
            ids_next = loadIdBatch(id_batch + 1);
        }
        const int id0 = pageOfEntry(e0), id1 = small_pages ? pageOfEntry(e0 + 1) : id0;
        if (copies_k) {
            // rows past the end of the sequence: as in prefillTiledKernel (their page exists, their scores are masked)
            if (!small_pages) {
                pend_src = k_head + (id0 * a.k_batch_stride + ((t & block_mask) + half_rows) * a.k_row_stride) * static_cast<int64_t>(sizeof(S));
            } else { // pages of 8 tokens: this wavefront's eight rows are one page
                pend_src = k_head + (copy_half ? id1 : id0) * a.k_batch_stride * static_cast<int64_t>(sizeof(S));
            }
            pend_dst = (2 * (step & 1) + copy_tile) * kTileChunksK + 64 * 8 * copy_half, pend_live = ~0u;
            return;
        }
        uint4 *v_dst = &lds.v[step & 1][copy_tile * kTileChunksV + 64 * copy_half * kHalfV];
        if (t + kTileTokens <= kv_len && !small_pages) {
            pend_src = v_head + (id0 * a.v_batch_stride + ((t & block_mask) + half_rows) * a.v_row_stride) * static_cast<int64_t>(sizeof(S));
            pend_dst = 4 * kTileChunksK + (2 * (step & 1) + copy_tile) * kTileChunksV + 64 * 8 * copy_half, pend_live = ~0u;
            return;
        }
        // last tile of the sequence, or two pages per tile: rows past the sequence are zeroed
        const int row0 = small_pages ? 0 : (t & block_mask);
#pragma unroll 1
        for (int n = 0; n < kHalfV; ++n) {
            const int i = __builtin_amdgcn_readfirstlane(n);
            const int slot = 64 * (copy_half * kHalfV + i) + own;
            const int row = vRowOfSlot(slot);
            const int page = (small_pages && row >= 8) ? id1 : id0;
            const int page_row = small_pages ? (row & 7) : row0 + row;
            const char *src = v_head + (page * a.v_batch_stride + page_row * a.v_row_stride) * static_cast<int64_t>(sizeof(S))
                            + 16 * vChunkOfSlot(slot);
            if (t + row < kv_len) {
                loadLane16ToLds(src, v_dst + 64 * i);
            } else {
                uint32_t zero = 0;
                asm volatile("" : "+v"(zero)); // not four registers of zeros for the whole loop
                v_dst[64 * i + own] = make_uint4(zero, zero, zero, zero);
            }
        }
    };
    auto awaitStage = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    // What the wavefronts hand over in the middle of a step passes through LDS only: the direct loads of the next stage
    // stay in flight across this barrier.
    auto ldsBarrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // ---- P.V side: rows of half w / 4, columns of quarter w % 4 ----
    const int half = w >> 2, quarter = w & 3;
    f32x4 o[4][kCols]; // o[i][e][rr] = O[row 64 half + 16 i + 4g + rr][column 16 (kCols quarter + e) + c]
    f32x4 ol = f32x4{0.f, 0.f, 0.f, 0.f}; // denominators of the wavefront's own rows 16 w + 4g + rr
    float m = -INFINITY, shift = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int e = 0; e < kCols; ++e) {
            o[i][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *LdsPiece;
    const auto v_read_base = (__attribute__((address_space(3))) char *)lds.v
                           + 16 * ((g >> 1) * 8 * G::kChunksPerRowV + (4 * (g & 1) + (c >> 2)) * 2 + ((c & 3) >> 1)) + 8 * (c & 1)
                           + 256 * kCols * quarter;
    // slots of chunk g of row c in either part of a K tile; chunk 4 kk + g is 4 (kk % 4) XORed and 16 (kk / 4) added
    const int k_first = 64 * c + (g ^ c), k_last = 64 * 16 + 8 * c + (g ^ (c >> 1));
    const float unit = a.scale_log2;
    const float lazy = kLazyLog2 / unit;
    // what the last of the wavefront's rows sees, which is the most any of them does (0 if it has no rows)
    const int wave_row0 = block_row0 + 16 * w;
    const int wave_sees = __builtin_amdgcn_readfirstlane(wave_row0 < total_rows ? visibleTokens(span, min(wave_row0 + 15, last_row) / a.group) : 0);

    auto computeStep = [&](int buf, int t0) {
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        {
            constexpr int kAheadK = 3; // two wavefronts of the SIMD take turns; a fourth would be spilled
            constexpr int kOperandsK = 2 * G::kLoadsK;
            // operand idx: the 32 dimensions kk = idx / 2 of tile idx % 2 (neighbours go to different accumulators), added in
            // the order of prefillTiledKernel, so that the outputs of the two are the same bits. Four lane addresses would
            // serve the sixteen dimensions of the first part of a row: each is formed from the one before, one is live.
            int first = 16 * k_first;
            asm volatile("" : "+v"(first));
            auto readK = [&](int idx) {
                const int kk = idx / 2;
                if (idx % 2 == 0 && kk > 0 && kk < 16) {
                    first ^= 16 * (4 * (kk % 4) ^ 4 * ((kk - 1) % 4));
                    asm volatile("" : "+v"(first));
                }
                const int at = kk < 16 ? first + 16 * 16 * (kk / 4) : 16 * (k_last ^ (4 * (kk % 4)));
                return *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(lds.k[buf] + idx % 2 * kTileChunksK) + at);
            };
            uint4 kf[kAheadK];
#pragma unroll
            for (int i = 0; i < kAheadK; ++i) {
                kf[i] = readK(i);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, kAheadK, 0);
#pragma unroll
            for (int idx = 0; idx < kOperandsK; ++idx) {
                const uint4 cur = kf[idx % kAheadK];
                if (idx + kAheadK < kOperandsK) {
                    kf[idx % kAheadK] = readK(idx + kAheadK);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                s[idx % 2] = T::mfmaK32(cur, q_reg[idx / 2], s[idx % 2]);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (idx % 4 == 3) {
                    issueSlot(idx / 4);
                }
            }
            static_assert(kOperandsK / 4 == kHalfK, "a place in the step for every load instruction of a stage");
        }

        // the causal mask, in every step: 16 vector instructions beside some 3 000 clocks; a branch around them costs
        // registers across it
        const int sees = visible - t0 - 4 * g;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                s[tt][rr] = 16 * tt + rr >= sees ? -INFINITY : s[tt][rr];
            }
        }
        float mx = maxOf(maxOf(s[0][0], s[0][1]), s[0][2]);
        mx = maxOf(maxOf(mx, s[0][3]), s[1][0]);
        mx = maxOf(maxOf(mx, s[1][1]), s[1][2]);
        mx = maxOf(mx, s[1][3]);
        const bool moves = __builtin_amdgcn_ballot_w64(mx > m + lazy) != 0; // some row's reference point
        if (moves) {
            mx = maxAcrossTokenGroups(mx);
            const float m_new = maxOf(m, mx);
            const float alpha = m_new > m ? fastExp2((m - m_new) * unit) : 1.0f;
            m = m_new;
            shift = m_new == -INFINITY ? 0.0f : -m_new * unit;
            int own = lane; // addresses formed where they are used, as in loadStage
            asm volatile("" : "+v"(own));
            if (own < 16) {
                reinterpret_cast<float *>(&lds.alpha[w][0])[own] = alpha;
            }
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                ol[rr] *= __shfl(alpha, 4 * (own >> 4) + rr, 64);
            }
        }
        if (lane == 0) {
            reinterpret_cast<int *>(lds.update)[w] = t0 >= wave_sees ? kUnseen : moves ? kRescales : kAdds;
        }
        uint32_t wds[4];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const f32x4 x = s[tt];
            wds[2 * tt] = T::pack2(fastExp2(__builtin_fmaf(x[0], unit, shift)), fastExp2(__builtin_fmaf(x[1], unit, shift)));
            wds[2 * tt + 1] = T::pack2(fastExp2(__builtin_fmaf(x[2], unit, shift)), fastExp2(__builtin_fmaf(x[3], unit, shift)));
        }
        const uint4 p_own = make_uint4(wds[0], wds[1], wds[2], wds[3]);
        lds.p[w][lane] = p_own;
        uint32_t one2 = T::pack2(1.0f, 1.0f);
        asm volatile("" : "+v"(one2)); // four registers for this instruction, not for the whole loop
        ol = T::mfmaK32(p_own, make_uint4(one2, one2, one2, one2), ol);
        ldsBarrier();

        const int4 update_lanes = lds.update[half];
        const int update[4] = {__builtin_amdgcn_readfirstlane(update_lanes.x), __builtin_amdgcn_readfirstlane(update_lanes.y),
                               __builtin_amdgcn_readfirstlane(update_lanes.z), __builtin_amdgcn_readfirstlane(update_lanes.w)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (__builtin_expect(update[i] == kRescales, 0)) {
                int own = lane;
                asm volatile("" : "+v"(own));
                const float4 f = lds.alpha[4 * half + i][own >> 4];
#pragma unroll
                for (int e = 0; e < kCols; ++e) {
                    o[i][e][0] *= f.x;
                    o[i][e][1] *= f.y;
                    o[i][e][2] *= f.z;
                    o[i][e][3] *= f.w;
                }
            }
        }
        uint4 p_op[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p_op[i] = lds.p[4 * half + i][lane];
        }
        auto readV = [&](int e) {
            const auto base = v_read_base + buf * (2 * kTileChunksV * 16) + 256 * e;
            const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsPiece>(base)));
            const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<LdsPiece>(base + kTileChunksV * 16)));
            return make_uint4(lo.x, lo.y, hi.x, hi.y);
        };
        // Two columns at a time, the next two requested before them; an operand lasts four matrix instructions. Rows that see
        // nothing of the step leave it out: their probabilities are zeros, but 0 * inf is NaN, and V may hold anything at
        // tokens that come after theirs.
        uint4 vf[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            vf[i] = readV(i);
        }
#pragma unroll
        for (int e = 0; e < kCols; e += 2) {
            const uint4 cur[2] = {vf[0], vf[1]};
            if (e + 2 < kCols) {
                vf[0] = readV(e + 2);
                vf[1] = readV(e + 3);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (__builtin_expect(update[i] != kUnseen, 1)) {
                    o[i][e] = T::mfmaK32(p_op[i], cur[0], o[i][e]);
                    o[i][e + 1] = T::mfmaK32(p_op[i], cur[1], o[i][e + 1]);
                }
            }
        }
    };

    // ---- pipeline ----
    loadStage(0);
#pragma unroll
    for (int i = 0; i < kHalfK; ++i) {
        issueSlot(i);
    }
    awaitStage();
    __syncthreads();
    for (int j = 0; j < n_steps; ++j) {
        if (j + 1 < n_steps) {
            loadStage(j + 1);
        } else {
            pend_live = 0;
        }
        computeStep(j & 1, j * BN);
        awaitStage();
        __syncthreads();
    }

    // ---- normalise and store: denominators to the wavefronts that hold the columns, the rows through the tile buffers
    // (nothing is in flight, everybody is past the last barrier of the loop) ----
    if (c == 0) {
        lds.denominator[w][g] = make_float4(ol[0], ol[1], ol[2], ol[3]);
    }
    __syncthreads();
    static_assert(sizeof(lds.k) + sizeof(lds.v) >= kLatentRows * VHEAD * 2, "the tile buffers hold the output rows");
    unsigned short *stage = reinterpret_cast<unsigned short *>(&lds);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 l = lds.denominator[4 * half + i][g];
        const float inv_l[4] = {1.0f / (l.x + 1e-6f), 1.0f / (l.y + 1e-6f), 1.0f / (l.z + 1e-6f), 1.0f / (l.w + 1e-6f)};
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            unsigned short *row = stage + (64 * half + 16 * i + 4 * g + rr) * VHEAD + 16 * kCols * quarter + c;
#pragma unroll
            for (int e = 0; e < kCols; ++e) {
                row[16 * e] = static_cast<unsigned short>(T::packProducts(o[i][e][rr], 0.0f, inv_l[rr]));
            }
        }
    }
    __syncthreads();
    static_assert(G::kChunksPerRowV == 64, "a wavefront stores one row at a time");
    for (int i = 0; i < kLatentRows / kWaves; ++i) {
        const int local_row = w * (kLatentRows / kWaves) + i;
        const int row = block_row0 + local_row;
        if (row >= total_rows) {
            break;
        }
        const int token = row / a.group;
        if (visibleTokens(span, token) <= 0) {
            continue;
        }
        const int head = kv_head * a.group + (row - token * a.group);
        const uint4 x = *reinterpret_cast<const uint4 *>(stage + local_row * VHEAD + 8 * lane);
        S *o_ptr = static_cast<S *>(a.out) + (span.q_start + token) * a.o_stride + head * a.o_head_stride;
        *reinterpret_cast<uint4 *>(o_ptr + 8 * lane) = x;
    }
}

} // namespace op::paged_attention_prefill::amd

#endif
