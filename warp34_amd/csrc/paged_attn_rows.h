// Paged GQA decode / verify attention over pages whose rows are read as stored: 16-bit rows
// (FP16 or BF16 storage, identity transform) and the 8-bit rows FP8-E4M3-256 and Q8_0-64, for
// gfx950.  Same work decomposition, chunk geometry, wave merge and split-K partial format as
// the TQ4 kernel in paged_attn.hip (which includes this file); only the per-unit body differs:
//   * the keys are dealt to the waves in halves of 16 tokens; the 16 K rows and 16 V rows of a half
//     go straight from the pages into the wave's private LDS area (LDS-direct loads, one half
//     ahead), laid out so that the operand reads do not conflict (RowsLds);
//   * S^T = K Q^T: A operand = 16 K rows read from LDS, B operand = the query rows, loaded
//     once in MFMA layout.  8-bit codes are widened to fp16 in registers (exact) and the fp32
//     block scales are applied to per-block partial scores, so K is never rounded;
//   * O^T += V^T P^T over the 16 keys of a half: each lane reads the 8-element slice of its 4 tokens
//     and transposes the 4x8 block in registers.  8-bit V is dequantised to fp16(d * code)
//     on the way, which is what the reference stages (op_paged_attn.cu:59-105).  16x16x16 MFMAs, or where
//     an operand has two parts 16x16x32 ones, whose upper 16 keys are the second part;
//   * BF16 storage: P is split into a bf16 high and low part (over the same value rows) so that the 8-bit
//     mantissa of bf16 does not limit the accuracy of the weighted sum;
//   * 8-bit layers may be stored rotated (WHT256 transform): the query rows are then rotated
//     once per tile and the output is rotated back once (op_kv_cache.cu:443-451,763-783).
// Replaces paged_attention_gqa_bf16_kernel (op_kv_cache.cu:873-1168) and the FP16, Q8_0 and
// FP8 branches of paged_attention_gqa_mma_f16_kernel (op_paged_attn.cu:186-588).
#pragma once

namespace w34 {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kKv16Waves = 8;
// The sparse kernel (qsa_sparse_rows.h) copies its rows through registers.  LDS row strides of 16-bit rows (512 B).  The key operand reads are 128 bits at (row n, piece b)
// for 16 rows x 4 pieces per instruction, the value reads 128 bits at (row 4 b + i, piece n): a
// probe of those two patterns measures the rate of a contiguous read at 544 / 608 / 672 bytes for
// the first and at 576 bytes for the second, 40 % less at 528.
constexpr int kKv16RowStride = 544;                      // key rows
constexpr int kKv16VRowStride = 576;                     // value rows
constexpr int kKv8RowStride = 272;                       // bytes: Q8_0 rows as stored, FP8 rows + 8 pad
constexpr int kKv16Stage = 16 * (kKv16RowStride + kKv16VRowStride);  // K half + V half: 17920 B per wave
constexpr int kKv16ColStride = 264;                      // dwords per column of a merge region (see kMergeColStride)
// byte offset of the (m, l) exchange table: behind both the staging areas and the merge regions
__host__ __device__ constexpr int kv16_ml_offset(int nt) {
    const int loop_bytes = kKv16Waves * kKv16Stage;
    const int region_bytes = kKv16Waves * (nt * 16 * kKv16ColStride) * 4;
    return loop_bytes > region_bytes ? loop_bytes : region_bytes;
}
__host__ __device__ constexpr int kv16_smem_bytes(int nt) {
    return kv16_ml_offset(nt) + (kKv16Waves + 1) * nt * 16 * 2 * 4 + 256;
}

// four E4M3 codes -> four fp16 values (exact)
__device__ __forceinline__ void fp8x4_to_h4(uint32_t w, uint32_t& lo, uint32_t& hi) {
    lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false));
    hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true));
}
// four int8 codes -> four fp16 values (exact): 0x6400 | (q + 128) is 1024 + (q + 128) in fp16
__device__ __forceinline__ void i8x4_to_h4(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const uint32_t u = w ^ 0x80808080u;
    const h2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - bias;
    const h2 c = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - bias;
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, c);
}
// four 8-bit codes -> fp32
template <bool FP8>
__device__ __forceinline__ void codes4_to_f32(uint32_t w, float (&f)[4]) {
    if constexpr (FP8) {
        const f2 a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
        const f2 c = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
        f[0] = a.x, f[1] = a.y, f[2] = c.x, f[3] = c.y;
    } else {
        f[0] = (float)(int8_t)(w & 0xFFu);
        f[1] = (float)(int8_t)((w >> 8) & 0xFFu);
        f[2] = (float)(int8_t)((w >> 16) & 0xFFu);
        f[3] = (float)(int8_t)(w >> 24);
    }
}

template <bool IS_BF16>
__device__ __forceinline__ f4 mfma_x32(u4 a, u4 b, f4 c) {
    if constexpr (IS_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    }
}
__device__ __forceinline__ f4 mfma_x16(u2v a, u2v b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, a), __builtin_bit_cast(h4, b), c, 0, 0, 0);
}
// two floats rounded to bf16 (nearest even), x in the lower half
__device__ __forceinline__ uint32_t pack_bf2(float x, float y) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, bf2));
}

// Staging area of one wave: the K half (16 rows), then the V half, as LDS-direct loads leave them.
//   16-bit rows: an instruction moves 1024 bytes = 2 rows (4 at head dimension 128).  Keys: the LDS
//     address advances by 64 (128) bytes more than that, and inside an instruction the 16-byte
//     pieces of row r are exchanged by r -- piece c of the row lies at c ^ 2 (r & 1) (c ^ 2 (r & 3)) --,
//     which the lanes do by loading from the exchanged address.  The 128-bit operand reads of 16 rows
//     then touch the banks in the same pattern as rows 544 bytes apart do.  Values: contiguous (a
//     read takes the same 256 bytes of four rows whose distance is a multiple of 256 bytes).
//   8-bit rows: contiguous, 272 (Q8_0) or 264 (FP8) bytes per row.
template <int KVF, int HD>
struct RowsLds {
    static constexpr bool kFp8 = KVF == WARP34_KV_FORMAT_FP8_E4M3;
    static constexpr bool k8 = kFp8 || KVF == WARP34_KV_FORMAT_Q8_0;
    static constexpr int kRowBytes = k8 ? (kFp8 ? 264 : 272) : 2 * HD;  // in memory
    static constexpr int kHalf = 16 * kRowBytes;                        // a half: 16 rows, contiguous in a page
    static constexpr int kLoads = (kHalf + 1023) / 1024;                // instructions per half
    static constexpr int kRowsPerLoad = k8 ? 0 : 1024 / kRowBytes;
    static constexpr int kKeyPad = k8 ? 0 : (HD == 256 ? 64 : 128);     // per instruction
    static constexpr int kKeyBytes = k8 ? (kHalf + 15) / 16 * 16 : kLoads * (1024 + kKeyPad);
    // after the loop the area holds the wave's merge region (16 columns) and 1 KB for transposing
    static constexpr int kColStride = HD + 8;                           // dwords, see kMergeColStride
    static constexpr int kRegion = 16 * kColStride * 4;
    static constexpr int kLoop = kKeyBytes + kHalf;
    static constexpr int kStage = kLoop > kRegion + 1024 ? kLoop : kRegion + 1024;
    static_assert(kStage % 16 == 0 && (kColStride * 4) % 256 == 32, "alignment, bank pattern of the merge reads");
};
// LDS of a workgroup with NT column tiles: [staging areas][query operands][(m, l) tables]
template <int KVF, int HD>
__host__ __device__ constexpr int rows_q_offset() {
    return kKv16Waves * RowsLds<KVF, HD>::kStage;
}
template <int KVF, int HD>
__host__ __device__ constexpr int rows_ml_offset(int nt) {
    // One tile of 16-bit rows has its query operands in registers from the start.  At head dimension 128 a workgroup then takes 77 KB
    // and two share a CU: a batch over four kv heads (512 workgroups) runs in one round.  us: 4 x 16 draft tokens on 1 000 / 4 000 /
    // 16 000 keys 14.6 / 24.3 / 53.8 -> 13.3 / 19.7 / 48.0, 8 x 8 14.6 / 29.8 / 64.7 -> 14.0 / 23.7 / 59.8.  A layer step, contexts from
    // an eighth of the length up, against one workgroup per CU: 8 x 16 on 6 000 32.8 -> 28.0, 12 x 16 on 16 000 101 -> 84, 15 x 16 142 -> 138
    // (with the tiles of a request on one XCD, see rows_key_groups: on two, 9 x 16 on 16 000 73.9 -> 82.5, 7 x 8 50.0 -> 53.3).
    return rows_q_offset<KVF, HD>() + (nt == 1 && !RowsLds<KVF, HD>::k8 ? 0 : nt * (HD / 32) * 1024);
}
template <int KVF, int HD>
__host__ __device__ constexpr int rows_smem_bytes(int nt) {
    return rows_ml_offset<KVF, HD>(nt) + kKv16Waves * nt * 16 * 2 * 4;
}

// Chunk grid, P.key_groups > 0: a workgroup's tile, kv head and chunk.  The tiles of a request read the same keys, and workgroups
// go round the XCDs in launch order: blockIdx.x = 8 x tile of the request + XCD, blockIdx.y = a group of keys (request x kv head x
// chunk) of each XCD, so that an XCD's L2 takes a group's keys in once.  False: no such group.
__device__ __forceinline__ bool rows_by_keys(const AttnParams& P, int& tile_z, int& kv_sub, int& chunk) {
    const int group = kXcds * (int)blockIdx.y + ((int)blockIdx.x & (kXcds - 1));
    if (group >= P.key_groups) return false;
    const int kv_subs = P.L.local_kv_heads * P.q_subgroups;
    const int req_head = small_div(group, P.max_chunks);
    const int req = small_div(req_head, kv_subs);
    chunk = group - req_head * P.max_chunks;
    kv_sub = req_head - req * kv_subs;
    tile_z = req * P.bal_tiles + ((int)blockIdx.x >> 3);
    return true;
}

// Chunk grid, P.first_round > 0: the tile of a workgroup where the requests go by length: the longest in the first round of
// workgroups, one per CU, longest first; the others, which share the CUs with them, shortest first, so that the shortest meets the
// longest.  In the requests' own order two long ones may meet on a CU and are done long after the others.  Lane r holds request r,
// at most 64.
__device__ __forceinline__ int rows_longest_first(const AttnParams& P, int lane, int tile_z) {
    const int n = P.B.num_reqs;
    const int place = small_div(tile_z, P.bal_tiles);
    const int len = lane < n ? P.B.seq_lens_after[lane] : 0;
    int longer = 0;  // requests before this lane's
    for (int r = 0; r < n; ++r) {
        const int other = __builtin_amdgcn_readlane(len, r);
        longer += other > len || (other == len && r < lane) ? 1 : 0;
    }
    const int want = place < P.first_round ? place : n - 1 - (place - P.first_round);
    const unsigned long long mine = __ballot(lane < n && longer == want);
    return (int)__builtin_ctzll(mine) * P.bal_tiles + (tile_z - place * P.bal_tiles);
}

// One LDS-direct load instruction: lane l's 16 bytes from base + voffset + IMM to lds_addr + IMM + 16 l.
template <bool STREAM, int IMM>
__device__ __forceinline__ void lds_load_piece(uint32_t voffset, const uint8_t* sbase, uint32_t lds_addr) {
    if constexpr (STREAM) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3 nt"
                     : : "v"(voffset), "s"(sbase), "s"(lds_addr), "n"(IMM) : "memory");
    } else {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3"
                     : : "v"(voffset), "s"(sbase), "s"(lds_addr), "n"(IMM) : "memory");
    }
}
// One half (16 rows): instruction i moves bytes 1024 i .. 1024 i + 1023 to lds_addr + (1024 + PAD) i.
template <bool STREAM, int BYTES, int PAD, int I = 0>
__device__ __forceinline__ void lds_load_half(uint32_t voffset, const uint8_t* sbase, uint32_t lds_addr, int lane) {
    if constexpr (1024 * I < BYTES) {
        constexpr int kImm = 1024 * (I & 3), kBase = 1024 * (I & ~3);  // the immediate holds 12 bits
        if (BYTES - 1024 * I >= 1024 || lane < (BYTES - 1024 * I) / 16)
            lds_load_piece<STREAM, kImm>(voffset, sbase + kBase, lds_addr + (uint32_t)(kBase + PAD * I));
        lds_load_half<STREAM, BYTES, PAD, I + 1>(voffset, sbase, lds_addr, lane);
    }
}

// KVF is the storage format of both slabs.  16-bit pages: TQ doubles as the storage type (F16
// query/output over FP16 pages, BF16 over BF16 pages).  8-bit pages: the MFMAs run in fp16 and
// a BF16 query is converted once.
// NT: 16-column tiles per workgroup.  A verify step has more than 16 query columns per kv head; with two
// tiles the keys are read, and 8-bit codes widened, once for 32 columns.  The accumulators take 64 NT
// registers, so the query operands stay in LDS for NT = 2 and are read again for every half.  Head
// dimension 256 only: at 128 the merge of the waves (2 us per tile) outweighs the keys read once more
// (launch_rows_balanced).
// Bound: one workgroup per CU streams about 20 bytes per ns, what the memory delivers; below some 100 MB the
// launch is the chain arguments - plan - block table - first rows (7 us to the first product), the
// streaming, and the merge of the waves (2.3 us per tile).
// BAL: the tile and its unit range come from `item` (balanced decode, see bal_for_each_piece)
// instead of blockIdx.
// VRES (8-bit rows stored rotated): the value operand is fp16(d * code) and, as the upper 16 keys of the
// same MFMA with the same weights, its rounding residual.  A scale block
// of a rotated row with large entries holds few distinct codes, so part of the fp16 rounding of
// d * code is common to the block, and the inverse rotation of the finished row would gather
// that common part into a single channel.
// HD: the head dimension, 256 or -- 16-bit rows only (op_kv_cache.cu:1227) -- 128.  At 128 a row is
// one 128-element half: four QK operands instead of eight, eight value tiles instead of sixteen,
// and lanes 0-31 carry a finished row.  The split-K partial records keep their 256-float stride.
// MAPPED: chunk grid whose workgroups go by keys or by length (rows_by_keys, rows_longest_first), else in launch order.
// PLAIN: chunk grid in launch order of a batch without masks and window, all q heads of a kv head in a tile, queries as given, page strides below 4 GiB
// (plain_rows): what follows from the host's bounds on it is worked out while the lengths travel.  STREAM: and one tile per request.
template <typename TQ, int NT, int KVF, bool BAL, bool VRES = false, bool STREAM = BAL, int HD = kHeadDim, bool MAPPED = false, bool PLAIN = false>
__device__ __forceinline__ void rows_tile(const AttnParams& P, uint8_t* smem, const BalItem& item) {
    static_assert(!VRES || KVF == WARP34_KV_FORMAT_FP8_E4M3 || KVF == WARP34_KV_FORMAT_Q8_0, "residual operand: 8-bit rows");
    using M = RowsLds<KVF, HD>;
    constexpr bool K8 = M::k8;
    constexpr bool FP8 = M::kFp8;
    static_assert(HD == 256 || (HD == 128 && !K8), "head dimension 128: 16-bit rows only");
    static_assert(NT == 1 || (BAL && HD == 256), "several column tiles: balanced form, head dimension 256");
    constexpr int kM = HD / 32;   // QK operands (32 elements each) per row
    constexpr int kH = HD / 128;  // 128-element halves of a row
    static_assert(K8 || KVF == TQ::kStorageFormat, "16-bit pages are read in the query type");
    constexpr bool IS_BF16 = !K8 && TQ::kStorageFormat == WARP34_KV_FORMAT_BF16;
    constexpr bool Q_BF16 = TQ::kStorageFormat == WARP34_KV_FORMAT_BF16;
    constexpr int kWaves = kKv16Waves;
    constexpr int kRowBytes = M::kRowBytes;

    int tid = (int)threadIdx.x;
    // The next piece works its lane values out again: the compiler kept addresses and the sign bits of the query
    // rotation in registers across the pieces, which the loop over the keys then did not have.  Q8_0 with two
    // column tiles: 256 registers and 10 spilled, reloaded behind the first row loads and waiting for them;
    // now 246 and none, 20 requests x 4 tokens on 3K to 16K keys 57.1 -> 52.5 us.
    if constexpr (BAL) asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int b = lane >> 4;
    const warp34_kv_layer_layout& L = P.L;
    const warp34_attention_batch& B = P.B;

    int tile_z = BAL ? item.req : (int)blockIdx.z;  // tile index (see locate_tile)
    int kv_sub = (int)blockIdx.y, chunk = BAL ? 0 : (int)blockIdx.x;
    if constexpr (MAPPED) {
        if (P.key_groups > 0 && !rows_by_keys(P, tile_z, kv_sub, chunk)) return;
        if constexpr (HD != kHeadDim) {
            if (P.first_round > 0) tile_z = rows_longest_first(P, lane, tile_z);
        }
    }
    const int kv_head = PLAIN ? kv_sub : small_div(kv_sub, P.q_subgroups);
    const int q_head_base = PLAIN ? kv_sub * P.q_group : kv_head * P.gqa + (kv_sub - kv_head * P.q_subgroups) * P.q_group;

    // Query rows in MFMA B layout: lane (n, b) holds Q[column n][32 m + 8 b .. + 7] for m = 0..kM-1.
    // One tile of un-rotated queries comes straight from global memory into registers; the first
    // token of the tile is guessed so that these loads overlap the lookup, a wrong guess is corrected
    // after it.  Rotated queries and several tiles go through the LDS table below.
    const bool rot_q = !PLAIN && K8 && P.rot_q != 0;  // workgroup-uniform
    const bool q_direct = NT == 1 && !rot_q;
    const int tok_tile = BAL ? item.tok_tile : P.tok_tile;
    const int tok_guess = BAL ? item.rq_start + item.tile * tok_tile
                              : min((PLAIN ? STREAM : P.tiles_by_request != 0) ? tile_z : tile_z * tok_tile, B.total_tokens - 1);
    u4 bq[kM];
    auto load_q = [&](int tokbase) {
        const int t = div_q_group(n, P);
        const int a = n - t * P.q_group;
        const int tok = min(tokbase + t, B.total_tokens - 1);
        const uint16_t* qrow = P.q + ((size_t)tok * P.num_q_heads + (size_t)(q_head_base + a)) * HD;
#pragma unroll
        for (int m = 0; m < kM; ++m) bq[m] = *reinterpret_cast<const u4*>(qrow + 32 * m + 8 * b);
    };
    // PLAIN: the lengths and the block-table slice are asked for first, the query rows behind them.
    TileReq a_req{};
    int spec_slot_base = -1, spec_vec = -1, req_guess = tile_z;
    if constexpr (PLAIN) {
        if constexpr (STREAM) {
            a_req = TileReq{B.query_start_loc[tile_z], B.query_start_loc[tile_z + 1], B.seq_lens_after[tile_z], B.context_lens_before[tile_z], 1};
        } else {
            a_req = load_tile_req<true>(P, 0, lane);
            req_guess = min(fast_div(tile_z, P.bal_tiles), B.num_reqs - 1);
        }
        spec_slot_base = div_block(chunk * P.spec_upc * kUnit, P);
        const int slot = spec_slot_base + lane;
        if (slot < B.max_blocks_per_req) spec_vec = B.block_tables[(size_t)req_guess * B.max_blocks_per_req + slot];
    }
    if (q_direct) {
        load_q(tok_guess);
    } else {
#pragma unroll
        for (int m = 0; m < kM; ++m) bq[m] = u4{0u, 0u, 0u, 0u};
    }

    // Speculative block-table load, in flight together with the lookup: it assumes that the
    // request's length is the host's bound max_seq_len and, where a request may have several tiles, that all
    // requests have as many.  A wrong guess is fetched again below, so it changes the latency only, never the result.
    // (4 requests x 16 tokens on 1 000 keys, head dimension 128, with the producer: 18.5 -> 17.4 us a layer.)
    if constexpr (PLAIN) {
    } else if constexpr (BAL) {
        // the piece's first unit is known: its block-table slice is requested with the query rows
        spec_slot_base = div_block(item.u_begin * kUnit, P);
        const int slot = spec_slot_base + lane;
        if (slot < B.max_blocks_per_req) spec_vec = B.block_tables[(size_t)tile_z * B.max_blocks_per_req + slot];
    } else if (B.sliding_window <= 0 && B.max_seq_len > 0) {
        if (!P.tiles_by_request) req_guess = min(fast_div(tile_z, P.bal_tiles), B.num_reqs - 1);
        spec_slot_base = div_block(chunk * P.spec_upc * kUnit, P);
        const int slot = spec_slot_base + lane;
        if (slot < B.max_blocks_per_req)
            spec_vec = B.block_tables[(size_t)req_guess * B.max_blocks_per_req + slot];
    }
    // PLAIN: the first half of this wave if the request is as long as the host's bound, its place in its page, and the slabs
    uint32_t spec_in_page = 0;
    int spec_rel = 0;
    uint64_t k_slab = 0, v_slab = 0;
    if constexpr (PLAIN) {
        k_slab = L.k_base + (uint64_t)(uint32_t)kv_head * L.k_head_stride_bytes;
        v_slab = L.v_base + (uint64_t)(uint32_t)kv_head * L.v_head_stride_bytes;
        const int pos = chunk * P.spec_upc * kUnit + 16 * wave;
        const int slot = div_block(pos, P);
        spec_rel = slot - spec_slot_base;
        spec_in_page = (uint32_t)(pos - slot * L.block_size) * (uint32_t)kRowBytes;
        asm volatile("" : "+s"(spec_rel), "+s"(spec_in_page), "+s"(k_slab), "+s"(v_slab));
    }
    TileInfo ti;
    if constexpr (PLAIN && STREAM) {
        const int lo = __builtin_amdgcn_readfirstlane(a_req.lo), hi = __builtin_amdgcn_readfirstlane(a_req.hi);
        ti = TileInfo{hi > lo, tile_z, lo, hi, __builtin_amdgcn_readfirstlane(a_req.sa), __builtin_amdgcn_readfirstlane(a_req.cb), 0};
    } else if constexpr (PLAIN) {
        ti = locate_tile_of<true>(P, tile_z, lane, a_req);
    } else if constexpr (BAL) {
        ti = TileInfo{true, item.req, item.rq_start, item.rq_end, item.seq_after, item.ctx_before, item.tile};
    } else {
        ti = locate_tile(P, tile_z, lane);
    }
    if (!ti.hit) return;  // no such tile, empty or masked request: outputs untouched
    if (!BAL && ti.req != req_guess) spec_slot_base = -1;
    const int req = ti.req, rq_start = ti.rq_start, rq_end = ti.rq_end;
    const int seq_after = ti.seq_after, ctx_before = ti.ctx_before;
    const int tok0 = rq_start + ti.tile_in_req * tok_tile;
    if (q_direct) {
        if (tok0 != tok_guess) load_q(tok0);  // wave-uniform, rare
        if constexpr (K8 && Q_BF16) {
#pragma unroll
            for (int m = 0; m < kM; ++m)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t w = bq[m][k];
                    bq[m][k] = pack_h2(BF16::to_f32((uint16_t)(w & 0xFFFFu)), BF16::to_f32((uint16_t)(w >> 16)));
                }
        }
    }
    bool tok_ok[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int tok = tok0 + div_q_group(nt * 16 + n, P);
        tok_ok[nt] = tok < B.total_tokens && (BAL || PLAIN || B.valid_token_mask == nullptr ||
                                              B.valid_token_mask[min(tok, B.total_tokens - 1)] != 0);
    }
    int tile_tokens = rq_end - tok0;
    if (tile_tokens > tok_tile) tile_tokens = tok_tile;

    // Column info (per lane = per query column: visible key range; tile-wide: union and intersection
    // of the ranges).  Without a token mask and a window the tile-wide values follow from scalars
    // and the per-lane part waits until the first rows have been requested (see the TQ4 kernel).
    int col_lo[NT], col_hi[NT];
    bool col_ok[NT];
    int u_lo = 0x7fffffff, u_hi = -1;
    int i_lo = 0, i_hi = 0x7fffffff;
    uint32_t ok_mask[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        col_lo[nt] = 0;
        col_hi[nt] = -1;
        col_ok[nt] = false;
        ok_mask[nt] = 0u;
    }
    // (a balanced batch has neither, see launch_rows_balanced)
    const bool simple = BAL || PLAIN || (B.valid_token_mask == nullptr && B.sliding_window <= 0);
    auto column_info = [&](bool accumulate) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int col = nt * 16 + n;
            const int t = div_q_group(col, P);
            const int tok = tok0 + t;
            const bool ok = t < tile_tokens && tok_ok[nt];
            const int q_off = tok - rq_start;
            int mx = (B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW) ? seq_after - 1 : ctx_before + q_off;
            if (mx >= seq_after) mx = seq_after - 1;
            int mn = 0;
            if (!BAL && !PLAIN && B.sliding_window > 0) mn = max(0, ctx_before + q_off - B.sliding_window + 1);
            col_ok[nt] = ok;
            col_lo[nt] = ok ? mn : 0;
            col_hi[nt] = ok ? mx : -1;
            if (ok) {
                if (accumulate) {
                    i_lo = max(i_lo, mn);
                    i_hi = min(i_hi, mx);
                    if (mn <= mx) {
                        u_lo = min(u_lo, mn);
                        u_hi = max(u_hi, mx);
                    }
                }
            } else if (NT == 1) {
#pragma unroll
                for (int m = 0; m < kM; ++m) bq[m] = u4{0u, 0u, 0u, 0u};
            }
            ok_mask[nt] = (uint32_t)(__ballot(ok) & 0xFFFFull);
        }
    };
    if (simple) {
        if (tok0 >= B.total_tokens) return;  // no live column
        const int q_off0 = tok0 - rq_start;
        const bool window = B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW;
        int hi_first = window ? seq_after - 1 : ctx_before + q_off0;
        int hi_last = window ? seq_after - 1 : ctx_before + q_off0 + tile_tokens - 1;
        if (hi_first >= seq_after) hi_first = seq_after - 1;
        if (hi_last >= seq_after) hi_last = seq_after - 1;
        u_lo = 0;
        u_hi = hi_last >= 0 ? hi_last : -1;
        i_lo = 0;
        i_hi = hi_first;
    } else {
        column_info(true);
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            u_lo = min(u_lo, __shfl_xor(u_lo, off, 64));
            u_hi = max(u_hi, __shfl_xor(u_hi, off, 64));
            i_lo = max(i_lo, __shfl_xor(i_lo, off, 64));
            i_hi = min(i_hi, __shfl_xor(i_hi, off, 64));
        }
        uint32_t any = 0;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) any |= ok_mask[nt];
        if (any == 0u) return;
    }
    if (u_hi < 0) u_lo = 0;
    u_lo = __builtin_amdgcn_readfirstlane(u_lo);
    u_hi = __builtin_amdgcn_readfirstlane(u_hi);
    i_lo = __builtin_amdgcn_readfirstlane(i_lo);
    i_hi = __builtin_amdgcn_readfirstlane(i_hi);

    ChunkGeom g;
    int cu_first, cu_end;
    bool as_guessed = false;
    if constexpr (BAL) {
        // the plan counted the units of [0, u_hi]: the batch has no window and no token mask
        g = ChunkGeom{0, (u_hi >> 5) + 1, 0, item.n_chunks};
        cu_first = item.u_begin;
        cu_end = item.u_end;
    } else {
        if (u_lo == 0 && B.max_seq_len > 0 && u_hi == B.max_seq_len - 1) {
            g = ChunkGeom{0, P.spec_units, P.spec_upc, P.spec_chunks};  // as long as the host's bound
            as_guessed = true;
        } else {
            g = chunk_geom(u_lo, u_hi, P.max_chunks, P.few_chunks);
        }
        if (chunk >= g.n_chunks) return;
        cu_first = g.u_first + chunk * g.upc;
        cu_end = cu_first + g.upc;
        if (cu_end > g.u_first + g.n_units) cu_end = g.u_first + g.n_units;
    }

    // ---- staging: LDS-direct loads of half units, K and V one half ahead ------------------------------
    const uint8_t* k_base;
    const uint8_t* v_base;
    if constexpr (PLAIN) {
        k_base = reinterpret_cast<const uint8_t*>((uintptr_t)k_slab);
        v_base = reinterpret_cast<const uint8_t*>((uintptr_t)v_slab);
    } else {
        k_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.k_base) + (size_t)kv_head * L.k_head_stride_bytes;
        v_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.v_base) + (size_t)kv_head * L.v_head_stride_bytes;
    }
    uint8_t* stage = smem + wave * M::kStage;
    const uint8_t* k_rows = stage;
    const uint8_t* v_rows = stage + M::kKeyBytes;
    // (the dynamic LDS block starts at LDS address 0: the kernel has no static LDS, checked on the host)
    const uint32_t k_lds = (uint32_t)(wave * M::kStage), v_lds = k_lds + (uint32_t)M::kKeyBytes;
    const int32_t* req_blocks = B.block_tables + (size_t)req * B.max_blocks_per_req;
    int slot_base = div_block(cu_first * kUnit, P);
    int page_vec;
    // (one assembly statement with its own wait, see the TQ4 kernel: a compiler load here would put a
    // vmcnt(0) in front of every half)
    auto load_page_vec = [&]() {
        const int slot = slot_base + lane;
        int32_t ids = -1;
        if (slot < B.max_blocks_per_req) {
            const int32_t* src = req_blocks + slot;
            asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=v"(ids) : "v"(src) : "memory");
        }
        page_vec = ids;
    };
    // lane l of a load instruction fetches piece l of the 64 it moves; key rows of 16-bit pages with
    // their pieces exchanged (see RowsLds)
    uint32_t k_off = (uint32_t)lane * 16u;
    const uint32_t v_off = (uint32_t)lane * 16u;
    if constexpr (!K8) {
        constexpr int kPieces = kRowBytes / 16;
        const int r = lane / kPieces, c = lane % kPieces;
        k_off = (uint32_t)(r * kRowBytes + 16 * (c ^ (2 * (r & (M::kRowsPerLoad - 1)))));
    }
    const uint8_t* next_k;
    const uint8_t* next_v;
    // rows of the half with index hidx (16 tokens); halves outside the visible range read page 0
    auto locate_half = [&](int hidx) {
        const int pos = hidx * 16;
        const int page_slot = div_block(pos, P);
        const int in_page = pos - page_slot * L.block_size;
        int rel = page_slot - slot_base;
        if (rel >= 64) {  // wave-uniform, at most once per 64 slots
            slot_base = page_slot;
            load_page_vec();
            rel = 0;
        }
        const int32_t pg = __builtin_amdgcn_readlane(page_vec, rel);
        const bool live = pos <= u_hi && pos + 15 >= u_lo && pg >= 0;
        if constexpr (PLAIN) {
            const uint32_t in_bytes = (uint32_t)in_page * (uint32_t)kRowBytes;
            next_k = k_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.k_page_stride_bytes + in_bytes : 0);
            next_v = v_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.v_page_stride_bytes + in_bytes : 0);
            return;
        }
        next_k = k_base + (live ? (size_t)pg * L.k_page_stride_bytes + (size_t)in_page * L.k_token_stride_bytes : 0);
        next_v = v_base + (live ? (size_t)pg * L.v_page_stride_bytes + (size_t)in_page * L.v_token_stride_bytes : 0);
    };
    // STREAM: every key is read by exactly one workgroup (no request has more than one tile), and
    // the loads carry the non-temporal hint, which is worth 8 to 13 % on a plain streaming read of
    // HBM.  Tiles that share a request's keys keep ordinary loads: with the hint the lines are gone
    // when the next tile asks for them.
    auto issue_k = [&]() { lds_load_half<STREAM, M::kHalf, M::kKeyPad>(k_off, next_k, k_lds, lane); };
    auto issue_v = [&]() { lds_load_half<STREAM, M::kHalf, 0>(v_off, next_v, v_lds, lane); };

    f4 o_acc[NT][kH][8];
    float m_run[NT], l_run[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m_run[nt] = kNegBig;
        l_run[nt] = 0.f;
#pragma unroll
        for (int h = 0; h < kH; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) o_acc[nt][h][j] = f4{0.f, 0.f, 0.f, 0.f};
    }
    const float score_scale = B.sm_scale * kLog2e;
    // query operands of tile nt, step m: 1 KB each, lane l's 16 bytes at 16 l
    uint8_t* qtab = smem + rows_q_offset<KVF, HD>();
    auto q_operand = [&](int nt, int m) -> u4 {
        if constexpr (NT == 1) return bq[m];
        else return *reinterpret_cast<const u4*>(qtab + (nt * kM + m) * 1024 + 16 * lane);
    };
    // where this lane reads its key operands (row n, piece 4 m + b): the exchange of the pieces
    // touches bit 1 of the piece number (in b) and, at head dimension 128, bit 2 (in m)
    const uint8_t* ka_even = k_rows;
    const uint8_t* ka_odd = k_rows;
    if constexpr (!K8) {
        constexpr int kRpl = M::kRowsPerLoad;
        const uint8_t* row = k_rows + (n / kRpl) * (1024 + M::kKeyPad) + (n % kRpl) * kRowBytes;
        if constexpr (kRpl == 2) {
            ka_even = ka_odd = row + 16 * (b ^ (2 * (n & 1)));
        } else {
            const int swap = (n >> 1) & 1;
            ka_even = row + 16 * (b ^ (2 * (n & 1))) + 64 * swap;
            ka_odd = row + 16 * (b ^ (2 * (n & 1))) - 64 * swap;
        }
    }

    // One 16-token half.  MASKED = false (wave-uniform): every token is visible to every live column.
    auto process_half = [&](int pos0, const bool MASKED, const bool HAS_NEXT) {
        wait_vm<M::kLoads>();  // this half's keys have landed, its values may still be in flight
        f4 s_acc[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) s_acc[nt] = f4{0.f, 0.f, 0.f, 0.f};
        u4 ka[kM];
        if constexpr (K8) {
            // Codes of row n, elements 32 m + 8 b .. + 7, widened to fp16; one partial score per
            // scale block (FP8: 2 blocks of 128 = m / 4; Q8_0: 4 blocks of 64 = m / 2), combined
            // with the fp32 scales of this lane's 4 tokens.
            constexpr int kBlocks = FP8 ? 2 : 4;
            constexpr int kMPerBlock = 8 / kBlocks;
            uint32_t kc[8][2];
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int off = FP8 ? 32 * m + 8 * b : 68 * (m >> 1) + 4 + 32 * (m & 1) + 8 * b;
                const uint32_t* src = reinterpret_cast<const uint32_t*>(k_rows + n * kRowBytes + off);
                kc[m][0] = src[0];
                kc[m][1] = src[1];
            }
            float dk[4][kBlocks];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int kb = 0; kb < kBlocks; ++kb)
                    dk[i][kb] = *reinterpret_cast<const float*>(k_rows + (4 * b + i) * kRowBytes +
                                                                (FP8 ? 256 + 4 * kb : 68 * kb));
            wait_lds_reads();
            if (HAS_NEXT) issue_k();  // located by the caller
#pragma unroll
            for (int kb = 0; kb < kBlocks; ++kb) {
                f4 part[NT];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) part[nt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int mm = 0; mm < kMPerBlock; ++mm) {
                    const int m = kb * kMPerBlock + mm;
                    uint32_t h0, h1, h2_, h3;
                    if constexpr (FP8) {
                        fp8x4_to_h4(kc[m][0], h0, h1);
                        fp8x4_to_h4(kc[m][1], h2_, h3);
                    } else {
                        i8x4_to_h4(kc[m][0], h0, h1);
                        i8x4_to_h4(kc[m][1], h2_, h3);
                    }
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        part[nt] = mfma_x32<false>(u4{h0, h1, h2_, h3}, q_operand(nt, m), part[nt]);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) s_acc[nt][i] += dk[i][kb] * part[nt][i];
            }
        } else {
#pragma unroll
            for (int m = 0; m < kM; ++m)
                ka[m] = *reinterpret_cast<const u4*>(((m & 1) ? ka_odd : ka_even) + 64 * m);
            wait_lds_reads();
            if (HAS_NEXT) issue_k();
#pragma unroll
            for (int m = 0; m < kM; ++m)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) s_acc[nt] = mfma_x32<IS_BF16>(ka[m], q_operand(nt, m), s_acc[nt]);
        }

        // ---- raw value rows of this lane's tokens 4b .. 4b + 3 ----
        if (HAS_NEXT) {
            wait_vm<M::kLoads>();  // the values have landed, the next half's keys may be in flight
        } else {
            wait_vm<0>();
        }
        u4 vr[K8 ? 1 : kH][4];
        uint32_t vc[K8 ? 2 : 1][4][2];
        float vd[K8 ? 2 : 1][4];
        if constexpr (K8) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint8_t* vrow = v_rows + (4 * b + i) * kRowBytes;
                    const int blk = 2 * h + (n >> 3);  // Q8_0 block of element 128 h + 8 n
                    const int off = FP8 ? 128 * h + 8 * n : 68 * blk + 4 + 8 * (n & 7);
                    const uint32_t* src = reinterpret_cast<const uint32_t*>(vrow + off);
                    vc[h][i][0] = src[0];
                    vc[h][i][1] = src[1];
                    vd[h][i] = *reinterpret_cast<const float*>(vrow + (FP8 ? 256 + 4 * h : 68 * blk));
                }
        } else {
#pragma unroll
            for (int h = 0; h < kH; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    vr[h][i] = *reinterpret_cast<const u4*>(v_rows + (4 * b + i) * kRowBytes + 256 * h + 16 * n);
        }
        wait_lds_reads();
        if (HAS_NEXT) issue_v();
        // rows outside [u_lo, u_hi] count as zeros: unwritten pool memory may hold NaN patterns,
        // and 0 * NaN would poison the P V product
        if (MASKED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int pos = pos0 + 4 * b + i;
                const bool row_ok = pos >= u_lo && pos <= u_hi;
                if constexpr (K8) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        vc[h][i][0] = row_ok ? vc[h][i][0] : 0u;
                        vc[h][i][1] = row_ok ? vc[h][i][1] : 0u;
                        vd[h][i] = row_ok ? vd[h][i] : 0.f;
                    }
                } else {
#pragma unroll
                    for (int h = 0; h < kH; ++h)
#pragma unroll
                        for (int k = 0; k < 4; ++k) vr[h][i][k] = row_ok ? vr[h][i][k] : 0u;
                }
            }
        }

        // ---- online softmax over this lane's 4 tokens ----
        // The weights; two operands (BF16: high and low part of a probability; VRES: the values' rounding residuals) are the halves
        // of one product of 32 keys: the 16x16x32 MFMA takes the time of a 16x16x16 one (17.6 cycles each).  us: 16 requests x 4
        // tokens on 8 000 keys, bf16 56.3 -> 55.1, rotated Q8_0 58.6 -> 56.6, rotated FP8 54.5 -> 53.5.
        constexpr bool kTwo = IS_BF16 || VRES;
        u4 pb[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            // (the MASKED tests sit outside the unrolled loops: one wave-uniform branch per block)
            float sc[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = s_acc[nt][i] * score_scale;
            if (MASKED) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int pos = pos0 + 4 * b + i;
                    const bool vis = (BAL || pos >= col_lo[nt]) && pos <= col_hi[nt];  // (dead columns: col_hi = -1)
                    sc[i] = vis ? sc[i] : kNegBig;
                }
            }
            const float mx = max_over_rows(max3(max3(sc[0], sc[1], sc[2]), sc[3], sc[3]));
            const float m_new = fmaxf(m_run[nt], mx);
            const float alpha = __builtin_amdgcn_exp2f(m_run[nt] - m_new);
            m_run[nt] = m_new;
            float p[4];
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(sc[i] - m_new);
            if (MASKED) {
#pragma unroll
                for (int i = 0; i < 4; ++i) p[i] = sc[i] > 0.5f * kNegBig ? p[i] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) psum += p[i];
            // (without a weight so far the sums are zero; at head dimension 128 the test costs more than the products: 21.2 -> 21.6 us a draft layer)
            const bool scale = alpha != 1.0f && (HD != kHeadDim || l_run[nt] != 0.f);
            l_run[nt] = l_run[nt] * alpha + psum;
            if (__ballot(scale) != 0ull) {
#pragma unroll
                for (int h = 0; h < kH; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j) o_acc[nt][h][j] *= alpha;
            }
            if constexpr (IS_BF16) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint32_t hi = pack_bf2(p[2 * k], p[2 * k + 1]);
                    pb[nt][k] = hi;
                    pb[nt][2 + k] = pack_bf2(p[2 * k] - __uint_as_float(hi << 16), p[2 * k + 1] - __uint_as_float(hi & 0xFFFF0000u));
                }
            } else {
                pb[nt][0] = pack_h2(p[0], p[1]);
                pb[nt][1] = pack_h2(p[2], p[3]);
                pb[nt][2] = pb[nt][0];
                pb[nt][3] = pb[nt][1];
            }
        }

        // ---- O^T += V^T P^T: row r = n of MFMA (h, j) is head dimension 128 h + 8 n + j; its operand
        // holds that element of tokens 4b .. 4b + 3 ----
#pragma unroll
        for (int h = 0; h < kH; ++h) {
            u4 a_v[8];  // (the upper half: the same values again for BF16, the residuals for VRES)
            if constexpr (K8) {
                // fp16(d * code), the value the reference stages (op_paged_attn.cu:59-105)
                float vf[4][8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float f0[4], f1[4];
                    codes4_to_f32<FP8>(vc[h][i][0], f0);
                    codes4_to_f32<FP8>(vc[h][i][1], f1);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        vf[i][k] = vd[h][i] * f0[k];
                        vf[i][4 + k] = vd[h][i] * f1[k];
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (VRES) {
                        uint32_t hi0, lo0, hi1, lo1;
                        split_h2(vf[0][j], vf[1][j], hi0, lo0);
                        split_h2(vf[2][j], vf[3][j], hi1, lo1);
                        a_v[j] = u4{hi0, hi1, lo0, lo1};
                    } else {
                        a_v[j] = u4{pack_h2(vf[0][j], vf[1][j]), pack_h2(vf[2][j], vf[3][j]), 0u, 0u};
                    }
                }
            } else {
                // the 4x8 block of 16-bit values is transposed in registers
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    // 16-bit element j of the four token slices -> (t0,t1), (t2,t3)
                    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
                    const uint32_t t01 = __builtin_amdgcn_perm(vr[h][1][j >> 1], vr[h][0][j >> 1], sel);
                    const uint32_t t23 = __builtin_amdgcn_perm(vr[h][3][j >> 1], vr[h][2][j >> 1], sel);
                    a_v[j] = u4{t01, t23, t01, t23};
                }
            }
            if constexpr (VRES) settle(a_v);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    f4& o = o_acc[nt][h][j];
                    if constexpr (kTwo) {
                        o = mfma_x32<IS_BF16>(a_v[j], pb[nt], o);
                    } else {
                        o = mfma_x16(u2v{a_v[j][0], a_v[j][1]}, u2v{pb[nt][0], pb[nt][1]}, o);
                    }
                }
        }
    };

    // Halves are dealt to the waves round robin, a fixed rule (the result must not depend on timing).
    const int h_end = min(2 * cu_end, (u_hi >> 4) + 1);  // (the last unit may end with an invisible half)
    int hidx = 2 * cu_first + wave;
    if (slot_base == spec_slot_base) {
        page_vec = spec_vec;
    } else {
        load_page_vec();
    }
    // The query operands are touched again after the first rows have been requested (dead columns
    // are zeroed).  Loads return in order: a wait for them placed behind the row loads would wait
    // for the rows too, so the compiler is made to finish them here, where they have long landed.
    // (On every path: the compiler does not connect this test of q_direct with the one at the loads,
    // and would otherwise wait for them once more inside the loop.)
    if constexpr (NT == 1) {
#pragma unroll
        for (int m = 0; m < kM; ++m) asm volatile("" : "+v"(bq[m]));
    }
    asm volatile("" ::"v"(page_vec));
    auto first_rows = [&]() {
        if (hidx < h_end) {
            if (PLAIN && as_guessed && slot_base == spec_slot_base && ti.req == req_guess) {  // (spec_rel < 64: eight halves from the chunk's start on)
                const int32_t pg = __builtin_amdgcn_readlane(page_vec, spec_rel);
                next_k = k_base + (pg >= 0 ? (uint64_t)(uint32_t)pg * (uint32_t)L.k_page_stride_bytes + spec_in_page : 0);
                next_v = v_base + (pg >= 0 ? (uint64_t)(uint32_t)pg * (uint32_t)L.v_page_stride_bytes + spec_in_page : 0);
            } else {
                locate_half(hidx);
            }
            issue_k();
            issue_v();
        }
    };
    if (q_direct) {
        first_rows();
        if (simple) column_info(false);
    } else {
        // The query table: one column per wave at a time, lane l holds elements 4 l .. 4 l + 3 =
        // one half of operand (m = l / 8, k-block (l / 2) % 4).  (The rows are requested behind the
        // query loads: a wait for those would wait for the rows as well.)
        if (simple) column_info(false);
        constexpr int kCols = 16 * NT / kWaves;
        uint2 raw[kCols];
#pragma unroll
        for (int c = 0; c < kCols; ++c) {
            const int col = wave + c * kWaves;
            const int t = div_q_group(col, P);
            const int a = col - t * P.q_group;
            raw[c] = uint2{0u, 0u};
            if (4 * lane < HD && t < tile_tokens) {
                const int tok = min(tok0 + t, B.total_tokens - 1);
                raw[c] = *reinterpret_cast<const uint2*>(P.q + ((size_t)tok * P.num_q_heads + (size_t)(q_head_base + a)) * HD +
                                                         4 * lane);
            }
        }
#pragma unroll
        for (int c = 0; c < kCols; ++c) asm volatile("" ::"v"(raw[c].x), "v"(raw[c].y));
        first_rows();
#pragma unroll
        for (int c = 0; c < kCols; ++c) {
            const int col = wave + c * kWaves;
            uint2 packed = raw[c];
            if constexpr (K8) {
                float v[4] = {TQ::to_f32((uint16_t)(raw[c].x & 0xFFFFu)), TQ::to_f32((uint16_t)(raw[c].x >> 16)),
                              TQ::to_f32((uint16_t)(raw[c].y & 0xFFFFu)), TQ::to_f32((uint16_t)(raw[c].y >> 16))};
                if (rot_q) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = apply_sign(v[k], 4 * lane + k);
                    wht256_wave<NT == 2>(v, lane);
                }
                packed.x = pack_h2(v[0], v[1]);
                packed.y = pack_h2(v[2], v[3]);
            }
            if (4 * lane < HD)
                *reinterpret_cast<uint2*>(qtab + ((col >> 4) * kM + (lane >> 3)) * 1024 +
                                          16 * (16 * ((lane >> 1) & 3) + (col & 15)) + 8 * (lane & 1)) = packed;
        }
        __syncthreads();
        if constexpr (NT == 1) {
#pragma unroll
            for (int m = 0; m < kM; ++m) bq[m] = *reinterpret_cast<const u4*>(qtab + m * 1024 + 16 * lane);
        }
    }
    while (hidx < h_end) {
        const int next_h = hidx + kWaves;
        const bool has_next = next_h < h_end;
        if (has_next) locate_half(next_h);
        const int pos0 = hidx * 16;
        process_half(pos0, !(pos0 >= i_lo && pos0 + 15 <= i_hi), has_next);
        hidx = next_h;
    }
    wait_vm<0>();  // nothing of this wave may still be on its way into LDS when the areas are reused

#pragma unroll
    for (int nt = 0; nt < NT; ++nt) l_run[nt] = sum_over_rows(l_run[nt]);

    // ---- merge of the waves' states (same scheme and region layout as the TQ4 kernel) ----
    // A wave stores one tile of its O as it stands in its own staging area, which nobody else
    // touches; after a barrier wave c adds up column c (and c + 8) of the eight regions, each weighted
    // by 2^(m_w - m_tot), one 128-bit piece per lane and region, and brings the sums into element
    // order through the 1 KB its staging area has left behind the region.
    constexpr int kColStride = M::kColStride;
    float* mlbuf = reinterpret_cast<float*>(smem + rows_ml_offset<KVF, HD>(NT));
    if (b == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            mlbuf[(wave * NT * 16 + nt * 16 + n) * 2 + 0] = m_run[nt];
            mlbuf[(wave * NT * 16 + nt * 16 + n) * 2 + 1] = l_run[nt];
        }
    }
    // element e = 128 h + 8 r + j sits in slot ((h*8 + j)*4 + (r >> 2))*4 + (r & 3): of element 4 lane (the next ones: + 16 each)
    const int merge_e = (4 * lane) & (HD - 1);  // (lanes beyond the row repeat its start and store nothing)
    const int merge_slot = (((merge_e >> 7) * 8 + (merge_e & 7)) * 4 + (merge_e >> 5 & 3)) * 4 + (merge_e >> 3 & 3);
    // finishes column `col` from its sums v (element order of the head dimension) and its state
    auto finish_column = [&](int col, float (&v)[4], float m_col, float l_col) {
        const int t = div_q_group(col, P);
        const int a = col - t * P.q_group;
        const size_t row = (size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + a);
        if (BAL ? item.n_chunks > 1 : P.max_chunks > 1) {
            const size_t prow = BAL ? bal_partial_row(item.slot, (int)gridDim.y, kv_sub, 16 * NT, col)
                                    : row * P.max_chunks + chunk;
            float* dst = P.part_acc + prow * kHeadDim;
            if (4 * lane < HD) *reinterpret_cast<f4*>(dst + 4 * lane) = f4{v[0], v[1], v[2], v[3]};
            if (lane == 0) {
                *reinterpret_cast<f4*>(P.part_ml + prow * 4) = f4{m_col, l_col, (float)g.n_chunks, 0.f};
            }
        } else {
            const float inv = l_col > 0.f ? 1.0f / l_col : 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[k] *= inv;
                asm("" : "+v"(v[k]));  // rounded before the conversion to fp16, as where a merge kernel finishes the row
            }
            if (K8 && P.rot_out) {  // rotated V rows: one inverse rotation of the finished row
                wht256_wave<NT == 2>(v, lane);
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = apply_sign(v[k], 4 * lane + k);
            }
            store_out_row<TQ, HD>(P, row, lane, v);
        }
    };
    float* region = reinterpret_cast<float*>(stage);
    float* tbuf = region + 16 * kColStride;
    // (rolled loops: this code runs once per workgroup, and a workgroup of a small batch waits for its
    // instructions to come from memory)
#pragma unroll 1
    for (int nt = 0; nt < NT; ++nt) {
        if (nt > 0) __syncthreads();  // the previous tile's regions have been read
        uint32_t live = 0;
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            if (k != nt) continue;  // wave-uniform
            live = ok_mask[k];
            if ((live >> n) & 1u) {
                float* c = region + n * kColStride;
#pragma unroll
                for (int h = 0; h < kH; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j) *reinterpret_cast<f4*>(c + ((h * 8 + j) * 4 + b) * 4) = o_acc[k][h][j];
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int col = wave; col < 16; col += kWaves) {
            if (!((live >> col) & 1u)) continue;
            float mw[kWaves], lw[kWaves];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const f2 r = *reinterpret_cast<const f2*>(mlbuf + (w * NT * 16 + nt * 16 + col) * 2);
                mw[w] = r[0];
                lw[w] = r[1];
            }
            float m_col = kNegBig, l_col = 0.f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) m_col = fmaxf(m_col, mw[w]);
            f4 tot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const float wgt = __builtin_amdgcn_exp2f(mw[w] - m_col);
                l_col += lw[w] * wgt;
                // (head dimension 128: the upper lanes read what the lower ones read and drop it)
                tot += *reinterpret_cast<const f4*>(smem + w * M::kStage + (col * kColStride + ((4 * lane) & (HD - 1))) * 4) * wgt;
            }
            *reinterpret_cast<f4*>(tbuf + 4 * lane) = tot;
            float v[4];  // the reads follow the write of the same wave in LDS order
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = tbuf[merge_slot + 16 * k];
            finish_column(nt * 16 + col, v, m_col, l_col);
        }
    }
}

template <typename TQ, int KVF, bool VRES, int HD = kHeadDim>
__global__ __launch_bounds__(kKv16Waves * 64, 1) void paged_attn_rows_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    // (one body per kind of load: a branch around the loads themselves keeps the compiler from
    // scheduling them freely and loses what the hint gains)
    if (P.tiles_by_request != 0 && P.q_subgroups == 1) {  // uniform for the grid
        rows_tile<TQ, 1, KVF, false, VRES, true, HD>(P, smem, BalItem{});
    } else {
        rows_tile<TQ, 1, KVF, false, VRES, false, HD>(P, smem, BalItem{});
    }
}
// Without masks and windows, in launch order, see plain_rows; the bits of the kernel above.
template <typename TQ, int KVF, int HD, bool ONE_TILE>
__global__ __launch_bounds__(kKv16Waves * 64, 1) void paged_attn_rows_plain_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    rows_tile<TQ, 1, KVF, false, false, ONE_TILE, HD, false, true>(P, smem, BalItem{});
}
// The chunk grid by keys or by length.  (A kernel of its own: with the order worked out in the other, or a third body in it, chunks of 130 tokens
// over bf16 pages, which stay in launch order, took 4 to 5 % longer with the same instructions in the loop: 67.9 -> 71.8 us.)
template <typename TQ, int KVF, bool VRES, int HD = kHeadDim>
__global__ __launch_bounds__(kKv16Waves * 64, 1) void paged_attn_rows_mapped_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    rows_tile<TQ, 1, KVF, false, VRES, false, HD, true>(P, smem, BalItem{});
}

template <typename TQ, int NT, int KVF, bool VRES, bool STREAM, int HD = kHeadDim>
__global__ __launch_bounds__(kKv16Waves * 64, 1) void paged_attn_rows_balanced_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    bal_for_each_piece<(NT > 1 || (VRES && !STREAM)), kFewChunksRows, kGridUnitsRows>(
        P, [&](const BalItem& it) { rows_tile<TQ, NT, KVF, true, VRES, STREAM, HD>(P, smem, it); },
        [&] {
            const AttnParams A = kernel_params_again();
            // (several tiles per request: ordinary loads)
            bal_short_piece(A, [&](const BalItem& it) { rows_tile<TQ, 1, KVF, true, VRES, false, HD>(A, smem, it); });
        });
}

}  // namespace w34
