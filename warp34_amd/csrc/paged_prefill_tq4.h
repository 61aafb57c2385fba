// Chunked-prefill attention over TQ4 pages in tiles of 128 query rows (batches of fewer than 250 wide tiles, see
// launch_prefill_tq4, and the shared-prefix pass), and what it shares with the wide kernel (paged_prefill_wide.h): every K/V unit is
// dequantised ONCE per workgroup and shared by all waves through LDS.
// Replaces paged_attention_prefill_mma_f16_kernel + launch_prefill
// (op_paged_attn.cu:594-1128,1220-1259).  Included by paged_attn.hip.
//
// Workgroup = 12 waves = one tile of 128 query rows (128 / q_group consecutive tokens of ONE
// request x q_group heads of one kv head); wave w < 8 owns rows 16 w .. 16 w + 15 as the 16 columns
// of its MFMA results (S^T = K Q'^T, O^T += V^T P^T, as in the decode kernel, so the softmax
// state is one scalar pair per lane), waves 8-11 load and dequantise.  The workgroup walks the request's keys in 32-token
// units with a three-stage software pipeline and ONE barrier per unit:
//   load   : unit u+3, 16-byte pieces of the raw K / V rows, global -> registers
//   commit : unit u+2, registers -> raw LDS buffer
//   dequant: unit u+1, raw LDS -> fp16 centroids through the pair table, written in the
//            layouts the MFMAs read: K as [token][256] rows (544-byte stride), V transposed as
//            [dim][32 key slots] with the 16-byte pieces XOR-swizzled, scales as fp32
//   compute: unit u, 16 QK + 32 PV MFMAs per wave, operands read with 128-bit LDS loads
// Scales are not applied per element: K scales multiply the two half-row partial scores,
// V scales are folded into the probabilities, exactly as in the decode kernel.
#pragma once

namespace w34 {

constexpr int kPfWaves = 8;
constexpr int kPfRows = 128;                                  // query rows per workgroup
constexpr int kPfKStride = 544;                               // bytes per dequantised K row (measured: 128-bit reads of 16 rows at this stride do not conflict; 528, 560, 576 do)
constexpr int kPfKBytes = 32 * kPfKStride;                    // 16896
constexpr int kPfVBytes = 256 * 64;                           // V^T: 256 rows x 32 halves
constexpr int kPfScaleBytes = 8 * 32 * 4;                     // per token: K d0, K d1, V d0, V d1 (Q8_0: K d0-d3, V d0-d3)
constexpr int kPfDeqBytes = kPfKBytes + kPfVBytes + kPfScaleBytes;
// LDS map per page format: [table (TQ4 only)] [2 dequantised units] [2 raw units]
template <int KVF>
struct PfLds {
    static constexpr bool kFp8 = KVF == WARP34_KV_FORMAT_FP8_E4M3;
    static constexpr bool k16 = KVF == WARP34_KV_FORMAT_FP16 || KVF == WARP34_KV_FORMAT_BF16;
    static constexpr bool kQ8 = KVF == WARP34_KV_FORMAT_Q8_0;
    static constexpr int kRowBytes = k16 ? 512 : kFp8 ? 264 : kQ8 ? 272 : kTq4RowBytes;
    static constexpr int kRun = 16 * kRowBytes;                // 16 rows: 2112 B / 4224 B / 4352 B / 8192 B
    static constexpr int kRaw = 4 * kRun;                      // K rows 0-31, V rows 0-31
    static constexpr int kDeqBase = (kFp8 || k16 || kQ8) ? 0 : kLutBytes;
    static constexpr int kRawBase = kDeqBase + 2 * kPfDeqBytes;
    static constexpr int kEpilogue = kPfWaves * 16 * 260 * 4;  // the output transpose regions
};
constexpr int kPfSmem = PfLds<WARP34_KV_FORMAT_TQ4>::kRawBase + 2 * PfLds<WARP34_KV_FORMAT_TQ4>::kRaw + 256;
static_assert(kPfSmem >= PfLds<WARP34_KV_FORMAT_TQ4>::kEpilogue && kPfSmem <= 160 * 1024, "prefill LDS budget");
static_assert(PfLds<WARP34_KV_FORMAT_TQ4>::kRaw == kStageTq4, "TQ4 raw unit");
static_assert(kPfWaves * 16 * 264 * 2 <= 2 * kPfDeqBytes, "query staging must fit in the dequant buffers");

typedef __attribute__((address_space(3))) uint32_t lds_u32;

// 16x16x32 MFMA on fp16 or bf16 operands given as raw bits
template <bool IS_BF16>
__device__ __forceinline__ f4 pf_mfma32(h8 a, h8 b, f4 c) {
    if constexpr (IS_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
}

__device__ __forceinline__ float max2(float a, float b) {  // (see max3)
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// High and low fp16 operands of the weights p0 d0 | p1 d1
__device__ __forceinline__ void weight_h2(float p0, float p1, float d0, float d1, uint32_t& hi, uint32_t& lo) {
    split_weights(mul_legacy(p0, d0), mul_legacy(p1, d1), hi, lo);
}

// Which tile a workgroup takes: the n-th longest of the batch.  A causal tile's length is known up to a
// tile as (context / tile_tok) + its index in the request; the host knows neither the requests'
// contexts nor their numbers of new tokens.  In launch order -- requests one after the other, short
// tiles first -- a batch of 1 to 2 tiles per CU ended with long tiles started late: three requests of
// 1365, 722 and 1214 new tokens on 1 600 to 1 700 of context (416 tiles of 52 to 94 units, 115 per CU)
// needed the time of 176 units.  Tiles of equal length go round the requests, which
// also puts the requests of an even batch on XCDs of their own.  Lane r holds request r: at most 64.
struct PfTile {
    int req, tile;
};
__device__ __forceinline__ PfTile pf_longest_first(const AttnParams& P, int lane, int rank) {
    const warp34_attention_batch& B = P.B;
    int first = 0, count = 0;  // the request's tiles have the lengths first .. first + count - 1
    if (lane < B.num_reqs && (B.valid_req_mask == nullptr || B.valid_req_mask[lane] != 0)) {
        const int q_len = B.query_start_loc[lane + 1] - B.query_start_loc[lane];
        const int ctx = B.context_lens_before != nullptr ? B.context_lens_before[lane] : B.seq_lens_after[lane] - q_len;
        count = q_len > 0 ? (q_len + P.tok_tile - 1) / P.tok_tile : 0;
        first = ctx > 0 ? ctx / P.tok_tile : 0;
    }
    auto wave_sum = [&](int x) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
        return __builtin_amdgcn_readfirstlane(x);
    };
    auto longer = [&](int length) {  // tiles of at least this length
        return wave_sum(max(0, min(count, first + count - length)));
    };
    int lo = 0, hi = first + count;  // longer(lo) > rank, longer(hi) <= rank
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) hi = max(hi, __shfl_xor(hi, off, 64));
    hi = __builtin_amdgcn_readfirstlane(hi);
    if (longer(0) <= rank) return PfTile{-1, 0};
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (longer(mid) > rank) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    // the (rank - longer(hi))-th request that has a tile of length lo
    const unsigned long long has = __ballot(first <= lo && lo < first + count);
    const int nth = rank - longer(hi);
    const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
    const unsigned long long mine = __ballot(((has >> lane) & 1ull) != 0 && before == nth);
    const int req = (int)__builtin_ctzll(mine);
    return PfTile{req, lo - __builtin_amdgcn_readlane(first, req)};
}

// Waves 0-7 only multiply (16 columns each); waves 8-11 load and dequantise the next unit, a whole 16-row run each.  Every
// SIMD then holds two multiplying waves and one dequantising wave whose instruction streams never wait
// for each other's results inside an iteration.
// SPLIT: blockIdx.x = tile * P.pf_split + part; a workgroup takes one of P.pf_split equal
// parts of the tile's units and leaves un-normalised partial records (slot P.pf_slot_base + part
// of every row, the decode kernels' format) for the merge kernel.
template <typename TQ, bool SPLIT>
__global__ __launch_bounds__(12 * 64, 1) void paged_prefill_tq4_kernel(const AttnParams P) {
    using M = PfLds<WARP34_KV_FORMAT_TQ4>;
    constexpr int kPfDeqBase = M::kDeqBase, kPfRawBase = M::kRawBase, kPfRawBytes = M::kRaw;
    constexpr int kRunB = M::kRun;
    extern __shared__ __align__(16) uint8_t smem[];
    // (the pair table is addressed absolutely: the dynamic block starts at LDS address 0 because the
    // kernel has no static LDS, which the host checks before the first launch)

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int b = lane >> 4;
    const bool producer = wave >= kPfWaves;  // wave-uniform
    const warp34_kv_layer_layout& L = P.L;
    const warp34_attention_batch& B = P.B;

    // ---- tile identification ----
    // SPLIT: blockIdx = (tile x part, kv head x q subgroup, 0).  Else the grid holds (tiles of a request, kv
    // heads x q subgroups, requests) workgroups; taken in launch order they get the tiles longest first,
    // the heads of a tile next to each other.  More than 64 requests: in grid order.
    int req = (int)blockIdx.z, kv_sub = (int)blockIdx.y;
    int tile_x = SPLIT ? (int)blockIdx.x / P.pf_split : (int)(gridDim.x - 1 - blockIdx.x);
    const int part_x = SPLIT ? (int)blockIdx.x - tile_x * P.pf_split : 0;
    if (!SPLIT && B.num_reqs <= 64) {
        const uint32_t at = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const uint32_t rank = at / gridDim.y;
        kv_sub = (int)(at - rank * gridDim.y);
        const PfTile t = pf_longest_first(P, lane, (int)rank);
        if (t.req < 0) return;
        req = t.req;
        tile_x = t.tile;
    }
    const int kv_head = fast_div(kv_sub, P.q_subgroups);
    const int q_head_base = kv_head * P.gqa + (kv_sub - kv_head * P.q_subgroups) * P.q_group;
    if (B.valid_req_mask != nullptr && B.valid_req_mask[req] == 0) return;
    const int rq_start = B.query_start_loc[req];
    const int rq_end = B.query_start_loc[req + 1];
    const int seq_after = B.seq_lens_after[req];
    const int ctx_before = B.context_lens_before != nullptr ? B.context_lens_before[req]
                                                            : seq_after - (rq_end - rq_start);
    const int tile_tok = P.tok_tile;  // 128 / q_group
    const int tok0 = rq_start + tile_x * tile_tok;
    if (tok0 >= rq_end || tok0 >= B.total_tokens) return;
    int tile_tokens = rq_end - tok0;
    if (tile_tokens > tile_tok) tile_tokens = tile_tok;
    if (tile_tokens > B.total_tokens - tok0) tile_tokens = B.total_tokens - tok0;

    // ---- the pair table (64 lane replicas, as in the decode kernel) ----
    if (tid < kPfWaves * 64) {
        const int e = tid >> 1;
        const uint32_t v = centroid_bits((uint32_t)e & 15u) | centroid_bits((uint32_t)e >> 4) << 16;
        u4 vv = {v, v, v, v};
        u4* dst = reinterpret_cast<u4*>(smem + e * 256 + (tid & 1) * 128);
#pragma unroll
        for (int k = 0; k < 8; ++k) dst[k] = vv;
    }

    // ---- key range of every column; workgroup-wide unit range ----
    const int q_off0 = tok0 - rq_start;
    auto range_hi = [&](int q_off) {
        int mx = (B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW) ? seq_after - 1 : ctx_before + q_off;
        return mx >= seq_after ? seq_after - 1 : mx;
    };
    auto range_lo = [&](int q_off) {
        return B.sliding_window > 0 ? max(0, ctx_before + q_off - B.sliding_window + 1) : 0;
    };
    const int lo_all = range_lo(q_off0);
    const int hi_all = range_hi(q_off0 + tile_tokens - 1);
    int u_first = lo_all >> 5;
    int n_units = hi_all >= lo_all ? (hi_all >> 5) - u_first + 1 : 0;
    if constexpr (SPLIT) {  // this workgroup's part of the units
        const int per_part = (n_units + P.pf_split - 1) / P.pf_split;
        const int first = part_x * per_part;
        int n = n_units - first;
        n = n < 0 ? 0 : (n > per_part ? per_part : n);
        u_first += first;
        n_units = n;
    }

    const int my_col = 16 * wave + n;
    const int my_t = div_q_group(my_col, P);
    const int my_tok = tok0 + my_t;
    const bool col_ok = my_t < tile_tokens &&
                        (B.valid_token_mask == nullptr || B.valid_token_mask[min(my_tok, B.total_tokens - 1)] != 0);
    const int col_lo = col_ok ? range_lo(q_off0 + my_t) : 0;
    const int col_hi = col_ok ? range_hi(q_off0 + my_t) : -1;
    const uint32_t ok_mask = (uint32_t)(__ballot(col_ok) & 0xFFFFull);
    int i_lo = col_ok ? col_lo : 0, i_hi = col_ok ? col_hi : 0x7fffffff;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        i_lo = max(i_lo, __shfl_xor(i_lo, off, 64));
        i_hi = min(i_hi, __shfl_xor(i_hi, off, 64));
    }
    i_lo = __builtin_amdgcn_readfirstlane(i_lo);
    i_hi = __builtin_amdgcn_readfirstlane(i_hi);

    // ---- rotated, scaled queries of this wave's 16 columns -> LDS -> MFMA B operands ----
    constexpr int kQStride = 264;
    _Float16* qbuf = reinterpret_cast<_Float16*>(smem + kPfDeqBase) + wave * 16 * kQStride;
    const float q_scale = B.sm_scale * kLog2e * kLutInvGain;
    const bool rot_q = P.rot_q != 0;
    const bool rot_out = P.rot_out != 0;
    if (!producer) {
        uint2 q_raw[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int col = 16 * wave + c;
            const int t = div_q_group(col, P);
            const int a = col - t * P.q_group;
            const int tok = min(tok0 + t, B.total_tokens - 1);
            const uint16_t* qrow = P.q + ((size_t)tok * P.num_q_heads + (size_t)(q_head_base + a)) * kHeadDim;
            q_raw[c] = *reinterpret_cast<const uint2*>(qrow + 4 * lane);
        }
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            float v[4];
            v[0] = TQ::to_f32((uint16_t)(q_raw[c].x & 0xFFFFu));
            v[1] = TQ::to_f32((uint16_t)(q_raw[c].x >> 16));
            v[2] = TQ::to_f32((uint16_t)(q_raw[c].y & 0xFFFFu));
            v[3] = TQ::to_f32((uint16_t)(q_raw[c].y >> 16));
            if (rot_q) {  // keys stored rotated: rotate the query rows
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = apply_sign(v[k], 4 * lane + k);
                wht256_wave(v, lane);
            }
            uint2 packed = {0u, 0u};  // dead columns: zero query
            if ((ok_mask >> c) & 1u) {
                packed.x = pack_h2(v[0] * q_scale, v[1] * q_scale);
                packed.y = pack_h2(v[2] * q_scale, v[3] * q_scale);
            }
            *reinterpret_cast<uint2*>(qbuf + c * kQStride + 4 * lane) = packed;
        }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    h8 bq[2][4];  // [half of the head dim][32-wide k step]: Q'[col n][128 h + 32 m + 8 b ..]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < 4; ++m)
            bq[h][m] = producer ? h8{} : *reinterpret_cast<const h8*>(qbuf + n * kQStride + 128 * h + 32 * m + 8 * b);

    // ---- loader ----
    // A unit is four runs of 16 rows: K rows 0-15, K rows 16-31, V rows 0-15, V rows 16-31.  A run is 2112 B = 132 16-byte
    // pieces: one run per dequantising wave, two pieces per lane, lanes 0-3 also carry the tail pieces 128-131.
    const uint8_t* k_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.k_base) +
                            (size_t)kv_head * L.k_head_stride_bytes;
    const uint8_t* v_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.v_base) +
                            (size_t)kv_head * L.v_head_stride_bytes;
    const int32_t* req_blocks = B.block_tables + (size_t)req * B.max_blocks_per_req;
    const int ld_run = (wave - kPfWaves) & 3;
    const bool ld_is_v = ld_run >= 2;
    const uint8_t* ld_base = ld_is_v ? v_base : k_base;
    const uint64_t ld_page_stride = ld_is_v ? L.v_page_stride_bytes : L.k_page_stride_bytes;
    const uint64_t ld_tok_stride = ld_is_v ? L.v_token_stride_bytes : L.k_token_stride_bytes;
    const uint32_t ld_lane_off = (uint32_t)(16 * lane);
    const uint32_t ld_tail_off = (uint32_t)(2048 + 16 * (lane & 3));
    const uint32_t ld_commit0 = (uint32_t)(ld_run * kRunB) + ld_lane_off;
    const uint32_t ld_commit1 = (uint32_t)(ld_run * kRunB) + ld_tail_off;
    u4 pf[3];
    // page id of unit k (relative to u_first) for this wave's run; -1 = nothing to fetch.
    // Only groups that overlap the visible key range are fetched: block-table entries beyond
    // the request's pages are unspecified.
    auto load_page = [&](int k) -> int32_t {
        const int pos = (u_first + k) * kUnit + 16 * (ld_run & 1);
        const int slot = __builtin_amdgcn_readfirstlane(div_block(pos, P));
        const bool live = k < n_units && pos <= hi_all && pos + 15 >= lo_all && slot < B.max_blocks_per_req;
        int32_t pg = -1;
        if (live) pg = req_blocks[slot];
        return pg;  // wave-uniform value in a vector register: made scalar where it is used, an iteration later
    };
    auto issue_loads = [&](int k, int32_t pg) {
        const int pos = (u_first + k) * kUnit + 16 * (ld_run & 1);
        const int slot = __builtin_amdgcn_readfirstlane(div_block(pos, P));
        const int in_page = pos - slot * L.block_size;
        size_t off = 0;  // missing page: rows of page 0, every one of them is masked
        if (pg >= 0) off = (size_t)pg * ld_page_stride + (size_t)in_page * ld_tok_stride;
        const uint8_t* src = ld_base + off;
        pf[0] = *(global_cu4*)(src + ld_lane_off);
        pf[1] = *(global_cu4*)(src + ld_tail_off);
        pf[2] = *(global_cu4*)(src + ld_lane_off + 1024);
    };
    auto commit_loads = [&](int buf) {
        uint8_t* raw = smem + kPfRawBase + buf * kPfRawBytes;
        *reinterpret_cast<u4*>(raw + ld_commit0) = pf[0];
        if (lane < 4) *reinterpret_cast<u4*>(raw + ld_commit1) = pf[1];
        *reinterpret_cast<u4*>(raw + ld_commit0 + 1024) = pf[2];
    };

    // ---- dequantiser ----
    // A raw row is 33 dwords; dwords 0 and 16 hold two scale bytes and two code bytes each.
    // They are fused into one synthetic dword [code bytes 0,1 | code bytes 62,63], which leaves
    // exactly 32 four-code-byte items per row:
    //   item 0      : alignbit(dword 16, dword 0, 16)  -> elements 0..3 and 124..127
    //   item j 1..15: dword j                          -> elements 8 j - 4 .. 8 j + 3
    //   item j 16..31: dword j + 1                     -> elements 8 j .. 8 j + 7
    // K: 32 rows x 32 items = four per thread (item idx = thread + 256 i: row idx >> 5, j = idx & 31);
    //    the four looked-up pairs are written as two 8-byte stores into the row-major fp16 tile.
    // V: 16 token pairs x 32 items = two per thread (pair p = thread & 15, j = (thread >> 4) + 16 i).  Tokens
    //    2p, 2p+1 sit in key slots 8 b' + 4 s + {0,1} (+2 for odd p), s = p >> 3, b' = (p >> 1) & 3;
    //    element d lives in V^T row d, 16-byte piece b' ^ ((d >> 1) & 3).  Lanes whose
    //    (lane >> 4) is odd write the odd elements first so that a 32-lane write pass covers
    //    32 banks.
    const uint32_t lut_lane = (uint32_t)lane << 2;
    auto item_src = [](int j, uint32_t (&src)[2], uint32_t& shift) {
        // byte offsets of the two dwords inside the row, and the alignbit shift
        if (j == 0) {
            src[0] = 0;
            src[1] = 64;
            shift = 16;
        } else {
            const int w = j < 16 ? j : j + 1;
            src[0] = src[1] = 4u * (uint32_t)w;
            shift = 0;
        }
    };
    constexpr int kDqThreads = 256;
    constexpr int kKItems = 1024 / kDqThreads, kVItems = 512 / kDqThreads;
    const int dq_tid = (tid - kPfWaves * 64) & 255;
    uint32_t k_src[kKItems][2], k_shift[kKItems], k_dst[kKItems][2];
#pragma unroll
    for (int it = 0; it < kKItems; ++it) {
        const int idx = dq_tid + kDqThreads * it;
        const int r = idx >> 5, j = idx & 31;
        uint32_t src[2];
        item_src(j, src, k_shift[it]);
        k_src[it][0] = (uint32_t)(r * kTq4RowBytes) + src[0];
        k_src[it][1] = (uint32_t)(r * kTq4RowBytes) + src[1];
        const int d_lo = j == 0 ? 0 : j < 16 ? 8 * j - 4 : 8 * j;   // element of code byte 0
        const int d_hi = j == 0 ? 124 : d_lo + 4;                    // element of code byte 2
        k_dst[it][0] = (uint32_t)(r * kPfKStride + 2 * d_lo);
        k_dst[it][1] = (uint32_t)(r * kPfKStride + 2 * d_hi);
    }
    const int nibsel = (lane >> 4) & 1;
    uint32_t v_src[kVItems][2], v_shift[kVItems], v_dst[kVItems][4];
#pragma unroll
    for (int vi = 0; vi < kVItems; ++vi) {
        const int p = dq_tid & 15, j = (dq_tid >> 4) + (kDqThreads / 16) * vi;  // (j keeps the parity of lane >> 4)
        uint32_t src[2];
        item_src(j, src, v_shift[vi]);
        v_src[vi][0] = (uint32_t)(kPfRawBytes / 2 + (2 * p) * kTq4RowBytes) + src[0];
        v_src[vi][1] = (uint32_t)(kPfRawBytes / 2 + (2 * p) * kTq4RowBytes) + src[1];
        const int bp = (p >> 1) & 3, s = p >> 3;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = j == 0 ? (q < 2 ? 2 * q : 120 + 2 * q) : (j < 16 ? 8 * j - 4 : 8 * j) + 2 * q;
            v_dst[vi][q] = (uint32_t)(kPfKBytes + d * 64 + 16 * (bp ^ ((d >> 1) & 3)) + 8 * s + 4 * (p & 1) + 64 * nibsel);
        }
    }
    // ---- per-wave attention state ----
    f4 o_acc[2][8];
    // Until every live column has a maximum (`started`) that of a column without one is 0, and so is its sum (see the decode kernel).
    bool started = false;
    float m_run = 0.f, l_run = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) o_acc[h][j] = f4{0.f, 0.f, 0.f, 0.f};

    // Three phases, each a batch of independent LDS operations: all raw reads, all table reads,
    // all writes.  (Written item by item, every item's reads would have to wait for the previous
    // item's writes: the compiler cannot prove that they do not alias.)
    auto dequant_unit = [&](int rawbuf, int deqbuf) {
        const uint32_t raw = (uint32_t)(kPfRawBase + rawbuf * kPfRawBytes);
        const uint32_t deq = (uint32_t)(kPfDeqBase + deqbuf * kPfDeqBytes);
        // ---- phase 1: raw dwords ----
        uint32_t kw0[kKItems], kw1[kKItems];
#pragma unroll
        for (int it = 0; it < kKItems; ++it) {
            kw0[it] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + k_src[it][0]));
            kw1[it] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + k_src[it][1]));
        }
        uint32_t a0[kVItems], a1[kVItems], b0[kVItems], b1[kVItems];
#pragma unroll
        for (int vi = 0; vi < kVItems; ++vi) {
            a0[vi] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + v_src[vi][0]));
            a1[vi] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + v_src[vi][1]));
            b0[vi] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + v_src[vi][0] + kTq4RowBytes));
            b1[vi] = *reinterpret_cast<lds_cu32*>((uintptr_t)(raw + v_src[vi][1] + kTq4RowBytes));
        }
        // scales: thread x * 32 + r (x = 0: K d0, 1: K d1, 2: V d0, 3: V d1) of the first two dequantising waves
        uint16_t scale_bits = 0;
        if (dq_tid < 128) {
            const int x = dq_tid >> 5, r = dq_tid & 31;
            scale_bits = *reinterpret_cast<const uint16_t*>(smem + raw + (x >> 1) * (kPfRawBytes / 2) +
                                                            r * kTq4RowBytes + (x & 1) * 66);
        }
        // ---- phase 2: table reads ----
        uint2 k_lo[kKItems], k_hi[kKItems];
#pragma unroll
        for (int it = 0; it < kKItems; ++it) {
            const uint32_t word = __builtin_amdgcn_alignbit(kw1[it], kw0[it], k_shift[it]);
            k_lo[it].x = lut_read(word, lut_lane, 0x0c0c0400u);
            k_lo[it].y = lut_read(word, lut_lane, 0x0c0c0500u);
            k_hi[it].x = lut_read(word, lut_lane, 0x0c0c0600u);
            k_hi[it].y = lut_read(word, lut_lane, 0x0c0c0700u);
        }
        uint32_t vx0[kVItems][4], vx1[kVItems][4];
#pragma unroll
        for (int vi = 0; vi < kVItems; ++vi) {
            const uint32_t wa = __builtin_amdgcn_alignbit(a1[vi], a0[vi], v_shift[vi]);
            const uint32_t wb = __builtin_amdgcn_alignbit(b1[vi], b0[vi], v_shift[vi]);
            // byte q of ev / od = (even / odd element of token 2p) | (same of token 2p+1) << 4
            const uint32_t ev = (wa & 0x0F0F0F0Fu) | ((wb << 4) & 0xF0F0F0F0u);
            const uint32_t od = ((wa >> 4) & 0x0F0F0F0Fu) | (wb & 0xF0F0F0F0u);
            const uint32_t first = nibsel ? od : ev;   // elements of parity nibsel, stored at v_dst
            const uint32_t second = nibsel ? ev : od;  // the other parity, one V^T row (64 B) away
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t sel = 0x0c0c0400u + ((uint32_t)q << 8);
                vx0[vi][q] = lut_read(first, lut_lane, sel);
                vx1[vi][q] = lut_read(second, lut_lane, sel);
            }
        }
        // ---- phase 3: writes ----
#pragma unroll
        for (int it = 0; it < kKItems; ++it) {
            *reinterpret_cast<uint2*>(smem + deq + k_dst[it][0]) = k_lo[it];
            *reinterpret_cast<uint2*>(smem + deq + k_dst[it][1]) = k_hi[it];
        }
#pragma unroll
        for (int vi = 0; vi < kVItems; ++vi)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t addr = deq + v_dst[vi][q];
                *reinterpret_cast<uint32_t*>(smem + addr) = vx0[vi][q];
                *reinterpret_cast<uint32_t*>(smem + (addr ^ 64u)) = vx1[vi][q];
            }
        if (dq_tid < 128) {
            *reinterpret_cast<float*>(smem + deq + kPfKBytes + kPfVBytes + 4 * dq_tid) =
                (float)__builtin_bit_cast(_Float16, scale_bits);
        }
    };

    auto compute_unit = [&](int deqbuf, int t0, const bool MASKED) {
        const uint8_t* kb = smem + kPfDeqBase + deqbuf * kPfDeqBytes;
        const uint8_t* vb = kb + kPfKBytes;
        const float* sc = reinterpret_cast<const float*>(vb + kPfVBytes);
        float score[8];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            h8 a[2][4];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    a[h][m] = *reinterpret_cast<const h8*>(kb + (16 * s + n) * kPfKStride + 2 * (128 * h + 32 * m + 8 * b));
            // (the scale reads are issued with the operand reads, ahead of the MFMAs)
            const f4 kd0 = *reinterpret_cast<const f4*>(sc + 16 * s + 4 * b);
            const f4 kd1 = *reinterpret_cast<const f4*>(sc + 32 + 16 * s + 4 * b);
            f4 s_acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h) s_acc[h] = pf_mfma32<false>(a[h][m], bq[h][m], s_acc[h]);
#pragma unroll
            for (int i = 0; i < 4; ++i)  // minus the running maximum; the wide kernel's order of operations, so its bits
                score[4 * s + i] = __builtin_fmaf(kd1[i], s_acc[1][i], __builtin_fmaf(kd0[i], s_acc[0][i], -m_run));
        }
        // (the MASKED tests sit outside the unrolled loops: one wave-uniform branch per block)
        if (MASKED) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int pos = t0 + 16 * (t >> 2) + 4 * b + (t & 3);
                score[t] = (col_ok && pos >= col_lo && pos <= col_hi) ? score[t] : kNegBig;
            }
        }
        // online softmax, log2 domain; key slot j of this lane = token 16 (j >> 2) + 4 b + (j & 3).  See kPfSlack.
        const float mx = max3(max3(max3(score[0], score[1], score[2]), score[3], score[4]), score[5], max2(score[6], score[7]));
        float slack = kPfSlack;
        if (__ballot(mx > 0.f) != 0ull) {  // one value scale of the unit per lane
            const bool large = __ballot(!(fabsf(sc[64 + lane]) <= kPfSlackScale)) != 0ull;
            slack = large || (MASKED && !(t0 >= col_lo && t0 + kUnit - 1 <= col_hi)) ? 0.f : kPfSlack;
        }
        const bool raise = !started || __ballot(mx > slack) != 0ull;
        if (raise) {
            const float m = max_over_rows(mx);
            const bool empty = !(sum_over_rows(l_run) > 0.f), any = m > 0.5f * kNegBig;
            started = started || (!MASKED && __ballot(!any) == 0ull);  // (a unit that every live column sees)
            const float up = empty ? (any ? m : 0.f) : m > slack ? m : 0.f;
            const float alpha = empty ? 1.f : __builtin_amdgcn_exp2f(-up);
            m_run += up;
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < 8; ++t) score[t] -= up;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 8; ++j) o_acc[h][j] *= alpha;
        }
        float p[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) p[t] = __builtin_amdgcn_exp2f(score[t]);
        l_run += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        u4 pb[2], pb_lo[2];  // high and low operands per half of the head dimension
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f4 da = *reinterpret_cast<const f4*>(sc + 64 + 32 * h + 4 * b);
            const f4 db = *reinterpret_cast<const f4*>(sc + 64 + 32 * h + 16 + 4 * b);
            // high and low fp16 operand (see split_weights): one rounding of p * d would be shared by the
            // whole 128-element scale block
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const f4 d = k < 2 ? da : db;
                uint32_t whi, wlo;
                weight_h2(p[2 * k], p[2 * k + 1], d[2 * (k & 1)], d[2 * (k & 1) + 1], whi, wlo);
                pb[h][k] = whi;
                pb_lo[h][k] = wlo;
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            h8 a[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int d = 128 * h + 16 * j + n;
                a[j] = *reinterpret_cast<const h8*>(vb + d * 64 + 16 * (b ^ ((d >> 1) & 3)));
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) o_acc[h][j] = pf_mfma32<false>(a[j], __builtin_bit_cast(h8, pb[h]), o_acc[h][j]);
            // the low-order operands in a pass of their own: a tile's two MFMAs are then eight
            // instructions apart instead of back to back (the second waits for the first's result)
#pragma unroll
            for (int j = 0; j < 8; ++j) o_acc[h][j] = pf_mfma32<false>(a[j], __builtin_bit_cast(h8, pb_lo[h]), o_acc[h][j]);
        }
    };

    // ---- pipeline ----
    __syncthreads();  // table complete; query staging (aliases the dequant buffers) consumed
    // Between two barriers the dequantising waves commit unit it + 2, request unit it + 3 and dequantise unit it + 1 into
    // buffer (it + 1) & 1, the multiplying waves work on unit it in buffer it & 1.
    if (producer) {
        const int32_t pg_first = __builtin_amdgcn_readfirstlane(load_page(0));
        int32_t pg_next = load_page(1);
        if (n_units > 0) issue_loads(0, pg_first);
        for (int it = -2; it < n_units; ++it) {
            if (it + 2 < n_units) commit_loads((it + 2) & 1);
            // The page id of unit it + 4 is requested BEFORE the key loads of unit it + 3: a
            // write to its register after them would have to wait for all of them to return.
            const int32_t pg_s = __builtin_amdgcn_readfirstlane(pg_next);
            pg_next = load_page(it + 4);
            if (it + 3 < n_units) issue_loads(it + 3, pg_s);
            if (it + 1 >= 0 && it + 1 < n_units) dequant_unit((it + 1) & 1, (it + 1) & 1);
            __syncthreads();
        }
        return;  // the epilogue has no workgroup barrier
    }
    __builtin_amdgcn_s_setprio(1);  // (measured: none 8.20 ms, the multiplying waves 8.04, the dequantising waves 8.65)
    for (int it = -2; it < n_units; ++it) {
        if (it >= 0) {
            const int t0 = (u_first + it) * kUnit;
            compute_unit(it & 1, t0, !(t0 >= i_lo && t0 + kUnit - 1 <= i_hi));
        }
        __syncthreads();
    }
    __builtin_amdgcn_s_setprio(0);

    // ---- epilogue: normalise, transpose through LDS, rotate back, store ----
    l_run = sum_over_rows(l_run);
    float* reg = reinterpret_cast<float*>(smem) + wave * 16 * 260;
    const float inv = SPLIT ? 1.0f : (l_run > 0.f ? kLutInvGain / l_run : 0.f);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j)
            *reinterpret_cast<f4*>(reg + n * 260 + 128 * h + 16 * j + 4 * b) = o_acc[h][j] * inv;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    for (int c = 0; c < 16; ++c) {
        if (!((ok_mask >> c) & 1u)) continue;
        const int col = 16 * wave + c;
        const int t = div_q_group(col, P);
        const int a = col - t * P.q_group;
        const f4 x = *reinterpret_cast<const f4*>(reg + c * 260 + 4 * lane);
        float o[4] = {x[0], x[1], x[2], x[3]};
        if constexpr (SPLIT) {
            // un-normalised, rotated, still carrying the table gain: the merge kernel finishes
            const size_t row = (size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + a);
            const size_t prow = row * P.part_stride + (size_t)(P.pf_slot_base + part_x);
            *reinterpret_cast<f4*>(P.part_acc + prow * kHeadDim + 4 * lane) = x;
            const float l_c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l_run), c));
            // (a record without keys must not set the row's maximum)
            const float m_c = l_c == 0.f ? kNegBig : __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_run), c));
            if (lane == 0) *reinterpret_cast<f4*>(P.part_ml + prow * 4) = f4{m_c, l_c, (float)P.pf_split, 0.f};
            continue;
        }
        if (rot_out) {  // values stored rotated: rotate the finished row back
            wht256_wave(o, lane);
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * lane + k);
        }
        const size_t row = (size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + a);
        store_out_row<TQ>(P, row, lane, o);
    }
}

}  // namespace w34
