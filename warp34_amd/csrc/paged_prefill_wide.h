// Chunked-prefill attention over TQ4, FP8-E4M3, Q8_0, FP16 or BF16 pages: tiles of 256 (or 128) query rows.
// Replaces paged_attention_prefill_mma_f16_kernel + launch_prefill (op_paged_attn.cu:594-1128,1220-1259).  Included by
// paged_attn.hip.
//
// Workgroup = 8 waves, two per SIMD, up to 256 registers each.  Wave w owns the query rows 16 NC w .. + 16 NC - 1 as NC column
// tiles of its 16x16x32 MFMA results (S^T = K Q'^T, O^T += V^T P^T: the softmax state is one scalar pair per lane and column
// tile).  The workgroup walks the request's keys in 32-token units, one barrier per unit; between two barriers
//   rows of unit u + 2 travel from the pages to LDS (LDS-direct loads: no register holds them),
//   unit u + 1 is dequantised from LDS into the key and value tiles the MFMAs read (dq), and
//   unit u is multiplied: 16 operands of 16 bytes per lane for S, 16 for O, each used for NC MFMAs (2 NC for O where the weights have
//   a low-order operand).
// What bounds it: the SIMD's issue.  Vector and MFMA instructions of its two waves hardly overlap on this part (measured: 16.6
// cycles per 16x16x32 MFMA plus 2.5 to 4.3 per vector instruction, exp 8.3), so a unit costs the sum of both; LDS is busy 30 %
// of the cycles.  Hence two column tiles per wave: the operand reads, the dequantiser, the addresses and the barrier of a
// unit are paid once per 256 rows instead of once per 128 (the form this one replaces).  What does not fit 256 registers then
// is kept out of them: raw rows and run addresses in LDS, addresses of a lane worked out again for every unit (pw_lane), no
// scale or operand read earlier than the latency asks for.  The softmax of a unit that raises no column's maximum needs no
// exchange between lanes: the score sum starts at minus the running maximum, and one ballot tells.
// Measured, 4 x 2 048 tokens on 16 384 (2.34 TFLOP), us, against 128-row tiles on the same box: Q8_0 3 923 -> 2 374, FP8 3 610 ->
// 2 215, FP16 3 678 -> 2 242, BF16 4 164 -> 2 751, TQ4 3 610 (128-row tiles with separate dequantising waves) -> 3 118.
// Measured out: the two waves of a SIMD taking turns between MFMA and vector phases, six barriers per unit: 15 to 25 %
// slower; the dequantiser in opposite order in them: 8 % slower; priorities: within 1 %.
#pragma once

namespace w34 {

// Query rows of a workgroup with NC column tiles of 16 per wave
constexpr int pw_rows(int nc) { return kPfWaves * 16 * nc; }

typedef __attribute__((address_space(3))) const f4 lds_cf4;
typedef __attribute__((address_space(3))) const f2 lds_cf2;
typedef __attribute__((address_space(3))) u2v lds_u2;
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) const uint16_t lds_cu16;
__device__ __forceinline__ h8 pw_read_h8(uint32_t addr) { return *reinterpret_cast<lds_ch8*>((uintptr_t)addr); }
__device__ __forceinline__ f4 pw_read_f4(uint32_t addr) { return *reinterpret_cast<lds_cf4*>((uintptr_t)addr); }

__device__ __forceinline__ u2v pw_read_u2(uint32_t addr) { return *reinterpret_cast<__attribute__((address_space(3))) const u2v*>((uintptr_t)addr); }

// The lane, worked out where it is asked for: what follows from it is not kept in registers between the units.
__device__ __forceinline__ int pw_lane() {
    int none = 0;
    asm volatile("" : "+s"(none));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, (uint32_t)none));
}
// LDS-direct loads of 16 bytes per lane: piece i goes to lds_addr + 1024 i (M0 and the loads in one statement:
// the compiler does not know that M0 holds a value between two)
template <int PIECES>
__device__ __forceinline__ void pw_load_lds(uint32_t voffset, const uint8_t* sbase, uint32_t lds_addr) {
    static_assert(PIECES == 1 || PIECES == 2 || PIECES == 4, "pieces per call");
    if constexpr (PIECES == 1) {
        asm volatile(
            "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1"
            :
            : "v"(voffset), "s"(sbase), "s"(lds_addr)
            : "memory");
    } else if constexpr (PIECES == 2) {
        asm volatile(
            "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:1024"
            :
            : "v"(voffset), "s"(sbase), "s"(lds_addr)
            : "memory");
    } else {
        asm volatile(
            "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:1024\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:2048\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:3072"
            :
            : "v"(voffset), "s"(sbase), "s"(lds_addr)
            : "memory");
    }
}

// LDS: PfLds' map, the run offsets of eight waves behind the raw units
template <int KVF>
constexpr int pw_smem() {
    constexpr int loop = PfLds<KVF>::kRawBase + 2 * PfLds<KVF>::kRaw + kPfWaves * 512;
    constexpr int bytes = loop > PfLds<KVF>::kEpilogue ? loop : PfLds<KVF>::kEpilogue;
    static_assert(bytes <= 160 * 1024, "wide tile LDS budget");
    return bytes;
}

// The work of one workgroup: tile_tok tokens of the request from its token tile_tok0 on x the heads of kv_sub (16 NC columns per
// wave).
// VF (8-bit value rows stored rotated): the value tile holds code / kVfGain (exact: a power of two) and the block scales go into
// the weights, p * d * kVfGain, as a high and a low fp16 operand, as for TQ4 rows: fp16(d * code) rounds partly alike across a
// scale block that holds few distinct codes, and the inverse rotation of the finished row would gather that common part into
// one channel.  The block scales are small (amax / 448, amax / 127): without the gain the low-order operand, 2^-12
// of the weight, would fall into fp16's subnormal range.
template <typename TQ, int KVF, int NC, bool VF>
__device__ __forceinline__ void pw_tile(const AttnParams& P, uint8_t* smem, int req, int kv_sub, int tile_tok0, int tile_tok) {
    using M = PfLds<KVF>;
    constexpr bool FP8 = M::kFp8;
    constexpr bool K16 = M::k16;  // 16-bit rows, read as stored: the MFMAs run in the storage type
    constexpr bool Q8 = M::kQ8;   // Q8_0 rows: the key tile holds the codes, the value tile fp16(d * code) unless VF
    static_assert(!VF || FP8 || Q8, "scales in the probabilities: 8-bit rows only");
    constexpr float kVfGain = FP8 ? 256.0f : 128.0f;
    constexpr bool TQ4F = !FP8 && !K16 && !Q8;
    constexpr bool IS_BF16 = KVF == WARP34_KV_FORMAT_BF16;
    static_assert(!K16 || KVF == TQ::kStorageFormat, "16-bit pages are read in the query type");
    constexpr int kPfDeqBase = M::kDeqBase, kPfRawBase = M::kRawBase, kPfRawBytes = M::kRaw;
    constexpr int kRowB = M::kRowBytes, kRunB = M::kRun;
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int b = lane >> 4;
    const warp34_kv_layer_layout& L = P.L;
    const warp34_attention_batch& B = P.B;

    const int kv_head = fast_div(kv_sub, P.q_subgroups);
    const int q_head_base = kv_head * P.gqa + (kv_sub - kv_head * P.q_subgroups) * P.q_group;
    if (B.valid_req_mask != nullptr && B.valid_req_mask[req] == 0) return;
    const int rq_start = B.query_start_loc[req];
    const int rq_end = B.query_start_loc[req + 1];
    const int seq_after = B.seq_lens_after[req];
    const int ctx_before = B.context_lens_before != nullptr ? B.context_lens_before[req]
                                                            : seq_after - (rq_end - rq_start);
    const int tok0 = rq_start + tile_tok0;
    if (tok0 >= rq_end || tok0 >= B.total_tokens) return;
    int tile_tokens = rq_end - tok0;
    if (tile_tokens > tile_tok) tile_tokens = tile_tok;
    if (tile_tokens > B.total_tokens - tok0) tile_tokens = B.total_tokens - tok0;

    // ---- the pair table (64 lane replicas, as in the decode kernel) ----
    if (TQ4F) {
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
    const int u_first = lo_all >> 5;
    const int n_units = hi_all >= lo_all ? (hi_all >> 5) - u_first + 1 : 0;

    // column n of column tile g of this wave is row 16 (2 wave + g) + n of the workgroup
    uint32_t ok_mask[NC];
    int i_lo = 0, i_hi = 0x7fffffff;
#pragma unroll
    for (int g = 0; g < NC; ++g) {
        const int my_t = div_q_group(16 * (NC * wave + g) + n, P);
        const int my_tok = tok0 + my_t;
        const bool ok = my_t < tile_tokens &&
                        (B.valid_token_mask == nullptr || B.valid_token_mask[min(my_tok, B.total_tokens - 1)] != 0);
        ok_mask[g] = (uint32_t)(__ballot(ok) & 0xFFFFull);
        if (ok) {
            i_lo = max(i_lo, range_lo(q_off0 + my_t));
            i_hi = min(i_hi, range_hi(q_off0 + my_t));
        }
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        i_lo = max(i_lo, __shfl_xor(i_lo, off, 64));
        i_hi = min(i_hi, __shfl_xor(i_hi, off, 64));
    }
    i_lo = __builtin_amdgcn_readfirstlane(i_lo);
    i_hi = __builtin_amdgcn_readfirstlane(i_hi);

    // ---- rotated, scaled queries of this wave's columns -> LDS -> MFMA B operands ----
    constexpr int kQStride = 264;
    _Float16* qbuf = reinterpret_cast<_Float16*>(smem + kPfDeqBase) + wave * 16 * kQStride;
    const float q_scale = B.sm_scale * kLog2e * (TQ4F ? kLutInvGain : 1.0f);
    const bool rot_q = !K16 && P.rot_q != 0;
    const bool rot_out = !K16 && P.rot_out != 0;
    h8 bq[NC][2][4];  // [column tile][half of the head dim][32-wide k step]: Q'[col n][128 h + 32 m + 8 b ..]
#pragma unroll
    for (int g = 0; g < NC; ++g) {
        uint2 q_raw[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int col = 16 * (NC * wave + g) + c;
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
            if ((ok_mask[g] >> c) & 1u) {
                if constexpr (K16) {
                    packed = q_raw[c];  // as given: the scores are scaled after the MFMAs
                } else if constexpr (FP8 || Q8) {
                    // the softmax factor is applied with the fp32 key scales: an un-rotated fp16
                    // query enters the MFMAs exactly as given
                    packed.x = pack_h2(v[0], v[1]);
                    packed.y = pack_h2(v[2], v[3]);
                } else {
                    packed.x = pack_h2(v[0] * q_scale, v[1] * q_scale);
                    packed.y = pack_h2(v[2] * q_scale, v[3] * q_scale);
                }
            }
            *reinterpret_cast<uint2*>(qbuf + c * kQStride + 4 * lane) = packed;
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_wave_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < 4; ++m)
                bq[g][h][m] = *reinterpret_cast<const h8*>(qbuf + n * kQStride + 128 * h + 32 * m + 8 * b);
        // (the next column tile's rows go through the same 16-row buffer)
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_wave_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
    }

    // ---- loader: a unit's four runs of 16 rows (K rows 0-15, 16-31, V rows 0-15, 16-31), two waves a run ----
    const int ld_run = wave >> 1, ld_half = wave & 1;
    const uint8_t* ld_base;
    uint64_t ld_page_stride;
    {
        const bool is_v = ld_run >= 2;
        ld_base = reinterpret_cast<const uint8_t*>((uintptr_t)(is_v ? L.v_base : L.k_base)) +
                  (size_t)kv_head * (is_v ? L.v_head_stride_bytes : L.k_head_stride_bytes);
        ld_page_stride = is_v ? L.v_page_stride_bytes : L.k_page_stride_bytes;
    }
    const int32_t* req_blocks = B.block_tables + (size_t)req * B.max_blocks_per_req;
    // Byte offsets of this wave's runs of 64 units, in LDS: a run's address then costs one broadcast read (worked out by scalar
    // instructions for every unit: 560 to 840 of its 7 100 cycles; in vector registers there is no room).
    // Only runs that overlap the visible key range are looked up: block-table entries beyond the request's
    // pages are unspecified.  The others read rows of page 0, every one of which is masked.
    const uint32_t runs = (uint32_t)(kPfRawBase + 2 * kPfRawBytes + wave * 512);
    auto run_offset = [&](int k) __attribute__((always_inline)) -> u2v {  // of unit k, units in order
        if ((k & 63) == 0) {
            const int l = pw_lane();
            const int pos = (u_first + k + l) * kUnit + 16 * (ld_run & 1);
            const int slot = div_block(pos, P);
            uint64_t off = 0;
            if (k + l < n_units && pos <= hi_all && pos + 15 >= lo_all && slot < B.max_blocks_per_req) {
                const int32_t pg = req_blocks[slot];
                if (pg >= 0) off = (uint64_t)(uint32_t)pg * ld_page_stride + (uint64_t)((uint32_t)(pos - slot * L.block_size) * (uint32_t)kRowB);
            }
            *reinterpret_cast<lds_u2*>((uintptr_t)(runs + 8 * l)) = u2v{(uint32_t)off, (uint32_t)(off >> 32)};
        }
        return pw_read_u2(runs + 8 * (k & 63));
    };
    auto scalar_offset = [](u2v off) __attribute__((always_inline)) {
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)off[1]) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)off[0]);
    };
    auto issue_loads = [&](int k, uint64_t off) __attribute__((always_inline)) {
        // this wave's share of the run
        constexpr int kShare = K16 ? 4096 : FP8 ? 2112 : Q8 ? 2176 : 1024;
        const uint8_t* src = ld_base + off + ld_half * kShare;
        const uint32_t v = 16 * (uint32_t)pw_lane();
        const uint32_t dst = (uint32_t)(kPfRawBase + (k & 1) * kPfRawBytes + ld_run * kRunB + ld_half * kShare);
        if constexpr (K16) {
            pw_load_lds<4>(v, src, dst);
        } else if constexpr (FP8 || Q8) {
            pw_load_lds<2>(v, src, dst);
            if (v < (Q8 ? 128u : 64u)) pw_load_lds<1>(v, src + 2048, dst + 2048);
        } else {
            pw_load_lds<1>(v, src, dst);
            if (ld_half == 0 && v < 64u) pw_load_lds<1>(v, src + 2048, dst + 2048);  // pieces 128 to 131 of the run
        }
    };

    // ---- dequantiser: raw rows of unit u -> the tiles the MFMAs read, in kDqStages steps ----
    // The steps are dealt out between the MFMAs of the value product (compute_unit): a step reads what an earlier
    // one requested.  Key tile: rows of 256 fp16 / bf16, kPfKStride apart.  Value tile: V^T, row d (64 bytes, 32 key
    // slots) in place d ^ (d >> 3 & 1), its 16-byte piece b in place b ^ (d >> 1 & 3): neither the operand reads nor the
    // stores of token pairs conflict.  Tokens 2p, 2p + 1 sit in key slots 8 b + 4 s + {0,1} (+2 for odd p), s = p >> 3,
    // b = (p >> 1) & 3.
    constexpr int kDqStages = 9;
    uint32_t dk[8], dv[8], ds[4];
    auto dq = [&](int u, int stage, int t) __attribute__((always_inline)) {  // t: the thread
        const uint32_t raw = (uint32_t)(kPfRawBase + (u & 1) * kPfRawBytes);
        const uint32_t deq = (uint32_t)(kPfDeqBase + (u & 1) * kPfDeqBytes);
        const uint32_t deq_v = deq + (uint32_t)kPfKBytes, deq_s = deq_v + (uint32_t)kPfVBytes;
        const int p = t & 15;  // value token pair
        if constexpr (TQ4F) {
            // A raw row is 33 dwords; dwords 0 and 16 hold two scale bytes and two code bytes each.  They are fused into
            // one item, which leaves 32 items of four code bytes per row:
            //   item 0      : alignbit(dword 16, dword 0, 16)  -> elements 0..3 and 124..127
            //   item j 1..15: dword j                          -> elements 8 j - 4 .. 8 j + 3
            //   item j 16..31: dword j + 1                     -> elements 8 j .. 8 j + 7
            // (the second dword of a pair, 64 bytes on, is used by item 0 only)
            // K: item j of rows r and r + 16.  V: item jv of tokens 2p, 2p + 1; a table byte = (element of token 2p) |
            // (same of token 2p + 1) << 4 looks the pair up.
            const uint32_t lut_lane = ((uint32_t)t & 63u) << 2;
            const uint32_t r = (uint32_t)t >> 5, j = (uint32_t)t & 31u, jv = (uint32_t)t >> 4;
            if (stage == 0) {
                const uint32_t src = raw + r * kTq4RowBytes + 4u * (j + (j >= 16u ? 1u : 0u));
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    dk[i] = *reinterpret_cast<lds_cu32*>((uintptr_t)(src + i * 16 * kTq4RowBytes));
                    dk[2 + i] = *reinterpret_cast<lds_cu32*>((uintptr_t)(src + 64 + i * 16 * kTq4RowBytes));
                }
            } else if (stage == 1) {
                const uint32_t src = raw + (uint32_t)(kPfRawBytes / 2) + 2u * p * kTq4RowBytes + 4u * (jv + (jv >= 16u ? 1u : 0u));
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    dv[i] = *reinterpret_cast<lds_cu32*>((uintptr_t)(src + i * kTq4RowBytes));
                    dv[2 + i] = *reinterpret_cast<lds_cu32*>((uintptr_t)(src + 64 + i * kTq4RowBytes));
                }
                // scales, 32 x + row: K d0, K d1, V d0, V d1 (four threads work out the same one: cheaper than a branch)
                const uint32_t x = ((uint32_t)t >> 5) & 3u;
                ds[0] = *reinterpret_cast<lds_cu16*>((uintptr_t)(raw + (x >> 1) * (uint32_t)(kPfRawBytes / 2) + (x & 1u) * 66u +
                                                                 ((uint32_t)t & 31u) * kTq4RowBytes));
            } else if (stage == 2 || stage == 3) {
                const int i = stage - 2;
                const uint32_t word = __builtin_amdgcn_alignbit(dk[2 + i], dk[i], j == 0 ? 16u : 0u);
                uint32_t w[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) w[q] = lut_read(word, lut_lane, 0x0c0c0400u + ((uint32_t)q << 8));
                // (dk[0 .. 1], dk[2 .. 3] are still needed for i = 1: results of row r go to dk[4 .. 7])
#pragma unroll
                for (int q = 0; q < 4; ++q) dk[i == 0 ? 4 + q : q] = w[q];
            } else if (stage == 4) {
                const uint32_t shift = jv == 0 ? 16u : 0u;
                const uint32_t wa = __builtin_amdgcn_alignbit(dv[2], dv[0], shift);
                const uint32_t wb = __builtin_amdgcn_alignbit(dv[3], dv[1], shift);
                dv[0] = (wa & 0x0F0F0F0Fu) | ((wb << 4) & 0xF0F0F0F0u);         // even elements
                dv[1] = ((wa >> 4) & 0x0F0F0F0Fu) | (wb & 0xF0F0F0F0u);         // odd elements
            } else if (stage == 5) {
                const uint32_t ev = dv[0], od = dv[1];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t sel = 0x0c0c0400u + ((uint32_t)q << 8);
                    dv[q] = lut_read(ev, lut_lane, sel);
                    dv[4 + q] = lut_read(od, lut_lane, sel);
                }
            } else if (stage == 6) {
                const uint32_t dst = deq + r * kPfKStride + 16u * j - (j - 1u < 15u ? 8u : 0u);
                const uint32_t dst_hi = dst + (j == 0 ? 248u : 8u);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int at = i == 0 ? 4 : 0;
                    *reinterpret_cast<lds_u2*>((uintptr_t)(dst + i * 16 * kPfKStride)) = u2v{dk[at], dk[at + 1]};
                    *reinterpret_cast<lds_u2*>((uintptr_t)(dst_hi + i * 16 * kPfKStride)) = u2v{dk[at + 2], dk[at + 3]};
                }
            } else if (stage == 7 || stage == 8) {
                // even elements d = base + 2 q (item 0: 0, 2, 124, 126); the odd one's row is the neighbour
                const bool hi = stage == 8;
                const uint32_t base = 8u * jv - (jv - 1u < 15u ? 4u : 0u) + (hi && jv == 0 ? 120u : 0u);
                const uint32_t x = (base + (hi ? 4u : 0u)) >> 3 & 1u;
                const uint32_t at = deq_v + 64u * (base + x) + 8u * ((uint32_t)p >> 3) + 4u * ((uint32_t)p & 1u) +
                                    16u * ((((uint32_t)p >> 1) & 3u) ^ (base >> 1 & 3u));
#pragma unroll
                for (int q = hi ? 2 : 0; q < (hi ? 4 : 2); ++q) {
                    *reinterpret_cast<lds_u32*>((uintptr_t)((at ^ (16u * q)) + 128u * q)) = dv[q];
                    *reinterpret_cast<lds_u32*>((uintptr_t)((at ^ (16u * q) ^ 64u) + 128u * q)) = dv[4 + q];
                }
                if (hi && wave < 2) *reinterpret_cast<lds_f32*>((uintptr_t)(deq_s + 4u * ((uint32_t)t & 127u))) = (float)__builtin_bit_cast(_Float16, (uint16_t)ds[0]);
            }
        } else {
            // K: pieces g and g + 16 (eight elements each) of row r.  V: elements 8 j .. 8 j + 7 of tokens 2p, 2p + 1.
            // Value rows outside the visible key range become zeros: unwritten pool memory may hold NaN codes, and
            // 0 * NaN would poison the value product.
            const uint32_t r = (uint32_t)t >> 4, g = (uint32_t)t & 15u, j = (uint32_t)t >> 4;
            const uint8_t* rawp = smem + raw;
            const uint8_t* krow = rawp + r * kRowB;
            const uint8_t* vrow = rawp + kPfRawBytes / 2 + 2u * p * kRowB;
            const int pos = (u_first + u) * kUnit + 2 * p;
            auto keep = [&](int at) { return at >= lo_all && at <= hi_all ? ~0u : 0u; };
            auto store_k = [&](int piece, u4 w) {
                *reinterpret_cast<u4*>(smem + deq + r * kPfKStride + 16u * (g + 16u * piece)) = w;
            };
            auto store_v = [&](int e, uint32_t pair) {
                const uint32_t at = deq_v + 512u * j + 64u * (j & 1u) + 16u * (((uint32_t)p >> 1) & 3u) + 8u * ((uint32_t)p >> 3) + 4u * ((uint32_t)p & 1u);
                *reinterpret_cast<lds_u32*>((uintptr_t)((at ^ (64u * (e & 1) + 16u * (e >> 1))) + 128u * (e >> 1))) = pair;
            };
            if constexpr (K16) {
                if (stage == 0) {
                    const u4 w = *reinterpret_cast<const u4*>(krow + 16u * g), w1 = *reinterpret_cast<const u4*>(krow + 16u * g + 256u);
#pragma unroll
                    for (int i = 0; i < 4; ++i) dk[i] = w[i], dk[4 + i] = w1[i];
                } else if (stage == 1) {
                    const u4 a = *reinterpret_cast<const u4*>(vrow + 16u * j), c = *reinterpret_cast<const u4*>(vrow + kRowB + 16u * j);
#pragma unroll
                    for (int i = 0; i < 4; ++i) dv[i] = a[i], dv[4 + i] = c[i];
                } else if (stage == 2) {
                    store_k(0, u4{dk[0], dk[1], dk[2], dk[3]});
                } else if (stage == 3) {
                    store_k(1, u4{dk[4], dk[5], dk[6], dk[7]});
                } else if (stage == 4) {
                    const uint32_t a = keep(pos), c = keep(pos + 1);
#pragma unroll
                    for (int i = 0; i < 4; ++i) dv[i] &= a, dv[4 + i] &= c;
                } else {
                    const int i = stage - 5;
                    store_v(2 * i, __builtin_amdgcn_perm(dv[4 + i], dv[i], 0x05040100u));
                    store_v(2 * i + 1, __builtin_amdgcn_perm(dv[4 + i], dv[i], 0x07060302u));
                }
            } else {
                // FP8: 256 codes, then fp32 d0, d1.  Q8_0: four blocks of {fp32 d, 64 codes}.
                // Keys: the tile holds the codes (exact in fp16) and the scores take the fp32 block scales, which carry the
                // softmax factor: keys rounded to fp16(d * code) move a score by ~2e-3 when the row has outlier channels.
                // Values: fp16(d * code), every element rounded on its own; VF: code / kVfGain (exact for FP8's power
                // of two; the weights carry d * kVfGain).
                constexpr uint32_t kScales = Q8 ? 128u : 64u;  // key scales of a unit
                const uint32_t si = (uint32_t)t & ((VF ? 2u : 1u) * kScales - 1u);
                if (stage == 0) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const uint32_t pc = g + 16u * i;
                        const uint8_t* c = Q8 ? krow + 68u * (pc >> 3) + 4u + 8u * (pc & 7u) : krow + 8u * pc;
                        dk[2 * i] = *reinterpret_cast<const uint32_t*>(c);
                        dk[2 * i + 1] = *reinterpret_cast<const uint32_t*>(c + 4);
                    }
                    // key scales, x 32 + row (VF: then the value scales)
                    // (several threads work out the same one: cheaper than a branch)
                    const uint32_t x = (si & (kScales - 1u)) >> 5;
                    const uint8_t* row = rawp + (VF && si >= kScales ? kPfRawBytes / 2 : 0) + (si & 31u) * kRowB;
                    ds[0] = *reinterpret_cast<const uint32_t*>(row + (Q8 ? 68u * x : 256u + 4u * x));
                } else if (stage == 1) {
                    const uint8_t* c = Q8 ? vrow + 68u * (j >> 3) + 4u + 8u * (j & 7u) : vrow + 8u * j;
                    const uint8_t* sc = Q8 ? vrow + 68u * (j >> 3) : vrow + 256u + 4u * (j >> 4);
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        dv[2 * i] = *reinterpret_cast<const uint32_t*>(c + i * kRowB);
                        dv[2 * i + 1] = *reinterpret_cast<const uint32_t*>(c + i * kRowB + 4);
                        ds[1 + i] = *reinterpret_cast<const uint32_t*>(sc + i * kRowB);
                    }
                } else if (stage == 2 || stage == 3) {
                    const int i = stage - 2;
                    uint32_t h0, h1, h2_, h3;
                    if constexpr (FP8) {
                        fp8x4_to_h4(dk[2 * i], h0, h1);
                        fp8x4_to_h4(dk[2 * i + 1], h2_, h3);
                    } else {
                        i8x4_to_h4(dk[2 * i], h0, h1);
                        i8x4_to_h4(dk[2 * i + 1], h2_, h3);
                    }
                    store_k(i, u4{h0, h1, h2_, h3});
                } else if (stage == 4) {
                    const uint32_t a = keep(pos), c = keep(pos + 1);
                    dv[0] &= a, dv[1] &= a, ds[1] &= a;
                    dv[2] &= c, dv[3] &= c, ds[2] &= c;
                } else {
                    const int h = (stage - 5) >> 1, half = (stage - 5) & 1;  // two of the four elements of code dword h
                    float fa[4], fb[4];
                    codes4_to_f32<FP8>(dv[h], fa);
                    codes4_to_f32<FP8>(dv[2 + h], fb);
                    const float da = VF ? 1.0f / kVfGain : __uint_as_float(ds[1]), db = VF ? 1.0f / kVfGain : __uint_as_float(ds[2]);
#pragma unroll
                    for (int k = 2 * half; k < 2 * half + 2; ++k) store_v(4 * h + k, pack_h2(da * fa[k], db * fb[k]));
                    if (stage == 8) {
                        float d = __uint_as_float(ds[0]) * q_scale;
                        if constexpr (VF) {
                            const float dv_ = __uint_as_float(ds[0] & keep((u_first + u) * kUnit + (int)(si & 31u))) * kVfGain;
                            d = si >= kScales ? dv_ : d;
                        }
                        *reinterpret_cast<lds_f32*>((uintptr_t)(deq_s + 4u * si)) = d;
                    }
                }
            }
        }
    };

    // ---- per-wave attention state ----
    f4 o_acc[NC][2][8];
    float m_run[NC], l_run[NC];
#pragma unroll
    for (int g = 0; g < NC; ++g) {
        m_run[g] = 0.f, l_run[g] = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) o_acc[g][h][j] = f4{0.f, 0.f, 0.f, 0.f};
    }
    // addresses of a lane's operands and scales (worked out again for each unit)
    auto key_lane = [&]() __attribute__((always_inline)) {
        const uint32_t l = (uint32_t)pw_lane();
        return (uint32_t)kPfDeqBase + (l & 15u) * (uint32_t)kPfKStride + (l & 48u);
    };
    auto value_lane = [&]() __attribute__((always_inline)) {
        const uint32_t l = (uint32_t)pw_lane(), vn = l & 15u;
        return (uint32_t)(kPfDeqBase + kPfKBytes) + (vn ^ (vn >> 3)) * 64u + 16u * ((l >> 4) ^ ((vn >> 1) & 3u));
    };
    auto scale_lane = [&]() __attribute__((always_inline)) {
        return (uint32_t)(kPfDeqBase + kPfKBytes + kPfVBytes) + ((uint32_t)pw_lane() & 48u);
    };

    // A operands (16 bytes per lane) are read a few steps ahead: a step is one operand and its MFMAs
    constexpr int KRING = NC == 1 ? 6 : VF ? 3 : 4, VRING = NC == 1 ? 6 : VF ? 2 : TQ4F ? 3 : 4;
    h8 kring[KRING], vring[VRING];
    uint32_t k_at = 0;
    auto read_k = [&](int at) __attribute__((always_inline)) {  // step at: token half at / 8, k step at % 8
        kring[at % KRING] = pw_read_h8(k_at + (at >> 3) * 16 * kPfKStride + 64 * (at & 7));
    };
    uint32_t v_at = 0;
    auto read_v = [&](int at) __attribute__((always_inline)) {  // step at: channels 16 at ..
        vring[at % VRING] = pw_read_h8(v_at + at * 1024);
    };
    // Until every live column has a maximum (`started`) that of a column without one is 0, and so is its sum (see the decode kernel).
    bool started = false;
    auto compute_unit = [&](int u, const bool masked, auto&& after_keys) __attribute__((always_inline)) {
        const int deqbuf = u & 1, t0 = (u_first + u) * kUnit;
        const uint32_t sc = scale_lane() + deqbuf * kPfDeqBytes;
        // Scores minus the running maximum, then weights, of key slots 2k (pe) and 2k + 1 (po).  As vectors: the operands of the
        // second value product take their places without a move.
        f4 pe[NC], po[NC];
        auto get = [&](int g, int t) __attribute__((always_inline)) { return t & 1 ? po[g][t >> 1] : pe[g][t >> 1]; };
        auto put = [&](int g, int t, float x) __attribute__((always_inline)) {
            if (t & 1) po[g][t >> 1] = x;
            else pe[g][t >> 1] = x;
        };
        // ---- S = K Q ----
        constexpr int kBlocks = K16 ? 1 : Q8 ? 4 : 2;  // key scale blocks of a row = partial scores
        constexpr int kSteps = 8 / kBlocks;
        f4 part[2][NC], kd;
        auto score = [&](int at) __attribute__((always_inline)) {  // block at of the unit's 2 * kBlocks: its partial scores join the sums
            const int s = at / kBlocks;
#pragma unroll
            for (int g = 0; g < NC; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float from = at % kBlocks ? get(g, 4 * s + i) : -m_run[g];
                    put(g, 4 * s + i, __builtin_fmaf(part[at & 1][g][i], K16 ? q_scale : kd[i], from));
                }
        };
#pragma unroll
        for (int at = 0; at < 16; ++at) {
            const int blk = at / kSteps;  // block of the unit
            if (at + KRING - 1 < 16) read_k(at + KRING - 1);
#pragma unroll
            for (int g = 0; g < NC; ++g)
                part[blk & 1][g] = pf_mfma32<IS_BF16>(kring[at % KRING], bq[g][(at & 7) >> 2][at & 3],
                                                      at % kSteps ? part[blk & 1][g] : f4{0.f, 0.f, 0.f, 0.f});
            if (blk > 0 && at % kSteps == 0) score(blk - 1);
            // (read as soon as the previous block's are used: a read takes about 130 cycles to arrive)
            if (!K16 && at % kSteps == 0) kd = pw_read_f4(sc + 128 * (blk % kBlocks) + 64 * (blk / kBlocks));
            __builtin_amdgcn_sched_barrier(0);
        }
        score(2 * kBlocks - 1);
        after_keys();
        __builtin_amdgcn_sched_barrier(0);
        // key slot j of this lane = token 16 (j >> 2) + 4 b + (j & 3)
        bool sees_all[NC] = {};  // (masked units) the column sees the whole unit
        if (masked) {
            const int l = pw_lane();  // (worked out where it is needed: few units come here)
#pragma unroll
            for (int g = 0; g < NC; ++g) {
                const int my_t = div_q_group(16 * (NC * wave + g) + (l & 15), P);
                const bool ok = ((ok_mask[g] >> (l & 15)) & 1u) != 0;
                const int lo = range_lo(q_off0 + my_t) - t0 - 4 * (l >> 4);
                const int hi = ok ? range_hi(q_off0 + my_t) - t0 - 4 * (l >> 4) : -1000;
                if constexpr (TQ4F) sees_all[g] = lo + 4 * (l >> 4) <= 0 && hi + 4 * (l >> 4) >= kUnit - 1;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int at = 16 * (t >> 2) + (t & 3);
                    put(g, t, at >= lo && at <= hi ? get(g, t) : kNegBig);
                }
            }
        }
        // ---- online softmax, log2 domain ----
        float mx[NC];
#pragma unroll
        for (int g = 0; g < NC; ++g)
            mx[g] = max3(max3(max3(pe[g][0], po[g][0], pe[g][1]), po[g][1], pe[g][2]), po[g][2], max2(pe[g][3], po[g][3]));
        // A column's maximum stays where it is until a unit exceeds it by kPfSlack (see there): most units need no exchange between lanes
        // and leave the sums alone.
        // (One weight operand: every unit that exceeds it.  That form keeps its text: with the comparisons of the other Q8_0 batches take 10 % longer.)
        constexpr bool kLazy = TQ4F || IS_BF16;
        float slack[NC];
#pragma unroll
        for (int g = 0; g < NC; ++g) slack[g] = kPfSlack;
        if constexpr (TQ4F) {
            if (__ballot(max2(mx[0], mx[NC - 1]) > 0.f) != 0ull) {  // one value scale of the unit per lane
                const uint32_t l = (uint32_t)pw_lane();
                const float d = *reinterpret_cast<__attribute__((address_space(3))) const float*>((uintptr_t)(sc - (l & 48u) + 256u + 4u * l));
                const bool large = __ballot(!(fabsf(d) <= kPfSlackScale)) != 0ull;
#pragma unroll
                for (int g = 0; g < NC; ++g) slack[g] = large || (masked && !sees_all[g]) ? 0.f : kPfSlack;
            }
        }
        if (!started || (kLazy ? __ballot(mx[0] > slack[0] || mx[NC - 1] > slack[NC - 1])
                               : __ballot(max2(mx[0], mx[NC - 1]) > 0.f)) != 0ull) {
            float least = -kNegBig;
#pragma unroll
            for (int g = 0; g < NC; ++g) {
                const float m = max_over_rows(mx[g]);
                least = fminf(least, m);
                const bool empty = !(sum_over_rows(l_run[g]) > 0.f);
                const float up = empty ? (m > 0.5f * kNegBig ? m : 0.f) : !kLazy ? fmaxf(m, 0.f) : m > slack[g] ? m : 0.f;
                const float alpha = empty ? 1.f : __builtin_amdgcn_exp2f(-up);
                m_run[g] += up;
                l_run[g] *= alpha;
                pe[g] -= up, po[g] -= up;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j) o_acc[g][h][j] *= alpha;
            }
            started = started || (!masked && __ballot(!(least > 0.5f * kNegBig)) == 0ull);  // (a unit that every live column sees)
        }
#pragma unroll
        for (int g = 0; g < NC; ++g) {
#pragma unroll
            for (int t = 0; t < 8; ++t) put(g, t, __builtin_amdgcn_exp2f(get(g, t)));
            const f4 sum = pe[g] + po[g];
            l_run[g] += (sum[0] + sum[1]) + (sum[2] + sum[3]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- O += V P ----
        v_at = value_lane() + deqbuf * kPfDeqBytes;
#pragma unroll
        for (int j = 0; j < VRING - 1; ++j) read_v(j);
        // Weight operands.  TQ4: the value scales ride on the weights, one high and one low fp16 operand per scale block
        // (weight_h2); those of the second block are made between the MFMAs of the first.  Rotated 8-bit rows: the same,
        // each block's made in front of its MFMAs.  BF16: the bits of a probability that bf16 does not keep go into
        // a second operand.  Else one operand.
        constexpr bool kTwo = TQ4F || VF || IS_BF16;
        u4 pw[NC], pw_lo[NC];
        constexpr int kVBlocks = Q8 ? 4 : 2;
        constexpr int kTiles = 16 / kVBlocks;  // value tiles (16 channels) per scale block
        f4 vd[2];  // value scales of a block, four tokens each
        auto read_vd = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) vd[h] = pw_read_f4(sc + (Q8 ? 512 : 256) + 128 * blk + 64 * h);
        };
        auto weights = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f4 d = vd[h];
#pragma unroll
                for (int g = 0; g < NC; ++g)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        uint32_t hi, lo;
                        weight_h2(pe[g][2 * h + k], po[g][2 * h + k], d[2 * k], d[2 * k + 1], hi, lo);
                        pw[g][2 * h + k] = hi, pw_lo[g][2 * h + k] = lo;
                    }
            }
        };
        if constexpr (TQ4F || VF) {
            read_vd(0);
        } else {
#pragma unroll
            for (int g = 0; g < NC; ++g)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if constexpr (IS_BF16) {
                        const uint32_t h0 = BF16::from_f32(pe[g][k]), h1 = BF16::from_f32(po[g][k]);
                        const uint32_t l0 = BF16::from_f32(pe[g][k] - BF16::to_f32((uint16_t)h0));
                        const uint32_t l1 = BF16::from_f32(po[g][k] - BF16::to_f32((uint16_t)h1));
                        pw[g][k] = h0 | (h1 << 16);
                        pw_lo[g][k] = l0 | (l1 << 16);
                    } else {
                        pw[g][k] = pack_h2(pe[g][k], po[g][k]);
                    }
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        int dq_t = 0;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (VF && j > 0 && j % kTiles == 0) read_vd(j / kTiles);  // (read ahead, they do not fit the registers)
            if ((TQ4F || VF) && j % kTiles == 0) weights();
            if (j + VRING - 1 < 16) read_v(j + VRING - 1);
            if (TQ4F && j == kTiles - 1) read_vd(1);
#pragma unroll
            for (int lo = 0; lo < (kTwo ? 2 : 1); ++lo)
#pragma unroll
                for (int g = 0; g < NC; ++g) {
                    f4& o = o_acc[g][j >> 3][j & 7];
                    o = pf_mfma32<IS_BF16>(vring[j % VRING], __builtin_bit_cast(h8, lo ? pw_lo[g] : pw[g]), o);
                }
            // the next unit's tiles: the steps go where registers are free (the thread is worked out here: what follows
            // from it is not kept between the units)
            if (TQ4F ? j == 8 || j == 11 : j == (VF ? 7 : 0)) dq_t = 64 * wave + pw_lane();
            constexpr int kStageTq4[16] = {-1, -1, -1, -1, -1, -1, -1, -1, 0, 2, 3, 6, 4, 5, 7, 8};
            constexpr int kStageVf[16] = {-1, -1, -1, -1, -1, -1, -1, 0, 2, 3, 1, 4, 5, 6, 7, 8};
            constexpr int kStage[16] = {0, 1, -1, -1, 2, -1, 3, -1, 4, -1, 5, -1, 6, 7, -1, 8};
            const int stage = TQ4F ? kStageTq4[j] : VF ? kStageVf[j] : kStage[j];
            if (stage >= 0) dq(u + 1, stage, dq_t);
            if (TQ4F && j == 11) dq(u + 1, 1, dq_t);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- pipeline ----
    __syncthreads();  // table complete; query staging (aliases the dequant buffers) consumed
    if (n_units > 0) issue_loads(0, scalar_offset(run_offset(0)));
    wait_vm<0>();
    __syncthreads();
    if (n_units > 1) issue_loads(1, scalar_offset(run_offset(1)));
    if (n_units > 0) {
#pragma unroll
        for (int i = 0; i < kDqStages; ++i) dq(0, i, (int)threadIdx.x);
    }
    wait_vm<0>();
    __syncthreads();
    uint64_t next_off = n_units > 2 ? scalar_offset(run_offset(2)) : 0;
    for (int u = 0; u < n_units; ++u) {
        k_at = key_lane() + (u & 1) * kPfDeqBytes;
#pragma unroll
        for (int at = 0; at < KRING - 1; ++at) read_k(at);
        // rows of unit u + 2 travel while unit u is multiplied and unit u + 1 dequantised (behind the last unit: left-over rows)
        if (u + 2 < n_units) issue_loads(u + 2, next_off);
        const u2v off = run_offset(u + 3);  // (behind the last unit: not used)
        const int t0 = (u_first + u) * kUnit;
        compute_unit(u, !(t0 >= i_lo && t0 + kUnit - 1 <= i_hi), [&]() __attribute__((always_inline)) { next_off = scalar_offset(off); });
        wait_vm<0>();
        __syncthreads();
    }

    // ---- epilogue: normalise, transpose through LDS, rotate back, store ----
    const int e_lane = pw_lane(), e_n = e_lane & 15, e_b = e_lane >> 4;
    float* reg = reinterpret_cast<float*>(smem) + wave * 16 * 260;
#pragma unroll
    for (int g = 0; g < NC; ++g) {
        l_run[g] = sum_over_rows(l_run[g]);
        const float inv = l_run[g] > 0.f ? (TQ4F ? kLutInvGain : 1.0f) / l_run[g] : 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                *reinterpret_cast<f4*>(reg + e_n * 260 + 128 * h + 16 * j + 4 * e_b) = o_acc[g][h][j] * inv;
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_wave_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        for (int c = 0; c < 16; ++c) {
            if (!((ok_mask[g] >> c) & 1u)) continue;
            const int col = 16 * (NC * wave + g) + c;
            const int t = div_q_group(col, P);
            const int a = col - t * P.q_group;
            const f4 x = *reinterpret_cast<const f4*>(reg + c * 260 + 4 * e_lane);
            float o[4] = {x[0], x[1], x[2], x[3]};
            if (rot_out) {  // values stored rotated: rotate the finished row back
                wht256_wave(o, e_lane);
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * e_lane + k);
            }
            const size_t row = (size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + a);
            store_out_row<TQ>(P, row, e_lane, o);
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_wave_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
    }
}

// Workgroup -> tile.  The batch's tiles of 256 rows, longest first (pf_longest_first), the heads of a tile next to each
// other.  A last, partly filled round of workgroups over the kPwCus CUs would cost as much as a full one: as many of its tiles as
// there are CUs left over are cut into two tiles of 128 rows, which take about 0.65 of the time of a whole one (Q8_0 0.73, FP8
// and FP16 0.69, TQ4 and BF16 0.63): the longest ones while the batch fits one round (they end last), else the shortest ones (they
// start last).
// A tile whose request ends inside its first half runs as one of 128 rows: the other half's products would be those of dead
// columns.  us a layer step, 128-row tiles of their own kernel / whole tiles only / this: 32 requests x 40 tokens, two q heads
// per kv head, on 240 to 940 keys: Q8_0 90 / 109 / 86, FP8 86 / 105 / 82, FP16 84 / 99 / 77; 300 x 33 to 60 733 / 920 / 700.
// More than 64 requests: no ranks.  The workgroups of a request one after the other, its last tile first, which share its keys;
// but by tile index, all requests' first tiles first, where a request's tiles would meet the same parts of the chip over and over
// (workgroups go round 8 XCDs and their shader engines): with two tiles, one whole and one short, half of the XCDs get the whole
// ones only; with 24 and more a shader engine keeps seeing the same index, behind the end of most requests.  us, the former order /
// the latter: Q8_0 100 x 33 to 48 tokens, eight q heads per kv head, 213 / 183, bf16 128 x 129, two q heads, 869 / 816, Q8_0
// 70 x 100 to 1 000 (32 tiles) 2 440 / 1 697; 80 x 20 to 300 (10 tiles) on 1 500 to 5 200 keys 1 389 / 1 512.
// Requests of different lengths: whole tiles of the longest would be the batch's time, so they are cut too (pw_long_tiles).
constexpr int kPwCus = kChipCus;
// What a tile of a request takes, in units of its length (pf_longest_first): lane r holds request r.
struct PwRequest {
    int first, count;  // lengths first + 1 .. first + count
    // tiles of at least this length, and what they take
    __device__ __forceinline__ int from(int length) const { return max(0, min(count, first + count + 1 - length)); }
    __device__ __forceinline__ float work(int n) const { return (float)n * ((float)(first + count) - 0.5f * (float)(n - 1)); }
};
// How many tiles, of the longest, are cut into halves because the others would be done long before them: all that are longer than
// three quarters of the longest, if there are few enough for their halves to run at once, and if by list scheduling (a tile
// begins when what comes before it, spread over the CUs, is done; a half takes 0.7) the batch then ends before the longest whole tile
// would.  us, whole tiles only / this: four requests of 1 024 tokens, eight q heads per kv head, one on 16 000 keys and three on 2 000:
// FP8 871 / 686, Q8_0 961 / 797, FP16 810 / 682, BF16 1 023 / 750.
__device__ __forceinline__ int pw_long_tiles(const AttnParams& P, int lane, int kv_subs, int tiles) {
    const warp34_attention_batch& B = P.B;
    if (B.num_reqs < 2 || B.sliding_window > 0 || B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW) return 0;
    PwRequest mine{0, 0};
    if (lane < B.num_reqs && (B.valid_req_mask == nullptr || B.valid_req_mask[lane] != 0)) {
        const int q_len = B.query_start_loc[lane + 1] - B.query_start_loc[lane];
        const int ctx = B.context_lens_before != nullptr ? B.context_lens_before[lane] : B.seq_lens_after[lane] - q_len;
        mine.count = q_len > 0 ? (q_len + P.tok_tile - 1) / P.tok_tile : 0;
        mine.first = ctx > 0 ? ctx / P.tok_tile : 0;
    }
    int longest = mine.count > 0 ? mine.first + mine.count : 0;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) longest = max(longest, __shfl_xor(longest, off, 64));
    longest = __builtin_amdgcn_readfirstlane(longest);
    const int cut_from = longest - (longest >> 2) + 1;
    // up to and with the shortest tile of this lane's request: workgroups, what they take, the batch's cut tiles
    int before = 0, cut = 0;
    float work = 0.0f;
    for (int r = 0; r < B.num_reqs; ++r) {
        const PwRequest other{__builtin_amdgcn_readlane(mine.first, r), __builtin_amdgcn_readlane(mine.count, r)};
        const int n = other.from(mine.first + 1), n_cut = other.from(cut_from), halved = min(n, n_cut);
        before += n + halved;
        work += other.work(n) + 0.4f * other.work(halved);
        cut += n_cut;
    }
    cut = __builtin_amdgcn_readfirstlane(cut) * kv_subs;
    if (cut > kPwCus / 2 || cut >= tiles) return 0;
    float end = 0.0f;
    if (mine.count > 0) {
        const float own = (float)(mine.first + 1);
        end = before * kv_subs > kPwCus ? work * (float)kv_subs / (float)kPwCus + own : own;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) end = fmaxf(end, __shfl_xor(end, off, 64));
    return __ballot(end < 0.95f * (float)longest) != 0ull ? cut : 0;
}
constexpr int kPwTq4Tiles = 250;  // TQ4 pages: from this many 256-row tiles on (see launch_prefill_tq4)
template <typename TQ, int KVF, bool VF>
__global__ __launch_bounds__(kPfWaves * 64, 1) void paged_prefill_wide_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int kv_subs = P.L.local_kv_heads * P.q_subgroups;
    const int tiles_x = P.bal_tiles;  // 256-row tiles of the longest request
    const int wg = (int)(blockIdx.x + gridDim.x * blockIdx.y);
    int req, kv_sub, tile, half = -1;
    if (P.B.num_reqs <= 64) {
        int tiles = 0;  // of 256 rows, all heads of the batch
        {
            const int r = (int)threadIdx.x & 63;
            if (r < P.B.num_reqs && (P.B.valid_req_mask == nullptr || P.B.valid_req_mask[r] != 0)) {
                const int q_len = P.B.query_start_loc[r + 1] - P.B.query_start_loc[r];
                tiles = q_len > 0 ? (q_len + P.tok_tile - 1) / P.tok_tile : 0;
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) tiles += __shfl_xor(tiles, off, 64);
            tiles = __builtin_amdgcn_readfirstlane(tiles) * kv_subs;
        }
        const int last = tiles % kPwCus;
        const int spare = min(last, last == 0 ? 0 : kPwCus - last);
        const int longest = tiles > kPwCus / 2 ? pw_long_tiles(P, (int)threadIdx.x & 63, kv_subs, tiles) : 0;
        const bool from_front = tiles < kPwCus || longest > 0;
        const int cut = longest == 0 ? spare : tiles < kPwCus ? max(longest, spare) : longest;
        if (wg >= tiles + cut) return;
        int at = wg;  // the tile
        if (from_front) {
            if (wg < 2 * cut) at = wg >> 1, half = wg & 1;
            else at = wg - cut;
        } else if (wg >= tiles - cut) {
            const int h = wg - (tiles - cut);
            at = tiles - cut + (h >> 1), half = h & 1;
        }
        const int rank = at / kv_subs;
        kv_sub = at - rank * kv_subs;
        const PfTile t = pf_longest_first(P, (int)threadIdx.x & 63, rank);
        if (t.req < 0) return;
        req = t.req;
        tile = t.tile;
    } else {
        const int per_req = tiles_x * kv_subs, per_tile = P.B.num_reqs * kv_subs;
        if (tiles_x <= 2 || tiles_x >= 24) {
            tile = wg / per_tile;
            if (tile >= tiles_x) return;
            const int at = wg - tile * per_tile;
            req = at / kv_subs;
            kv_sub = at - req * kv_subs;
        } else {
            req = wg / per_req;
            if (req >= P.B.num_reqs) return;
            const int in_req = wg - req * per_req;
            kv_sub = in_req / tiles_x;
            tile = tiles_x - 1 - (in_req - kv_sub * tiles_x);
        }
    }
    const int half_tok = P.tok_tile >> 1, tok0 = tile * P.tok_tile + (half > 0 ? half_tok : 0);
    const int left = P.B.query_start_loc[req + 1] - P.B.query_start_loc[req] - tok0;
    if (half < 0 && left > half_tok) {
        pw_tile<TQ, KVF, 2, VF>(P, smem, req, kv_sub, tok0, P.tok_tile);
    } else {
        pw_tile<TQ, KVF, 1, VF>(P, smem, req, kv_sub, tok0, half_tok);
    }
}

}  // namespace w34
