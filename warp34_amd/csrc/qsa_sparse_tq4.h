// QSA sparse paged attention over TQ4 pages for gfx950: every query token attends over its own
// list of selected 4-token groups (ops/op_qsa.cu:716-1158, 1446-1571 of the reference).
//
// The streaming core is the one of the dense TQ4 decode kernel (pair table in LDS, S^T = K Q'^T
// and O^T += V^T P^T on v_mfma_f32_16x16x32_f16, one query column per lane); what differs is where
// the keys come from.  A 32-token unit is eight selected groups; a group is four consecutive rows
// of one page, 528 bytes = 33 16-byte pieces: one LDS-direct load of 33 lanes from a wave-uniform address, and the unit
// lies in LDS in the layout the core expects.
// What bounds it: two dependent memory round trips (the list, the rows), the table and one or two units per
// wave for a small batch; the instructions of the unit for a large one (eight units a wave).  Hence: the list entries
// of eight units in one load, K rows asked for before V rows and the next unit's before this one's products, table reads
// a batch ahead of the MFMAs, one barrier before the loop and one behind it.  us a call, 513 groups, against rows through
// registers, K and V waited for together, two barriers on either side: 16 tokens 19.6 -> 17.4, 64 30.6 -> 25.8, 256
// 85 -> 66; 16 tokens x 64 groups 12.6 -> 11.2; with the table written without bank conflicts (build_pair_table; 16 bytes every 128
// before) 16.7, 25.7, 67 and 9.8.
//
//   grid  = (query tokens, kv heads x q subgroups, splits), block = 8 waves
//   split = an equal share of the token's units; every split writes an (m, l) record (l = 0
//           without work), the merge kernel adds them up.  One split finishes in the kernel.
//   tail  = rotate back, sigmoid gate, fp16 rounding, optional H64 / 8 over every 64-element
//           block of the rounded row (ops/hadamard_inline.cuh:11-50)
//
// Included by paged_attn.hip after the dense kernels (shares their device helpers).
#pragma once

namespace w34 {

constexpr int kQsaWaves = 8;
// LDS: the pair table, the waves' staging areas (after the loop: merge regions), the query rows, (m, l) of the waves
constexpr int kQsaQStride = 264;
constexpr int kQsaQBase = kLutBytes + kQsaWaves * kStageTq4;
constexpr int kQsaMlBase = kQsaQBase + 16 * kQsaQStride * 2;
constexpr int kQsaSmem = kQsaMlBase + kQsaWaves * 16 * 2 * 4;
constexpr int kQsaGroupBytes = 4 * kTq4RowBytes;  // 33 pieces of 16 bytes
constexpr int kQsaMaxSplits = 16;

struct QsaParams {
    warp34_kv_layer_layout L;
    const uint16_t* gate;  // may be null
    uint16_t* out;
    const uint8_t* valid_token_mask;  // may be null
    float* part_acc;  // [rows][n_splits][256]
    float* part_ml;   // [rows][n_splits][4]: m, l, -, -
    int had64;
    int groups_per_page;
    int gpp_shift;  // log2(groups_per_page), or -1 when it is not a power of two
    float sm_scale;
    float out_scale;  // factor of the un-normalised sums (the table gain of the TQ4 form, else 1)
    int rot_q;        // row-format form: K rows are stored rotated, rotate the query rows
    int rot_out;      // V rows are stored rotated: rotate the finished row back
};

// Leading arguments of the two attention kernels: in scalar registers when a wave starts, so the list, its counts and the query rows are
// asked for at once (behind the argument block: 16 tokens of 513 groups, TQ4, 16.5 us a call instead of 15.8).
#define QSA_LEAD                                                                                                                  \
    const int32_t *__restrict__ sel_phys, const int32_t *__restrict__ sel_log, const int32_t *__restrict__ num_sel,               \
        const int32_t *__restrict__ seq_pos_of, const uint16_t *__restrict__ q_in, int select_k, int guess, uint32_t shape, int num_q_heads
// shape: q_group (5 bits), splits (5 bits), q_subgroups.  guess: units (halves) of a split of a full list.
struct QsaShape {
    int q_group, n_splits, q_subgroups;
    __host__ static uint32_t pack(int q_group, int n_splits, int q_subgroups) { return (uint32_t)(q_group | n_splits << 5 | q_subgroups << 10); }
    __device__ explicit QsaShape(uint32_t x) : q_group((int)(x & 31u)), n_splits((int)(x >> 5 & 31u)), q_subgroups((int)(x >> 10)) {}
};
static_assert(kQsaMaxSplits < 32, "splits in five bits");
// (the compiler would load the rest of the arguments where they are used; here they are on their way beside the list)
__device__ __forceinline__ void qsa_have_arguments(const QsaParams& P) {
    asm volatile("" ::"s"(P.L.k_base), "s"(P.L.v_base), "s"(P.L.k_page_stride_bytes), "s"(P.L.v_page_stride_bytes), "s"(P.L.k_head_stride_bytes),
                 "s"(P.L.v_head_stride_bytes), "s"(P.L.k_token_stride_bytes), "s"(P.L.v_token_stride_bytes), "s"(P.valid_token_mask),
                 "s"(P.groups_per_page), "s"(P.gpp_shift), "s"(P.sm_scale));
}

// The end of a row: v = element 4 lane + k of the normalised sum in the rotated domain.
__device__ __forceinline__ uint2 qsa_load_gate(const uint16_t* gate, size_t row, int lane) {
    return gate != nullptr ? *reinterpret_cast<const uint2*>(gate + row * kHeadDim + 4 * lane) : uint2{0u, 0u};
}
// g: the row's gate values (qsa_load_gate, requested by the caller ahead of the sums)
__device__ __forceinline__ void qsa_finish_row(float (&v)[4], int lane, size_t row, bool rotate,
                                               bool has_gate, uint2 g, bool had64, uint16_t* out) {
    if (rotate) {
        wht256_wave(v, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = apply_sign(v[k], 4 * lane + k);
    }
    if (has_gate) {
        const float gv[4] = {F16::to_f32((uint16_t)(g.x & 0xFFFFu)), F16::to_f32((uint16_t)(g.x >> 16)),
                             F16::to_f32((uint16_t)(g.y & 0xFFFFu)), F16::to_f32((uint16_t)(g.y >> 16))};
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] *= 1.0f / (1.0f + expf(-gv[k]));
    }
    uint16_t h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) h[k] = F16::from_f32(v[k]);
    if (had64) {
        // H64 / 8 over the 16 lanes that hold one 64-element block, on the rounded values, sums in
        // fp32 in the reference's order
        float x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = F16::to_f32(h[k]);
        const float a0 = x[0] + x[1], a1 = x[0] - x[1], a2 = x[2] + x[3], a3 = x[2] - x[3];
        x[0] = a0 + a2;
        x[1] = a1 + a3;
        x[2] = a0 - a2;
        x[3] = a1 - a3;
        wht_stage<1>(x, lane);
        wht_stage<2>(x, lane);
        wht_stage<4>(x, lane);
        wht_stage<8>(x, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) h[k] = F16::from_f32(x[k] * 0.125f);
    }
    uint2 o;
    o.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    o.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
    *reinterpret_cast<uint2*>(out + row * kHeadDim + 4 * lane) = o;
}

__global__ __launch_bounds__(kQsaWaves * 64, 1) void qsa_sparse_tq4_kernel(QSA_LEAD, const QsaParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    // lut_read() addresses the table absolutely: the dynamic block starts at LDS address 0 because
    // the kernel has no static LDS (checked on the host before the first launch)
    uint8_t* stage_all = smem + kLutBytes;

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int b = lane >> 4;
    const warp34_kv_layer_layout& L = P.L;

    const int tok = (int)blockIdx.x;
    const int kv_sub = (int)blockIdx.y;
    const int split = (int)blockIdx.z;
    const QsaShape S(shape);
    const int kv_head = fast_div(kv_sub, S.q_subgroups);
    const int q_head_base = kv_sub * S.q_group;  // (a kv head's q heads are its subgroups')

    // ---- this token's list ------------------------------------------------------------------------
    // The counts and the list entries of this wave's first eight units (lane l: group l & 7 of unit l >> 3) are requested
    // together: where the wave's units start is guessed from the list's capacity (exact when the list is full, the
    // common case) and the entries are fetched again when the guess is wrong, so the guess changes the latency only.
    const int32_t* tok_phys = sel_phys + (size_t)tok * select_k;
    const int32_t* tok_log = sel_log + (size_t)tok * select_k;
    const int unit_guess = split * guess + wave;
    int list_id = -1, list_lg = 0;
    auto load_list = [&](int first_unit, int end) {
        const int gi = (first_unit + kQsaWaves * (lane >> 3)) * 8 + (lane & 7);
        list_id = -1, list_lg = 0;
        if (gi < end) {
            list_id = tok_phys[gi];
            list_lg = tok_log[gi];
        }
    };
    load_list(unit_guess, select_k);
    const int a_sel = num_sel[tok], a_pos = seq_pos_of[tok];

    // ---- query rows of this wave's columns (column c = q head q_head_base + c, c < q_group) ----------
    constexpr int kColsPerWave = 16 / kQsaWaves;
    uint2 q_raw[kColsPerWave];
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c) {
        const int col = wave + c * kQsaWaves;
        q_raw[c] = uint2{0u, 0u};
        if (col < S.q_group) {
            const uint16_t* qrow = q_in + ((size_t)tok * num_q_heads + (size_t)(q_head_base + col)) * kHeadDim;
            q_raw[c] = *reinterpret_cast<const uint2*>(qrow + 4 * lane);
        }
    }
    qsa_have_arguments(P);
    int a_live = 1;
    if (P.valid_token_mask != nullptr) a_live = (int)P.valid_token_mask[tok];
    build_pair_table(smem, tid, wave);

    int n_sel = __builtin_amdgcn_readfirstlane(a_live) != 0 ? __builtin_amdgcn_readfirstlane(a_sel) : 0;
    if (n_sel > select_k) n_sel = select_k;
    if (n_sel < 0) n_sel = 0;
    const int seq_pos = __builtin_amdgcn_readfirstlane(a_pos);
    const int n_units = (n_sel + 7) >> 3;
    const int upc = fast_div(n_units + S.n_splits - 1, S.n_splits);
    const int cu_first = split * upc;
    int cu_end = cu_first + upc;
    if (cu_end > n_units) cu_end = n_units;

    // ---- staging machinery ------------------------------------------------------------------------
    const uint8_t* k_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.k_base) + (size_t)kv_head * L.k_head_stride_bytes;
    const uint8_t* v_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.v_base) + (size_t)kv_head * L.v_head_stride_bytes;
    uint8_t* stage = stage_all + wave * kStageTq4;
    const uint32_t stage_addr = (uint32_t)(kLutBytes + wave * kStageTq4);
    // Of this lane's entry of the list: byte offsets of the group's rows in the K and the V slab, and its first key position
    // (or a position that is never visible).  A skipped group reads group 0 of page 0: any TQ4 bytes dequantise to
    // finite values, and every key of such a group is masked.
    uint64_t k_off = 0, v_off = 0;
    int pos_vec = 0x3fffffff;
    auto locate_list = [&](int first_unit) {
        const int gi = (first_unit + kQsaWaves * (lane >> 3)) * 8 + (lane & 7);
        const bool skip = gi >= n_sel || list_id < 0;
        const int gid = skip ? 0 : list_id;
        // pages of 2^k tokens (the usual case): shift and mask
        const int pg = P.gpp_shift >= 0 ? gid >> P.gpp_shift : gid / P.groups_per_page;
        const uint32_t row = (uint32_t)(gid - pg * P.groups_per_page) * 4u;
        k_off = (uint64_t)(uint32_t)pg * L.k_page_stride_bytes + (uint64_t)row * L.k_token_stride_bytes;
        v_off = (uint64_t)(uint32_t)pg * L.v_page_stride_bytes + (uint64_t)row * L.v_token_stride_bytes;
        pos_vec = skip ? 0x3fffffff : 4 * list_lg;
    };
    // The K or the V rows of the wave's unit j: eight LDS-direct loads of one group each.
    auto issue_loads = [&](int j, uint64_t off, const uint8_t* base, uint32_t lds) __attribute__((always_inline)) {
        const uint32_t lane16 = 16u * (uint32_t)lane;
        if (lane < kQsaGroupBytes / 16) {
#pragma unroll
            for (int gi = 0; gi < 8; ++gi) {
                const int at = 8 * (j & 7) + gi;
                const uint64_t o = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(off >> 32), at) << 32) |
                                   (uint32_t)__builtin_amdgcn_readlane((int)off, at);
                asm volatile(
                    "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                    "global_load_lds_dwordx4 %0, %1"
                    :
                    : "v"(lane16), "s"(base + o), "s"(lds + gi * kQsaGroupBytes)
                    : "memory");
            }
        }
    };
    auto issue_k = [&](int j) __attribute__((always_inline)) { issue_loads(j, k_off, k_base, stage_addr); };
    auto issue_v = [&](int j) __attribute__((always_inline)) { issue_loads(j, v_off, v_base, stage_addr + 2 * kRunBytes); };
    constexpr int kLoads = 8;  // load instructions of a unit's K (or V) rows

    const int unit0 = cu_first + wave;
    if (unit0 != unit_guess) load_list(unit0, n_sel);  // wave-uniform
    locate_list(unit0);
    // (the compiler's own loads end here, where they have landed: a wait for one of them behind the rows, which return in
    // order, would wait for the rows too)
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c) asm volatile("" ::"v"(q_raw[c].x), "v"(q_raw[c].y));
    asm volatile("" ::"v"(pos_vec));
    if (unit0 < cu_end) issue_k(0);

    // ---- rotated, scaled fp16 queries to LDS, then the B operands of the QK MFMAs -----------------
    constexpr int kQStride = kQsaQStride;
    _Float16* qlds = reinterpret_cast<_Float16*>(smem + kQsaQBase);
    const float q_scale = P.sm_scale * kLog2e * kLutInvGain;
    // up to eight columns: columns 8-15 repeat them and take the low-order part of the weights (see the dense kernel)
    const bool pack = S.q_group <= 8;
    static_assert(kQsaWaves == 8 && kColsPerWave == 2, "a packed tile's mirror column col + 8 belongs to the wave of col");
    uint2 packed_prev = {0u, 0u};
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c) {
        const int col = wave + c * kQsaWaves;
        if (pack && c == 1) {
            *reinterpret_cast<uint2*>(qlds + col * kQStride + 4 * lane) = packed_prev;
            continue;
        }
        float qv[4] = {F16::to_f32((uint16_t)(q_raw[c].x & 0xFFFFu)), F16::to_f32((uint16_t)(q_raw[c].x >> 16)),
                       F16::to_f32((uint16_t)(q_raw[c].y & 0xFFFFu)), F16::to_f32((uint16_t)(q_raw[c].y >> 16))};
        if (col < S.q_group) {  // wave-uniform; dead columns stay zero
#pragma unroll
            for (int k = 0; k < 4; ++k) qv[k] = apply_sign(qv[k], 4 * lane + k);
            wht256_wave(qv, lane);
        }
        uint2 packed;
        packed.x = pack_h2(qv[0] * q_scale, qv[1] * q_scale);
        packed.y = pack_h2(qv[2] * q_scale, qv[3] * q_scale);
        *reinterpret_cast<uint2*>(qlds + col * kQStride + 4 * lane) = packed;
        packed_prev = packed;
    }
    if (unit0 < cu_end) issue_v(0);
    __syncthreads();  // the table and the query rows are complete
    h8 bq[8];
    {
        const int kb = 8 * (b & 1) + 4 * (b >> 1);
        const uint8_t* qrow = reinterpret_cast<const uint8_t*>(qlds + n * kQStride);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int D = kb + m;
            u2v lo = *reinterpret_cast<const u2v*>(qrow + (D > 0 ? 16 * D - 8 : 0));
            u2v hi = *reinterpret_cast<const u2v*>(qrow + (D > 0 ? 16 * D : 248));  // (D = 0: see tq4_fuse)
            bq[m] = __builtin_bit_cast(h8, u4{lo[0], lo[1], hi[0], hi[1]});
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) bq[4 + m] = *reinterpret_cast<const h8*>(qrow + 256 + 16 * (kb + m));
    }

    const uint32_t lut_lane = (uint32_t)lane << 2;
    const bool col_ok = (pack ? n & 7 : n) < S.q_group;
    f4 o_acc[2][8];
    float m_run = kNegBig, l_run = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) o_acc[h][j] = f4{0.f, 0.f, 0.f, 0.f};

    // One 32-token unit.  gp0 / gp1: first key position of the groups that hold this lane's key
    // slots 0-3 / 4-7 (group 4 (b & 1) + (b >> 1), and that group + 2).
    auto process_unit = [&](int gp0, int gp1, const bool MASKED, const bool HAS_NEXT, int j_next) {
        const uint8_t* k_rows = stage;
        const uint8_t* v_rows = stage + 2 * kRunBytes;
        wait_vm<kLoads>();  // the K rows have landed (the V rows may still be on their way)
        float sc[8];
        uint32_t kw[2][8], ks[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int arow = unit_token(s, n >> 2, n & 3);
            const uint32_t* row32 = reinterpret_cast<const uint32_t*>(k_rows + arow * kTq4RowBytes);
#pragma unroll
            for (int mf = 0; mf < 8; ++mf) kw[s][mf] = row32[tq4_qk_dword(mf >> 2, mf & 3, b)];
            kw[s][0] = tq4_fuse(row32[16], kw[s][0], b == 0);
            // (the two scales of a token in one register: lane n reads token n & 3, see the dense kernel)
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(k_rows + unit_token(s, b, n & 3) * kTq4RowBytes);
            const uint32_t mine = __builtin_amdgcn_perm(r32[16], r32[0], 0x07060100u);
            ks[s][0] = row_bcast<0>(mine);
            ks[s][1] = row_bcast<1>(mine);
            ks[s][2] = row_bcast<2>(mine);
            ks[s][3] = row_bcast<3>(mine);
        }
        wait_lds_reads();
        if (HAS_NEXT) issue_k(j_next);
        // eight batches of two operands, the table reads of a batch in front of the MFMAs of the one before
        constexpr int kQkOrder[8] = {0, 4, 1, 5, 2, 6, 3, 7};
        f4 s_acc[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) s_acc[s][0] = s_acc[s][1] = f4{0.f, 0.f, 0.f, 0.f};
        u4 qa[2][2];
        auto qk_reads = [&](int bt, u4 (&a)[2]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t w = kw[bt >> 2][kQkOrder[2 * (bt & 3) + k]];
                a[k][0] = lut_read(w, lut_lane, 0x0c0c0400u);
                a[k][1] = lut_read(w, lut_lane, 0x0c0c0500u);
                a[k][2] = lut_read(w, lut_lane, 0x0c0c0600u);
                a[k][3] = lut_read(w, lut_lane, 0x0c0c0700u);
            }
        };
        qk_reads(0, qa[0]);
#pragma unroll
        for (int bt = 0; bt < 8; ++bt) {
            if (bt + 1 < 8) qk_reads(bt + 1, qa[(bt + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int mf = kQkOrder[2 * (bt & 3) + k];
                f4& acc = s_acc[bt >> 2][mf >> 2];
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, qa[bt & 1][k]), bq[mf], acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sc[4 * s + i] = __builtin_fmaf(s_acc[s][1][i], half_hi_to_f32(ks[s][i]), mul_by_half_lo(s_acc[s][0][i], ks[s][i]));
        if (MASKED) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int pos = (t < 4 ? gp0 : gp1) + (t & 3);
                sc[t] = (col_ok && pos <= seq_pos) ? sc[t] : kNegBig;
            }
        }
        if (HAS_NEXT) {
            wait_vm<kLoads>();  // the V rows have landed; the next K rows may be on their way
        } else {
            wait_vm<0>();
        }
        // Per token: the two scales in one register (lane n reads those of token n & 7 and hands them round inside its row of lanes),
        // the dword of the first half-row that holds this lane's codes (dword n, see tq4_fuse) and that of the second.
        uint32_t vsc[8], vw[2][8];
        {
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(v_rows + unit_token((n >> 2) & 1, b, n & 3) * kTq4RowBytes);
            const uint32_t mine_sc = __builtin_amdgcn_perm(r32[16], r32[0], 0x07060100u);
            vsc[0] = row_bcast<0>(mine_sc);
            vsc[1] = row_bcast<1>(mine_sc);
            vsc[2] = row_bcast<2>(mine_sc);
            vsc[3] = row_bcast<3>(mine_sc);
            vsc[4] = row_bcast<4>(mine_sc);
            vsc[5] = row_bcast<5>(mine_sc);
            vsc[6] = row_bcast<6>(mine_sc);
            vsc[7] = row_bcast<7>(mine_sc);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const uint32_t* row32 = reinterpret_cast<const uint32_t*>(v_rows + unit_token(t >> 2, b, t & 3) * kTq4RowBytes) + n;
                vw[0][t] = tq4_fuse(row32[16], row32[0], n == 0);
                vw[1][t] = row32[17];
            }
        }
        wait_lds_reads();
        if (HAS_NEXT) issue_v(j_next);
        float p[8];
        {
            float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
            mx = max_over_rows(mx);
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            float psum = 0.f;
#pragma unroll
            for (int t = 0; t < 8; ++t) p[t] = __builtin_amdgcn_exp2f(sc[t] - m_new);
            if (MASKED) {
#pragma unroll
                for (int t = 0; t < 8; ++t) p[t] = sc[t] > 0.5f * kNegBig ? p[t] : 0.f;
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) psum += p[t];
            const bool scale = alpha != 1.0f && l_run != 0.f;  // (without a weight so far the sums are zero)
            l_run = l_run * alpha + psum;
            if (__ballot(scale) != 0ull) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j) o_acc[h][j] *= alpha;
            }
        }
        // probability times the half-row scale of the value row, as a high and a low fp16 operand (split_weights): one rounding
        // would be shared by the whole scale block.  (Masked tokens have p == 0; a garbage scale must not reach the weights.)
        if (MASKED) {
#pragma unroll
            for (int t = 0; t < 8; ++t) vsc[t] = p[t] > 0.f ? vsc[t] : 0u;
        }
        u4 ph[2], pl[2];
        uint32_t lo[2][4], hi[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float w[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) w[t] = h == 0 ? mul_by_half_lo(p[t], vsc[t]) : mul_by_half_hi(p[t], vsc[t]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t whi, wlo;
                split_weights(w[2 * k], w[2 * k + 1], whi, wlo);
                ph[h][k] = pack && (n & 8) ? wlo : whi;
                pl[h][k] = wlo;
                const uint32_t wa = vw[h][2 * k], wb = vw[h][2 * k + 1];
                lo[h][k] = (wa & 0x0F0F0F0Fu) | ((wb << 4) & 0xF0F0F0F0u);
                hi[h][k] = ((wa >> 4) & 0x0F0F0F0Fu) | (wb & 0xF0F0F0F0u);
            }
        }
        // four batches of four value tiles, the table reads of a batch in front of the MFMAs of the one before
        u4 va[2][4];
        auto pv_reads = [&](int bt, u4 (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int j = 4 * (bt & 1) + jj;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    a[jj][k] = lut_read((j & 1) ? hi[bt >> 1][k] : lo[bt >> 1][k], lut_lane, 0x0c0c0400u + ((uint32_t)(j >> 1) << 8));
            }
        };
        pv_reads(0, va[0]);
#pragma unroll
        for (int bt = 0; bt < 4; ++bt) {
            if (bt + 1 < 4) pv_reads(bt + 1, va[(bt + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int part = 0; part < 2; ++part) {  // (a pass of its own: a tile's two MFMAs are not back to back)
                if (part == 1 && pack) continue;
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    f4& o = o_acc[bt >> 1][4 * (bt & 1) + jj];
                    o = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, va[bt & 1][jj]),
                                                              __builtin_bit_cast(h8, part ? pl[bt >> 1] : ph[bt >> 1]), o, 0, 0, 0);
                }
            }
        }
    };

    int unit = unit0;
    for (int j = 0; unit < cu_end; ++j) {
        const int next_unit = unit + kQsaWaves;
        const int ga = 8 * (j & 7) + 4 * (b & 1) + (b >> 1);
        const int gp0 = __shfl(pos_vec, ga, 64);
        const int gp1 = __shfl(pos_vec, ga + 2, 64);
        // interior unit: all eight groups present and wholly in front of the token's position
        const bool interior = __ballot((lane >> 3) == (j & 7) && pos_vec + 3 > seq_pos) == 0ull;
        if ((j & 7) == 7 && next_unit < cu_end) {  // the next eight units' entries
            load_list(next_unit, n_sel);
            locate_list(next_unit);
            asm volatile("" ::"v"(pos_vec));
        }
        process_unit(gp0, gp1, !interior, next_unit < cu_end, j + 1);
        unit = next_unit;
    }

    // ---- merge the waves' states through LDS (layout as in the dense kernel) -------------------------
    // (one barrier: every wave leaves its state in its own staging area, the adding wave weighs them)
    if (pack) add_mirror_columns(o_acc);
    l_run = sum_over_rows(l_run);
    constexpr int kRegion = 8 * kMergeColStride;
    static_assert(kRegion * 4 == kStageTq4, "a wave's merge region is its own staging area");
    float* xbuf = reinterpret_cast<float*>(stage_all);
    float* tbuf = reinterpret_cast<float*>(smem) + wave * 256;  // the table is dead behind the barrier
    float* mlbuf = reinterpret_cast<float*>(smem + kQsaMlBase);
    if (b == 0) {
        mlbuf[(wave * 16 + n) * 2 + 0] = m_run;
        mlbuf[(wave * 16 + n) * 2 + 1] = l_run;
    }
    auto store_region = [&](int half) {
        float* c = xbuf + wave * kRegion + (n & 7) * kMergeColStride;
        if (pack) {  // (half 0)
            if (col_ok) store_packed_column(c, o_acc, n, b);
            return;
        }
        if ((n >> 3) != half || !col_ok) return;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) *reinterpret_cast<f4*>(c + ((h * 8 + j) * 4 + b) * 4) = o_acc[h][j];
    };
    store_region(0);

    static_assert(kQsaWaves == 8, "a wave adds up one column of a pass");
    __syncthreads();
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        if (8 * half >= S.q_group) break;  // the same in every wave
        if (half == 1) {
            __syncthreads();  // the first pass has read the regions
            store_region(1);
            __syncthreads();
        }
        const int col = 8 * half + wave;
        if (col >= S.q_group) continue;
        const size_t row = (size_t)tok * num_q_heads + (size_t)(q_head_base + col);
        uint2 g = {0u, 0u};
        if (S.n_splits == 1) g = qsa_load_gate(P.gate, row, lane);
        float mw[kQsaWaves], lw[kQsaWaves];
#pragma unroll
        for (int w = 0; w < kQsaWaves; ++w) {
            const f2 r = *reinterpret_cast<const f2*>(mlbuf + (w * 16 + col) * 2);
            mw[w] = r[0];
            lw[w] = r[1];
        }
        float m_col = kNegBig, l_col = 0.f;
#pragma unroll
        for (int w = 0; w < kQsaWaves; ++w) m_col = fmaxf(m_col, mw[w]);
        f4 tot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kQsaWaves; ++w) {
            const float wgt = __builtin_amdgcn_exp2f(mw[w] - m_col);
            l_col += lw[w] * wgt;
            tot += *reinterpret_cast<const f4*>(xbuf + w * kRegion + wave * kMergeColStride + 4 * lane) * wgt;
        }
        // into the element order of the head dimension (the reads follow the write of the same wave in LDS order)
        *reinterpret_cast<f4*>(tbuf + 4 * lane) = tot;
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = tbuf[tq4_merge_slot(lane) + 16 * k];
        if (S.n_splits > 1) {
            const size_t prow = row * S.n_splits + split;
            *reinterpret_cast<f4*>(P.part_acc + prow * kHeadDim + 4 * lane) = f4{v[0], v[1], v[2], v[3]};
            if (lane == 0) *reinterpret_cast<f4*>(P.part_ml + prow * 4) = f4{m_col, l_col, 0.f, 0.f};
        } else {
            if (!(l_col > 0.f)) {  // masked token or no visible key: a row of (positive) zeros
                *reinterpret_cast<uint2*>(P.out + row * kHeadDim + 4 * lane) = uint2{0u, 0u};
                continue;
            }
            const float inv = kLutInvGain / l_col;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] *= inv;
            qsa_finish_row(v, lane, row, true, P.gate != nullptr, g, P.had64 != 0, P.out);
        }
    }
}

// One wave per (token, q head) row: lane s holds the record of split s (n_splits <= 16).  All arguments are in scalar registers when a
// wave starts: records, sums and gate are asked for at once.
__global__ __launch_bounds__(64) void qsa_sparse_merge_kernel(const float* __restrict__ part_ml, const float* __restrict__ part_acc,
                                                              const uint16_t* __restrict__ gate, uint16_t* __restrict__ out, int n_splits,
                                                              int rot_out, int had64, float out_scale) {
    const int lane = (int)threadIdx.x;
    const size_t row = (size_t)blockIdx.x;
    const float* ml = part_ml + row * n_splits * 4;
    const float* acc = part_acc + row * n_splits * kHeadDim;
    f4 rec = {kNegBig, 0.f, 0.f, 0.f};
    if (lane < n_splits) rec = *reinterpret_cast<const f4*>(ml + 4 * lane);
    const uint2 g = qsa_load_gate(gate, row, lane);
    f4 a[kQsaMaxSplits];
#pragma unroll
    for (int s = 0; s < kQsaMaxSplits; ++s) {
        a[s] = f4{0.f, 0.f, 0.f, 0.f};
        if (s < n_splits) a[s] = *reinterpret_cast<const f4*>(acc + (size_t)s * kHeadDim + 4 * lane);
    }
    float m_tot = rec[1] > 0.f ? rec[0] : kNegBig;
    m_tot = fmaxf(m_tot, lane_xor<1>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<2>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<4>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<8>(m_tot, lane));
    const float w_my = rec[1] > 0.f ? __builtin_amdgcn_exp2f(rec[0] - m_tot) : 0.f;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    float l_tot = 0.f;
#pragma unroll
    for (int s = 0; s < kQsaMaxSplits; ++s) {
        const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_my), s));
        const float ls = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rec[1]), s));
        if (s < n_splits && ws > 0.f) {  // wave-uniform
            l_tot += ls * ws;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] += a[s][k] * ws;
        }
    }
    if (!(l_tot > 0.f)) {  // masked token or no visible key: a row of (positive) zeros
        *reinterpret_cast<uint2*>(out + row * kHeadDim + 4 * lane) = uint2{0u, 0u};
        return;
    }
    const float inv = out_scale / l_tot;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] *= inv;
    qsa_finish_row(v, lane, row, rot_out != 0, gate != nullptr, g, had64 != 0, out);
}

}  // namespace w34
