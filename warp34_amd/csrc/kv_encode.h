// Row encoders of the paged KV formats for gfx950, shared by the append kernel and the fused
// QK-norm + RoPE + append kernels.  A row is encoded by one half of a wave64 (32 lanes); the
// arithmetic and the order of every sum follow the reference's 32-lane warp
// (op_kv_cache.cu:32-218, tq4_kv_common.cuh:54-107) and are bit-exact with the CPU restatement
// when the including file is built with -ffp-contract=off.
//
// Data layout: lane l32 holds the eight consecutive elements 8 l32 .. 8 l32 + 7 (the reference's
// lane holds l32 + 32 j).  Index bits 0-2 are then register bits and bits 3-7 lane bits.  The
// butterfly stages run in the reference's order (1, 2, 4, ..., 128, the scale on the last); its
// 32-element sums (one per register there: elements 32 j .. 32 j + 31) are four-lane groups
// here, all eight reduced by ONE pass of the same tree (xor 16, 8 across lanes; xor 4, 2, 1
// across registers); two neighbouring codes share a lane.  Every sum adds the same operands in
// the same order, so the bytes are those of the 32-lane form at half its instruction count.
#pragma once

#include "kv_common.h"

namespace w34 {

// (float)(1.0 / sqrt((double)x)) for a normal x: the hardware's reciprocal root (within 1 ulp) and one second-order
// correction in double precision, 8 double-precision instructions instead of 35 (the append of 4 096 tokens
// 9.1 -> 8.8 us).  1 / sqrt(x) of a float x is never nearer than 2^-51.7 (relative) to the middle of two floats, and
// over all significands of two binades and starting values up to 2 ulp off both forms round to the same float
// (checked on the host).
__device__ __forceinline__ float rsqrt_rn_normal(float x) {
    const double y = (double)__builtin_amdgcn_rsqf(x);
    const double r = __builtin_fma(-(y * y), (double)x, 1.0);
    return (float)__builtin_fma(y, r * __builtin_fma(r, 0.375, 0.5), y);
}
// the same for every x
__device__ __forceinline__ float rsqrt_rn(float x) {
    if (x >= 1.17549435e-38f && x <= 3.402823466e38f) return rsqrt_rn_normal(x);
    return (float)(1.0 / sqrt((double)x));
}

// 32-lane xor butterfly sum, offsets 16,8,4,2,1 (tq4_kv_common.cuh:54-60); cross-lane moves are
// DPP / lane-swap VALU operations (lane_xor), not LDS permutes.
__device__ __forceinline__ float half_wave_sum(float v, int lane) {
    v += lane_xor<16>(v, lane);
    v += lane_xor<8>(v, lane);
    v += lane_xor<4>(v, lane);
    v += lane_xor<2>(v, lane);
    v += lane_xor<1>(v, lane);
    return v;
}

// One butterfly stage across lanes: lanes with bit H clear take x + x[lane ^ H], the others
// x[lane ^ H] - x (tq4_kv_common.cuh:75-107).  flip = sign bit in the lanes with bit H set.
template <int H>
__device__ __forceinline__ float wht_lane_stage(float val, uint32_t flip, int lane) {
    static_assert(H == 1 || H == 2 || H == 8, "stages with one lane move per value");
    return lane_xor<H>(val, lane) + __uint_as_float(__float_as_uint(val) ^ flip);
}
// The same with H = 4: the sum goes to the groups of four lanes with the bit clear, the difference to the others; two
// instructions a value, where the exchange alone takes two.  (The compiler does not see that the statement reads and writes
// across lanes: the waits stand in it.)
__device__ __forceinline__ void wht_lane_stage4(float (&v)[8]) {
    float r[8];
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %8, %8 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %9, %9 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %2, %10, %10 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %3, %11, %11 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %4, %12, %12 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %5, %13, %13 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %6, %14, %14 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %7, %15, %15 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_sub_f32_dpp %0, %8, %8 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %1, %9, %9 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %2, %10, %10 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %3, %11, %11 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %4, %12, %12 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %5, %13, %13 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %6, %14, %14 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %7, %15, %15 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "s_nop 1"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = r[j];
}
// The same with H = 16, for two values a, b at a time: exchanged halves put a's two rows of lanes (and b's) side by side, the sum
// and the difference are the results of both rows, and a second exchange brings them back: four instructions for two values.
// (The append of 4 096 tokens, TQ4, with both stages in this form: 8.8 -> 8.4 us.)
__device__ __forceinline__ void wht_lane_stage16(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    const float sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // even rows: of a, odd rows: of b
    const float diff = __uint_as_float(r[0]) - __uint_as_float(r[1]);
    const auto o = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(diff), false, false);
    a = __uint_as_float(o[0]);
    b = __uint_as_float(o[1]);
}

// stages 1, 2, 4 of the 256-point Walsh-Hadamard transform: registers
__device__ __forceinline__ void wht_register_stages(float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
        const float a = v[j], b = v[j + 1];
        v[j] = a + b;
        v[j + 1] = a - b;
    }
#pragma unroll
    for (int g = 0; g < 8; g += 4) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float a = v[g + i], b = v[g + i + 2];
            v[g + i] = a + b;
            v[g + i + 2] = a - b;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = v[i], b = v[i + 4];
        v[i] = a + b;
        v[i + 4] = a - b;
    }
}
// The transform with the 1/16 scale on the last stage; v[j] = x[8 l32 + j] on entry and y[8 l32 + j] on return.
__device__ __forceinline__ void wht256(float (&v)[8], int lane) {
    wht_register_stages(v);
    // stages 8 .. 128: lanes (each stage over all eight registers: independent instructions
    // between a write and the cross-lane read of it)
    const uint32_t f1 = (uint32_t)(lane & 1) << 31, f2 = (uint32_t)(lane & 2) << 30, f8 = (uint32_t)(lane & 8) << 28;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = wht_lane_stage<1>(v[j], f1, lane);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = wht_lane_stage<2>(v[j], f2, lane);
    wht_lane_stage4(v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = wht_lane_stage<8>(v[j], f8, lane);
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
        wht_lane_stage16(v[j], v[j + 1]);
        v[j] *= 0.0625f;
        v[j + 1] *= 0.0625f;
    }
}
// sign[i] * x[i], then the transform
__device__ __forceinline__ void sign_wht256(float (&v)[8], int lane) {
    const int l32 = lane & 31;
    const uint32_t sb = sign_word(l32 >> 2) >> (8 * (l32 & 3));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(__float_as_uint(v[j]) ^ (((sb >> j) & 1u) << 31));
    wht256(v, lane);
}
// Sixteen times the transform, negated in the lanes where wht256_flipped() says so: a lane stage is then one instruction a value,
// x +- x[lane ^ H] (the exact form's difference is x[lane ^ H] - x in the lanes with bit H set, the same but for its sign).  A
// zero may have the other sign than the exact form's.
__device__ __forceinline__ constexpr bool wht256_flipped(int lane) { return __builtin_popcount(lane & 11) & 1; }
__device__ __forceinline__ void wht256_times16_flipped(float (&v)[8], int lane) {
    wht_register_stages(v);
    const float s1 = (lane & 1) ? -1.0f : 1.0f, s2 = (lane & 2) ? -1.0f : 1.0f, s8 = (lane & 8) ? -1.0f : 1.0f;
    // (a value is read across lanes two instructions behind its write at the earliest)
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %0, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %2, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %3, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %4, %4, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %5, %5, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %6, %6, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %7, %7, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %0, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %2, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %3, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %4, %4, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %5, %5, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %6, %6, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %7, %7, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])
        : "v"(s1), "v"(s2));
    wht_lane_stage4(v);
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %0, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %2, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %3, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %4, %4, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %5, %5, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %6, %6, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %7, %7, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])
        : "v"(s8));
#pragma unroll
    for (int j = 0; j < 8; j += 2) wht_lane_stage16(v[j], v[j + 1]);
}

// sums of the eight 32-element groups: lanes 4 g .. 4 g + 3 receive the sum of group g, added
// in the order of the 32-lane butterfly (element e with e ^ 16, then ^ 8, ^ 4, ^ 2, ^ 1).  FLIPPED: of values negated in the lanes
// of wht256_flipped(), where lane ^ 2 and lane ^ 1 are the other way; the sums come out negated in the same lanes.
template <bool FLIPPED = false>
__device__ __forceinline__ float group32_sums(const float (&p)[8], int lane) {
    float t[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = FLIPPED ? lane_xor<2>(p[r], lane) - p[r] : p[r] + lane_xor<2>(p[r], lane);
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = FLIPPED ? lane_xor<1>(t[r], lane) - t[r] : t[r] + lane_xor<1>(t[r], lane);
    const float a0 = t[0] + t[4], a1 = t[1] + t[5], a2 = t[2] + t[6], a3 = t[3] + t[7];
    const float b0 = a0 + a2, b1 = a1 + a3;
    return b0 + b1;
}

// (((0 + S0) + S1) + S2) + S3 over the four groups of a 16-lane row, in every lane of the row
__device__ __forceinline__ float row_sum_of_groups(float s, int lane) {
    float x = 0.0f + s;  // the reference accumulates from +0: a sum of -0 terms ends as +0
    x = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x114, 0xF, 0xF, false)) + s;  // row_shr:4
    x = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x114, 0xF, 0xF, false)) + s;
    x = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x114, 0xF, 0xF, false)) + s;
    // lanes 12-15 of the row hold the total; hand it to the whole row
    return __int_as_float(__builtin_amdgcn_ds_bpermute((lane | 12) << 2, __float_as_int(x)));
}

// Codes of a lane's eight elements -- the number of boundaries below the value (op_kv_cache.cu:186-189) --
// and their centroids.  64 equal cells of 1 / 120.25 around zero, of which no one holds two boundaries and no boundary is
// within a quarter of a cell of an edge: the cell of u (rounded as it may be) names the one boundary u has to be
// compared with and the code below it.  The cell tables are held across the lanes and fetched with ds_bpermute
// (no memory access); what the first two fetches give is the lane of the third, 16 + code.
// Instruction-bound: 4 096 tokens x 2 heads of K and V, us a call: 9.7 with a binary search (two thresholds by selection, two
// fetched), 9.1 with this.
constexpr float kCellsPerUnit = 120.25f, kCellOfZero = 31.5f;
constexpr uint64_t tq4_cells_with_boundary() {
    uint64_t cells = 0;
    for (int k = 0; k < 15; ++k) cells |= 1ull << (int)(kBoundaries[k] * kCellsPerUnit + kCellOfZero);
    return cells;
}
// Where u is rounded across the edge of a cell, both cells give the same code only while no boundary is near the edge; the first and the
// last cell also take what saturates (and NaN), so they hold none.
constexpr bool tq4_boundaries_inside_cells() {
    for (int k = 0; k < 15; ++k) {
        const float at = kBoundaries[k] * kCellsPerUnit + kCellOfZero, in_cell = at - (float)(int)at;
        if (!(at >= 1.0f && at < 63.0f && in_cell >= 0.25f && in_cell <= 0.75f)) return false;
    }
    return __builtin_popcountll(tq4_cells_with_boundary()) == 15;
}
static_assert(tq4_boundaries_inside_cells(), "every boundary in a cell of its own, away from its edges");
// What a lane of the encoder holds throughout, from one table of constants (two loads that are on their way beside those of the
// row; worked out, 45 vector instructions of a wave's 433).
struct __attribute__((aligned(16))) Tq4Lane {
    uint32_t sign[4];  // of elements 8 l32 + 2 k (bit 15) and + 2 k + 1 (bit 31): the signs of the rotation, set where negative
    float boundary;    // lane i: of cell i the boundary in it (or +inf)
    int at;            // 4 (16 + number of boundaries below cell i)
    float centroid;    // i % 16
    float scale;       // 1/16, negated in the lanes of wht256_flipped()
};
struct Tq4LaneTable {
    Tq4Lane lane[64];
};
constexpr Tq4LaneTable make_tq4_lane_table() {
    Tq4LaneTable t{};
    constexpr uint64_t kCells = tq4_cells_with_boundary();
    int below = 0;
    for (int i = 0; i < 64; ++i) {
        Tq4Lane& l = t.lane[i];
        for (int k = 0; k < 4; ++k) {
            const int e = 8 * (i & 31) + 2 * k;
            const uint32_t even = kSignMask[e >> 5] >> (e & 31) & 1u, odd = kSignMask[(e + 1) >> 5] >> ((e + 1) & 31) & 1u;
            l.sign[k] = even << 15 | odd << 31;
        }
        const bool has = (kCells >> i) & 1u;
        l.boundary = has ? kBoundaries[below] : __builtin_inff();
        l.at = 4 * (16 + below);
        below += has ? 1 : 0;
        l.centroid = kCentroids[i & 15];
        l.scale = wht256_flipped(i) ? -0.0625f : 0.0625f;
    }
    return t;
}
__device__ __constant__ constexpr Tq4LaneTable kTq4LaneTable = make_tq4_lane_table();
__device__ __forceinline__ const uint4* tq4_lane_entry(int lane) { return reinterpret_cast<const uint4*>(&kTq4LaneTable.lane[lane]); }
__device__ __forceinline__ Tq4Lane tq4_lane_of(const uint4 a, const uint4 b) {  // the entry's two halves
    return Tq4Lane{{a.x, a.y, a.z, a.w}, __uint_as_float(b.x), (int)b.y, __uint_as_float(b.z), __uint_as_float(b.w)};
}
__device__ __forceinline__ Tq4Lane tq4_lane(int lane) {
    const uint4* src = tq4_lane_entry(lane);
    return tq4_lane_of(src[0], src[1]);
}
__device__ __forceinline__ void tq4_codes(const float (&v)[8], float inv_norm, const Tq4Lane& tab, uint32_t& halves_lo,
                                          uint32_t& halves_hi, float (&c)[8]) {
    int at[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float u = v[j] * inv_norm;
        // four times the cell: the byte address ds_bpermute takes, which ignores its two low bits.  The conversion saturates at 0 and
        // 255, NaN to 0 (a NaN is above no boundary); whether it rounds or truncates is an eighth of a cell.
        const uint32_t cell = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(u, 4.0f * kCellsPerUnit, 4.0f * kCellOfZero), 0u, 0u);
        const float t = __int_as_float(__builtin_amdgcn_ds_bpermute((int)cell, __float_as_int(tab.boundary)));
        const int below = __builtin_amdgcn_ds_bpermute((int)cell, tab.at);
        at[j] = below + ((u > t) ? 4 : 0);  // 4 (16 + code)
        c[j] = __int_as_float(__builtin_amdgcn_ds_bpermute(at[j], __float_as_int(tab.centroid)));
    }
    // nibble pairs (even element low), two bytes per half: 4 (code bytes) + what the sixteens add up to
    constexpr int kSixteens = 64 * (1 + 16) * (1 + 256);
    const int p0 = at[0] + 16 * at[1], p1 = at[2] + 16 * at[3], p2 = at[4] + 16 * at[5], p3 = at[6] + 16 * at[7];
    halves_lo = (uint32_t)(p0 + 256 * p1 - kSixteens) >> 2;
    halves_hi = (uint32_t)(p2 + 256 * p3 - kSixteens) >> 2;
}

// TQ4 encode of one 256-wide row, v[j] = sign * x[8 l32 + j] (op_kv_cache.cu:152-218).  The 132 row
// bytes are assembled in `row` (LDS, private to this half-wave).  Lanes 0-15 hold the first
// scale block, lanes 16-31 the second: one instruction stream computes both norms and scales.
__device__ __forceinline__ void tq4_store_codes(uint8_t* row, int l32, uint32_t lo, uint32_t hi) {
    // byte m of a 64-byte block holds elements 2m (low nibble) and 2m + 1 (high nibble):
    // elements 8 l32 .. + 7 are bytes 4 (l32 % 16) .. + 3 of block l32 / 16
    uint8_t* wdst = row + 66 * (l32 >> 4) + 2 + 4 * (l32 & 15);
    *reinterpret_cast<uint16_t*>(wdst) = (uint16_t)lo;
    *reinterpret_cast<uint16_t*>(wdst + 2) = (uint16_t)hi;
}
__device__ __forceinline__ void tq4_encode_row_exact(float (&v)[8], int lane, const Tq4Lane& tab, uint8_t* row) {
    const int l32 = lane & 31;
    wht256(v, lane);

    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = v[j] * v[j];
    const float s_sq = row_sum_of_groups(group32_sums(p, lane), lane);
    // (an infinite sum has the reciprocal root 0)
    const float inv_norm = (s_sq > 1e-20f && s_sq <= 3.402823466e38f) ? (0.7071067811865475f * rsqrt_rn_normal(s_sq)) : 0.0f;

    float c[8];
    uint32_t lo, hi;
    tq4_codes(v, inv_norm, tab, lo, hi, c);
    tq4_store_codes(row, l32, lo, hi);

    float pv[8], pc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        pv[j] = v[j] * c[j];
        pc[j] = c[j] * c[j];
    }
    const float vc_dot = row_sum_of_groups(group32_sums(pv, lane), lane);
    const float c_sq = row_sum_of_groups(group32_sums(pc, lane), lane);
    if ((l32 & 15) == 0) {
        const float d = (c_sq > 1e-10f) ? (vc_dot / c_sq) : 0.0f;
        *reinterpret_cast<uint16_t*>(row + 66 * (l32 >> 4)) = F16::from_f32(d);
    }
}
// The same bytes at 55 instructions less: the transform's shorter form, whose values y are 16 v, some of them negated.  Powers of two and
// signs go through products and sums unchanged while nothing is infinite and nothing that counts is subnormal; rows for which
// that is not so (by their sum of squares) take the exact form, all rows of a wave together.
__device__ __forceinline__ void tq4_encode_row(const float (&x)[8], int lane, const Tq4Lane& tab, uint8_t* row) {
    const int l32 = lane & 31;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = x[j];
    wht256_times16_flipped(v, lane);

    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = v[j] * v[j];
    const float s_sq256 = row_sum_of_groups(group32_sums(p, lane), lane);
    if (__builtin_expect(__ballot(!(s_sq256 >= 1e-15f && s_sq256 <= 3.402823466e38f)) != 0ull, 0)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[j];
        tq4_encode_row_exact(v, lane, tab, row);
        return;
    }
    const float inv_norm = 0.7071067811865475f * rsqrt_rn_normal(s_sq256 * 0.00390625f);

    float c[8];
    uint32_t lo, hi;
    tq4_codes(v, inv_norm * tab.scale, tab, lo, hi, c);
    tq4_store_codes(row, l32, lo, hi);

    float pv[8], pc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        pv[j] = v[j] * c[j];
        pc[j] = c[j] * c[j];
    }
    const float vc_dot = row_sum_of_groups(group32_sums<true>(pv, lane) * tab.scale, lane);
    const float c_sq = row_sum_of_groups(group32_sums(pc, lane), lane);
    if ((l32 & 15) == 0) {
        const float d = (c_sq > 1e-10f) ? (vc_dot / c_sq) : 0.0f;
        *reinterpret_cast<uint16_t*>(row + 66 * (l32 >> 4)) = F16::from_f32(d);
    }
}

// TQ4 without the rotation (op_kv_cache.cu:219-264): the block quantiser on the raw 128-element
// blocks of the row, v[j] = x[8 l32 + j]; lanes 0-15 hold block 0, lanes 16-31 block 1 (absent at
// head dimension 128: those lanes carry zeros and their bytes are not stored).  The reference sums
// with block_reduce_sum_128 (tq4_kv_common.cuh:109-124): the 32-lane butterfly inside each warp,
// then the same butterfly over the four warp sums in lanes 0-3 of a warp whose other lanes hold
// +0 -- three additions of +0, then (s0 + s2) + (s1 + s3).
__device__ __forceinline__ float block128_sum(const float (&p)[8], int lane) {
    float t = group32_sums(p, lane);  // lanes 4 g .. 4 g + 3: the sum of warp g of the row
    t = ((t + 0.0f) + 0.0f) + 0.0f;   // (a sum that is -0 ends as +0, as in the reference)
    t = t + lane_xor<8>(t, lane);     // s0 + s2 (lanes of warps 0, 2), s1 + s3 (warps 1, 3)
    return t + lane_xor<4>(t, lane);
}

__device__ __forceinline__ void tq4_encode_row_plain(const float (&v)[8], int lane, const Tq4Lane& tab, uint8_t* row) {
    const int l32 = lane & 31;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = v[j] * v[j];
    const float norm_x = __builtin_sqrtf(block128_sum(p, lane));
    const float inv_norm = (norm_x > 1e-12f) ? (0.7071067811865475f / norm_x) : 0.0f;
    float c[8];
    uint32_t lo, hi;
    tq4_codes(v, inv_norm, tab, lo, hi, c);
    // ("q = b + 1 for the last boundary b below u" over ascending boundaries = the number of boundaries below u)
    tq4_store_codes(row, l32, lo, hi);

    float pv[8], pc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        pv[j] = v[j] * c[j];
        pc[j] = c[j] * c[j];
    }
    const float xc_dot = block128_sum(pv, lane);
    const float c_sq = block128_sum(pc, lane);
    if ((l32 & 15) == 0) {
        const float d = (c_sq > 1e-12f) ? (xc_dot / c_sq) : 0.0f;
        *reinterpret_cast<uint16_t*>(row + 66 * (l32 >> 4)) = F16::from_f32(d);
    }
}

// fp32 -> OCP FP8 E4M3, round to nearest even, saturating at +-448, NaN -> 0x7f
// (__nv_cvt_float2_to_fp8x2(.., __NV_SATFINITE, __NV_E4M3) in op_kv_cache.cu:83-86).  Integer
// arithmetic, so the bits do not depend on a hardware conversion mode.
__device__ __forceinline__ uint32_t f32_to_e4m3(float f) {
    const uint32_t u = __float_as_uint(f);
    const uint32_t sign = (u >> 24) & 0x80u;
    const uint32_t ax = u & 0x7fffffffu;
    if (ax > 0x7f800000u) return sign | 0x7fu;
    const float a = __uint_as_float(ax);
    if (a >= 448.0f) return sign | 0x7eu;
    if (a < 0.015625f) return sign | (uint32_t)rintf(a * 512.0f);  // multiples of 2^-9
    uint32_t r = (ax + 0x7ffffu + ((ax >> 20) & 1u)) >> 20;
    r -= (127u - 7u) << 3;
    return sign | (r > 0x7eu ? 0x7eu : r);
}

// 8-bit rows of a 256-wide head, identity transform; lane l32 holds elements 8 l32 .. 8 l32 + 7.
//   FP8:  264 B = 256 codes, then fp32 d0 (elements 0..127) and d1; d = amax / 448
//         (op_kv_cache.cu:104-138)
//   Q8_0: 272 B = 4 x {fp32 d, 64 int8}; d = amax / 127, q = clamp(roundf(x / d))
//         (op_kv_cache.cu:32-62)
// max() is exact and order-free, so only the element-wise arithmetic has to follow the source.
__device__ __forceinline__ void fp8_encode_row(const float (&v)[8], int lane, uint8_t* row) {
    const int l32 = lane & 31;
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    amax = fmaxf(amax, lane_xor<8>(amax, lane));
    amax = fmaxf(amax, lane_xor<4>(amax, lane));
    amax = fmaxf(amax, lane_xor<2>(amax, lane));
    amax = fmaxf(amax, lane_xor<1>(amax, lane));
    const float d = amax * (1.0f / 448.0f);
    const float inv_d = (d > 1e-30f) ? (1.0f / d) : 0.0f;
    uint32_t w0 = 0, w1 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        w0 |= f32_to_e4m3(v[j] * inv_d) << (8 * j);
        w1 |= f32_to_e4m3(v[4 + j] * inv_d) << (8 * j);
    }
    *reinterpret_cast<uint2*>(row + 8 * l32) = uint2{w0, w1};
    if ((l32 & 15) == 0) *reinterpret_cast<float*>(row + 256 + 4 * (l32 >> 4)) = d;
}

__device__ __forceinline__ void q8_encode_row(const float (&v)[8], int lane, uint8_t* row) {
    const int l32 = lane & 31;
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    amax = fmaxf(amax, lane_xor<4>(amax, lane));
    amax = fmaxf(amax, lane_xor<2>(amax, lane));
    amax = fmaxf(amax, lane_xor<1>(amax, lane));
    const float d = amax / 127.0f;
    const float inv_d = (d > 1e-12f) ? (1.0f / d) : 0.0f;
    uint32_t w0 = 0, w1 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float q0 = fminf(127.0f, fmaxf(-127.0f, roundf(v[j] * inv_d)));
        const float q1 = fminf(127.0f, fmaxf(-127.0f, roundf(v[4 + j] * inv_d)));
        w0 |= ((uint32_t)(int)q0 & 0xffu) << (8 * j);
        w1 |= ((uint32_t)(int)q1 & 0xffu) << (8 * j);
    }
    uint8_t* blk = row + 68 * (l32 >> 3);
    *reinterpret_cast<uint32_t*>(blk + 4 + 8 * (l32 & 7)) = w0;
    *reinterpret_cast<uint32_t*>(blk + 8 + 8 * (l32 & 7)) = w1;
    if ((l32 & 7) == 0) *reinterpret_cast<float*>(blk) = d;
}

// Encodes one 256-wide row held as v[j] = x[8 l32 + j] (not yet transformed) in `format` /
// `transform`, assembles it in the half-wave's LDS area `row` (272 bytes, 8-byte aligned) and
// stores it at dst (nothing is stored for dst == nullptr).  16-bit formats are stored directly.
// Rotated 8-bit rows are the un-rotated encoders applied to the transformed row
// (op_kv_cache.cu:36-44,71-99: the same scale and code arithmetic; max is order-free).  The
// caller guarantees what the append entry points check: head_dim 256, TQ4 with WHT256, 8-bit
// rows 4-byte aligned.
// tab: tq4_lane(lane) for TQ4 rows, requested well before (not looked at otherwise).
// ROTATED_TQ4: the caller knows that the row is one; a kernel that holds this form alone needs fewer registers.
template <bool ROTATED_TQ4 = false>
__device__ __forceinline__ void encode_store_row(float (&v)[8], int format, int transform, int lane, const Tq4Lane& tab,
                                                 uint8_t* row, uint8_t* dst) {
    const int l32 = lane & 31;
    int n_dwords = 33;
    if constexpr (!ROTATED_TQ4) {
        if (format == WARP34_KV_FORMAT_FP16 || format == WARP34_KV_FORMAT_BF16) {
            if (dst == nullptr) return;
            uint16_t* d16 = reinterpret_cast<uint16_t*>(dst) + 8 * l32;
#pragma unroll
            for (int j = 0; j < 8; ++j) d16[j] = (format == WARP34_KV_FORMAT_BF16) ? BF16::from_f32(v[j]) : F16::from_f32(v[j]);
            return;
        }
    }
    if (ROTATED_TQ4 || format == WARP34_KV_FORMAT_TQ4) {
        if (ROTATED_TQ4 || transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = __uint_as_float(__float_as_uint(v[j]) ^ ((j & 1 ? tab.sign[j >> 1] : tab.sign[j >> 1] << 16) & 0x80000000u));
            tq4_encode_row(v, lane, tab, row);
        } else {
            tq4_encode_row_plain(v, lane, tab, row);
        }
    } else {
        if (transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256) sign_wht256(v, lane);
        if (format == WARP34_KV_FORMAT_FP8_E4M3) {
            fp8_encode_row(v, lane, row);
            n_dwords = 66;
        } else {
            q8_encode_row(v, lane, row);
            n_dwords = 68;
        }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (dst == nullptr) return;  // a half that only keeps the other half's cross-lane steps company
    if ((reinterpret_cast<uintptr_t>(dst) & 3u) == 0) {
        const uint32_t* r32 = reinterpret_cast<const uint32_t*>(row);
        uint32_t* d32 = reinterpret_cast<uint32_t*>(dst);
        for (int i = l32; i < n_dwords; i += 32) d32[i] = r32[i];
    } else {  // TQ4 rows promise 2-byte alignment only
        const uint16_t* r16 = reinterpret_cast<const uint16_t*>(row);
        uint16_t* d16 = reinterpret_cast<uint16_t*>(dst);
        for (int i = l32; i < 2 * n_dwords; i += 32) d16[i] = r16[i];
    }
}

// v[j] = x[l32 + 32 j] (one element per lane and register, as a kernel holds a row whose pairs
// (i, i + 128) it has just rotated) -> v[j] = x[8 l32 + j], through 1 KB of LDS private to the
// half-wave.  Whole-wave call.
__device__ __forceinline__ void strided_to_consecutive(float (&v)[8], int lane, float* xpose) {
    const int l32 = lane & 31;
#pragma unroll
    for (int j = 0; j < 8; ++j) xpose[l32 + 32 * j] = v[j];
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const float4 a = *reinterpret_cast<const float4*>(xpose + 8 * l32);
    const float4 b = *reinterpret_cast<const float4*>(xpose + 8 * l32 + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// ---- host-side checks shared by the entry points that write rows ----
inline bool format_supported_for_write(int format, int transform, int head_dim) {
    if (format == WARP34_KV_FORMAT_FP16 || format == WARP34_KV_FORMAT_BF16) {
        return transform == WARP34_KV_TRANSFORM_IDENTITY;
    }
    if (format == WARP34_KV_FORMAT_TQ4) {
        // rotated at head dimension 256 with the WHT-256 transform; every other combination is the
        // plain block quantiser, one block per 128 elements (op_kv_cache.cu:152,219)
        return head_dim == 256 || head_dim == 128;
    }
    if (format == WARP34_KV_FORMAT_Q8_0 || format == WARP34_KV_FORMAT_FP8_E4M3) {
        // the tail-anchor layers of the default policy store these un-rotated (cache.rs:87-109);
        // the rotated variant is what op_kv_cache.cu:36-44,71-99 accepts as well
        return head_dim == 256 && (transform == WARP34_KV_TRANSFORM_IDENTITY ||
                                   transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256);
    }
    return false;
}

inline bool is_8bit_format(int format) {
    return format == WARP34_KV_FORMAT_Q8_0 || format == WARP34_KV_FORMAT_FP8_E4M3;
}

// Q8_0 and FP8 rows carry fp32 scales (alignof 4, tq4_kv_common.cuh:28-46) and are stored with
// 32-bit stores.
inline bool rows_aligned_for_write(const warp34_kv_layer_layout* l) {
    if (is_8bit_format(l->k_format) &&
        ((l->k_base | l->k_page_stride_bytes | l->k_head_stride_bytes | l->k_token_stride_bytes) & 3u)) {
        return false;
    }
    if (is_8bit_format(l->v_format) &&
        ((l->v_base | l->v_page_stride_bytes | l->v_head_stride_bytes | l->v_token_stride_bytes) & 3u)) {
        return false;
    }
    return true;
}


}  // namespace w34
