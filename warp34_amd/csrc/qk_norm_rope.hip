// QK RMSNorm + RoPE over packed bf16 rows for gfx950, optionally fused with the append of the
// rotated K row and the V row into the paged KV cache: the producer side of the KV path, one
// HBM round trip instead of two (operator, then append).
//
// Replaces qk_norm_rope_bf16_warp and its four entry points (ops/op_dflash2.cu:338-418,
// 1251-1410).  The reference's fused cache write takes BF16 pages only (op_dflash2.cu:1326-1333);
// here the cache may also be TQ4 + WHT256, FP8-E4M3 or Q8_0 at head_dim 256, encoded by the same
// row encoders as the append kernel, so a fused write equals operator + append bit for bit.
//
// Mapping: one wave per work item, two items' worth of lanes: lanes 0-31 and lanes 32-63 each
// play the reference's 32-thread warp.  A Q item handles two Q heads; a KV item handles one K
// head (lanes 0-31: norm, rotation, cache row or in-place store) and, when the cache is
// written, the V row of the same kv head (lanes 32-63).
//
// Numerics (bit-exact contract with the CPU restatement, file built with -ffp-contract=off):
// fp32 in source order; sum of squares in the order of reduce_sum256_exact_warp
// (op_dflash2.cu:30-39); rsqrt(x) computed as (float)(1.0 / sqrt((double)x)); bf16 RNE.
#include "kv_encode.h"

namespace w34 {

struct NormRopeParams {
    uint16_t* q_out;       // [rows, q_heads * dim] or null (Q in place)
    const void* table;     // [table_rows, dim]: cos (dim/2) | sin (dim/2)
    warp34_kv_layer_layout L;
    int table_rows;
    float eps;
};

// A call over a few rows is a chain of memory round trips: the leading arguments are in scalar registers when a wave starts, so
// position, slot, row and weights are asked for at once, and the table's row as soon as the position is there (before: arguments,
// position, row, weights and table, for head sizes other than 256 the row a second time).  us: four draft blocks of sixteen
// tokens over 16 + 4 heads of 128, with their attention, 24.1 before / 21.7 a layer; 8 192 tokens over 16 + 2 heads of 256 to
// rotated TQ4 pages 40.8 / 36.2.
// HD: the head size where it is known at compile time (256 or 128: no bounds tests, the second pass reuses the values of the
// first), else 0.  PAGES: what the rows may go to besides q_out and the packed rows.
enum NormRopePages { kBf16Pages, kRotatedTq4Pages, kQuantisedPages };
template <bool TABLE_F32, int HD, NormRopePages PAGES>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(const int32_t* __restrict__ positions, const int32_t* __restrict__ slots,
                                                           uint16_t* qkv,  // [rows, (q_heads + 2 kv_heads) * dim] bf16
                                                           const uint16_t* __restrict__ qw, const uint16_t* __restrict__ kw, int rows,
                                                           int q_heads, int kv_heads, int dim_arg, const NormRopeParams P) {
    constexpr bool QUANT = PAGES != kBf16Pages;
    static_assert(!QUANT || HD == 256, "quantised pages: head size 256");
    __shared__ __align__(8) uint8_t rows_lds[QUANT ? 4 : 1][2][272];
    __shared__ __align__(16) float xpose_lds[QUANT ? 4 : 1][2][256];  // register layout of the rotation -> the encoder's
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = lane_id();
    const int half_id = lane >> 5;
    const int l32 = lane & 31;
    // Items are ordered KV items of all rows first, then the Q items: the long items (norm +
    // two row encodes) start first and every workgroup holds items of one kind.
    const int q_items = (q_heads + 1) >> 1;
    int row, it;
    {
        const long long n_kv_items = (long long)rows * kv_heads, item = (long long)blockIdx.x * 4 + wave;
        const bool kv = item < n_kv_items;
        const long long n = kv ? item : item - n_kv_items;
        const int per_row = kv ? kv_heads : q_items;
        if (n < (1 << 21) && per_row > 0) {  // (uniform: exact by the float quotient and one correction)
            row = __builtin_amdgcn_readfirstlane((int)((float)(int)n * __builtin_amdgcn_rcpf((float)per_row)));
            const int r = (int)n - row * per_row;
            row += r >= per_row ? 1 : r < 0 ? -1 : 0;
        } else {
            row = per_row > 0 ? (int)(n / per_row) : rows;
        }
        if (row >= rows) return;
        it = (int)(n - (long long)row * per_row) + (kv ? q_items : 0);
    }
    const int pos = positions[row];

    const int dim = HD ? HD : dim_arg, half = dim >> 1;
    const size_t row_elems = (size_t)(q_heads + 2 * kv_heads) * dim;
    uint16_t* row_base = qkv + (size_t)row * row_elems;

    // Both halves of the wave run the same instruction stream (the cross-lane steps want the
    // whole wave): the half without a head of its own (the V half of a KV item, the second half
    // of the last Q item when q_heads is odd) computes on a row it may read and stores nothing.
    const bool is_q = it < q_items;
    const bool is_v_half = !is_q && half_id == 1;
    const int kv_head = is_q ? 0 : it - q_items;
    int head = is_q ? 2 * it + half_id : q_heads + kv_head;
    const bool has_head = is_q ? head < q_heads : !is_v_half;
    if (is_q && head >= q_heads) head = q_heads - 1;

    // V half: its "head" is the V row of the kv head (read-only)
    uint16_t* src = row_base + (size_t)(is_v_half ? q_heads + kv_heads + kv_head : head) * dim;
    const uint16_t* w = is_q ? qw : kw;

    // sum of squares, element c = l32 + 32 k in register k (op_dflash2.cu:362-380)
    constexpr int kPairs = HD ? HD / 64 : 4;  // pairs (c, half + c) of a lane
    uint16_t raw16[8], w16[2 * kPairs];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int c = l32 + 32 * k;
        raw16[k] = (HD ? c < HD : c < dim) ? src[c] : (uint16_t)0;
    }
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
        const int c = l32 + 32 * k;
        w16[k] = w16[kPairs + k] = 0;
        if (HD || c < half) {
            w16[k] = w[c];
            w16[kPairs + k] = w[half + c];
        }
    }
    const int slot = (!is_q && slots != nullptr) ? slots[row] : -1;
    // (the compiler would load these only where they are used, behind the checks)
    asm volatile("" ::"s"(pos), "s"(P.table), "s"(P.table_rows), "s"(P.q_out), "s"(P.L.k_base), "s"(P.L.v_base), "s"(P.L.k_page_stride_bytes),
                 "s"(P.L.k_head_stride_bytes), "s"(P.L.k_token_stride_bytes), "s"(P.L.block_size));
    const bool to_cache = slot >= 0;  // wave-uniform
    if (pos < 0 || pos >= P.table_rows) return;  // op_dflash2.cu:356
    float cosine[kPairs], sine[kPairs];
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
        const int c = l32 + 32 * k;
        cosine[k] = sine[k] = 0.0f;
        if (HD || c < half) {
            if constexpr (TABLE_F32) {
                const float* t = reinterpret_cast<const float*>(P.table) + (size_t)pos * dim;
                cosine[k] = t[c];
                sine[k] = t[half + c];
            } else {
                const uint16_t* t = reinterpret_cast<const uint16_t*>(P.table) + (size_t)pos * dim;
                cosine[k] = BF16::to_f32(t[c]);
                sine[k] = BF16::to_f32(t[half + c]);
            }
        }
    }
    Tq4Lane tab{};
    if (QUANT && to_cache && (PAGES == kRotatedTq4Pages || P.L.k_format == WARP34_KV_FORMAT_TQ4)) tab = tq4_lane(lane);  // (used by the row encoder)

    float raw[8], sq[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        raw[k] = BF16::to_f32(raw16[k]);
        sq[k] = raw[k] * raw[k];
    }
    float s = ((sq[0] + sq[4]) + (sq[2] + sq[6])) + ((sq[1] + sq[5]) + (sq[3] + sq[7]));
    s = half_wave_sum(s, lane);
    const float mean = s / (float)dim + P.eps;
    const float inv = rsqrt_rn(mean);

    // rotated values of this lane: out[c] and out[half + c] for c = l32, l32 + 32, ... < half
    float lo[kPairs], hi[kPairs];
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
        const int c = l32 + 32 * k;
        lo[k] = hi[k] = 0.0f;
        if (HD || c < half) {
            const float x_lo = raw[k];  // element l32 + 32 k, of every head size
            const float x_hi = HD ? raw[(k + kPairs) & 7] : BF16::to_f32(src[half + c]);
            const float a = BF16::to_f32(BF16::from_f32(x_lo * inv * BF16::to_f32(w16[k])));
            const float b = BF16::to_f32(BF16::from_f32(x_hi * inv * BF16::to_f32(w16[kPairs + k])));
            const float ac = a * cosine[k], bs = b * sine[k], bc = b * cosine[k], as = a * sine[k];
            lo[k] = BF16::to_f32(BF16::from_f32(ac - bs));
            hi[k] = BF16::to_f32(BF16::from_f32(bc + as));
        }
    }

    if (to_cache) {
        // rotated K (lanes 0-31) and the V row as it is (lanes 32-63) into the cache; the packed
        // row keeps its K (op_dflash2.cu:387-416)
        const int page = slot / P.L.block_size, off = slot - page * P.L.block_size;
        uint8_t* dst = reinterpret_cast<uint8_t*>((uintptr_t)(is_v_half ? P.L.v_base : P.L.k_base)) +
                       (size_t)page * (is_v_half ? P.L.v_page_stride_bytes : P.L.k_page_stride_bytes) +
                       (size_t)kv_head * (is_v_half ? P.L.v_head_stride_bytes : P.L.k_head_stride_bytes) +
                       (size_t)off * (is_v_half ? P.L.v_token_stride_bytes : P.L.k_token_stride_bytes);
        if constexpr (QUANT) {
            // Quantised pages: head_dim 256, K and V in the same format and transform (host
            // check), so both halves take the same path through the encoder.  Element
            // l32 + 32 j is lo[j] for j < 4 and hi[j - 4] above.
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = is_v_half ? raw[j] : (j < 4 ? lo[j & 3] : hi[j & 3]);
            strided_to_consecutive(v, lane, xpose_lds[wave][half_id]);
            encode_store_row<PAGES == kRotatedTq4Pages>(v, P.L.k_format, P.L.k_transform, lane, tab, rows_lds[wave][half_id], dst);
        } else {  // both slabs are BF16 (host check)
            uint16_t* d16 = reinterpret_cast<uint16_t*>(dst);
            if (is_v_half) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int c = l32 + 32 * k;
                    if (HD ? c < HD : c < dim) d16[c] = raw16[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < kPairs; ++k) {
                    const int c = l32 + 32 * k;
                    if (HD || c < half) {
                        d16[c] = BF16::from_f32(lo[k]);
                        d16[half + c] = BF16::from_f32(hi[k]);
                    }
                }
            }
        }
        return;
    }
    if (!has_head) return;
    uint16_t* dst = (is_q && P.q_out != nullptr) ? P.q_out + ((size_t)row * q_heads + head) * dim : src;
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
        const int c = l32 + 32 * k;
        if (HD || c < half) {
            dst[c] = BF16::from_f32(lo[k]);
            dst[half + c] = BF16::from_f32(hi[k]);
        }
    }
}

static bool norm_rope_args_ok(const warp34_exec* ex, const void* qkv, const int32_t* positions, const void* qw,
                              const void* kw, const void* table, int rows, int q_heads, int kv_heads, int dim,
                              int table_rows, float eps) {
    return ex && qkv && positions && qw && kw && table && rows >= 0 && q_heads >= 0 && kv_heads > 0 &&
           q_heads % kv_heads == 0 && dim > 0 && dim <= 256 && dim % 2 == 0 && table_rows > 0 && eps > 0.0f &&
           eps <= 3.402823466e38f;  // finite: NaN fails the first comparison, +inf this one
}

template <bool TABLE_F32>
static int launch_norm_rope(const warp34_exec* ex, void* qkv, void* q_out, const int32_t* positions, const void* qw,
                            const void* kw, const void* table, const warp34_kv_layer_layout* layout,
                            const int32_t* write_slot_mapping, int rows, int q_heads, int kv_heads, int dim,
                            int table_rows, float eps) {
    NormRopeParams P{};
    P.q_out = (uint16_t*)q_out;
    P.table = table;
    if (layout != nullptr) P.L = *layout;
    P.table_rows = table_rows;
    P.eps = eps;
    const long long items = (long long)rows * ((q_heads + 1) / 2 + kv_heads);
    const unsigned grid = (unsigned)((items + 3) / 4);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, (hipStream_t)ex->stream, positions, write_slot_mapping, (uint16_t*)qkv,
                           (const uint16_t*)qw, (const uint16_t*)kw, rows, q_heads, kv_heads, dim, P);
    };
    if (layout != nullptr && layout->k_format != WARP34_KV_FORMAT_BF16) {
        const bool rotated_tq4 = layout->k_format == WARP34_KV_FORMAT_TQ4 && layout->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256;
        rotated_tq4 ? launch(qk_norm_rope_kernel<TABLE_F32, 256, kRotatedTq4Pages>) : launch(qk_norm_rope_kernel<TABLE_F32, 256, kQuantisedPages>);
    } else if (dim == 256) {
        launch(qk_norm_rope_kernel<TABLE_F32, 256, kBf16Pages>);
    } else if (dim == 128) {
        launch(qk_norm_rope_kernel<TABLE_F32, 128, kBf16Pages>);
    } else {
        launch(qk_norm_rope_kernel<TABLE_F32, 0, kBf16Pages>);
    }
    return (int)hipGetLastError();
}

}  // namespace w34

using namespace w34;

// op_dflash2.cu:1251-1278 (bf16 cos|sin table)
extern "C" int warp34_dflash_qk_norm_rope_bf16(const warp34_exec* ex, void* qkv, const int32_t* positions,
                                               const void* qw, const void* kw, const void* table, int rows,
                                               int q_heads, int kv_heads, int dim, int table_rows, float eps) {
    if (!norm_rope_args_ok(ex, qkv, positions, qw, kw, table, rows, q_heads, kv_heads, dim, table_rows, eps))
        return (int)hipErrorInvalidValue;
    if (rows == 0) return 0;
    return launch_norm_rope<false>(ex, qkv, nullptr, positions, qw, kw, table, nullptr, nullptr, rows, q_heads,
                                   kv_heads, dim, table_rows, eps);
}

// op_dflash2.cu:1280-1308 (fp32 table, Q to a contiguous buffer when q_out != null)
extern "C" int warp34_dflash_qk_norm_rope_bf16_f32_table_qout(const warp34_exec* ex, void* qkv, void* q_out,
                                                              const int32_t* positions, const void* qw,
                                                              const void* kw, const void* table, int rows,
                                                              int q_heads, int kv_heads, int dim, int table_rows,
                                                              float eps) {
    if (!norm_rope_args_ok(ex, qkv, positions, qw, kw, table, rows, q_heads, kv_heads, dim, table_rows, eps) ||
        q_out == qkv)
        return (int)hipErrorInvalidValue;
    if (rows == 0) return 0;
    return launch_norm_rope<true>(ex, qkv, q_out, positions, qw, kw, table, nullptr, nullptr, rows, q_heads,
                                  kv_heads, dim, table_rows, eps);
}

// op_dflash2.cu:1395-1410
extern "C" int warp34_dflash_qk_norm_rope_bf16_f32_table(const warp34_exec* ex, void* qkv, const int32_t* positions,
                                                         const void* qw, const void* kw, const void* table,
                                                         int rows, int q_heads, int kv_heads, int dim,
                                                         int table_rows, float eps) {
    return warp34_dflash_qk_norm_rope_bf16_f32_table_qout(ex, qkv, nullptr, positions, qw, kw, table, rows, q_heads,
                                                          kv_heads, dim, table_rows, eps);
}

// op_dflash2.cu:1310-1345.  The reference accepts BF16 pages only; TQ4 + WHT256, FP8-E4M3 and
// Q8_0 pages (head_dim 256) are accepted here as well.
extern "C" int warp34_dflash_qk_norm_rope_kv_write_bf16_f32_table(
    const warp34_exec* ex, void* qkv, void* q_out, const int32_t* positions, const void* qw, const void* kw,
    const void* table, const warp34_kv_layer_layout* kv_layout, const int32_t* write_slot_mapping, int rows,
    int q_heads, int kv_heads, int dim, int table_rows, float eps) {
    if (!norm_rope_args_ok(ex, qkv, positions, qw, kw, table, rows, q_heads, kv_heads, dim, table_rows, eps) ||
        !kv_layout || !write_slot_mapping || q_out == qkv || kv_layout->k_base == 0 || kv_layout->v_base == 0 ||
        kv_layout->block_size <= 0 || kv_layout->local_kv_heads != kv_heads || kv_layout->head_dim != dim) {
        return (int)hipErrorInvalidValue;
    }
    const bool bf16_pages = kv_layout->k_format == WARP34_KV_FORMAT_BF16 && kv_layout->v_format == WARP34_KV_FORMAT_BF16;
    const int fmt = kv_layout->k_format;
    const bool quantised_pages =
        dim == 256 && (fmt == WARP34_KV_FORMAT_TQ4 || is_8bit_format(fmt)) && kv_layout->v_format == fmt &&
        kv_layout->v_transform == kv_layout->k_transform &&
        format_supported_for_write(fmt, kv_layout->k_transform, dim) && rows_aligned_for_write(kv_layout);
    if (!bf16_pages && !quantised_pages) return (int)hipErrorInvalidValue;
    if (rows == 0) return 0;
    return launch_norm_rope<true>(ex, qkv, q_out, positions, qw, kw, table, kv_layout, write_slot_mapping, rows,
                                  q_heads, kv_heads, dim, table_rows, eps);
}
