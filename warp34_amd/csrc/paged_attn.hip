// Paged GQA decode / verify attention for gfx950 with split-K across workgroups.
//
// Replaces the reference's paged_attention_gqa_mma_f16_kernel, its split-KV reduce kernel and
// the dispatcher (op_paged_attn.cu:186-588,1132-1218,1266-1448), and the bf16 decode kernel
// (op_kv_cache.cu:873-1241).  The dispatch table of the reference is NOT reproduced: it is
// tuned for 84-SM GDDR parts and leaves long contexts on a handful of CTAs.
//
// Work decomposition
//   tile  = up to TT consecutive query tokens of one request x the q heads of one kv head
//           (16*NT MFMA columns; decode: 1 token x 8 heads -> 8 of 16 columns used)
//   chunk = contiguous range of 32-token "units" of the tile's visible keys; one workgroup
//           (8 waves) per (chunk, kv head, tile).  The number of chunks of a tile depends only
//           on the tile's own key range and on a host cap derived from total_tokens and the
//           scratch size -- never on max_seq_len, max_blocks_per_req, physical page numbers or
//           local_kv_heads -- so outputs are bit-identical under page permutation, graph-bucket
//           bounds and head sharding (tests/tq4_vision_and_moe.rs:1089-1663).
//   unit  = 32 consecutive tokens handled by ONE wave start to finish: the raw K and V rows of
//           the unit go straight from the pages into the wave's private LDS area (LDS-direct
//           16-byte loads from a wave-uniform base, one unit ahead), the wave forms
//           S^T = K Q'^T with MFMA, does the online softmax in registers and accumulates
//           O^T += V^T P^T with MFMA.  Waves never synchronise inside the key loop; their
//           (m, l, O) states are merged once at the end.
//
// TQ4 specifics (row = [fp16 d0][64 B nibbles][fp16 d1][64 B nibbles], 132 B, 33 dwords):
//   * dequantisation is a 256-entry LDS table indexed by a code BYTE that returns the two
//     centroids as packed fp16.  The table is replicated once per lane (entry stride 256 B) so
//     that random indices never conflict and the address is a single v_perm_b32:
//     addr = (byte << 8) | (lane << 2);
//   * the per-128 scales are not applied per element: K scales multiply the two half-row
//     partial scores, V scales are folded into the probabilities (two P matrices);
//   * LDS reads must be dword aligned (misaligned ds_read_b32 is ~15x slower on this part)
//     but the first half of a row starts at byte 2.  The K path therefore treats the row as 33
//     aligned dwords and zeroes the query for the 8 nibble slots that hold scale bytes; the V
//     path builds dword column 0 as [codes 0-3 | codes 124-127] from dwords 0 and 16, every
//     other column is an aligned dword;
//   * attention runs in the rotated domain: Q' = WHT(sign*q) once per tile, the output is
//     un-rotated once at the end (op_kv_cache.cu:443-451,763-783).
//
// MFMA use: v_mfma_f32_16x16x32_f16.  A = K rows (QK) or V^T (PV) so that every lane owns one
// query column: softmax state and the O rescale are per-lane scalars.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "kv_common.h"

namespace w34 {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

// waves per workgroup of the TQ4 decode kernels: eight, two per SIMD (up to 256 registers each); the
// LDS holds the table, eight staging areas, the query operand tables and the (m, l) tables, of 160 KB
// 140 (one column tile) or 150 (two): one workgroup per CU
constexpr int kTq4Waves = 8;
constexpr int kUnit = 32;             // tokens per wave iteration
constexpr int kLutBytes = 256 * 256;  // 256 entries x 64 lane replicas x 4 B
constexpr int kRunBytes = 16 * kTq4RowBytes;  // 16 rows = 2112 B = 132 16-byte pieces
constexpr int kStageTq4 = 4 * kRunBytes;      // K rows 0-31 then V rows 0-31: 8448 B
// column stride of a merge region in dwords: 1 056 bytes, a stride at which 128-bit accesses of
// eight columns do not collide (measured; 1 040 bytes cost 40 % more)
constexpr int kMergeColStride = 264;
constexpr int kMergeFloats = kTq4Waves * 8 * kMergeColStride;  // one region of 8 columns per wave
constexpr int kQopBytes = 16 * 4 * 9 * 16;  // query operand table of a column tile: 16 columns x 4 k-blocks x 8 operands, 144 bytes apart
// nt: column tiles of a workgroup
__host__ __device__ constexpr int ml_offset_for(int nt) {  // (m, l) tables of the merge: behind everything the loop uses
    return kLutBytes + kTq4Waves * kStageTq4 + nt * kQopBytes;
}
__host__ __device__ constexpr int smem_bytes_for(int nt) {
    return ml_offset_for(nt) + (kTq4Waves + 1) * nt * 16 * 2 * 4;
}
static_assert(kMergeFloats * 4 <= kTq4Waves * kStageTq4, "merge regions alias the staging areas only");
static_assert(smem_bytes_for(2) <= 160 * 1024, "decode LDS budget");
constexpr int kXcds = 8;  // workgroups go round them in launch order
constexpr int kChipCus = 256;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegBig = -1.0e30f;  // "minus infinity" that stays finite under subtraction
// The table holds fp16(kLutGain * centroid); the gain is divided out of the query (K side)
// and of the final normalisation (V side).  1.908032 minimises the worst fp16 rounding error
// of the eight centroid magnitudes (9.4e-5 relative instead of 3.7e-4), which is what limits
// the accuracy of the scores.
constexpr float kLutGain = 1.908032f;
constexpr float kLutInvGain = 1.0f / kLutGain;

// Weights of two operands (TQ4, BF16): a column's running maximum is raised only by scores that exceed it by more than this (log2 domain), so
// a probability may be up to 2^8; its operands keep 22 (16) bits of it whatever its size, the sums are fp32.  Raising multiplies 64 sums per column
// tile, and of the first units nearly every one raises the maximum of some column of a wave.  TQ4 value scales ride on the probabilities: in a
// unit with a larger one than kPfSlackScale, where the weight could leave fp16's range, and where a column does not see the whole unit (what lies
// behind the sequence must not matter), the maximum is exact.  Per column, so that tiles of either size give the same bits.  (One fp16
// operand: exact as well, the largest probability is then 1 and rounds to itself; with the slack FP16 and Q8_0 batches came out 6 % further from 64
// bits, 3.24e-4 for 3.05e-4.)  us, maximum
// raised by every unit that exceeds it / now: 16 requests of 256 tokens on 2 048 keys BF16 224 / 199, TQ4 261 / 247, 4 of 700 on 6 000 BF16 507 / 459,
// TQ4 634 / 618, 8 of 2 048 on 16 384 TQ4 6 261 / 6 185.
constexpr float kPfSlack = 8.0f, kPfSlackScale = 255.0f;
constexpr uint32_t kSlackScaleBits = 0x5BF8u;  // kPfSlackScale in fp16

struct AttnParams {
    warp34_kv_layer_layout L;
    warp34_attention_batch B;
    const uint16_t* q;
    uint16_t* out;
    float* part_acc;  // [rows][max_chunks][256] or null
    float* part_ml;   // [rows][max_chunks][4]: m, l, chunk count, unused
    int num_q_heads;
    int gqa;          // q heads per kv head
    int q_group;      // q heads of one kv head handled by one workgroup (<= 16)
    int q_subgroups;  // gqa / q_group
    int tok_tile;     // query tokens per tile
    int max_chunks;   // cap on chunks per tile (1 = no split, scratch untouched)
    union {  // (in the place of one: as a word further on, 0.1 us of a 12.5 us call)
        int min_upc;      // balanced decode: minimum units per piece
        int few_chunks;   // chunk grid: chunk_count's line (few_chunks_of)
    };
    int tiles_by_request;  // 1: blockIdx.z is a request (no request has more than one tile)
    int rot_q;             // K rows are stored rotated (WHT-256 transform): rotate the query rows
    int rot_out;           // V rows are stored rotated: rotate the output back
    int32_t* bal_table;    // balanced decode: per query token {first partial slot, pieces, token of the tile, columns (0: bal_cols)}
    int bal_tiles;         // tiles per request (a bound); balanced decode: the plan's entries are request x tile
    union {
        int bal_aligned;    // balanced decode: no piece boundary inside a workgroup's share (few entries)
        int first_round;    // row formats, chunk grid: see rows_first_round
    };
    int piece_cost;        // balanced decode: what starting a piece costs, in units
    union {
        int bal_cols;      // balanced decode: columns of a partial slot, 16 x column tiles of the kernel
        int key_groups;    // row formats, chunk grid: see rows_key_groups
    };
    uint32_t block_magic;  // floor(2^32 / block_size), see div_block
    uint32_t q_group_magic;  // see div_q_group
    const uint16_t* gate;  // fp16 [tokens, q heads, 256] or null: out = fp16(out) * sigmoid(gate)
    union {  // (a longer argument block costs every kernel's start: 12 bytes more, a bf16 decode step 0.2 us of 20)
        // chunk geometry of a tile whose keys are exactly [0, max_seq_len): worked out on the host, so a
        // request that is as long as the host's bound needs no division on the device
        struct {
            int spec_units, spec_upc, spec_chunks;
        };
        // balanced verify: a batch of up to short_units units runs as tiles of 16 columns (bal_short_piece); -1: none does
        struct {
            int short_units, short_tiles, short_tok_tile;
        };
    };
    // Partial records: part_stride slots per output row.  Slots [0, max_chunks) belong to the
    // split-K chunks of the decode kernels; a shared-prefix pass (tile kernel over the keys every
    // request of the batch has in common) owns slots [pf_slot_base, pf_slot_base + pf_split), and
    // the decode kernel then starts at key *key_floor.
    int part_stride;
    int pf_split, pf_slot_base;
    const int32_t* key_floor;
    // TQ4 decode kernels: a 32-token unit never straddles two pages (the page size is a multiple of
    // 32) and both page strides fit 32 bits, so a unit's four runs follow from ONE block-table entry
    // and two 32 x 32-bit products
    int unit_in_page;
    // Balanced decode: the chunk grid's cap on chunks per request, for batches it may serve (grid_decode_serves); 0: none.  (A word of its own: a
    // launch may take a kernel that reads short_units.)
    int grid_chunks;
};

// A finished output row leaves the kernels here: lane l holds channels 4 l .. 4 l + 3.  With a gate
// (the gated full-attention layers, model/forward.rs:1192-1211) the stored value is the attention
// output rounded to its 16-bit type and then passed through the gate operator's arithmetic
// (ops/op_norms_rope_act.cu:742-759), so it has the bits of the two calls in sequence.
// HD: the head dimension (lanes beyond a 128-element row store nothing).
// gate_values: the row's, loaded here or asked for ahead (load_out_gate) by a kernel that waits for something else anyway.
template <typename TQ, int HD, typename GateFn>
__device__ __forceinline__ void store_out_row_by(const AttnParams& P, size_t row, int lane, const float (&o)[4], GateFn&& gate_values) {
    if (HD < 256 && 4 * lane >= HD) return;
    uint16_t h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) h[k] = TQ::from_f32(o[k]);
    if (P.gate != nullptr) {
        const uint2 g = gate_values();
        const uint16_t gb[4] = {(uint16_t)g.x, (uint16_t)(g.x >> 16), (uint16_t)g.y, (uint16_t)(g.y >> 16)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            h[k] = TQ::from_f32(gate_product(TQ::to_f32(h[k]), F16::to_f32(gb[k])));
        }
    }
    uint2 ob;
    ob.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    ob.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
    *reinterpret_cast<uint2*>(P.out + row * HD + 4 * lane) = ob;
}
template <typename TQ, int HD = kHeadDim>
__device__ __forceinline__ void store_out_row(const AttnParams& P, size_t row, int lane, const float (&o)[4]) {
    store_out_row_by<TQ, HD>(P, row, lane, o, [&] { return *reinterpret_cast<const uint2*>(P.gate + row * HD + 4 * lane); });
}
template <typename TQ, int HD = kHeadDim>
__device__ __forceinline__ void store_out_row(const AttnParams& P, size_t row, int lane, const float (&o)[4], uint2 g) {
    store_out_row_by<TQ, HD>(P, row, lane, o, [&] { return g; });
}
template <int HD = kHeadDim>
__device__ __forceinline__ uint2 load_out_gate(const uint16_t* gate, size_t row, int lane) {
    if (gate == nullptr || (HD < 256 && 4 * lane >= HD)) return uint2{0u, 0u};
    return *reinterpret_cast<const uint2*>(gate + row * HD + 4 * lane);
}


// token of k-slot (s, b, i) inside a unit: spreads the four 4-row groups of an MFMA over LDS
// banks so that neither the K-row reads nor the V-column reads conflict.
__device__ __forceinline__ constexpr int unit_token(int s, int b, int i) {
    return 16 * (b & 1) + 8 * s + 4 * (b >> 1) + i;
}

// chunk geometry of a tile
// a / b for 0 <= a < 2^21 and 0 < b: the float quotient is within one of the exact result,
// one correction step makes it exact.  A runtime integer division costs ~40 dependent
// instructions on this hardware, and the prologue and the per-unit address arithmetic
// divide by block sizes and group sizes that only the descriptors know.
__device__ __forceinline__ int small_div(int a, int b) {  // a < 2^21
    int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b));
    const int r = a - q * b;
    q += r >= b ? 1 : 0;
    q -= r < 0 ? 1 : 0;
    return q;
}
__device__ __forceinline__ int fast_div(int a, int b) { return a >= (1 << 21) ? a / b : small_div(a, b); }

// pos / block_size for 0 <= pos < 2^31 without a branch: the high word of pos * floor(2^32 / b)
// is the quotient or one less, one compare settles it.  The inner loops divide a token position
// by the page size for every group of 16 keys.
__device__ __forceinline__ int div_block(int pos, const AttnParams& P) {
    int q = (int)__umulhi((uint32_t)pos, P.block_magic);
    q += (pos - q * P.L.block_size >= P.L.block_size) ? 1 : 0;
    return q;
}
__host__ inline uint32_t block_magic_for(int block_size) {
    return block_size <= 1 ? 0xFFFFFFFFu : (uint32_t)((1ull << 32) / (uint32_t)block_size);
}

// column / q_group for the columns of a workgroup (at most 128, q_group at most 16): exact with
// ceil(2^16 / q_group), whose excess over 2^16 / q_group adds less than 128 * 16 / 2^16 of a group
__device__ __forceinline__ int div_q_group(int col, const AttnParams& P) {
    return (int)(((uint32_t)col * P.q_group_magic) >> 16);
}
__host__ inline uint32_t q_group_magic_for(int q_group) { return (65536u + (uint32_t)q_group - 1u) / (uint32_t)q_group; }

struct ChunkGeom {
    int u_first, n_units, upc, n_chunks;
};
// Smallest chunk: 256 tokens, one unit per wave.  7 to 12 % faster than 16 at 16K-32K keys, same as 4
constexpr int kMinUnitsPerChunk = 8;
// Split geometry is sized for the layout the path is built for, two kv heads per device: 128
// chunks (or shares) per kv head.  The counts below depend on the batch and on gqa only, never
// on local_kv_heads: a rank that holds one kv head of a sharded model computes every row with
// the same chunks, in the same order, as a rank that holds all of them (bit-identical outputs
// under head sharding, op_paged_attn.cu:1301-1304), at the price of half-filled compute units
// on such a rank.
constexpr int kTargetWorkgroupsPerHead = 128;
// Chunks of n_units units.  Up to `few` chunks (kFewChunks*) they are shorter: four units are one
// for the first wave of every SIMD, which then shares its issue slots with nobody, and one half unit per wave of a row format.
constexpr int kShortChunkUnits = 4;
__host__ __device__ constexpr int chunk_count(int n_units, int few) {
    const int whole = (n_units + kMinUnitsPerChunk - 1) / kMinUnitsPerChunk, quick = (n_units + kShortChunkUnits - 1) / kShortChunkUnits;
    return whole <= 1 || whole >= few ? whole : quick < few ? quick : few;
}
// us a layer step of one request, chunks of eight units / of four (merged by one wave per row on both sides): TQ4, 1 token on 600 keys
// 17.3 / 16.8, on 2 500 17.5 / 17.1, 4 tokens on 5 000 with 40 chunks 21.2 / 21.5; Q8_0 1 200 17.3 / 16.6, 5 000 18.3 / 17.3; FP16 2 500 17.0 / 15.6, 10 000
// with 79 chunks 18.4 / 18.8.
constexpr int kFewChunksTq4 = 24, kFewChunksRows = 32;
// More workgroups than the chip takes in one round cost more than shorter ones give, so all tiles of a kv head together have at most this many shorter
// chunks: 256 workgroups with four kv heads.  (The count must not depend on the kv heads: a rank that holds some of them has the chunks of all.)  us, chunks of
// eight units / of four without a limit / with it: 32 + 4 heads, TQ4 16 tokens on 3 000 keys 17.5 / 27.0 / 16.6, 8 on 6 000 17.7 / 27.2 / 16.9, 4 requests of 750 to 3 000
// 17.2 / 20.5 / 13.6; Q8_0 16 on 3 000 15.9 / 22.8 / 15.1.  What it costs two kv heads: TQ4 8 requests of 375 to 1 500 keys 14.7 / 12.2 / 12.9, Q8_0 14.7 / 11.7 / 12.0,
// BF16 10 of 402 to 1 592 16.4 / 12.7 / 14.1.  Half the limit spares eight kv heads the second round as well (TQ4 4 tokens of 64 + 8 heads on 6 000 keys 17.8 / 27.0 / 27.3,
// with half 17.1), but takes back a third of what one and two kv heads gain where it binds (Q8_0 7 requests of 507 to 1 705, 8 + 1 heads, 14.2 / 11.1 / 11.5, with half 12.8).
constexpr int kShortWorkgroupsPerHead = 64;
static_assert(kTargetWorkgroupsPerHead % kShortWorkgroupsPerHead == 0, "few_chunks_of: target = 128 / tiles");
__host__ __device__ constexpr int few_chunks_of(int few, int target) {
    const int share = target / (kTargetWorkgroupsPerHead / kShortWorkgroupsPerHead);
    return share < few ? share : few;
}
__device__ __forceinline__ ChunkGeom chunk_geom(int u_lo, int u_hi, int max_chunks, int few) {
    ChunkGeom g;
    g.u_first = u_lo >> 5;
    g.n_units = (u_hi >= u_lo) ? ((u_hi >> 5) - g.u_first + 1) : 0;
    int nc = chunk_count(g.n_units, few);
    if (nc > max_chunks) nc = max_chunks;
    if (nc < 1) nc = 1;
    g.upc = fast_div(g.n_units + nc - 1, nc);
    if (g.upc < 1) g.upc = 1;
    g.n_chunks = fast_div(g.n_units + g.upc - 1, g.upc);
    if (g.n_chunks < 1) g.n_chunks = 1;
    return g;
}

// The 256-point WHT of finished rows and queries: 60 instructions a row (128 with an exchange, two sums and a select per value and lane stage).
// A prefill wave rotates 64 rows: 16 requests of 256 tokens on 512 keys 116.6 / 107.7 us, 2 of 250 on 1 000 46.9 / 45.3.
// One lane stage, H = 1, 2 or 8: lanes with bit H clear take v + v[lane ^ H], the others v[lane ^ H] - v.
// SELECT: the same by both results and a choice, twelve instructions more in all and no sign to keep.  For the two-column-tile form of 8-bit rows: with
// the signs it spills 30 to 50 more scalars, also where nothing is rotated.  us a call, signs / choice: Q8_0 5 requests x 4 tokens on 2 000 keys 17.3 / 16.1, 24 tokens
// on 240 keys 14.3 / 13.0, FP8 16.4 / 15.8, 13.5 / 12.7.  The other forms are as fast with the signs or faster (rotated FP8, 8 x 8 tokens on 240 keys 14.4 / 14.8).
template <int H, bool SELECT = false>
__device__ __forceinline__ void wht_stage(float (&v)[4], int lane) {
    const uint32_t flip = (lane & H) ? 0x80000000u : 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float o = lane_xor<H>(v[k], lane);
        if constexpr (SELECT) v[k] = (lane & H) ? o - v[k] : v[k] + o;
        else v[k] = o + __uint_as_float(__float_as_uint(v[k]) ^ flip);
    }
}
// H = 4: the sum in the groups of four lanes with the bit clear, the difference in the others.  (The compiler does not see that the statement
// reads across lanes: the waits stand in it.)
__device__ __forceinline__ void wht_stage4(float (&v)[4]) {
    float r[4];
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %4, %4 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %5, %5 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %2, %6, %6 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %3, %7, %7 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_sub_f32_dpp %0, %4, %4 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %1, %5, %5 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %2, %6, %6 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_sub_f32_dpp %3, %7, %7 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "s_nop 1"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = r[k];
}
// H = 16 or 32, two values at a time: exchanged halves put both sides of a's pairs (and of b's) into the same lane, the sum and the difference
// are the results of both sides, and a second exchange brings them back.
template <int H>
__device__ __forceinline__ void wht_stage_pair(float& a, float& b) {
    const auto swap = [](float x, float y) {
        if constexpr (H == 16) return __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        else return __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    };
    const auto r = swap(a, b);
    const float sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const float diff = __uint_as_float(r[0]) - __uint_as_float(r[1]);
    const auto o = swap(sum, diff);
    a = __uint_as_float(o[0]);
    b = __uint_as_float(o[1]);
}

// 256-point WHT over one wave: element e = 4*lane + k, scaled by 1/16.
template <bool SELECT = false>
__device__ __forceinline__ void wht256_wave(float (&v)[4], int lane) {
    {
        const float a0 = v[0] + v[1], a1 = v[0] - v[1], a2 = v[2] + v[3], a3 = v[2] - v[3];
        v[0] = a0 + a2;
        v[1] = a1 + a3;
        v[2] = a0 - a2;
        v[3] = a1 - a3;
    }
    wht_stage<1, SELECT>(v, lane);
    wht_stage<2, SELECT>(v, lane);
    wht_stage4(v);
    wht_stage<8, SELECT>(v, lane);
    wht_stage_pair<16>(v[0], v[1]);
    wht_stage_pair<16>(v[2], v[3]);
    wht_stage_pair<32>(v[0], v[1]);
    wht_stage_pair<32>(v[2], v[3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] *= 0.0625f;
}

// Entry bits of a code: fp16(kLutGain * centroid), by two byte permutes over immediates (no constant-memory load on the critical path; a chain of selects
// is sixty instructions with branches).  Magnitude k is that of centroids 8 + k and 7 - k.
__host__ __device__ constexpr uint32_t centroid_bits_of(int code) { return __builtin_bit_cast(uint16_t, (_Float16)(kLutGain * kCentroids[code])); }
__host__ __device__ constexpr uint32_t magnitude_bytes(int first, int shift) {  // byte `shift / 8` of four magnitudes
    uint32_t r = 0;
    for (int k = 0; k < 4; ++k) r |= (centroid_bits_of(8 + first + k) >> shift & 0xFFu) << (8 * k);
    return r;
}
__device__ __forceinline__ uint32_t centroid_bits(uint32_t code) {
    constexpr uint32_t lo0 = magnitude_bytes(0, 0), lo4 = magnitude_bytes(4, 0), hi0 = magnitude_bytes(0, 8), hi4 = magnitude_bytes(4, 8);
    const bool negative = (code & 8u) == 0u;
    const uint32_t k = (negative ? ~code : code) & 7u;
    return __builtin_amdgcn_perm(lo4, lo0, k | 0x0c0c0c00u) | __builtin_amdgcn_perm(hi4, hi0, k << 8 | 0x0c0c000cu) | (negative ? 0x8000u : 0u);
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    f2 f = {a, b};
    h2 h = __builtin_convertvector(f, h2);
    return __builtin_bit_cast(uint32_t, h);
}
// Two fp16 operands for one fp32 weight pair: hi = fp16(w), lo = fp16(w - hi).  A value scale
// that is folded into the probabilities (w = p * d) reaches every element of a 128-wide scale
// block through ONE number; rounded to fp16 once, its error is the same for the whole block,
// and the inverse rotation gathers such a block-wide error into a single output channel
// (channel c ^ 128 of a channel c with large values).  With the low-order operand the weight
// carries 22 bits and that error disappears; the price is a second MFMA per value tile.
__device__ __forceinline__ void split_h2(float a, float b, uint32_t& hi, uint32_t& lo) {
    const h2 h = __builtin_convertvector(f2{a, b}, h2);
    hi = __builtin_bit_cast(uint32_t, h);
    // lo = fp16(a - hi.x) | fp16(b - hi.y) << 16: one mixed-precision FMA per half (x * 1 - h with
    // h read as fp16), the same value as widening, subtracting (exact) and rounding
    uint32_t l;
    asm("v_fma_mixlo_f16 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(l) : "v"(a), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(l) : "v"(b), "v"(hi));
    lo = l;
}
// An MFMA may read a register two wait states after a vector instruction has written it.  The compiler
// keeps that distance for its own instructions but does not see through an assembly statement, so
// the low-order operands pass through settle() on their way to the MFMAs.
__device__ __forceinline__ void settle(u2v (&a)[8]) {
    asm("s_nop 1" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]));
}
__device__ __forceinline__ void settle(u4 (&a)[8]) {
    asm("s_nop 1" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]));
}
// The same for the weights of TQ4 rows, where issue and not registers is short: v_fma_mix_f32 and v_cvt_pk_f16_f32 issue every 4 cycles, v_fma_mixlo_f16 /
// mixhi, which do both, every 8.  (Written as fma, the compiler widens the halves with instructions of their own.)
__device__ __forceinline__ void split_weights(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = pack_h2(a, b);
    float r0, r1;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(r0) : "v"(a), "v"(hi));
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r1) : "v"(b), "v"(hi));
    lo = pack_h2(r0, r1);
}
// a * (fp16 half of w) as one mixed-precision FMA that reads the half in place (v_fma_mix_f32 with
// a zero addend; written as an fma so that the compiler forms it and places the wait states that
// separate it from the instruction that produced a).  A product of -0 comes out as +0.
__device__ __forceinline__ float mul_by_half_lo(float a, uint32_t w) {
    return __builtin_fmaf(a, (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu)), 0.0f);
}
__device__ __forceinline__ float mul_by_half_hi(float a, uint32_t w) {
    return __builtin_fmaf(a, (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)), 0.0f);
}
// the larger ones of two pairs of 16-bit numbers
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    typedef uint16_t us2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, a), __builtin_bit_cast(us2, b)));
}
// maximum of three finite values in one instruction (fmaxf would first quiet each operand); the
// operands must come from ordinary vector instructions: the compiler places no wait states in
// front of an assembly statement that reads the result of an MFMA
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float half_lo_to_f32(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu));
}
__device__ __forceinline__ float half_hi_to_f32(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
}
// max / sum over the four 16-lane rows of a wave, result in every lane (pure VALU on gfx950)
__device__ __forceinline__ float max_over_rows(float x) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_over_rows(float x) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Table lookup: the dequantisation table sits at LDS address 0 (it is the start of the dynamic
// LDS block and the kernel has no static LDS), so the v_perm_b32 result IS the address.
typedef __attribute__((address_space(3))) const uint32_t lds_cu32;
typedef __attribute__((address_space(3))) const h8 lds_ch8;
typedef __attribute__((address_space(1))) const u4 global_cu4;
__device__ __forceinline__ uint32_t lut_read(uint32_t code_word, uint32_t lut_lane, uint32_t sel) {
    const uint32_t addr = __builtin_amdgcn_perm(code_word, lut_lane, sel);
    return *reinterpret_cast<lds_cu32*>((uintptr_t)addr);
}

// The pair table, by 512 threads: entry e = (gain*centroid[e & 15], gain*centroid[e >> 4]) as packed fp16, 64 copies of 4 bytes.
// Thread t writes the 16-byte slots t + 512 i (conflict-free), i.e. entries (t >> 4) + 32 i:
// their low code (t >> 4) & 15 is the thread's own, their high code (t >> 8) + 2 i is the
// same in the whole wave, one of two immediates.
__device__ __forceinline__ void build_pair_table(uint8_t* smem, int tid, int wave) {
    const uint32_t lo = centroid_bits((uint32_t)tid >> 4 & 15u);
    const bool odd = (wave >> 2) != 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t v = lo | (odd ? centroid_bits_of(2 * i + 1) << 16 : centroid_bits_of(2 * i) << 16);
        *reinterpret_cast<u4*>(smem + (tid + 512 * i) * 16) = u4{v, v, v, v};
    }
}

// element index (0..255) of nibble i of aligned dword D of a TQ4 row, -1 for scale nibbles
__device__ __forceinline__ constexpr int tq4_dword_elem(int D, int i) {
    if (D == 0) return i >= 4 ? i - 4 : -1;
    if (D < 16) return 8 * D - 4 + i;
    if (D == 16) return i < 4 ? 124 + i : -1;
    return 128 + 8 * (D - 17) + i;
}
// dword read by k-block bk for QK MFMA m (0..3) of half h.  The k-blocks of
// lanes 0-31 (bk 0,1) sit 8 dwords apart, which keeps the 32 simultaneous reads on 32 banks.
// Dword 0 holds four codes behind a scale and dword 16 four in front of one: the two make one operand of eight codes
// (tq4_fuse; a fifth MFMA for dword 16 alone and its four look-ups before).
__device__ __forceinline__ constexpr int tq4_qk_dword(int h, int m, int bk) {
    return (h == 0 ? 0 : 17) + 8 * (bk & 1) + 4 * (bk >> 1) + m;
}
// The code dword of the lanes with first: elements 0..3 and 124..127; the others: dword d as it is.
__device__ __forceinline__ uint32_t tq4_fuse(uint32_t d16, uint32_t d, bool first) {
    return __builtin_amdgcn_alignbit(d16, d, first ? 16u : 0u);
}
// element index of V^T row r, nibble j, half h (PV MFMA output row -> head dimension)
__device__ __forceinline__ constexpr int tq4_pv_elem(int h, int j, int r) {
    if (h == 1) return 128 + 8 * r + j;
    if (r == 0) return j < 4 ? j : 120 + j;
    return 8 * r - 4 + j;
}

// Elements 4 lane .. 4 lane + 3 in the order of the code dwords: twice the dword inside its half-row plus the half of it.  (Lanes 0 and 31, elements 0..3 and
// 124..127, are the halves of the fused dword, see tq4_fuse.)
__device__ __forceinline__ int tq4_half_dword(int lane) { return lane < 32 ? (lane == 0 || lane == 31 ? lane & 1 : lane + 1) : lane - 32; }
// Merge regions: slot of element 4 lane; element 4 lane + k: + 16 k (inverse of tq4_pv_elem).  (Worked out element by element, with a branch for
// each kind of lane, it was 150 instructions in front of the workgroup's barrier.)
__device__ __forceinline__ int tq4_merge_slot(int lane) {
    const int i = tq4_half_dword(lane), r = i >> 1;
    return (((lane >> 5) * 8 + 4 * (i & 1)) * 4 + (r >> 2)) * 4 + (r & 3);
}

constexpr int kMergeGroups = 16;
// Up to this many chunks one wave per row adds them up (split_merge_few_kernel); kMergeFewRows where it stands for four waves, not sixteen
// (merge_small_groups).  us a call, sixteen waves / one: nine to sixteen chunks, one request of 2 000 keys TQ4 11.7 / 11.3, Q8_0 11.2 / 10.8, of 1 000
// 16 tokens BF16 13.0 / 12.4; twenty and more TQ4 3 500 keys 12.4 / 12.6, 8 000 12.8 / 13.2, Q8_0 5 000 12.2 / 12.5, 8 000 13.7 / 14.0.  Four waves / one, 21
// chunks: TQ4 6 requests x 4 tokens on 8 000 keys, 8 + 2 heads, 22.3 / 21.5; of 32 rows the same.
constexpr int kMergeFew = 16, kMergeFewRows = 32;
constexpr int kMergeMaxPerGroup = 16;  // at most 256 partials per row

// ---- balanced decode ----------------------------------------------------------------------------
// A decode or verify batch (no window, no token mask) is cut into equal shares of 32-token units,
// one share per workgroup, whatever the lengths of the requests.  A request with more query tokens
// than a tile holds has several tiles; entry e of the plan is tile e % T of request e / T, T =
// P.bal_tiles (1 for a decode step; tiles a request does not have are entries without units).
// The units of all entries are laid end to end and workgroup x owns units [x S, (x + 1) S).  A share
// that crosses an entry boundary is worked off piece by piece.  Piece (x, e) gets partial slot
// x + e: both grow along the pieces, so the slots are unique and those of one entry are
// consecutive, first_wg(e) + e .. last_wg(e) + e.  The workgroup that owns an entry's first
// piece records {first slot, number of pieces, token of the tile} for each of the tile's
// query tokens in a per-token table for the merge kernel; the tokens of entries without work
// are recorded by workgroup (0, 0): pieces = 0 for a live request without visible keys (output
// zeros), -1 for a masked one and for tokens behind the last request (output untouched).
// Few entries (P.bal_aligned): every entry is cut into equal pieces of its own, no workgroup has two
// pieces.  The start of a piece is a chain of memory round trips and its end a merge of the waves,
// together more than a workgroup's streaming when the batch is small, and the call lasts as long as
// the workgroup that goes through it twice.  With n entries on G workgroups rounding to whole pieces
// costs about n / 2G of the streaming, so for many entries the shares that cross boundaries are
// better.  Slot of a piece: its workgroup.
// Starting a piece (table, query rotation, first loads, merge of the waves) costs about as much
// as P.piece_cost units of streaming, so every entry is charged that many extra units in
// front of its real ones: a share that contains entry boundaries gets fewer keys.
__host__ __device__ __forceinline__ size_t bal_partial_row(int slot, int kv_subs, int kv_sub, int cols, int col) {
    return ((size_t)slot * kv_subs + kv_sub) * cols + col;
}

// A decode batch (kGridDecodeReqs requests at most, one q subgroup) whose longest request is at most this many units is cut as the chunk grid cuts
// it, 128 / requests chunks each at most, and the chunk grid runs instead of the plan where the host's bound on the lengths says as
// much: the plan and the merge's table cost 2 to 3 us of a call.  Under a looser bound the plan runs and cuts the same way.  So a batch must not
// lose by the cut, whatever its lengths are:
// - Up to 16 requests (kAlignedReqs) the plan would cut a long request among short ones into pieces of kMinUnitsPerChunk.  A chunk is no longer
//   than that while the cap does not bind.  us a layer, attention alone, plan's own cut / this cut under the exact bound / under a loose one,
//   one long request and the others of one unit: TQ4 16 of up to 64 units 14.3 / 11.9 / 13.5, 12 of 80 14.3 / 12.0 / 13.7, 12 of 85 (ten chunks of nine
//   units) 14.3 / 14.1 / 15.5, 16 of 128 14.6 / 14.6 / 16.3; Q8_0 16 of 64 13.8 / 12.5 / 13.3, of 128 14.4 / 16.1 / 17.2; BF16 4 of 256 15.4 / 14.1 / 15.3, of
//   512 16.8 / 19.0 / 20.3.  All of the same length: TQ4 16 of 64 15.9 / 13.1 / 14.6, of 128 19.2 / 16.4 / 17.8, BF16 16 of 64 19.7 / 17.7 / 18.9.
// - With more requests the plan's shares cross from one into the next, which costs it 5 us more: `many` units in all.  TQ4 24 of 128, one long
//   23.7 / 18.7 / 20.4, all 26.0 / 21.0 / 22.3, 64 of 48 23.9 / 17.1 / 18.3.  Row formats turn earlier: BF16 33 of 62 22.5 / 18.8 / 20.3, of 77 22.6 / 21.6 / 23.2,
//   48 of 53 22.4 / 22.3 / 23.8; Q8_0 48 of 42 21.1 / 18.1 / 19.2, of 53 21.1 / 20.8 / 22.0.
constexpr int kGridDecodeReqs = 64, kAlignedReqs = 16;
constexpr int kGridUnitsTq4 = 3072, kGridUnitsRows = 2048;  // many
__host__ __device__ constexpr bool grid_decode_serves(long long longest, int reqs, int chunks, int many) {
    return reqs <= kAlignedReqs ? longest <= (long long)kMinUnitsPerChunk * chunks : longest * reqs <= many;
}

struct BalReq {  // entry base + lane of a group of 64
    int lo, hi;          // query tokens of the request
    int t_lo, t_hi;      // query tokens of the tile
    int sa, cb, units;
    int cost;  // units + P.piece_cost, 0 for an entry without work
    int live;  // has query tokens and is not masked
};
__device__ __forceinline__ BalReq bal_load_req(const AttnParams& P, int tiles, int tok_tile, int e) {
    const warp34_attention_batch& B = P.B;
    BalReq q{0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int r = tiles == 1 ? e : small_div(e, tiles);
    if (r >= B.num_reqs) return q;
    q.lo = B.query_start_loc[r];
    q.hi = B.query_start_loc[r + 1];
    q.sa = B.seq_lens_after[r];
    const int q_len = q.hi - q.lo;
    q.cb = B.context_lens_before != nullptr ? B.context_lens_before[r] : q.sa - q_len;
    const int first = (e - r * tiles) * tok_tile;  // the tile's first token inside the request
    q.t_lo = min(q.lo + first, max(q.lo, q.hi));
    q.t_hi = min(q.lo + first + tok_tile, max(q.lo, q.hi));
    const bool live = q.t_hi > q.t_lo && (B.valid_req_mask == nullptr || B.valid_req_mask[r] != 0);
    int last = (B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW) ? q.sa - 1 : q.cb + (q.t_hi - q.lo) - 1;
    if (last >= q.sa) last = q.sa - 1;
    q.units = (live && last >= 0) ? (last >> 5) + 1 : 0;
    q.cost = q.units > 0 ? q.units + P.piece_cost : 0;
    q.live = live ? 1 : 0;
    return q;
}
// inclusive prefix sum over the wave: four row shifts, then the totals of the rows before (DPP moves;
// lanes without a source add 0)
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
    return v;
}
// minimum over the wave, in lane 63
__device__ __forceinline__ int wave_min_last(int v) {
    constexpr int kNone = 0x7fffffff;
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x111, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x112, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x114, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x118, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x142, 0xA, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(kNone, v, 0x143, 0xC, 0xF, false));
    return v;
}
// units per share for a batch of `total` units over `groups` workgroups
__device__ __forceinline__ int bal_share(int total, int groups, int min_share) {
    const int s = fast_div(total + groups - 1, groups);
    return s < min_share ? min_share : s;
}

// One piece of work of the balanced decode kernel: units [u_begin, u_end) of tile `tile` of request
// `req`, the piece number `slot` (partials of a tile occupy consecutive slots) and the number of
// pieces the tile is cut into.
struct BalItem {
    int req, tile, tok_tile, rq_start, rq_end, seq_after, ctx_before;
    int u_begin, u_end, n_chunks, slot;
};

// Tile lookup shared by the kernels that do not split it around other work (see the TQ4
// decode kernel for the scheme): blockIdx.z counts tiles; request z when no request can have
// two tiles, a prefix sum over the requests' tile counts otherwise.
struct TileInfo {
    bool hit;
    int req, rq_start, rq_end, seq_after, ctx_before, tile_in_req;
};
// what the lookup reads of request base + lane
struct TileReq {
    int lo, hi, sa, cb, rm;
};
// PLAIN: the batch has context_lens_before and no request mask
template <bool PLAIN = false>
__device__ __forceinline__ TileReq load_tile_req(const AttnParams& P, int base, int lane) {
    const warp34_attention_batch& B = P.B;
    const int r = base + lane;
    const bool inb = r < B.num_reqs;
    TileReq q;
    q.lo = inb ? B.query_start_loc[r] : 0;
    q.hi = inb ? B.query_start_loc[r + 1] : 0;
    q.sa = inb ? B.seq_lens_after[r] : 0;
    q.cb = (inb && (PLAIN || B.context_lens_before != nullptr)) ? B.context_lens_before[r] : 0;
    q.rm = (inb && !PLAIN && B.valid_req_mask != nullptr) ? (int)B.valid_req_mask[r] : 1;
    return q;
}
// Tile tile_z by the requests' tile counts; q: the first 64 requests (load_tile_req), which a kernel with other work to do meanwhile
// asks for ahead.  The sum over the lanes by DPP moves; by LDS permutes, with the requests asked for here: us a call, 4 tokens each,
// Q8_0 1 request on 16 000 keys 18.8 -> 18.3, TQ4 20.0 -> 19.5, 1 on 1 000 16.6 -> 16.2.
template <bool PLAIN = false>
__device__ __forceinline__ TileInfo locate_tile_of(const AttnParams& P, int tile_z, int lane, TileReq q) {
    const warp34_attention_batch& B = P.B;
    TileInfo t{false, -1, 0, 0, 0, 0, 0};
    int tiles_before = 0;
    for (int base = 0; base < B.num_reqs; base += 64) {
        if (base > 0) q = load_tile_req<PLAIN>(P, base, lane);
        const int cnt = q.hi > q.lo ? fast_div(q.hi - q.lo + P.tok_tile - 1, P.tok_tile) : 0;
        const int incl = wave_incl_scan(cnt);
        const int first = tiles_before + incl - cnt;
        const unsigned long long hits = __ballot(cnt > 0 && tile_z >= first && tile_z < first + cnt);
        if (hits != 0ull) {
            const int src = __builtin_ctzll(hits);
            t.req = base + src;
            t.rq_start = __builtin_amdgcn_readlane(q.lo, src);
            t.rq_end = __builtin_amdgcn_readlane(q.hi, src);
            t.seq_after = __builtin_amdgcn_readlane(q.sa, src);
            t.ctx_before = PLAIN || B.context_lens_before != nullptr ? __builtin_amdgcn_readlane(q.cb, src)
                                                                     : t.seq_after - (t.rq_end - t.rq_start);
            t.tile_in_req = tile_z - __builtin_amdgcn_readlane(first, src);
            t.hit = __builtin_amdgcn_readlane(q.rm, src) != 0;
            return t;
        }
        tiles_before += __builtin_amdgcn_readlane(incl, 63);
    }
    return t;
}
__device__ __forceinline__ TileInfo locate_tile(const AttnParams& P, int tile_z, int lane) {
    const warp34_attention_batch& B = P.B;
    if (P.tiles_by_request) {
        TileInfo t{false, -1, 0, 0, 0, 0, 0};
        t.req = tile_z;
        const int lo = B.query_start_loc[tile_z];
        const int hi = B.query_start_loc[tile_z + 1];
        const int sa = B.seq_lens_after[tile_z];
        const int cb = B.context_lens_before != nullptr ? B.context_lens_before[tile_z] : 0;
        const int rm = B.valid_req_mask != nullptr ? (int)B.valid_req_mask[tile_z] : 1;
        t.rq_start = __builtin_amdgcn_readfirstlane(lo);
        t.rq_end = __builtin_amdgcn_readfirstlane(hi);
        t.seq_after = __builtin_amdgcn_readfirstlane(sa);
        t.ctx_before = B.context_lens_before != nullptr ? __builtin_amdgcn_readfirstlane(cb)
                                                        : t.seq_after - (t.rq_end - t.rq_start);
        t.hit = __builtin_amdgcn_readfirstlane(rm) != 0 && t.rq_end > t.rq_start;
        return t;
    }
    return locate_tile_of(P, tile_z, lane, load_tile_req(P, 0, lane));
}

// LDS-direct loads (gfx950): each active lane's 16 bytes go from global memory straight to LDS at
// m0 + OFFSET + lane * 16, without passing through registers; the immediate OFFSET is added to
// the global address as well.  Written as assembly so that
// the compiler does not know the instruction writes LDS: it would otherwise make every later
// table read (absolute addresses it cannot tell apart from the staging area) wait for the load
// unit.  The waits are placed by hand (wait_vm): loads return in order, so "all but the N most
// recent" is a safe condition whatever other loads the compiler has in flight.
// STREAM: the load carries the non-temporal hint (decode batches: every key is read by exactly one
// workgroup; a plain streaming read of HBM gains 8 to 13 % from the hint, the 32-sequence batch 2 %).
// One 16-row run (2112 bytes = 132 pieces of 16 bytes) is moved by three such instructions of 44
// lanes each, with M0 written once.
template <bool STREAM>
__device__ __forceinline__ void lds_load_run(uint32_t voffset, const uint8_t* sbase, uint32_t lds_addr) {
    if constexpr (STREAM) {
        asm volatile(
            "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:0 nt\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:704 nt\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:1408 nt"
            :
            : "v"(voffset), "s"(sbase), "s"(lds_addr)
            : "memory");
    } else {
        asm volatile(
            "s_mov_b32 m0, %2\n\ts_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:0\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:704\n\t"
            "global_load_lds_dwordx4 %0, %1 offset:1408"
            :
            : "v"(voffset), "s"(sbase), "s"(lds_addr)
            : "memory");
    }
}
// value of the lane eight places on inside the row of 16 lanes (DPP row_ror:8)
__device__ __forceinline__ float row_ror8(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true));
}
// lane L of every row of 16 lanes, in all lanes of that row (one VALU move)
template <int L>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + L, 0xF, 0xF, true);  // row_newbcast:L
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

// Packed tile: columns n and n + 8 += each other (the high-order and the low-order share of the weights), in both lanes.  (The empty statement keeps the
// sums here: moved behind a branch they would be an exchange and a sum.)
__device__ __forceinline__ void add_mirror_columns(f4 (&o)[2][8]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float x = o[h][j][k];
                x += row_ror8(x);
                asm volatile("" : "+v"(x));
                o[h][j][k] = x;
            }
}
// ... and a column's values into its merge region: lane n < 8 the value tiles with even j, lane n + 8 those with odd j.  (The comments in assembly keep
// the branches' stores apart: joined, they take an address inside the array, which then lies in scratch memory.)
__device__ __forceinline__ void store_packed_column(float* c, const f4 (&o)[2][8], int n, int b) {
    if (n < 8) {
#pragma unroll
        for (int t = 0; t < 16; t += 2) *reinterpret_cast<f4*>(c + (t * 4 + b) * 4) = o[t >> 3][t & 7];
        asm volatile("; even tiles");
    } else {
#pragma unroll
        for (int t = 1; t < 16; t += 2) *reinterpret_cast<f4*>(c + (t * 4 + b) * 4) = o[t >> 3][t & 7];
        asm volatile("; odd tiles");
    }
}

// The work of one workgroup on one tile.  BAL = false: the tile and the chunk come from
// blockIdx (grid = chunks x (kv head, q subgroup) x tiles).  BAL = true: they come from `item`
// (balanced decode: every workgroup owns an equal share of the batch's units).
//
// LDS: [pair table 64 KB][kTq4Waves staging areas of 8448 B][query operand table 9216 B][(m, l) tables].
// A staging area holds one 32-token unit as it lies in the pages, written by LDS-direct loads:
// K rows 0-31, then V rows 0-31, 132 bytes each (four runs of 16 rows = 2112 bytes).
// SP: the keys below `item.u_begin` belong to a shared-prefix pass (*P.key_floor, see AttnParams), tile and chunk are `item.req` and `item.slot`; a
// separate instantiation, so that the plain form carries no trace of it.
// NT: column tiles of 16 (two: batches with neither a token mask nor a window).
// PLAIN: split-K form of a batch whose requests have one tile of at most eight columns each, all q heads of a kv head in it, without masks and window, page
// strides below 4 GiB (plain_decode): what follows from the host's bounds on it is worked out while the lengths travel.
template <typename TQ, bool BAL, bool SP = false, bool STREAM = BAL, int NT = 1, bool PLAIN = false>
__device__ __forceinline__ void tq4_tile(const AttnParams& P, uint8_t* smem, const BalItem& item, bool build_table) {
    static_assert(!(SP && BAL), "shared-prefix pass: split-K form only");
    constexpr int kWaves = kTq4Waves;
    uint8_t* stage_all = smem + kLutBytes;

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;  // MFMA column = query row of this lane; also A-operand row
    const int b = lane >> 4;  // MFMA k-block / output row group
    const warp34_kv_layer_layout& L = P.L;
    const warp34_attention_batch& B = P.B;

    // ---- tile identification ---------------------------------------------------------------------
    // blockIdx.z counts TILES (groups of tok_tile consecutive query tokens of one request), so
    // every workgroup that is launched has work.  When no request can have more than one tile
    // (max_q_len <= tok_tile, e.g. decode) tile z is request z; otherwise the tile is located
    // with a prefix sum over the requests' tile counts.
    const int tile_z = BAL || SP ? item.req : (int)blockIdx.z;
    const int kv_sub = (int)blockIdx.y;
    const int kv_head = PLAIN ? kv_sub : small_div(kv_sub, P.q_subgroups);
    const int q_head_base = PLAIN ? kv_sub * P.q_group : kv_head * P.gqa + (kv_sub - kv_head * P.q_subgroups) * P.q_group;
    const int chunk = BAL ? 0 : SP ? item.slot : (int)blockIdx.x;

    // The request lookup goes first: its loads head the longest dependency chain of the prologue
    // (lengths -> chunk geometry -> page ids -> the first K / V loads).
    bool req_hit = false;
    int req = -1, rq_start = 0, rq_end = 0, seq_after = 0, ctx_before = 0, tile_in_req = 0;
    int spec_slot_base = -1, spec_vec = -1;
    int a_lo = 0, a_hi = 0, a_sa = 0, a_cb = 0, a_rm = 0;
    TileReq a_req;  // several tiles per request: as a_*, of request `lane`
    if constexpr (BAL) {
        req = item.req;
        rq_start = item.rq_start;
        rq_end = item.rq_end;
        seq_after = item.seq_after;
        ctx_before = item.ctx_before;
        tile_in_req = item.tile;
        req_hit = true;
        // the piece's first unit is known: its block-table slice is requested together with the
        // query rows
        spec_slot_base = div_block(item.u_begin * kUnit, P);
        const int slot = spec_slot_base + lane;
        if (slot < B.max_blocks_per_req) spec_vec = B.block_tables[(size_t)req * B.max_blocks_per_req + slot];
    } else {
        // a request by the launch geometry, or the guess that all requests have as many tiles as the longest
        req = PLAIN || P.tiles_by_request ? tile_z : min(fast_div(tile_z, P.bal_tiles), B.num_reqs - 1);
        // Speculative block-table load, in flight together with the request's lengths: it
        // assumes that the request's length is the host's bound max_seq_len.  When the guess is
        // wrong the ids are fetched again below, so it changes the latency only, never the result.
        if (PLAIN || (!SP && B.sliding_window <= 0 && B.max_seq_len > 0)) {
            spec_slot_base = div_block(chunk * P.spec_upc * kUnit, P);
            const int slot = spec_slot_base + lane;
            if (slot < B.max_blocks_per_req)
                spec_vec = B.block_tables[(size_t)req * B.max_blocks_per_req + slot];
        }
        // By requests: the same address in all lanes, so scalar loads, one per array and all on their way together with the block-table slice (in the
        // row formats vector loads took 2 to 4 % longer).  By tiles: one request per lane.
        if constexpr (PLAIN) {
            a_lo = B.query_start_loc[req];
            a_hi = B.query_start_loc[req + 1];
            a_sa = B.seq_lens_after[req];
            a_cb = B.context_lens_before[req];
            a_rm = 1;
        } else if (P.tiles_by_request) {
            a_lo = B.query_start_loc[req];
            a_hi = B.query_start_loc[req + 1];
            a_sa = B.seq_lens_after[req];
            a_cb = B.context_lens_before != nullptr ? B.context_lens_before[req] : 0;
            a_rm = B.valid_req_mask != nullptr ? (int)B.valid_req_mask[req] : 1;
        } else {
            a_req = load_tile_req(P, 0, lane);
        }
    }
    // While the request's lengths are on their way: the raw query rows of this wave's columns and
    // the table.  The first token of the tile is guessed (exact when every request has a whole
    // number of tiles); a wrong guess is corrected after the lookup.
    const int tok_guess = BAL ? item.rq_start + item.tile * P.tok_tile
                              : min(PLAIN || P.tiles_by_request ? tile_z : tile_z * P.tok_tile, B.total_tokens - 1);
    constexpr int kColsPerWave = (16 * NT + kWaves - 1) / kWaves;
    uint2 q_raw[kColsPerWave];
    auto load_q = [&](int tokbase) {
#pragma unroll
        for (int c = 0; c < (PLAIN ? 1 : kColsPerWave); ++c) {
            const int col = wave + c * kWaves;
            const int t = div_q_group(col, P);
            const int a = col - t * P.q_group;
            q_raw[c] = uint2{0u, 0u};
            if (col < 16 * NT && tokbase + t < B.total_tokens) {
                const uint16_t* qrow =
                    P.q + ((size_t)(tokbase + t) * P.num_q_heads + (size_t)(q_head_base + a)) * kHeadDim;
                q_raw[c] = *reinterpret_cast<const uint2*>(qrow + 4 * lane);
            }
        }
    };
    load_q(tok_guess);
    // validity of the token of this lane's column
    bool tok_ok = false;
    auto load_tok_ok_col = [&](int tokbase, int column) {
        const int tok = tokbase + div_q_group(column, P);
        tok_ok = tok < B.total_tokens &&
                 (PLAIN || B.valid_token_mask == nullptr || B.valid_token_mask[min(tok, B.total_tokens - 1)] != 0);
    };
    auto load_tok_ok = [&](int tokbase) {
        if constexpr (NT == 1) load_tok_ok_col(tokbase, n);
    };
    load_tok_ok(tok_guess);

    if (build_table) {
        static_assert(kWaves == 8, "table build: 512 threads");
        build_pair_table(smem, tid, wave);
    }

    // PLAIN: the first unit of this wave if the request is as long as the host's bound, its runs' places in the pages and the slabs
    const int simd = wave & 3, wslot = wave >> 2;
    uint32_t spec_in_page[2] = {0u, 0u};
    int spec_rel[2] = {0, 0};
    uint64_t k_slab = 0, v_slab = 0;
    if constexpr (PLAIN) {
        k_slab = L.k_base + (uint64_t)(uint32_t)kv_head * L.k_head_stride_bytes;
        v_slab = L.v_base + (uint64_t)(uint32_t)kv_head * L.v_head_stride_bytes;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int pos = (chunk * P.spec_upc + 4 * wslot + simd) * kUnit + 16 * r;
            const int slot = div_block(pos, P);
            spec_rel[r] = slot - spec_slot_base;
            spec_in_page[r] = (uint32_t)(pos - slot * L.block_size) * (uint32_t)kTq4RowBytes;
            asm volatile("" : "+s"(spec_rel[r]), "+s"(spec_in_page[r]));
        }
        asm volatile("" : "+s"(k_slab), "+s"(v_slab));
    }
    if (!BAL && (PLAIN || P.tiles_by_request)) {
        rq_start = __builtin_amdgcn_readfirstlane(a_lo);
        rq_end = __builtin_amdgcn_readfirstlane(a_hi);
        seq_after = __builtin_amdgcn_readfirstlane(a_sa);
        ctx_before = PLAIN || B.context_lens_before != nullptr ? __builtin_amdgcn_readfirstlane(a_cb)
                                                               : seq_after - (rq_end - rq_start);
        req_hit = __builtin_amdgcn_readfirstlane(a_rm) != 0 && rq_end > rq_start;
    }
    if (!BAL && !PLAIN && !P.tiles_by_request) {
        const TileInfo ti = locate_tile_of(P, tile_z, lane, a_req);
        if (ti.req != req) spec_slot_base = -1;
        req = ti.req;
        rq_start = ti.rq_start;
        rq_end = ti.rq_end;
        seq_after = ti.seq_after;
        ctx_before = ti.ctx_before;
        tile_in_req = ti.tile_in_req;
        req_hit = ti.hit;
    }
    if (!req_hit) return;  // no such tile, empty or masked request: outputs untouched
    const int tok0 = rq_start + tile_in_req * P.tok_tile;
    if (tok0 != tok_guess) {  // wave-uniform, rare
        load_q(tok0);
        load_tok_ok(tok0);
    }

    int tile_tokens = rq_end - tok0;
    if (tile_tokens > P.tok_tile) tile_tokens = P.tok_tile;

    // A tile with at most eight columns (a decode step of up to eight query heads per kv head) runs
    // "packed": columns 8-15 repeat columns 0-7 -- same query, same scores, same probabilities -- and
    // carry the LOW-order fp16 part of the value weights where columns 0-7 carry the high-order
    // part, so one MFMA per value tile does the work of two.  The two halves are added up before
    // the waves merge.
    const bool pack = PLAIN || (NT == 1 && tile_tokens * P.q_group <= 8);  // wave-uniform
    const int ncol = pack ? (n & 7) : n;             // the query column this lane works for
    if (pack && ncol != n) load_tok_ok_col(tok0, ncol);

    // Column info: per lane (= per query column) the visible key range, and for the tile the union
    // and the intersection of the ranges.  Without a token mask and a window -- the common case --
    // the tile-wide values follow from scalars (every token of the tile is live, the ranges start
    // at 0 and their ends grow with the token: the union is the last token's range, the
    // intersection the first one's), and the per-lane part waits until the first loads are out.
    int col_lo = 0, col_hi = -1;
    bool col_ok = false;
    int col_hi2 = -1;  // (two column tiles) of column 16 + n
    bool col_ok2 = false;
    int u_lo = 0x7fffffff, u_hi = -1;  // union of the visible ranges
    int i_lo = 0, i_hi = 0x7fffffff;   // intersection of the visible ranges
    uint32_t ok_mask = 0u;             // bit c: column c is live (wave-uniform)
    const bool simple = PLAIN || NT > 1 || (B.valid_token_mask == nullptr && B.sliding_window <= 0);
    // keys below the floor were handled by the shared-prefix pass (a multiple of the unit size)
    int key_floor = 0;
    if constexpr (SP) key_floor = item.u_begin;
    auto column_info = [&](bool accumulate) {
        if constexpr (NT > 1) {
            auto last = [&](int col, bool& ok) {
                const int t = div_q_group(col, P), tok = tok0 + t;
                ok = t < tile_tokens && tok < B.total_tokens;
                const int mx = B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW ? seq_after - 1 : ctx_before + tok - rq_start;
                return ok ? min(mx, seq_after - 1) : -1;
            };
            col_lo = key_floor;
            col_hi = last(n, col_ok);
            col_hi2 = last(16 + n, col_ok2);
            ok_mask = (uint32_t)(__ballot(col_ok) & 0xFFFFull) | (uint32_t)(__ballot(col_ok2) & 0xFFFFull) << 16;
            return;
        }
        const int t = div_q_group(ncol, P);
        const int tok = tok0 + t;
        const bool ok = t < tile_tokens && tok_ok;
        const int q_off = tok - rq_start;
        int mx = (!PLAIN && B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW) ? seq_after - 1 : ctx_before + q_off;
        if (mx >= seq_after) mx = seq_after - 1;
        int mn = key_floor;
        if (!PLAIN && B.sliding_window > 0) mn = max(key_floor, ctx_before + q_off - B.sliding_window + 1);
        col_ok = ok;
        col_lo = ok ? mn : 0;
        col_hi = ok ? mx : -1;
        if (accumulate && ok) {
            i_lo = max(i_lo, mn);
            i_hi = min(i_hi, mx);
            if (mn <= mx) {
                u_lo = min(u_lo, mn);
                u_hi = max(u_hi, mx);
            }
        }
        ok_mask = (uint32_t)(__ballot(ok) & (pack ? 0xFFull : 0xFFFFull));  // mirror columns produce no output
    };
    if (simple) {
        if (tok0 >= B.total_tokens) return;  // no live column
        const int q_off0 = tok0 - rq_start;
        const bool window = !PLAIN && B.mask_mode == WARP34_ATTN_MASK_NONCAUSAL_WINDOW;
        int hi_first = window ? seq_after - 1 : ctx_before + q_off0;
        int hi_last = window ? seq_after - 1 : ctx_before + q_off0 + tile_tokens - 1;
        if (hi_first >= seq_after) hi_first = seq_after - 1;
        if (hi_last >= seq_after) hi_last = seq_after - 1;
        u_lo = key_floor;
        u_hi = hi_last >= key_floor ? hi_last : -1;
        i_lo = key_floor;
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
        if (ok_mask == 0u) return;  // whole tile masked: outputs untouched
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

    // ---- staging machinery ----------------------------------------------------------------------
    const uint8_t* k_base;
    const uint8_t* v_base;
    if constexpr (PLAIN) {
        k_base = reinterpret_cast<const uint8_t*>((uintptr_t)k_slab);
        v_base = reinterpret_cast<const uint8_t*>((uintptr_t)v_slab);
    } else {
        k_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.k_base) + (size_t)kv_head * L.k_head_stride_bytes;
        v_base = reinterpret_cast<const uint8_t*>((uintptr_t)L.v_base) + (size_t)kv_head * L.v_head_stride_bytes;
    }
    const uint32_t stage_addr = (uint32_t)(kLutBytes + wave * kStageTq4);  // LDS byte address (the block starts at 0)
    uint8_t* stage = stage_all + wave * kStageTq4;

    // The physical page ids come from ONE vector load per 64 block-table slots: lane l holds
    // the id of slot slot_base + l, a unit picks its two ids with readlane.  No scalar memory
    // loads remain in the loop (they share the LDS wait counter and would serialise it).
    const int32_t* req_blocks = B.block_tables + (size_t)req * B.max_blocks_per_req;
    int slot_base = div_block(cu_first * kUnit, P);
    int page_vec;
    // (Loaded and waited for in one assembly statement: were the load the compiler's, it would place
    // a vmcnt(0) in front of every readlane of page_vec -- once per unit -- and that wait, which
    // cannot tell the compiler's loads from the LDS-direct ones, would make every unit wait for all
    // the K / V data in flight.  The reload happens once per 64 block-table slots.)
    auto load_page_vec = [&]() {
        const int slot = slot_base + lane;
        int32_t ids = -1;
        if (slot < B.max_blocks_per_req) {
            const int32_t* src = req_blocks + slot;
            asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=v"(ids) : "v"(src) : "memory");
        }
        page_vec = ids;
    };
    // Runs that do not overlap the visible key range, or whose block-table entry is missing,
    // are read from page 0 of the slab instead: every row they deliver is masked, and any
    // TQ4 bytes dequantise to finite values.
    const uint8_t* nk[2];  // run bases of the unit that is loaded next (wave-uniform)
    const uint8_t* nv[2];
    auto locate_unit = [&](int unit) {
        if (P.unit_in_page) {  // uniform for the launch
            const int pos = unit * kUnit;
            const int page_slot = div_block(pos, P);
            const int in_page = pos - page_slot * L.block_size;
            int rel = page_slot - slot_base;
            if (rel >= 64) {  // wave-uniform, at most once per 64 slots
                slot_base = page_slot;
                load_page_vec();
                rel = 0;
            }
            const int32_t pg = __builtin_amdgcn_readlane(page_vec, rel);
            // (the unit overlaps the visible key range, so its page holds a visible key and its
            // block-table entry is a real page; rows of the unit outside the range are masked)
            const bool live = pg >= 0;
            const uint64_t tok_off = (uint64_t)((uint32_t)in_page * (uint32_t)kTq4RowBytes);
            const uint64_t koff = live ? (uint64_t)(uint32_t)pg * (uint32_t)L.k_page_stride_bytes + tok_off : 0;
            const uint64_t voff = live ? (uint64_t)(uint32_t)pg * (uint32_t)L.v_page_stride_bytes + tok_off : 0;
            nk[0] = k_base + koff;
            nk[1] = nk[0] + kRunBytes;
            nv[0] = v_base + voff;
            nv[1] = nv[0] + kRunBytes;
            return;
        }
#pragma unroll
        for (int gidx = 0; gidx < 2; ++gidx) {
            const int pos = unit * kUnit + 16 * gidx;
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
                const uint64_t tok_off = (uint64_t)((uint32_t)in_page * (uint32_t)kTq4RowBytes);
                nk[gidx] = k_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.k_page_stride_bytes + tok_off : 0);
                nv[gidx] = v_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.v_page_stride_bytes + tok_off : 0);
                continue;
            }
            const size_t koff = live ? (size_t)pg * L.k_page_stride_bytes + (size_t)in_page * L.k_token_stride_bytes : 0;
            const size_t voff = live ? (size_t)pg * L.v_page_stride_bytes + (size_t)in_page * L.v_token_stride_bytes : 0;
            nk[gidx] = k_base + koff;
            nv[gidx] = v_base + voff;
        }
    };
    // six load instructions per half unit: a 16-row run is 2112 bytes = 132 pieces of 16 bytes, moved
    // by three instructions of 44 lanes each (the instruction's immediate offset moves the global
    // AND the LDS address, so the rows arrive contiguous, as they lie in the page)
    const uint32_t lane16 = (uint32_t)lane * 16u;
    auto issue_k = [&]() {
        if (lane < 44) {
#pragma unroll
            for (int r = 0; r < 2; ++r) lds_load_run<STREAM>(lane16, nk[r], stage_addr + r * kRunBytes);
        }
    };
    auto issue_v = [&]() {
        if (lane < 44) {
#pragma unroll
            for (int r = 0; r < 2; ++r) lds_load_run<STREAM>(lane16, nv[r], stage_addr + (2 + r) * kRunBytes);
        }
    };
    constexpr int kLoadsPerHalf = 6;

    // Units are dealt to the waves by a fixed rule, never handed out dynamically: which wave
    // sums which keys decides the floating-point result, and the output has to be the same bits
    // on every run and under every page permutation.  The rule deals the units to the four
    // SIMDs in turn and, inside a SIMD, to its waves in turn (wave w runs on SIMD w mod 4): with
    // a wave count that is not a multiple of four the SIMDs still get equal shares.
    const int simd_waves = (kWaves - simd + 3) / 4;
    auto nth_unit = [&](int j) -> int { return cu_first + 4 * (wslot + simd_waves * j) + simd; };

    // first unit's K half goes in flight before the rest of the prologue
    int unit = nth_unit(0);
    if (slot_base == spec_slot_base) {
        page_vec = spec_vec;
    } else {
        load_page_vec();
    }
    // The raw query rows are consumed after the first K / V loads have gone out.  Loads return in
    // order, so a wait for them placed behind those loads would wait for the K / V data as well:
    // the (empty) statement makes the compiler finish its own loads here, where they have long landed.
#pragma unroll
    for (int c = 0; c < (PLAIN ? 1 : kColsPerWave); ++c) asm volatile("" ::"v"(q_raw[c].x), "v"(q_raw[c].y));
    if (unit < cu_end) {
        if (PLAIN && as_guessed) {  // (spec_rel < 64: the first eight units of a chunk, 256 tokens of pages of 16 and more)
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int32_t pg = __builtin_amdgcn_readlane(page_vec, spec_rel[r]);
                const bool live = unit * kUnit + 16 * r <= u_hi && pg >= 0;
                nk[r] = k_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.k_page_stride_bytes + spec_in_page[r] : 0);
                nv[r] = v_base + (live ? (uint64_t)(uint32_t)pg * (uint32_t)L.v_page_stride_bytes + spec_in_page[r] : 0);
            }
        } else {
            locate_unit(unit);
        }
        issue_k();  // (its V half follows below, behind the query operands)
    }
    if (simple) column_info(false);

    // ---- prologue: the query operand table ---------------------------------------------------------
    // B operands of the QK MFMAs, eight per lane (four for either half-row), in the order the loop reads
    // them: slot (n, b) holds 8 x 16 bytes.  Operand (h, m) of k-block b pairs with row dword D =
    // tq4_qk_dword(h, m, b); its eight elements (tq4_dword_elem) are contiguous in the query row: dword
    // D < 16 covers elements 8 D - 4 .. 8 D + 3 (D = 0: 0 .. 3 and 124 .. 127, see tq4_fuse), dword
    // 17 + k elements 128 + 8 k .. 128 + 8 k + 7.  A lane of the rotating wave holds elements
    // 4 lane .. 4 lane + 3 of its column, i.e. one half of one operand, and writes it there.
    // All the constant factors of the scores (softmax scale, log2 e, 1 / table gain) go into Q'.
    uint8_t* qop = stage_all + kWaves * kStageTq4;
    const float q_scale = B.sm_scale * kLog2e * kLutInvGain;
    // where this lane's four elements go: operand (k-block, mf) and which half of it
    int q_kb, q_mf, q_half;
    {
        const int i = tq4_half_dword(lane);
        const int Dh = i >> 1, grp = Dh >> 2;                               // dword inside its half-row, 4-dword group
        q_kb = grp == 1 ? 2 : grp == 2 ? 1 : grp;                           // groups 1 and 2 swapped
        q_mf = (Dh & 3) + (lane < 32 ? 0 : 4);
        q_half = i & 1;
    }
    static_assert(kColsPerWave == 2 * NT && kWaves == 8, "a packed tile's mirror column col + 8 belongs to the wave of col");
    uint2 packed_prev = {0u, 0u};
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c) {
        const int col = wave + c * kWaves;
        if (col < 16 * NT) {  // wave-uniform
            float q_rot[4];
            q_rot[0] = TQ::to_f32((uint16_t)(q_raw[c].x & 0xFFFFu));
            q_rot[1] = TQ::to_f32((uint16_t)(q_raw[c].x >> 16));
            q_rot[2] = TQ::to_f32((uint16_t)(q_raw[c].y & 0xFFFFu));
            q_rot[3] = TQ::to_f32((uint16_t)(q_raw[c].y >> 16));
            const bool okc = (ok_mask >> col) & 1u;
            uint2 packed = {0u, 0u};
            if (pack && c == 1) {  // mirror column: the operands of column col - 8
                packed = packed_prev;
            } else if (okc) {  // dead columns stay zero: no need to rotate them
                if (P.rot_q) {  // keys stored rotated (uniform for the launch)
#pragma unroll
                    for (int k = 0; k < 4; ++k) q_rot[k] = apply_sign(q_rot[k], 4 * lane + k);
                    wht256_wave(q_rot, lane);
                }
                packed.x = pack_h2(q_rot[0] * q_scale, q_rot[1] * q_scale);
                packed.y = pack_h2(q_rot[2] * q_scale, q_rot[3] * q_scale);
            }
            packed_prev = packed;
            uint8_t* slot0 = qop + (size_t)(col * 4) * 144;
            *reinterpret_cast<uint2*>(slot0 + q_kb * 144 + q_mf * 16 + q_half * 8) = packed;
        }
    }
    // The V half of the first unit is requested only now, about 1 us after its K half.  At one
    // sequence all 2048 waves of the chip start together: asked for at once, the first K and V
    // halves are 17 MB that arrive over 3 us in no useful order; with the V halves held back the
    // K halves are there after half of that, the first scores are computed while the V halves
    // travel, and the call is 0.3 to 0.7 us shorter (three boxes, three rounds each).  The order
    // of the requests -- K then V -- is what the waits in the loop count on, and stays.
    if (unit < cu_end) issue_v();
    __syncthreads();  // the pair table and the query operands are complete

    // ---- per-wave state -----------------------------------------------------------------------
    const uint32_t lut_lane = (uint32_t)lane << 2;  // byte 0 of every table address
    const uint8_t* my_qop = qop + (size_t)(n * 4 + b) * 144;
    const uint32_t qop_lane = (uint32_t)(kLutBytes + kWaves * kStageTq4 + (n * 4 + b) * 144);  // its LDS address
    h8 bq[8];  // the query operands of this lane stay in registers
    if constexpr (NT == 1) {
#pragma unroll
        for (int mf = 0; mf < 8; ++mf) bq[mf] = *reinterpret_cast<const h8*>(my_qop + 16 * mf);
    }

    // Until every live column of the tile has a maximum (`started`) that of a column without one is 0, and so is its sum.  (A unit that it sees need
    // not give it one: with infinite key scales its scores may all be minus infinity.)
    bool started = false, started2 = false;
    f4 o_acc[2][8];
    float m_run = 0.f, l_run = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) o_acc[h][j] = f4{0.f, 0.f, 0.f, 0.f};
    // (two column tiles) the second one's
    f4 o_acc2[2][8];
    float m_run2 = 0.f, l_run2 = 0.f;
    if constexpr (NT > 1) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) o_acc2[h][j] = f4{0.f, 0.f, 0.f, 0.f};
    }

    // rows of the staging area: K rows 0-31, then V rows 0-31, 132 bytes each
    const uint8_t* ka_lo = stage + unit_token(0, n >> 2, n & 3) * kTq4RowBytes;  // A row of sub-tile 0; sub-tile 1: + 8 rows
    const uint8_t* kt_lo = stage + unit_token(0, b, 0) * kTq4RowBytes;           // token of output row 4b; + 8 s + i rows
    const uint8_t* vt_lo = kt_lo + 2 * kRunBytes;
    const uint8_t* kt_n = kt_lo + (n & 3) * kTq4RowBytes;  // the token whose K scales this lane fetches (+ 8 s rows)
    const uint8_t* vt_n = vt_lo + (8 * ((n >> 2) & 1) + (n & 3)) * kTq4RowBytes;  // ... and V scales: token n & 7

    // one 32-token unit.  MASKED = false (wave-uniform) is the interior case: every token of the
    // unit is visible to every live column, so the compares / selects are branched over.
    // HAS_NEXT: the wave has another unit, whose two halves are requested as soon as the raw rows of
    // this unit's halves have been read out of the staging area.
    auto process_unit = [&](int t0, const bool MASKED, const bool HAS_NEXT) {
        // ---- raw K dwords and K scales -------------------------------------------------------------
        wait_vm<kLoadsPerHalf>();  // this unit's K half has landed (its V half may still be in flight)
        uint32_t kw[2][8], ksc[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint32_t* row32 = reinterpret_cast<const uint32_t*>(ka_lo + s * 8 * kTq4RowBytes);
#pragma unroll
            for (int mf = 0; mf < 8; ++mf) kw[s][mf] = row32[tq4_qk_dword(mf >> 2, mf & 3, b)];
            kw[s][0] = tq4_fuse(row32[16], kw[s][0], b == 0);
            // The two scales of token unit_token(s, b, i) in one register, d0 | d1 << 16.  The 16
            // lanes of a row need the same four tokens: lane n reads token n & 3 and the values
            // are handed round inside the row.
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(kt_n + 8 * s * kTq4RowBytes);
            const uint32_t mine = __builtin_amdgcn_perm(r32[16], r32[0], 0x07060100u);
            ksc[s][0] = row_bcast<0>(mine);
            ksc[s][1] = row_bcast<1>(mine);
            ksc[s][2] = row_bcast<2>(mine);
            ksc[s][3] = row_bcast<3>(mine);
        }
        wait_lds_reads();
        if (HAS_NEXT) issue_k();  // nk was located by the caller

        // ---- S^T = K Q'^T for the two 16-key sub-tiles ------------------------------------------
        // Eight batches of two operands (eight table reads, two MFMAs), software-pipelined: the
        // table reads of batch k + 1 are requested before the MFMAs of batch k are issued, so the
        // wave does not sit out the LDS latency of every batch.
        constexpr int kQkOrder[8] = {0, 4, 1, 5, 2, 6, 3, 7};
        // (log2 domain) minus the running maximum: the sum of the scaled partial scores of a token's half rows starts there
        auto score = [](const f4 (&part)[2], int i, uint32_t scales, float m) __attribute__((always_inline)) {
            return __builtin_fmaf(part[1][i], half_hi_to_f32(scales), __builtin_fmaf(part[0][i], half_lo_to_f32(scales), -m));
        };
        constexpr int kQkBatch = 2, kQkBatches = 16 / kQkBatch;
        float sc[8], sc2[8];
        if constexpr (NT == 1) {
        f4 s_acc[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) s_acc[s][0] = s_acc[s][1] = f4{0.f, 0.f, 0.f, 0.f};
        u4 qa[2][kQkBatch];
        auto qk_reads = [&](int bt, u4 (&a)[kQkBatch]) {
#pragma unroll
            for (int k = 0; k < kQkBatch; ++k) {
                const int at = kQkBatch * bt + k;
                const uint32_t w = kw[at >> 3][kQkOrder[at & 7]];
                a[k][0] = lut_read(w, lut_lane, 0x0c0c0400u);
                a[k][1] = lut_read(w, lut_lane, 0x0c0c0500u);
                a[k][2] = lut_read(w, lut_lane, 0x0c0c0600u);
                a[k][3] = lut_read(w, lut_lane, 0x0c0c0700u);
            }
        };
        qk_reads(0, qa[0]);
#pragma unroll
        for (int bt = 0; bt < kQkBatches; ++bt) {
            if (bt + 1 < kQkBatches) qk_reads(bt + 1, qa[(bt + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < kQkBatch; ++k) {
                const int at = kQkBatch * bt + k, s = at >> 3, mf = kQkOrder[at & 7], h = mf >> 2;
                s_acc[s][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, qa[bt & 1][k]), bq[mf],
                                                                    s_acc[s][h], 0, 0, 0);
            }
        }
        // rows 4b+i of the result are tokens unit_token(s, b, i); apply the K scales
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sc[4 * s + i] = score(s_acc[s], i, ksc[s][i], m_run);
        } else {
            // Eight steps of one operand each: eight table reads and the operands of both column tiles (from LDS: with
            // 128 accumulators they do not fit the registers) a step ahead, four MFMAs.
            f4 s_acc[2][2][2];  // [column tile][sub-tile][half row]
#pragma unroll
            for (int g2 = 0; g2 < 2; ++g2)
#pragma unroll
                for (int s = 0; s < 2; ++s) s_acc[g2][s][0] = s_acc[g2][s][1] = f4{0.f, 0.f, 0.f, 0.f};
            u4 ka[2][2];
            h8 qb[2][2];
            auto reads = [&](int st, u4 (&a)[2], h8 (&q)[2]) {
                const int mf = kQkOrder[st];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint32_t w = kw[s][mf];
                    a[s][0] = lut_read(w, lut_lane, 0x0c0c0400u);
                    a[s][1] = lut_read(w, lut_lane, 0x0c0c0500u);
                    a[s][2] = lut_read(w, lut_lane, 0x0c0c0600u);
                    a[s][3] = lut_read(w, lut_lane, 0x0c0c0700u);
                }
#pragma unroll
                for (int g2 = 0; g2 < 2; ++g2) q[g2] = *reinterpret_cast<lds_ch8*>((uintptr_t)(qop_lane + (uint32_t)(g2 * kQopBytes + 16 * mf)));
            };
            reads(0, ka[0], qb[0]);
#pragma unroll
            for (int st = 0; st < 8; ++st) {
                if (st + 1 < 8) reads(st + 1, ka[(st + 1) & 1], qb[(st + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                const int h = kQkOrder[st] >> 2;
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int g2 = 0; g2 < 2; ++g2)
                        s_acc[g2][s][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, ka[st & 1][s]), qb[st & 1][g2],
                                                                                s_acc[g2][s][h], 0, 0, 0);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sc[4 * s + i] = score(s_acc[0][s], i, ksc[s][i], m_run);
                    sc2[4 * s + i] = score(s_acc[1][s], i, ksc[s][i], m_run2);
                }
        }
        if (MASKED) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int pos = t0 + unit_token(t >> 2, b, t & 3);
                const bool vis = col_ok && pos >= col_lo && pos <= col_hi;
                sc[t] = vis ? sc[t] : kNegBig;
                if constexpr (NT > 1) sc2[t] = pos >= col_lo && pos <= col_hi2 ? sc2[t] : kNegBig;
            }
        }

        // ---- raw V dwords of this lane's 8 tokens ------------------------------------------
        if (HAS_NEXT) {
            wait_vm<kLoadsPerHalf>();  // the V half has landed; the next K half may be in flight
        } else {
            wait_vm<0>();
        }
        // per token: the two scales (d0 | d1 << 16), the dword of the first half-row that holds this
        // lane's codes (dword n; for n = 0 codes 0-3 and 124-127 are put together from dwords 0 and
        // 16) and the dword of the second half-row
        uint32_t vsc[8], vw[2][8];
        {
            // lane n reads dwords 0 and 16 of token n & 7 (of the eight this row of lanes works on)
            // and hands the scale pair round inside the row
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(vt_n);
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
                // (dwords 16 + n and 17 + n by one instruction; the former counts for n = 0 only)
                const uint32_t* row32 = reinterpret_cast<const uint32_t*>(vt_lo + (8 * (t >> 2) + (t & 3)) * kTq4RowBytes) + n;
                vw[0][t] = tq4_fuse(row32[16], row32[0], n == 0);
                vw[1][t] = row32[17];
            }
        }
        wait_lds_reads();
        if (HAS_NEXT) issue_v();

        // ---- online softmax (log2 domain), per lane = per query column: scores -> probabilities ----
        // A column's maximum stays where it is until a unit exceeds it by kPfSlack: most units need no exchange between lanes
        // and leave the sums alone, and a probability of up to 2^8 keeps its 22 bits.  us, this, eight instead of nine operands (tq4_fuse) and split_weights, before /
        // now: one token on 131 072 keys 26.5 / 25.9 a layer, eight layers of one on 1 200 126.3 / 124.2, 32 requests of 1 000 to 64 000 125.4 / 124.2.  Exact where that could leave fp16's range, and where the
        // column does not see the whole unit (what lies behind the sequence must not matter).
        auto softmax = [&](float (&x)[8], float& m, float& l, f4 (&o)[2][8], int last, bool ok, bool& have) __attribute__((always_inline)) {
            const float mx = fmaxf(max3(x[0], x[1], x[2]), max3(x[3], x[4], max3(x[5], x[6], x[7])));
            if (!have || __ballot(mx > 0.f) != 0ull) {
                uint32_t d = 0;  // the largest scales
#pragma unroll
                for (int t = 0; t < 8; ++t) d = max_u16x2(d, vsc[t] & 0x7FFF7FFFu);
                const bool large = __ballot((d & 0xFFFFu) > kSlackScaleBits || (d >> 16) > kSlackScaleBits) != 0ull;
                const float slack = large || (MASKED && !(t0 >= col_lo && t0 + kUnit - 1 <= last)) ? 0.f : kPfSlack;
                if (!have || __ballot(mx > slack) != 0ull) {
                    const float top = max_over_rows(mx);
                    const bool empty = !(sum_over_rows(l) > 0.f), any = top > 0.5f * kNegBig;
                    have = __ballot(ok && empty && !any) == 0ull;
                    const float up = empty ? (any ? top : 0.f) : top > slack ? top : 0.f;
                    const float alpha = empty ? 1.f : __builtin_amdgcn_exp2f(-up);
                    m += up;
                    l *= alpha;
#pragma unroll
                    for (int t = 0; t < 8; ++t) x[t] -= up;
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int j = 0; j < 8; ++j) o[h][j] *= alpha;
                }
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) x[t] = __builtin_amdgcn_exp2f(x[t]);
            l += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        };
        softmax(sc, m_run, l_run, o_acc, col_hi, col_ok, started);
        if constexpr (NT > 1) softmax(sc2, m_run2, l_run2, o_acc2, col_hi2, col_ok2, started2);
        float(&p)[8] = sc;
        if constexpr (NT > 1) {
            float(&p2)[8] = sc2;
            if (MASKED) {
                // A token masked for one column tile only keeps its scales.  Where one is not finite, its product with that tile's weight of 0 would be
                // NaN: what the columns that see the token get of it, NaN in all channels of the half row, goes to their sums here, and
                // the scale counts as 0.  (A choice per tile in weights() instead, which few units need: whole call 508 / 513 us.)
                uint32_t bad = 0;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    vsc[t] = p[t] > 0.f || p2[t] > 0.f ? vsc[t] : 0u;
                    bad = max_u16x2(bad, vsc[t] & 0x7FFF7FFFu);
                }
                if (__ballot((bad & 0xFFFFu) >= 0x7C00u || (bad >> 16) >= 0x7C00u) != 0ull) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t exponent = 0x7C00u << (16 * h);
                        float sees = 0.f, sees2 = 0.f;
#pragma unroll
                        for (int t = 0; t < 8; ++t) {
                            const bool finite = (vsc[t] & exponent) != exponent;
                            sees += finite ? 0.f : p[t];
                            sees2 += finite ? 0.f : p2[t];
                            vsc[t] &= finite ? 0xFFFFFFFFu : 0xFFFFu << (16 * (1 - h));
                        }
                        const float add = sum_over_rows(sees) == 0.f ? 0.f : __builtin_nanf(""), add2 = sum_over_rows(sees2) == 0.f ? 0.f : __builtin_nanf("");
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            o_acc[h][j] += add;
                            o_acc2[h][j] += add2;
                        }
                    }
                }
            }
            // Eight batches of two value tiles: eight table reads a batch ahead, eight MFMAs (high and low weights of two column tiles).
            // The weights and code words of a half row are made in front of its batches.
            u4 va[2][2];
            uint32_t lo[4], hi[4];
            u4 ph[2], pl[2];
            auto words = [&](int h) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t wa = vw[h][2 * k], wb = vw[h][2 * k + 1];
                    lo[k] = (wa & 0x0F0F0F0Fu) | ((wb << 4) & 0xF0F0F0F0u);
                    hi[k] = ((wa >> 4) & 0x0F0F0F0Fu) | (wb & 0xF0F0F0F0u);
                }
            };
            auto weights = [&](int h) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    auto w = [&](const float (&pr)[8], int t) { return h == 0 ? mul_by_half_lo(pr[t], vsc[t]) : mul_by_half_hi(pr[t], vsc[t]); };
                    uint32_t whi, wlo;
                    split_weights(w(p, 2 * k), w(p, 2 * k + 1), whi, wlo);
                    ph[0][k] = whi, pl[0][k] = wlo;
                    split_weights(w(p2, 2 * k), w(p2, 2 * k + 1), whi, wlo);
                    ph[1][k] = whi, pl[1][k] = wlo;
                }
            };
            auto pv_reads = [&](int bt, u4 (&a)[2]) __attribute__((always_inline)) {
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int k = 0; k < 4; ++k) a[jj][k] = lut_read(jj ? hi[k] : lo[k], lut_lane, 0x0c0c0400u + ((uint32_t)(bt & 3) << 8));
            };
            words(0);
            pv_reads(0, va[0]);
            weights(0);
#pragma unroll
            for (int bt = 0; bt < 8; ++bt) {
                const int h = bt >> 2;
                if (bt == 3) words(1);
                if (bt + 1 < 8) pv_reads(bt + 1, va[(bt + 1) & 1]);
                if (bt == 4) weights(1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    const int j = 2 * (bt & 3) + jj;
                    const h8 av = __builtin_bit_cast(h8, va[bt & 1][jj]);
                    o_acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, ph[0]), o_acc[h][j], 0, 0, 0);
                    o_acc2[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, ph[1]), o_acc2[h][j], 0, 0, 0);
                }
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    const int j = 2 * (bt & 3) + jj;
                    const h8 av = __builtin_bit_cast(h8, va[bt & 1][jj]);
                    o_acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, pl[0]), o_acc[h][j], 0, 0, 0);
                    o_acc2[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, pl[1]), o_acc2[h][j], 0, 0, 0);
                }
            }
            return;
        } else {
        // ---- O^T += V^T P^T ------------------------------------------------------------------
        // weights of each half: probability times the half-row scale of the value row, as a high
        // and a low fp16 operand (split_weights)
        if (MASKED) {
            // masked tokens have p == 0; their scale pair is zeroed so that a garbage scale (rows
            // beyond the sequence end) cannot inject NaN into the weights
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
                ph[h][k] = (pack && (n & 8)) ? wlo : whi;  // packed: the mirror columns take the low-order part
                pl[h][k] = wlo;
                const uint32_t wa = vw[h][2 * k], wb = vw[h][2 * k + 1];
                // byte q of lo / hi = (nibble 2q / 2q+1 of token a) | (same nibble of token b) << 4
                lo[h][k] = (wa & 0x0F0F0F0Fu) | ((wb << 4) & 0xF0F0F0F0u);
                hi[h][k] = ((wa >> 4) & 0x0F0F0F0Fu) | (wb & 0xF0F0F0F0u);
            }
        }
        // four batches of four value tiles (16 table reads, eight MFMAs), pipelined like the QK batches
        u4 va[2][4];
        auto pv_reads = [&](int bt, u4 (&a)[4]) {
            const int h = bt >> 1;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int j = 4 * (bt & 1) + jj;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t src = (j & 1) ? hi[h][k] : lo[h][k];
                    const uint32_t sel = 0x0c0c0400u + ((uint32_t)(j >> 1) << 8);
                    a[jj][k] = lut_read(src, lut_lane, sel);
                }
            }
        };
        pv_reads(0, va[0]);
#pragma unroll
        for (int bt = 0; bt < 4; ++bt) {
            if (bt + 1 < 4) pv_reads(bt + 1, va[(bt + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
            const int h = bt >> 1;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int j = 4 * (bt & 1) + jj;
                const h8 av = __builtin_bit_cast(h8, va[bt & 1][jj]);
                o_acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, ph[h]), o_acc[h][j], 0, 0, 0);
            }
            if (!pack) {
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const int j = 4 * (bt & 1) + jj;
                    const h8 av = __builtin_bit_cast(h8, va[bt & 1][jj]);
                    o_acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(h8, pl[h]), o_acc[h][j], 0, 0, 0);
                }
            }
        }
        }
    };

    for (int j = 0; unit < cu_end; ++j) {
        const int next_unit = nth_unit(j + 1);
        const bool has_next = next_unit < cu_end;
        if (has_next) locate_unit(next_unit);
        const int t0 = unit * kUnit;
        const bool masked = !(t0 >= i_lo && t0 + kUnit - 1 <= i_hi);
        // The two waves of a SIMD take turns at the higher issue priority, unit by unit: left alone,
        // the arbiter favours the older wave every time and the younger one finishes its units late.
        if ((j + wslot) & 1) {
            __builtin_amdgcn_s_setprio(1);
        } else {
            __builtin_amdgcn_s_setprio(0);
        }
        process_unit(t0, masked, has_next);
        unit = next_unit;
    }
    __builtin_amdgcn_s_setprio(0);
    wait_vm<0>();  // nothing of this wave may still be on its way into LDS when the areas are reused

    if (pack) add_mirror_columns(o_acc);

    // ---- combine the per-lane partial sums of l over the four k-block lanes of a column ------
    l_run = sum_over_rows(l_run);
    if (l_run == 0.f) m_run = kNegBig;  // (no visible key: must not set the column's maximum)
    if constexpr (NT > 1) {
        l_run2 = sum_over_rows(l_run2);
        if (l_run2 == 0.f) m_run2 = kNegBig;
    }

    // ---- merge the waves' states through LDS ---------------------------------------------------
    // Every wave publishes (m, l) and its O, as it stands, in its own region -- its own staging area,
    // which nobody else touches, so the stores need not wait for the other waves -- and after ONE
    // barrier wave c adds up column c of the eight regions, each weighted by 2^(m_w - m_tot), in wave
    // order.  A region holds eight columns: a tile with live columns in both halves (more than
    // eight columns, never a decode step) takes a second pass, two column tiles take up to four.
    // Region layout: column stride kMergeColStride dwords; inside a column the four values a lane
    // holds for one MFMA result (rows 4b..4b+3 of (h, j)) are contiguous at ((h*8 + j)*4 + b)*4,
    // so a lane stores them with one 128-bit write and the adding wave reads one 128-bit piece per
    // lane and region.  The sums reach the element order of the head dimension (lane l: elements
    // 4 l .. 4 l + 3) through a 1 KB transposition buffer per wave in the idle query operand table.
    constexpr int kColStride = kMergeColStride;
    constexpr int kRegion = 8 * kColStride;
    static_assert(kRegion * 4 == kStageTq4, "a wave's merge region is its own staging area");
    static_assert(kWaves * 1024 <= kQopBytes, "transposition buffers");
    float* xbuf = reinterpret_cast<float*>(stage_all);
    float* tbuf = reinterpret_cast<float*>(qop) + wave * 256;
    // [kWaves][16][2]: in an area of its own, a wave publishes its state while others are still in their loops
    float* mlbuf = reinterpret_cast<float*>(smem + ml_offset_for(NT));
    static_assert(kWaves * kRegion == kMergeFloats, "merge layout");
    constexpr int kCols = 16 * NT;
    if (b == 0) {
        mlbuf[(wave * kCols + n) * 2 + 0] = m_run;
        mlbuf[(wave * kCols + n) * 2 + 1] = l_run;
        if constexpr (NT > 1) {
            mlbuf[(wave * kCols + 16 + n) * 2 + 0] = m_run2;
            mlbuf[(wave * kCols + 16 + n) * 2 + 1] = l_run2;
        }
    }
    auto store_region = [&](int half) {
        float* c = xbuf + wave * kRegion + (n & 7) * kColStride;
        if (pack) {  // (half 0)
            if (col_ok) store_packed_column(c, o_acc, n, b);
        } else if ((n >> 3) == half && col_ok) {  // dead columns are never read back
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 8; ++j) *reinterpret_cast<f4*>(c + ((h * 8 + j) * 4 + b) * 4) = o_acc[h][j];
        }
    };
    const bool live0 = (ok_mask & 0xFFu) != 0u, live1 = (ok_mask >> 8) != 0u;  // the same in every wave
    // (two column tiles: a live column is in the first eight, the tile's live ones lie without a gap from column 0 on)
    store_region(NT > 1 || live0 ? 0 : 1);

    __syncthreads();  // every wave is done with the table, and the regions of the first pass are there
#pragma unroll 1
    for (int half = 0; half < (PLAIN ? 1 : 2 * NT); ++half) {
        if constexpr (PLAIN) {
        } else if constexpr (NT > 1) {
            if (((ok_mask >> (8 * half)) & 0xFFu) == 0u) break;
            if (half > 0) {
                __syncthreads();  // the pass before has read the regions
                if (half == 2) {  // on to the second column tile
                    col_ok = col_ok2;
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int j = 0; j < 8; ++j) o_acc[h][j] = o_acc2[h][j];
                }
                store_region(half & 1);
                __syncthreads();
            }
        } else {
            if (!(half ? live1 : live0)) continue;
            if (half == 1 && live0) {
                __syncthreads();  // the first pass has read the regions
                store_region(1);
                __syncthreads();
            }
        }
        const int col = 8 * half + wave;
        if (wave < 8 && ((ok_mask >> col) & 1u)) {
            size_t old_row = 0;
            f4 old_acc, old_rec;
            if constexpr (NT > 1) {
                const int t = div_q_group(col, P);
                old_row = ((size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + col - t * P.q_group)) * P.part_stride +
                          (size_t)(P.pf_slot_base + chunk);
                old_acc = *reinterpret_cast<const f4*>(P.part_acc + old_row * kHeadDim + 4 * lane);
                old_rec = *reinterpret_cast<const f4*>(P.part_ml + old_row * 4);
            }
            // state of the column in the eight waves (the same addresses in every lane)
            float mw[kWaves], lw[kWaves];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const f2 r = *reinterpret_cast<const f2*>(mlbuf + (w * kCols + col) * 2);
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
                tot += *reinterpret_cast<const f4*>(xbuf + w * kRegion + wave * kColStride + 4 * lane) * wgt;
            }
            *reinterpret_cast<f4*>(tbuf + 4 * lane) = tot;
            // element e = 4*lane + k is value (h, j, row r) with e = tq4_pv_elem(h, j, r); the reads
            // follow the write of the same wave in LDS order
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = tbuf[tq4_merge_slot(lane) + 16 * k];
            const int t = div_q_group(col, P);
            const int a = col - t * P.q_group;
            const size_t row = (size_t)(tok0 + t) * P.num_q_heads + (size_t)(q_head_base + a);
            if (NT > 1 || (BAL ? item.n_chunks > 1 : P.max_chunks > 1)) {
                // un-normalised, rotated, still carrying the table gain; the merge kernel finishes
                if constexpr (NT > 1) {
                    // The chunk joins a record of the shared prefix (asked for ahead of the sums above); the row has no other
                    // chunk records, which the first one of them says.
                    const float m = fmaxf(m_col, old_rec[0]);
                    const float w_new = __builtin_amdgcn_exp2f(m_col - m), w_old = __builtin_amdgcn_exp2f(old_rec[0] - m);
                    float* dst = P.part_acc + old_row * kHeadDim;
                    *reinterpret_cast<f4*>(dst + 4 * lane) = f4{v[0], v[1], v[2], v[3]} * w_new + old_acc * w_old;
                    if (lane == 0) {
                        *reinterpret_cast<f4*>(P.part_ml + old_row * 4) = f4{m, l_col * w_new + old_rec[1] * w_old, old_rec[2], 0.f};
                        if (chunk == 0) *reinterpret_cast<f4*>(P.part_ml + row * P.part_stride * 4) = f4{kNegBig, 0.f, 0.f, 0.f};
                    }
                    continue;
                }
                const size_t prow = BAL ? bal_partial_row(item.slot, (int)gridDim.y, kv_sub, 16, col)
                                        : row * (SP ? P.part_stride : P.max_chunks) + chunk;
                float* dst = P.part_acc + prow * kHeadDim;
                *reinterpret_cast<f4*>(dst + 4 * lane) = f4{v[0], v[1], v[2], v[3]};
                if (lane == 0) {
                    // (m, l, number of chunks of this row, -): one record per chunk, every record
                    // carries the count so the merge needs no dependent load
                    *reinterpret_cast<f4*>(P.part_ml + prow * 4) = f4{m_col, l_col, (float)g.n_chunks, 0.f};
                }
            } else {
                const float inv = l_col > 0.f ? kLutInvGain / l_col : 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] *= inv;
                if (P.rot_out) {  // values stored rotated
                    wht256_wave(v, lane);
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = apply_sign(v[k], 4 * lane + k);
                }
                store_out_row<TQ>(P, row, lane, v);
            }
        }
    }
}

template <typename TQ, bool SP = false>
__global__ __launch_bounds__(kTq4Waves * 64, 1) void paged_attn_tq4_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    // lut_read() addresses the table absolutely: the dynamic block starts at LDS address 0 because
    // the kernel has no static LDS (checked on the host before the first launch)
    // decode steps (no request has more than one tile): every key is read by one workgroup only,
    // the loads carry the streaming hint; one body per kind of load
    BalItem item{};
    if constexpr (SP) item.req = (int)blockIdx.z, item.slot = (int)blockIdx.x, item.u_begin = __builtin_amdgcn_readfirstlane(*P.key_floor);
    if (!SP && P.tiles_by_request != 0 && P.q_subgroups == 1) {  // uniform for the grid
        tq4_tile<TQ, false, SP, true>(P, smem, item, true);
    } else {
        tq4_tile<TQ, false, SP, false>(P, smem, item, true);
    }
}

// Decode steps without masks, see plain_decode; the bits of the general kernel.  What bounds a short one is the chain lengths - addresses - first rows: device
// timestamps, one token on 1 200 keys, from the wave's entry: lengths there 1.16 us, addresses 1.72, first rows asked for 2.17 in the general kernel, most of it
// scalar instructions, which eight waves issue one after the other.  us, general / this: one token on 1 200 keys, eight layers with their producers, 116.1 / 110.9, one on
// 131 072, four layers, 101.9 / 98.4.
template <typename TQ>
__global__ __launch_bounds__(kTq4Waves * 64, 1) void paged_attn_tq4_plain_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    tq4_tile<TQ, false, false, true, 1, true>(P, smem, BalItem{}, true);
}

// What the probe of a shared prefix leaves for the kernels behind it.
struct SpHeader {
    int32_t floor;   // keys [0, floor) are the shared prefix
    int32_t qsl[2];  // query_start_loc of the pseudo request: {0, total_tokens}
    int32_t seq;     // its seq_lens_after (= floor)
    int32_t ctx;     // its context_lens_before (= floor: every key visible to every token)
    int32_t wide;    // the private rest is for two column tiles, see kWidePrivateUnits
    int32_t pad[2];
};

// The private rest of a verify batch with more than 16 query columns per request and kv head: both column tiles in one workgroup, so that
// a key is looked up once for 32 columns (a wave's unit: 465 vector instructions and 96 MFMAs, one tile 330 and 48).  Issue bounds it, so the loads keep their
// plain form: with the streaming hint 3 % slower.  `wide` holds the geometry of that form, whose chunks join the prefix's records, for which there is room
// whatever their number; `P` that of the plain path, for a short rest (kWidePrivateUnits) and with nothing shared, where the batch has the plain path's bits.  us, 16 requests x 4 tokens on 262 144 keys, 200 000 of
// them shared, one column tile / two: whole call 524 / 486, on another box 534 / 512; this kernel 177 / 147.
template <typename TQ>
__global__ __launch_bounds__(kTq4Waves * 64, 1) void paged_attn_tq4_private_kernel(const AttnParams P, const AttnParams wide, const SpHeader* hdr,
                                                                                   int chunks, int tiles, int wide_chunks, int wide_tiles) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int wg = (int)blockIdx.x;
    BalItem item{};
    const int floor = hdr->floor, wide_rest = hdr->wide;
    item.u_begin = __builtin_amdgcn_readfirstlane(floor);
    if (__builtin_amdgcn_readfirstlane(wide_rest) != 0) {
        item.req = wg / wide_chunks;
        item.slot = wg - item.req * wide_chunks;
        if (item.req < wide_tiles) tq4_tile<TQ, false, true, false, 2>(wide, smem, item, true);
    } else {
        item.req = wg / chunks;
        item.slot = wg - item.req * chunks;
        if (item.req < tiles) tq4_tile<TQ, false, true, false, 1>(P, smem, item, true);
    }
}

// The argument block once more, from the kernel's argument segment: a second body of a kernel that reads its
// arguments here leaves the scalar registers of the first alone (shared, the scalars of both are loaded at
// the kernel's start and spilled).
__device__ __forceinline__ AttnParams kernel_params_again() {
    typedef const __attribute__((address_space(4))) AttnParams* Args;
    Args args = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return *(const AttnParams*)args;
}

// A batch of wide or several tiles that has little to read (P.short_units): its tiles have 16 columns, and every entry (at
// most 128) is cut into equal pieces of its own, so that a workgroup has at most one.  The second column tile costs 5 us
// per piece (query table, merge of the waves), the second piece of a share 8; reading the keys once for both
// tiles repays neither here.  The plan decides by the lengths it finds, not by the host's bound.  us, before the plan ->
// one plan for all -> now: 20 requests x 4 tokens over Q8_0 on 600 keys 31.5 -> 27.7 -> 18.4, on 1000 33.3 -> 28.4 ->
// 21.3; 40 x 4 on 1000 26.2 -> 32.2 -> 27.6; bf16 10 x 4 on 1000 23.4 -> 20.1 -> 18.0.  Longer batches: no change.
template <typename TileFn>
__device__ __forceinline__ void bal_short_piece(const AttnParams& P, TileFn&& tile) {
    const int lane = (int)threadIdx.x & 63;
    const int groups = (int)gridDim.x, wg = (int)blockIdx.x;
    const int entries = P.B.num_reqs * P.short_tiles;
    const BalReq q0 = bal_load_req(P, P.short_tiles, P.short_tok_tile, lane);
    const BalReq q1 = bal_load_req(P, P.short_tiles, P.short_tok_tile, 64 + lane);
    const auto record = [&](int tok, int first, int pieces, int tok_of_tile) {
        if (tok < P.B.total_tokens) *reinterpret_cast<int4*>(P.bal_table + 4 * (size_t)tok) = int4{first, pieces, tok_of_tile, 16};
    };
    const auto record_idle = [&](const BalReq& q, int e) {  // as in bal_for_each_piece
        if (e >= entries) return;
        if (q.units == 0) {
            for (int t = q.t_lo; t < q.t_hi; ++t) record(t, 0, q.live ? 0 : -1, 0);
        }
        if (e == entries - 1) {
            for (int t = max(q.hi, 0); t < P.B.total_tokens; ++t) record(t, 0, -1, 0);
        }
    };
    if (wg == 0 && blockIdx.y == 0 && threadIdx.x < 64) {
        record_idle(q0, lane);
        record_idle(q1, 64 + lane);
    }
    int longest = bal_share(__builtin_amdgcn_readlane(wave_incl_scan(q0.units + q1.units), 63), groups, kMinUnitsPerChunk);
    int pieces0, pieces1, incl0, incl1;
    for (;;) {
        pieces0 = q0.units > 0 ? fast_div(q0.units + longest - 1, longest) : 0;
        pieces1 = q1.units > 0 ? fast_div(q1.units + longest - 1, longest) : 0;
        incl0 = wave_incl_scan(pieces0);
        incl1 = __builtin_amdgcn_readlane(incl0, 63) + wave_incl_scan(pieces1);
        const int n = __builtin_amdgcn_readlane(incl1, 63);
        if (n <= groups) break;
        // at least to where the first entry has a piece less: requests of one length go from two pieces to one in
        // one step (13 requests x 10 tokens on 1000 keys: 35.8 us with steps of one)
        const int less0 = pieces0 > 1 ? fast_div(q0.units + pieces0 - 2, pieces0 - 1) : 0x7fffffff;
        const int less1 = pieces1 > 1 ? fast_div(q1.units + pieces1 - 2, pieces1 - 1) : 0x7fffffff;
        longest = max(longest + fast_div(longest * (n - groups), groups),
                      (int)__builtin_amdgcn_readlane(wave_min_last(min(less0, less1)), 63));
    }
    unsigned long long hits = __ballot(pieces0 > 0 && wg < incl0);
    const bool second = hits == 0ull;
    if (second) hits = __ballot(pieces1 > 0 && wg < incl1);
    if (hits == 0ull) return;
    const int src = __builtin_ctzll(hits);
    // (lane values picked one by one: a copy of the struct, first or second, would go through memory)
    const auto pick = [&](int a, int b) {
        return second ? __builtin_amdgcn_readlane(b, src) : __builtin_amdgcn_readlane(a, src);
    };
    const int n_pieces = pick(pieces0, pieces1), first = pick(incl0, incl1) - n_pieces, units = pick(q0.units, q1.units);
    const int per_piece = fast_div(units + n_pieces - 1, n_pieces);
    const int entry = second ? 64 + src : src;
    BalItem it;
    it.req = small_div(entry, P.short_tiles);
    it.tile = entry - it.req * P.short_tiles;
    it.tok_tile = P.short_tok_tile;
    it.rq_start = pick(q0.lo, q1.lo);
    it.rq_end = pick(q0.hi, q1.hi);
    it.seq_after = pick(q0.sa, q1.sa);
    it.ctx_before = pick(q0.cb, q1.cb);
    it.u_begin = (wg - first) * per_piece;
    it.u_end = min(it.u_begin + per_piece, units);
    it.n_chunks = n_pieces;
    it.slot = wg;
    const int tok = pick(q0.t_lo, q1.t_lo) + (int)threadIdx.x;
    if (wg == first && blockIdx.y == 0 && tok < pick(q0.t_hi, q1.t_hi)) record(tok, first, n_pieces, (int)threadIdx.x);
    tile(it);
}

// Balanced decode: grid = (groups, kv head x q subgroup).  Every wave computes the plan (the
// loads are the same addresses in every wave of the chip and stay in cache) and calls
// tile(piece) for the pieces of its workgroup's share, in order.
// SHORT: a batch that turns out short is left to short_batch().
// FEW, MANY: chunk_count's and grid_decode_serves' lines for the format.
template <bool SHORT, int FEW, int MANY, typename TileFn, typename ShortFn>
__device__ __forceinline__ void bal_for_each_piece(const AttnParams& P, TileFn&& tile, ShortFn&& short_batch) {
    const int lane = (int)threadIdx.x & 63;
    const int entries = P.B.num_reqs * P.bal_tiles;
    // the first 64 entries are loaded once: their lane values serve the total and the search for
    // the first piece (most workgroups have exactly one piece, most batches at most 64 entries)
    const BalReq q0 = bal_load_req(P, P.bal_tiles, P.tok_tile, lane);
    const int incl0 = wave_incl_scan(q0.cost);
    int total = __builtin_amdgcn_readlane(incl0, 63);
    if constexpr (SHORT) {
        // (a batch that may be short has at most 64 entries)
        if (total - P.piece_cost * (int)__popcll(__ballot(q0.units > 0)) <= P.short_units) {  // uniform for the grid
            short_batch();
            return;
        }
    }
    // wave 0 of workgroup (0, 0) records the tokens no workgroup will work on
    const bool recorder = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 64;
    auto record_idle = [&](const BalReq& q, int e) {
        if (!recorder || e >= entries) return;
        if (q.units == 0) {
            for (int t = q.t_lo; t < q.t_hi && t < P.B.total_tokens; ++t)
                *reinterpret_cast<int4*>(P.bal_table + 4 * (size_t)t) = int4{0, q.live ? 0 : -1, t - q.t_lo, 0};
        }
        if (e == entries - 1) {
            for (int t = max(q.hi, 0); t < P.B.total_tokens; ++t)
                *reinterpret_cast<int4*>(P.bal_table + 4 * (size_t)t) = int4{0, -1, 0, 0};
        }
    };
    record_idle(q0, lane);
    for (int base = 64; base < entries; base += 64) {
        const BalReq q = bal_load_req(P, P.bal_tiles, P.tok_tile, base + lane);
        record_idle(q, base + lane);
        total += __builtin_amdgcn_readlane(wave_incl_scan(q.cost), 63);
    }
    BalItem it{};
    it.tok_tile = P.tok_tile;
    int my_begin = 0, my_end = 0, piece_end = 0;  // (aligned: the one piece ends the share)
    int share = 1;
    // a batch that the chunk grid serves where the host's bound says so: its chunks, so that the bits do not depend on the bound
    bool as_grid = false;
    if constexpr (!SHORT) as_grid = P.grid_chunks > 0 && __ballot(!grid_decode_serves(q0.units, P.B.num_reqs, P.grid_chunks, MANY)) == 0ull;
    const bool aligned = P.bal_aligned || as_grid;
    if (aligned) {  // uniform for the grid; at most 64 entries
        // Units per piece: the smallest count found by a few steps from below for which the pieces fit
        // the grid.  (Every wave of the chip computes the same numbers.)
        const int groups = (int)gridDim.x;
        const int units = __builtin_amdgcn_readlane(wave_incl_scan(q0.units), 63);
        int pieces, incl;
        if (as_grid) {
            pieces = q0.units > 0 ? chunk_geom(0, 32 * q0.units - 1, P.grid_chunks, few_chunks_of(FEW, P.grid_chunks)).n_chunks : 0;
            incl = wave_incl_scan(pieces);
        } else {
            share = bal_share(units, groups, P.min_upc);
            for (;;) {
                pieces = q0.units > 0 ? fast_div(q0.units + share - 1, share) : 0;
                incl = wave_incl_scan(pieces);
                const int n = __builtin_amdgcn_readlane(incl, 63);
                if (n <= groups) break;
                share += fast_div(share * (n - groups), groups) + 1;
            }
        }
        const unsigned long long hits = __ballot(pieces > 0 && (int)blockIdx.x < incl);
        if (hits == 0ull) return;
        const int src = __builtin_ctzll(hits);
        const int n_pieces = __builtin_amdgcn_readlane(pieces, src);
        const int first = __builtin_amdgcn_readlane(incl, src) - n_pieces;
        const int e_units = __builtin_amdgcn_readlane(q0.units, src);
        const int per_piece = fast_div(e_units + n_pieces - 1, n_pieces);
        it.req = P.bal_tiles == 1 ? src : small_div(src, P.bal_tiles);
        it.tile = src - it.req * P.bal_tiles;
        it.rq_start = __builtin_amdgcn_readlane(q0.lo, src);
        it.rq_end = __builtin_amdgcn_readlane(q0.hi, src);
        it.seq_after = __builtin_amdgcn_readlane(q0.sa, src);
        it.ctx_before = __builtin_amdgcn_readlane(q0.cb, src);
        // equal pieces, none without units: n_pieces = ceil(e_units / share), so per_piece <= share and
        // (n_pieces - 1) * per_piece < e_units
        it.u_begin = ((int)blockIdx.x - first) * per_piece;
        it.u_end = min(it.u_begin + per_piece, e_units);
        it.n_chunks = n_pieces;
        it.slot = (int)blockIdx.x;
        const int tok = __builtin_amdgcn_readlane(q0.t_lo, src) + (int)threadIdx.x;
        if ((int)blockIdx.x == first && blockIdx.y == 0 && tok < __builtin_amdgcn_readlane(q0.t_hi, src) &&
            tok < P.B.total_tokens) {
            *reinterpret_cast<int4*>(P.bal_table + 4 * (size_t)tok) = int4{first, n_pieces, (int)threadIdx.x, 0};
        }
    } else {
        share = bal_share(total, (int)gridDim.x, P.min_upc + P.piece_cost);
        my_begin = (int)blockIdx.x * share;
        my_end = min(my_begin + share, total);
        if (my_begin >= total) return;
    }

    // The pieces of this share, in order.  Nothing but a few scalars stays live across a tile:
    // the 64-request group that holds the next piece is loaded and scanned again after each one.
    int base = 0, before = 0, taken = 0;  // group, units before it, pieces of it already done
    // next piece inside the group whose lane values are (q, incl); false: the group has none left
    auto scan_group = [&](const BalReq& q, int incl) -> bool {
        const int start = before + incl - q.units;  // of the real units, behind the charge
        unsigned long long hits = __ballot(q.units > 0 && start < my_end && start + q.units > my_begin);
        for (int skip = 0; skip < taken && hits != 0ull; ++skip) hits &= hits - 1ull;
        if (hits == 0ull) {
            before += __builtin_amdgcn_readlane(incl, 63);
            base += 64;
            taken = 0;
            return false;
        }
        const int src = __builtin_ctzll(hits);
        const int r_start = __builtin_amdgcn_readlane(start, src);
        const int r_units = __builtin_amdgcn_readlane(q.units, src);
        const int entry = base + src;
        it.req = P.bal_tiles == 1 ? entry : small_div(entry, P.bal_tiles);
        it.tile = entry - it.req * P.bal_tiles;
        it.rq_start = __builtin_amdgcn_readlane(q.lo, src);
        it.rq_end = __builtin_amdgcn_readlane(q.hi, src);
        it.seq_after = __builtin_amdgcn_readlane(q.sa, src);
        it.ctx_before = __builtin_amdgcn_readlane(q.cb, src);
        it.u_begin = max(my_begin, r_start) - r_start;
        it.u_end = min(my_end, r_start + r_units) - r_start;
        it.n_chunks = fast_div(r_start + r_units - 1, share) - fast_div(r_start, share) + 1;
        it.slot = (int)blockIdx.x + entry;
        piece_end = r_start + it.u_end;
        const int tok = __builtin_amdgcn_readlane(q.t_lo, src) + (int)threadIdx.x;
        if (it.u_begin == 0 && blockIdx.y == 0 && tok < __builtin_amdgcn_readlane(q.t_hi, src) &&
            tok < P.B.total_tokens) {  // first piece: one entry per query token
            *reinterpret_cast<int4*>(P.bal_table + 4 * (size_t)tok) = int4{it.slot, it.n_chunks, (int)threadIdx.x, 0};
        }
        ++taken;
        return true;
    };
    auto find_next = [&]() -> bool {
        while (base < entries && before < my_end) {
            const BalReq q = bal_load_req(P, P.bal_tiles, P.tok_tile, base + lane);
            if (scan_group(q, wave_incl_scan(q.cost))) return true;
        }
        return false;
    };
    bool have = aligned || scan_group(q0, incl0);
    if (!have) have = find_next();
    while (have) {
        tile(it);
        if (piece_end >= my_end) break;  // the share ends with this piece
        __syncthreads();  // the tile's merge regions alias what the next piece sets up
        have = find_next();
    }
}

template <typename TQ>
__global__ __launch_bounds__(kTq4Waves * 64, 1) void paged_attn_tq4_balanced_kernel(const AttnParams P) {
    extern __shared__ __align__(16) uint8_t smem[];
    // the pair table survives a piece (the merge regions lie in the staging areas): built once
    bool first = true;
    const auto piece = [&](const BalItem& it) {
        tq4_tile<TQ, true>(P, smem, it, first);
        first = false;
    };
    bal_for_each_piece<false, kFewChunksTq4, kGridUnitsTq4>(P, piece, [] {});
}

// One wave adds up the slices of a row's n_chunks chunks (at most SLOTS; lane s holds the record of chunk s), in the order in which ORDER waves
// and their sum through LDS do it: every bit is the same.
template <int SLOTS, int ORDER>
__device__ __forceinline__ f4 merge_slices(const f4& rec, int n_chunks, const f4 (&a)[SLOTS], int lane, float& l_tot) {
    const bool mine = lane < n_chunks && rec[1] > 0.f;
    float m_tot = mine ? fmaxf(rec[0], kNegBig) : kNegBig;
    m_tot = fmaxf(m_tot, lane_xor<1>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<2>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<4>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<8>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<16>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<32>(m_tot, lane));
    const float w = mine ? __builtin_amdgcn_exp2f(rec[0] - m_tot) : 0.f, l = rec[1];
    const unsigned long long live = __ballot(mine);
    f4 v[ORDER];
    float l_part[ORDER];
#pragma unroll
    for (int g = 0; g < ORDER; ++g) v[g] = f4{0.f, 0.f, 0.f, 0.f}, l_part[g] = 0.f;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        if ((live >> s) & 1ull) {  // uniform
            const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s));
            const float ls = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l), s));
            l_part[s % ORDER] = __builtin_fmaf(ls, ws, l_part[s % ORDER]);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[s % ORDER][k] = __builtin_fmaf(a[s][k], ws, v[s % ORDER][k]);
        }
    }
    f4 tot = {0.f, 0.f, 0.f, 0.f};
    l_tot = 0.f;
#pragma unroll
    for (int g = 0; g < ORDER; ++g) {
        tot += v[g];
        l_tot += l_part[g];
    }
    return tot;
}

// Merge for the balanced decode kernel: one workgroup of GROUPS waves per (token, q head) row; wave g
// sums the partials g, g + GROUPS, ... and the first wave adds up the waves.  The token's table entry
// says where the partials are; rows whose tile was not cut (one piece) were finished by the attention
// kernel, rows of live requests without visible keys are zero, rows of masked requests stay untouched.
// GROUPS: see merge_small_groups.
// A chain of three round trips, the table entry, the records and slices, the store: the arguments before the first are preloaded, and up to 16 pieces
// are added up by one wave without LDS.  us of a whole attention call, arguments in memory and all rows through LDS / now: TQ4, 24 requests of 3 000 to
// 9 000 keys 29.9 / 28.7; Q8_0, 16 requests of 1 000 to 12 000 32.7 / 31.1, 5 x 4 tokens on 500 to 3 000 17.6 / 16.6; FP8 17.3 / 15.9.
template <typename TQ, int HD, int GROUPS>
__global__ __launch_bounds__(GROUPS * 64) void balanced_merge_kernel(const int32_t* bal_table, const float* part_acc,
                                                                     const float* part_ml, int num_q_heads, int q_group, int kv_subs,
                                                                     int bal_cols, const uint16_t* gate, const AttnParams P, float out_scale,
                                                                     int rotate) {
    constexpr int kSlots = kMergeGroups * kMergeMaxPerGroup;  // partials of a row at most
    static_assert(GROUPS * 64 >= kSlots, "one record per thread");
    __shared__ f4 s_acc[GROUPS][64];
    __shared__ f4 s_rec[kSlots];
    __shared__ float s_red[GROUPS];
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int grp = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int head = (int)blockIdx.x, tok = (int)blockIdx.y;
    // (the leading arguments repeat fields of P: preloaded, so that the table entry is asked for at once)
    const size_t row = (size_t)tok * num_q_heads + head;
    const int4 entry = *reinterpret_cast<const int4*>(bal_table + 4 * (size_t)tok);  // same address in every lane
    uint2 g = {0u, 0u};
    if (grp == 0) {
        g = load_out_gate<HD>(gate, row, lane);
        asm volatile("" ::"s"(P.out), "s"(P.gate), "s"(out_scale), "s"(rotate));  // (on their way beside the entry, not where they are used)
    }
    const int kv_sub = small_div(head, q_group);  // = kv_head * q_subgroups + subgroup
    const int n_chunks = __builtin_amdgcn_readfirstlane(entry.y);
    if (n_chunks < 0 || n_chunks == 1) return;  // masked, or finished by the attention kernel
    if (n_chunks == 0) {                        // no visible key: zeros
        const float zero[4] = {0.f, 0.f, 0.f, 0.f};
        if (grp == 0) store_out_row<TQ, HD>(P, row, lane, zero, g);
        return;
    }
    const int col = entry.z * q_group + (head - kv_sub * q_group);
    const int cols = entry.w != 0 ? entry.w : bal_cols;
    const size_t prow0 = bal_partial_row(entry.x, kv_subs, kv_sub, cols, col);
    const size_t pstride = (size_t)kv_subs * cols;  // partial rows between consecutive slots
    if (n_chunks <= kMergeMaxPerGroup) {  // few: one wave, see split_merge_few_kernel
        if (grp != 0) return;
        f4 rec = {kNegBig, 0.f, 0.f, 0.f};
        if (lane < n_chunks) rec = *reinterpret_cast<const f4*>(part_ml + (prow0 + lane * pstride) * 4);
        f4 a[kMergeMaxPerGroup];
#pragma unroll
        for (int s = 0; s < kMergeMaxPerGroup; ++s) {
            a[s] = f4{0.f, 0.f, 0.f, 0.f};
            if (s < n_chunks && (HD == 256 || 4 * lane < HD))
                a[s] = *reinterpret_cast<const f4*>(part_acc + (prow0 + s * pstride) * kHeadDim + 4 * lane);
        }
        float l_tot;
        const f4 tot = merge_slices<kMergeMaxPerGroup, GROUPS>(rec, n_chunks, a, lane, l_tot);
        const float inv = l_tot > 0.f ? out_scale / l_tot : 0.f;
        float o[4] = {tot[0] * inv, tot[1] * inv, tot[2] * inv, tot[3] * inv};
        if (rotate) {
            wht256_wave(o, lane);
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * lane + k);
        }
        store_out_row<TQ, HD>(P, row, lane, o, g);
        return;
    }
    if (tid < n_chunks && tid < kSlots) s_rec[tid] = *reinterpret_cast<const f4*>(part_ml + (prow0 + tid * pstride) * 4);
    f4 a[kMergeMaxPerGroup];
    auto load_slices = [&](int first) {
#pragma unroll
        for (int k = 0; k < kMergeMaxPerGroup; ++k) {
            const int s = first + grp + k * GROUPS;
            a[k] = f4{0.f, 0.f, 0.f, 0.f};
            if (s < n_chunks && (HD == 256 || 4 * lane < HD))
                a[k] = *reinterpret_cast<const f4*>(part_acc + (prow0 + s * pstride) * kHeadDim + 4 * lane);
        }
    };
    load_slices(0);
    __syncthreads();
    float m_tot = kNegBig;
    for (int s = lane; s < n_chunks; s += 64) {
        const f4 r = s_rec[s];
        if (r[1] > 0.f) m_tot = fmaxf(m_tot, r[0]);
    }
    m_tot = fmaxf(m_tot, lane_xor<1>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<2>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<4>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<8>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<16>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<32>(m_tot, lane));
    f4 v = {0.f, 0.f, 0.f, 0.f};
    float l_part = 0.f;
    for (int first = 0;;) {
#pragma unroll
        for (int k = 0; k < kMergeMaxPerGroup; ++k) {
            const int s = first + grp + k * GROUPS;
            if (s < n_chunks) {
                const f4 r = s_rec[s];
                if (r[1] > 0.f) {
                    const float w = __builtin_amdgcn_exp2f(r[0] - m_tot);
                    l_part += r[1] * w;
                    v += a[k] * w;
                }
            }
        }
        first += kMergeMaxPerGroup * GROUPS;
        if (GROUPS == kMergeGroups || first >= n_chunks) break;
        load_slices(first);
    }
    s_acc[grp][lane] = v;
    if (lane == 0) s_red[grp] = l_part;
    __syncthreads();
    if (grp != 0) return;
    float l_tot = 0.f;
    f4 tot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < GROUPS; ++k) {
        tot += s_acc[k][lane];
        l_tot += s_red[k];
    }
    const float inv = l_tot > 0.f ? out_scale / l_tot : 0.f;
    float o[4] = {tot[0] * inv, tot[1] * inv, tot[2] * inv, tot[3] * inv};
    if (rotate) {
        wht256_wave(o, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * lane + k);
    }
    store_out_row<TQ, HD>(P, row, lane, o, g);
}

// Does a row's token belong to a request, and is it to be computed?  Lane r looks at request r; the first 64 requests' tokens are asked for by the
// constructor, together with what else the kernel needs: asked for one behind the other, and the gate behind the sums, they were three more round trips of
// a kernel that consists of one (us, eight layers of one token on 1 200 keys 113.5 / 109.7, four of one on 32 768 bf16 keys 78.5 / 77.5).  (First match wins.)
struct RowOwner {
    int lo, hi;
    __device__ __forceinline__ RowOwner(const int32_t* query_start_loc, int num_reqs, int lane) {
        const int r = min(lane, num_reqs - 1);
        lo = query_start_loc[r];
        hi = query_start_loc[r + 1];
    }
    __device__ __forceinline__ bool live(const warp34_attention_batch& B, int tok, int lane) const {
        if (B.valid_token_mask != nullptr && B.valid_token_mask[tok] == 0) return false;
        for (int base = 0; base < B.num_reqs; base += 64) {
            const int r = base + lane;
            const bool inb = r < B.num_reqs;
            const int first = base == 0 ? lo : inb ? B.query_start_loc[r] : 0;
            const int end = base == 0 ? hi : inb ? B.query_start_loc[r + 1] : 0;
            const unsigned long long hits = __ballot(inb && tok >= first && tok < end);
            if (hits != 0ull) return B.valid_req_mask == nullptr || B.valid_req_mask[base + __builtin_ctzll(hits)] != 0;
        }
        return false;
    }
};

// Merge of the split-K partials (op_paged_attn.cu:1132-1218): m_tot = max m_s,
// w_s = 2^(m_s - m_tot), out = sum acc_s w_s / sum l_s w_s, then one inverse rotation.
// One workgroup of GROUPS waves per (token, q head) row: the waves stride the chunks, each thread
// owns 4 of the 256 columns; the waves are summed through LDS.
// Everything the row needs (validity, chunk records, accumulators) is requested in ONE memory
// round trip: records and accumulators of all max_chunks slots (the first 16 GROUPS of them) are
// loaded speculatively and the slots beyond the row's chunk count are discarded with selects.
template <typename TQ, bool SP, int HD, int GROUPS>
__global__ __launch_bounds__(GROUPS * 64) void split_merge_kernel(const float* part_acc_in, const float* part_ml_in,
                                                                  int max_chunks_in, int num_q_heads_in, const int32_t* query_start_loc,
                                                                  const uint16_t* gate, int num_reqs, const AttnParams P, float out_scale,
                                                                  int rotate) {
    constexpr int kSlots = kMergeGroups * kMergeMaxPerGroup;
    static_assert(GROUPS * 64 >= kSlots, "one record per thread");
    __shared__ f4 s_acc[GROUPS][64];
    __shared__ f4 s_rec[kSlots];
    __shared__ float s_red[GROUPS];
    __shared__ int s_valid;
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int grp = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tok = (int)blockIdx.y;
    const warp34_attention_batch& B = P.B;
    // the leading arguments repeat fields of P: they are preloaded into scalar registers at wave launch, so the loads below do not wait for
    // the kernel-argument fetch
    const size_t row = (size_t)tok * num_q_heads_in + blockIdx.x;
    const float* ml = part_ml_in + row * max_chunks_in * 4;
    const float* acc = part_acc_in + row * max_chunks_in * kHeadDim;

    // speculative loads: chunk records (one per thread) and this thread's accumulator slices
    f4 rec = {kNegBig, 0.f, 0.f, 0.f};
    if (tid < max_chunks_in) rec = *reinterpret_cast<const f4*>(ml + 4 * tid);
    f4 a[kMergeMaxPerGroup];
    auto load_slices = [&](int first) {
#pragma unroll
        for (int k = 0; k < kMergeMaxPerGroup; ++k) {
            const int s = first + grp + k * GROUPS;
            a[k] = f4{0.f, 0.f, 0.f, 0.f};
            // (records keep a 256-float stride at every head dimension; lanes beyond the row load nothing)
            if (s < max_chunks_in && (HD == 256 || 4 * lane < HD))
                a[k] = *reinterpret_cast<const f4*>(acc + (size_t)s * kHeadDim + 4 * lane);
        }
    };
    load_slices(0);
    uint2 g = {0u, 0u};
    if (grp == 0) {
        const RowOwner owner(query_start_loc, num_reqs, lane);
        g = load_out_gate<HD>(gate, row, lane);
        asm volatile("" ::"s"(P.out), "s"(P.gate), "s"(out_scale), "s"(rotate));  // (on their way beside the slices, not where they are used)
        const bool live = owner.live(B, tok, lane);
        if (lane == 0) s_valid = live ? 1 : 0;
    }
    if (tid < kSlots) s_rec[tid] = rec;
    __syncthreads();
    if (!s_valid) return;  // masked row: output untouched (uniform for the block)
    int n_chunks = (int)s_rec[0][2];
    if (n_chunks > P.max_chunks) n_chunks = P.max_chunks;
    // slots of the row: its split-K chunks, then (SP, behind a gap) those of the shared-prefix pass
    auto live_slot = [&](int s) {
        if constexpr (SP) return s < n_chunks || (s >= P.pf_slot_base && s < P.pf_slot_base + P.pf_split);
        return s < n_chunks;
    };
    const int n_slots = __builtin_amdgcn_readfirstlane(SP ? max_chunks_in : n_chunks);

    // global maximum of m over chunks with l > 0 (every thread scans the LDS copy)
    float m_tot = kNegBig;
    for (int s = lane; s < n_slots; s += 64) {
        if (!live_slot(s)) continue;
        const f4 r = s_rec[s];
        if (r[1] > 0.f) m_tot = fmaxf(m_tot, r[0]);
    }
    m_tot = fmaxf(m_tot, lane_xor<1>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<2>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<4>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<8>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<16>(m_tot, lane));
    m_tot = fmaxf(m_tot, lane_xor<32>(m_tot, lane));

    f4 v = {0.f, 0.f, 0.f, 0.f};
    float l_part = 0.f;
    for (int first = 0;;) {
#pragma unroll
        for (int k = 0; k < kMergeMaxPerGroup; ++k) {
            const int s = first + grp + k * GROUPS;
            if (s < n_slots && live_slot(s)) {
                const f4 r = s_rec[s];
                if (r[1] > 0.f) {
                    const float w = __builtin_amdgcn_exp2f(r[0] - m_tot);
                    l_part += r[1] * w;
                    v += a[k] * w;
                }
            }
        }
        first += kMergeMaxPerGroup * GROUPS;
        if (GROUPS == kMergeGroups || first >= n_slots) break;
        load_slices(first);
    }
    s_acc[grp][lane] = v;
    if (lane == 0) s_red[grp] = l_part;
    __syncthreads();
    if (grp != 0) return;
    float l_tot = 0.f;
    f4 tot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < GROUPS; ++k) {
        tot += s_acc[k][lane];
        l_tot += s_red[k];
    }
    const float inv = l_tot > 0.f ? out_scale / l_tot : 0.f;
    float o[4] = {tot[0] * inv, tot[1] * inv, tot[2] * inv, tot[3] * inv};
    if (rotate) {
        wht256_wave(o, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * lane + k);
    }
    store_out_row<TQ, HD>(P, row, lane, o, g);
}

// The same for rows of at most SLOTS chunks: one wave per row, which holds all of its records' slices; the records reach the other lanes
// through scalar registers, no LDS and no barrier.
template <typename TQ, int HD, int SLOTS, int ORDER>
__global__ __launch_bounds__(64) void split_merge_few_kernel(const float* part_acc_in, const float* part_ml_in, int max_chunks_in,
                                                             int num_q_heads_in, const int32_t* query_start_loc, const uint16_t* gate,
                                                             int num_reqs, const AttnParams P, float out_scale, int rotate) {
    static_assert(SLOTS <= 64, "one record per lane");
    const int lane = (int)threadIdx.x;
    const int tok = (int)blockIdx.y;
    const warp34_attention_batch& B = P.B;
    const size_t row = (size_t)tok * num_q_heads_in + blockIdx.x;
    const float* ml = part_ml_in + row * max_chunks_in * 4;
    const float* acc = part_acc_in + row * max_chunks_in * kHeadDim;
    f4 rec = {kNegBig, 0.f, 0.f, 0.f};
    if (lane < max_chunks_in) rec = *reinterpret_cast<const f4*>(ml + 4 * lane);
    f4 a[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        a[s] = f4{0.f, 0.f, 0.f, 0.f};
        if (s < max_chunks_in && (HD == 256 || 4 * lane < HD)) a[s] = *reinterpret_cast<const f4*>(acc + (size_t)s * kHeadDim + 4 * lane);
    }
    const RowOwner owner(query_start_loc, num_reqs, lane);
    const uint2 g = load_out_gate<HD>(gate, row, lane);
    asm volatile("" ::"s"(P.out), "s"(P.gate), "s"(out_scale), "s"(rotate));  // (on their way beside the slices, not where they are used)
    if (!owner.live(B, tok, lane)) return;  // masked row: output untouched
    const int n_chunks = min((int)__int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(rec[2]))), max_chunks_in);
    float l_tot;
    const f4 tot = merge_slices<SLOTS, ORDER>(rec, n_chunks, a, lane, l_tot);
    const float inv = l_tot > 0.f ? out_scale / l_tot : 0.f;
    float o[4] = {tot[0] * inv, tot[1] * inv, tot[2] * inv, tot[3] * inv};
    if (rotate) {
        wht256_wave(o, lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = apply_sign(o[k], 4 * lane + k);
    }
    store_out_row<TQ, HD>(P, row, lane, o, g);
}

}  // namespace w34

#include "paged_attn_rows.h"
#include "paged_prefill_tq4.h"
#include "paged_prefill_wide.h"
#include "qsa_sparse_tq4.h"
#include "qsa_sparse_rows.h"

namespace w34 {

// ---- host side ---------------------------------------------------------------------------------
constexpr int kMaxChunksCap = 256;
// Cost of starting a piece of a balanced batch, in units of streaming: TQ4 builds its table and
// rotates the queries first.
constexpr int kTq4PieceCost = 32;
constexpr int kRowsPieceCost = 16;
// Smallest piece where a request has several tiles or column tiles and the batch is no short one (bal_short_piece).
// It counts where few keys meet many shares: Q8_0, 100 requests x 4 tokens on 200 keys 29.5 us with 4, 32.1 with 8, 36.7
// with 16; rotated Q8_0, 5 x 4 on 600 keys 14.9, 17.0, 17.3.  On longer contexts the same.
constexpr int kMinUnitsPerWidePiece = 4;
// A batch whose requests have several tiles goes to the chunk grid instead while it has no more 16-column
// tiles than this per kv head: the plan, the table and the merge launch cost 1 to 2 us of a call.  Layer steps over
// Q8_0 pages (contexts from a third of the length up), chunk grid against plan, us: 4 requests x 4 tokens (8 tiles) on
// 2000 keys 23.4 against 24.1, on 16000 32.5 against 34.5; 5 x 4 (10 tiles) on 2000 23.6 against 24.3, on 19000 37.6
// against 37.2; 12 x 4 on 800 23.8 against 24.4; 16 x 4 on 3000 31.6 against 31.4; 30 x 4 on 2000 38.9 against 39.7.  The
// line lies where the longest contexts turn (attention alone, 10 x 4 on 3K to 16K 54 against 35, 20 x 4 93 against 53).
// (Counts of tiles, not lengths: results do not depend on max_seq_len.)
// At head dimension 128 every such batch goes there: the plan has one column tile at that size (with two the merge of
// the waves outweighs the keys read once more) and is nowhere ahead.  Draft blocks, layer steps, contexts from an eighth of the length
// up: 3 x 8 on 2000 keys 16.2 against 19.8, 4 x 16 on 9000 24.3 against 34.2, 12 x 8 on 8000 32.9 against 44.6, 9 x 16 on 16000 69.6
// against 103, 16 x 16 99 against 174; 8 x 16 on 6000 each 45.7 against 51.1.
constexpr int kRowsGridTiles = 8;
// A decode batch at head dimension 128 (four q heads per kv head) goes to the chunk grid up to this many requests.
// Chunk grid against plan, four kv heads, us: 2 requests of 1000 keys 10.2 against 13.0, of 3K to 16K 11.6 against 15.0, of 5K to
// 60K 24.2 against 24.4; 3 requests 10.5 against 13.3, 17.9 against 20.7, 41 against 35; 4 requests 11.8 against 13.5, 24.1
// against 23.2, 59 against 45; 6 requests 11.7 against 13.6, 38 against 29.
// (Those with one workgroup per CU.  With two, layer steps: 2 requests of 1000 keys 14.5 against 19.3, of 3K to 16K 16.0 against 20.4, of 5K to
// 60K 25.1 against 25.1; 3 requests 14.7 against 19.5, 21.0 against 21.6, 40.4 against 37.0.)
constexpr int kRowsGridRequests128 = 3;
// Short batches (bal_short_piece): key and value rows of up to this many bytes per kv head, each counted once, for
// batches whose entries are cut into pieces of their own anyway and for others (whose workgroups mostly have
// two pieces).  Tiles of 16 against 32 columns, us: few entries, Q8_0 5 x 4 tokens on 800 to 8000 keys (12 MB) 21.2 against
// 22.0, 5 x 8 (24 MB) 27.4 against 25.0, bf16 10 x 4 on 2000 (21 MB) equal; others, Q8_0 20 x 4 on 2000 (22 MB) 26.7
// against 29.4, 32 x 4 on 300 to 3000 (29 MB) 36.6 against 32.9, bf16 20 x 4 on 1000 (21 MB) 24.4 against 29.5, on 300 to 3000
// (34 MB) 34.5 against 31.4.
constexpr int kShortBytesFew = 16 << 20;
constexpr int kShortBytes = 24 << 20;
constexpr int kShortMaxEntries = 128;  // of 16 columns: two per lane
// Up to here the chunk grid has one chunk per tile and its merge is not launched; a short batch whose requests
// are no longer has one piece per tile of the same 16 columns, and the bits are the same (5 x 4 tokens on 200 keys:
// 11.4 against 13.6 us).
constexpr int kShortGridKeys = (kMinUnitsPerChunk - 1) * kUnit;
// The most units that 64 entries of kShortGridKeys have make a short batch in every format.
static_assert(kShortMaxEntries / 2 * (kMinUnitsPerChunk - 1) <= kShortBytes / (64 * 2 * kHeadDim) &&
                  16 * (kMinUnitsPerChunk - 1) <= kShortBytesFew / (64 * 2 * kHeadDim),
              "the chunk grid stands in for short batches only");
static size_t partial_bytes(long long rows, int max_chunks) {
    return (size_t)rows * (size_t)max_chunks * (kHeadDim + 4) * sizeof(float);
}

// Cap on chunks per tile: a function of total_tokens (tiles), gqa (q subgroups per kv head) and, with too little of it, the scratch and
// the heads.  Then as many as it holds and the chip takes in one round (two kv heads: all), so that scratch for n chunks gives n, or the
// target halved until it fits.  us, scratch by the size query, halved / now: one token of 16 + 2 heads, 1 200 keys, TQ4 13.3 / 11.2 (eight of ten chunks), Q8_0
// 12.4 / 10.7, 10 000 keys TQ4 15.2 / 12.9 (64 of 79).  What halving is for: 8 MiB, 4 tokens of 32 + 4 heads on 32 000 keys, 63 chunks / 32: TQ4 35.6 / 26.8,
// Q8_0 35.6 / 28.6; 64 + 8 heads, 31 / 16: 48.6 / 36.0.
static long long one_round(long long tiles, int kv_subs) { return 2 * kTargetWorkgroupsPerHead / (tiles * kv_subs); }
static int chunk_target(long long tiles, int q_subgroups) {
    return (int)std::min<long long>(kMaxChunksCap, kTargetWorkgroupsPerHead / (std::max(tiles, 1ll) * std::max(q_subgroups, 1)));
}
static int choose_max_chunks(const warp34_exec* ex, int total_tokens, int num_q_heads, int tok_tile, int q_subgroups, int kv_subs) {
    if (ex->scratch_ptr == 0 || (ex->scratch_ptr & 15u) != 0u) return 1;
    const int tiles = (total_tokens + tok_tile - 1) / tok_tile;
    int want = chunk_target(tiles, q_subgroups);
    if (want < 2) return 1;
    const size_t one = partial_bytes((long long)total_tokens * num_q_heads, 1);
    if (one > 0 && ex->scratch_size / one < (size_t)want) {
        const int fit = (int)(ex->scratch_size / one);
        while (want > fit) want >>= 1;
        want = std::max(want, (int)std::min<long long>(fit, one_round(tiles, kv_subs)));
    }
    return want < 2 ? 1 : want;
}

// One attribute call per kernel instantiation and device.  The record is process-wide and
// lock-free: slot i belongs to the first kernel that claims it, bit d of its mask says that
// device d is configured.  Kernels that address their dequantisation table absolutely
// (lds_base_zero) also have their static LDS size checked here: it must be zero, so that the
// dynamic block starts at LDS address 0.
constexpr int kLdsRecordSlots = 128;
static std::atomic<const void*> g_lds_fn[kLdsRecordSlots];
static std::atomic<unsigned long long> g_lds_devs[kLdsRecordSlots];

template <typename KernelT>
static int ensure_dynamic_lds(KernelT kernel, int bytes, bool lds_base_zero = false) {
    int dev = 0;
    hipError_t rc = hipGetDevice(&dev);
    if (rc != hipSuccess) return (int)rc;
    const void* fn = (const void*)kernel;
    int slot = -1;
    for (int i = 0; i < kLdsRecordSlots; ++i) {
        const void* cur = g_lds_fn[i].load(std::memory_order_acquire);
        if (cur == nullptr) {
            const void* expect = nullptr;
            if (g_lds_fn[i].compare_exchange_strong(expect, fn, std::memory_order_acq_rel)) cur = fn;
            else cur = expect;
        }
        if (cur == fn) {
            slot = i;
            break;
        }
    }
    const bool tracked = slot >= 0 && dev >= 0 && dev < 64;
    if (tracked && ((g_lds_devs[slot].load(std::memory_order_acquire) >> dev) & 1ull)) return 0;
    if (lds_base_zero) {
        hipFuncAttributes attr;
        rc = hipFuncGetAttributes(&attr, fn);
        if (rc != hipSuccess) return (int)rc;
        if (attr.sharedSizeBytes != 0) return (int)hipErrorInvalidConfiguration;
    }
    rc = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (rc != hipSuccess) return (int)rc;
    if (tracked) g_lds_devs[slot].fetch_or(1ull << dev, std::memory_order_release);
    return 0;
}

// Decode batches of several requests take the balanced path: no request has more than one
// tile, no window, no token mask (the plan counts units of [0, last key]), usable scratch.
static bool balanced_decode_applicable(const warp34_exec* ex, const warp34_attention_batch* batch,
                                       int tiles_by_request, int force_single) {
    return tiles_by_request && batch->num_reqs >= 2 && !force_single && batch->sliding_window <= 0 &&
           batch->valid_token_mask == nullptr && batch->total_tokens <= 65535 && ex->scratch_ptr != 0 && (ex->scratch_ptr & 15u) == 0u;
}
// The chunk grid's cap on chunks per request of a decode batch that it may serve in the plan's place (grid_decode_serves): one round of
// workgroups; 0: not such a batch.
static int decode_grid_chunks(const warp34_exec* ex, const warp34_attention_batch* batch, int num_q_heads, int q_subgroups) {
    if (q_subgroups != 1 || batch->num_reqs < 2 || batch->num_reqs > kGridDecodeReqs) return 0;
    const int chunks = kTargetWorkgroupsPerHead / batch->num_reqs;
    return partial_bytes((long long)batch->total_tokens * num_q_heads, chunks) <= ex->scratch_size ? chunks : 0;
}
static bool decode_on_grid(const warp34_attention_batch* batch, int chunks, int many) {
    return chunks > 0 && batch->max_seq_len > 0 &&
           grid_decode_serves(((long long)batch->max_seq_len + kUnit - 1) / kUnit, batch->num_reqs, chunks, many);
}
// shares of a balanced decode batch per (kv head, q subgroup): a function of gqa only
static int balanced_groups(int q_subgroups) {
    int groups = kTargetWorkgroupsPerHead / (q_subgroups > 0 ? q_subgroups : 1);
    if (groups > kMergeGroups * kMergeMaxPerGroup - 1) groups = kMergeGroups * kMergeMaxPerGroup - 1;
    return groups < 1 ? 1 : groups;
}

// Entries that are cut into pieces of their own, see the plan.  Up to one entry per eight workgroups:
// five requests of 3K to 21K keys (10 entries on 128) 29.7 -> 28.7 us; 32 requests of 1K to 64K keys
// 136 -> 149 us, they keep the shares that cross boundaries.
static int balanced_aligned(long long entries, int groups) {
    return entries <= 64 && entries * 8 <= groups ? 1 : 0;
}

// The second launch of a split batch: one workgroup per row.  Sixteen waves per row have all partials of
// a long sequence in flight at once; from 32 rows per kv head on the workgroups are many and the
// partials of a row few, and four waves per row start sooner (two kv heads, 80 rows of 25 partials: 6.9 ->
// 5.2 us; 512 rows: 8.9 -> 5.8; four kv heads, 1 024 rows of ten: 11.5 -> 4.9; but 16 rows of 128
// partials: 5.2 -> 6.8).  At the line, one request of 4 tokens (32 rows): 64 partials, 32 768 keys, whole call 23.2 us with
// sixteen waves, 23.6 with four; 6 partials, 1500 keys, 16.9 and 16.7.  24 rows of 64 partials: 21.3 and 21.7; 64 rows of 32:
// 28.4 and 28.4.  Rows per kv head, not rows: a rank with one kv head adds in the same order.
static bool merge_small_groups(const AttnParams& P) { return (long long)P.B.total_tokens * P.gqa >= 32; }

template <typename TQ, int HD>
static int launch_balanced_merge(const AttnParams& P, int kv_subs, float out_scale, hipStream_t stream) {
    const dim3 grid((unsigned)P.num_q_heads, (unsigned)P.B.total_tokens);
    const int groups = merge_small_groups(P) ? 4 : kMergeGroups;
    const auto kernel = groups == 4 ? balanced_merge_kernel<TQ, HD, 4> : balanced_merge_kernel<TQ, HD, kMergeGroups>;
    hipLaunchKernelGGL(kernel, grid, dim3((unsigned)groups * 64), 0, stream, (const int32_t*)P.bal_table, (const float*)P.part_acc,
                       (const float*)P.part_ml, P.num_q_heads, P.q_group, kv_subs, P.bal_cols, P.gate, P, out_scale, P.rot_out);
    return (int)hipGetLastError();
}

template <typename TQ, bool SP, int HD>
static int launch_split_merge(const AttnParams& P, int slots, float out_scale, hipStream_t stream) {
    const dim3 grid((unsigned)P.num_q_heads, (unsigned)P.B.total_tokens);
    if constexpr (!SP) {
        const auto few = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(64), 0, stream, (const float*)P.part_acc, (const float*)P.part_ml, slots, P.num_q_heads,
                               P.B.query_start_loc, P.gate, P.B.num_reqs, P, out_scale, P.rot_out);
            return (int)hipGetLastError();
        };
        if (slots <= (merge_small_groups(P) ? kMergeFewRows : kMergeFew)) {
            if (merge_small_groups(P))
                return slots <= 8           ? few(split_merge_few_kernel<TQ, HD, 8, 4>)
                       : slots <= kMergeFew ? few(split_merge_few_kernel<TQ, HD, kMergeFew, 4>)
                                            : few(split_merge_few_kernel<TQ, HD, kMergeFewRows, 4>);
            return slots <= 8 ? few(split_merge_few_kernel<TQ, HD, 8, kMergeGroups>)
                              : few(split_merge_few_kernel<TQ, HD, kMergeFew, kMergeGroups>);
        }
    }
    if (merge_small_groups(P)) {
        hipLaunchKernelGGL((split_merge_kernel<TQ, SP, HD, 4>), grid, dim3(4 * 64), 0, stream, (const float*)P.part_acc,
                           (const float*)P.part_ml, slots, P.num_q_heads, P.B.query_start_loc, P.gate, P.B.num_reqs, P, out_scale, P.rot_out);
    } else {
        hipLaunchKernelGGL((split_merge_kernel<TQ, SP, HD, kMergeGroups>), grid, dim3(kMergeGroups * 64), 0, stream,
                           (const float*)P.part_acc, (const float*)P.part_ml, slots, P.num_q_heads, P.B.query_start_loc, P.gate, P.B.num_reqs, P,
                           out_scale, P.rot_out);
    }
    return (int)hipGetLastError();
}

// Tiles of a request, and of the batch, at most: the grid's z.  sum_r ceil(q_r / tok_tile) is bounded by
// total_tokens / tok_tile + num_reqs and by what num_reqs requests of max_q_len tokens have.  The workgroups of tiles that
// do not exist come behind the real ones, which fill the chip: a round of their own.  us, the first bound alone / both: TQ4, 4
// tokens each, 1 request on 16 000 keys 21.2 / 19.8, 4 on 4 000 20.6 / 19.1, 8 on 8 000 28.2 / 26.8.
static int tiles_per_request_bound(const warp34_attention_batch& B, const AttnParams& P) {
    return B.max_q_len > 0 ? (int)(((long long)B.max_q_len + P.tok_tile - 1) / P.tok_tile) : 1;
}
static int tiles_bound(const warp34_attention_batch& B, const AttnParams& P) {
    if (P.tiles_by_request) return B.num_reqs;
    const long long by_tokens = (long long)(B.total_tokens / P.tok_tile) + B.num_reqs;
    const long long by_requests = (long long)B.num_reqs * tiles_per_request_bound(B, P);
    return (int)(B.max_q_len > 0 && by_requests < by_tokens ? by_requests : by_tokens);
}

// P.spec_* = chunk_geom(0, max_seq_len - 1, P.max_chunks, P.few_chunks), worked out on the host
static void fill_spec_geometry(AttnParams& P, int max_seq_len) {
    if (max_seq_len <= 0) return;
    P.spec_units = ((max_seq_len - 1) >> 5) + 1;
    int nc = chunk_count(P.spec_units, P.few_chunks);
    if (nc > P.max_chunks) nc = P.max_chunks;
    if (nc < 1) nc = 1;
    P.spec_upc = (P.spec_units + nc - 1) / nc;
    if (P.spec_upc < 1) P.spec_upc = 1;
    P.spec_chunks = (P.spec_units + P.spec_upc - 1) / P.spec_upc;
    if (P.spec_chunks < 1) P.spec_chunks = 1;
}

// ---- shared-prefix pass (verify batches whose requests share their leading pages) ----
// The host cannot see the block tables, so a one-workgroup kernel finds the common leading run:
// the pages that every request's block table holds at the same index and that lie below every
// request's first query position (every query of the batch sees all of their keys).  It leaves
// the length in tokens (a multiple of the unit; 0 below kSpMinTokens) and the descriptor of one
// pseudo request -- all query tokens of the batch over exactly those keys -- in the header (SpHeader).
constexpr int kSpMinTokens = 4096;
// Units behind the prefix, counted once per column tile pair, from which on the private rest is for two column tiles.  A key is looked up once for both, but
// the four columns of a wave are added up and joined to the records one after the other: about 6 us a call, which a short rest does not earn back.
// Counted on the device from the lengths themselves, and not by the kv heads that a rank holds, so that results depend on neither the bounds nor
// the sharding.  us a call, two kv heads of 8 query heads, one tile / two: 4 tokens each, 16 requests with 2 976 units in all 116.3 / 122.9, 8 with
// 5 008 108.7 / 111.9, 4 with 7 680 84.1 / 81.8, 16 with 9 984 128.7 / 122.5; 8 requests of 8 tokens with 2 752 149.1 / 149.1, with 7 744 158.7 / 153.1.
// What other numbers of kv heads give up for that: one, 8 x 4 tokens with 5 008 103.9 / 99.4; four, 6 x 4 with 1 872 118.8 / 126.9, 12 x 4 with 3 744 201.8 / 197.0.
constexpr int kWidePrivateUnits = 6144;

// wide_tok_tile: tokens of two column tiles
__global__ __launch_bounds__(1024) void shared_prefix_probe_kernel(const warp34_attention_batch B, int block_size, int wide_tok_tile,
                                                                   SpHeader* hdr) {
    __shared__ int s_first_diff, s_min_ctx, s_private;
    const int tid = (int)threadIdx.x;
    if (tid == 0) {
        s_first_diff = B.max_blocks_per_req;
        s_min_ctx = 0x7fffffff;
        s_private = 0;
    }
    __syncthreads();
    const auto tokens_of = [&](int r) { return B.query_start_loc[r + 1] - B.query_start_loc[r]; };
    const auto context_of = [&](int r, int q_len) { return B.context_lens_before != nullptr ? B.context_lens_before[r] : B.seq_lens_after[r] - q_len; };
    int my_q = 0, my_ctx = 0;  // of request tid
    for (int r = tid; r < B.num_reqs; r += 1024) {
        const int q_len = tokens_of(r), ctx = context_of(r, q_len);
        atomicMin(&s_min_ctx, ctx < 0 ? 0 : ctx);
        if (r == tid) my_q = q_len, my_ctx = ctx;
    }
    __syncthreads();
    int max_pages = s_min_ctx / block_size;  // pages that lie entirely below every first query position
    if (max_pages > B.max_blocks_per_req) max_pages = B.max_blocks_per_req;
    // one request per wave (r = 1 + wave, + 16, ...), sixteen pages per lane and round trip: the
    // loads of a batch are independent of each other
    const int wave = tid >> 6, lane = tid & 63;
    int first_diff = 0x7fffffff;
    for (int r = 1 + wave; r < B.num_reqs; r += 16) {
        const int32_t* row = B.block_tables + (size_t)r * B.max_blocks_per_req;
        for (int base = lane; base < max_pages; base += 16 * 64) {
            int32_t mine[16], ref[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int p = base + 64 * k;
                const int pc = p < max_pages ? p : 0;
                mine[k] = row[pc];
                ref[k] = B.block_tables[pc];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int p = base + 64 * k;
                if (p < max_pages && mine[k] != ref[k] && p < first_diff) first_diff = p;
            }
        }
    }
    if (first_diff != 0x7fffffff) atomicMin(&s_first_diff, first_diff);
    __syncthreads();
    const int pages = s_first_diff < max_pages ? s_first_diff : max_pages;
    int floor = (pages * block_size) & ~(kUnit - 1);
    if (floor < kSpMinTokens) floor = 0;
    // units behind the prefix, one column tile pair's by one
    int units = 0;
    for (int r = tid; r < B.num_reqs; r += 1024) {
        const int q_len = r == tid ? my_q : tokens_of(r), ctx = r == tid ? my_ctx : context_of(r, q_len);
        const long long mine = (long long)((q_len + wide_tok_tile - 1) / wide_tok_tile) * (((ctx + q_len - 1) >> 5) - (floor >> 5) + 1);
        units = (int)min((long long)kWidePrivateUnits, units + (q_len > 0 && mine > 0 ? mine : 0ll));
    }
    if (units > 0) atomicAdd(&s_private, units);
    __syncthreads();
    if (tid == 0) {
        hdr->wide = floor != 0 && s_private >= kWidePrivateUnits ? 1 : 0;
        hdr->floor = floor;
        hdr->qsl[0] = 0;
        hdr->qsl[1] = B.total_tokens;
        hdr->seq = floor;
        hdr->ctx = floor;
    }
}

// Batches that may take the pass: several requests, a few query tokens each (a verify step),
// long contexts, plain causal masking.  (Decode batches keep the balanced shares; the pass costs
// two small launches and wide partial records when nothing is shared.)
static bool shared_prefix_applicable(const warp34_attention_batch* b, int q_group, int force_single) {
    return !force_single && b->num_reqs >= 4 && b->max_q_len >= 2 && b->max_q_len <= kPfRows / q_group &&
           b->total_tokens >= 16 && b->max_seq_len >= 8 * kSpMinTokens && b->sliding_window <= 0 &&
           b->mask_mode == WARP34_ATTN_MASK_CAUSAL && b->valid_token_mask == nullptr && b->valid_req_mask == nullptr &&
           b->context_lens_before != nullptr && (q_group & (q_group - 1)) == 0;
}
// parts of the prefix per tile: a function of the batch and of gqa only, never of the number of
// local kv heads (a rank with one kv head must produce the bits of a rank with two)
static int shared_prefix_parts(int total_tokens, int q_group, int q_subgroups) {
    const int tiles = (total_tokens + kPfRows / q_group - 1) / (kPfRows / q_group) * q_subgroups;
    int parts = (kTargetWorkgroupsPerHead + tiles - 1) / tiles;  // about one workgroup per CU at two kv heads
    return parts < 1 ? 1 : (parts > 32 ? 32 : parts);
}

// Batches for the kernels that know this of them.
static bool plain_batch(const AttnParams& P) {
    const warp34_attention_batch& B = P.B;
    return P.q_subgroups == 1 && B.max_seq_len > 0 && B.sliding_window <= 0 && B.valid_token_mask == nullptr && B.valid_req_mask == nullptr &&
           B.context_lens_before != nullptr && P.L.k_page_stride_bytes <= 0xFFFFFFFFull && P.L.v_page_stride_bytes <= 0xFFFFFFFFull;
}
static bool plain_decode(const AttnParams& P) {
    return plain_batch(P) && P.tiles_by_request != 0 && P.B.max_q_len * P.q_group <= 8 && P.B.mask_mode == WARP34_ATTN_MASK_CAUSAL;
}
// Row formats: 8-bit rows, and 16-bit rows of several tiles per request (one tile: within 1 %, the rows themselves are what takes the time).  us, general / plain: eight layers
// of one token on 1 200 keys Q8_0 116.0 / 110.9, FP8 119.2 / 113.4, with their producers; four requests of 1 000 to 3 000 Q8_0 93.4 / 86.6; one token on 20 000 Q8_0
// 120.9 / 113.6; 4 tokens on 2 000 Q8_0 127.8 / 121.1; five layers of 4 x 16 draft tokens 115.3 / 114.2.
static bool plain_rows(const AttnParams& P) { return plain_batch(P) && P.key_groups == 0 && P.first_round == 0 && P.rot_q == 0; }

template <typename TQ>
static int launch_tq4(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                      const warp34_attention_batch* batch, const void* q, void* out, int num_q_heads,
                      int force_single, const void* gate) {
    AttnParams P{};
    P.L = *layout;
    P.B = *batch;
    P.block_magic = block_magic_for(layout->block_size);
    P.q = (const uint16_t*)q;
    P.out = (uint16_t*)out;
    P.gate = (const uint16_t*)gate;
    P.rot_q = layout->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    P.rot_out = layout->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    P.num_q_heads = num_q_heads;
    P.gqa = num_q_heads / layout->local_kv_heads;
    int q_group = P.gqa;
    if (q_group > 16) {
        for (int d = 16; d >= 1; --d)
            if (P.gqa % d == 0) {
                q_group = d;
                break;
            }
    }
    P.q_group = q_group;
    P.q_group_magic = q_group_magic_for(q_group);
    P.q_subgroups = P.gqa / q_group;
    // One column tile (16 query columns) per workgroup; two behind a shared prefix (paged_attn_tq4_private_kernel).
    P.tok_tile = 16 / q_group;
    if (P.tok_tile < 1) P.tok_tile = 1;
    P.unit_in_page = (layout->block_size % kUnit == 0 && layout->k_page_stride_bytes <= 0xFFFFFFFFull &&
                      layout->v_page_stride_bytes <= 0xFFFFFFFFull)
                         ? 1
                         : 0;
    P.tiles_by_request = (batch->max_q_len > 0 && batch->max_q_len <= P.tok_tile) ? 1 : 0;
    const int kv_subs = layout->local_kv_heads * P.q_subgroups;
    // decode batches: the plan's records and table fit
    const int plan_groups = balanced_groups(P.q_subgroups);
    const size_t plan_rows = bal_partial_row(plan_groups + batch->num_reqs, kv_subs, 0, 16, 0);
    const bool plan = balanced_decode_applicable(ex, batch, P.tiles_by_request, force_single) &&
                      partial_bytes((long long)plan_rows, 1) + (size_t)batch->total_tokens * 16 <= ex->scratch_size;
    const int decode_chunks = plan ? decode_grid_chunks(ex, batch, num_q_heads, P.q_subgroups) : 0;
    const bool on_grid = decode_on_grid(batch, decode_chunks, kGridUnitsTq4);
    P.max_chunks = force_single ? 1
                   : on_grid    ? decode_chunks
                                : choose_max_chunks(ex, batch->total_tokens, num_q_heads, P.tok_tile, P.q_subgroups, kv_subs);
    P.part_acc = nullptr;
    P.part_ml = nullptr;
    const long long rows = (long long)batch->total_tokens * num_q_heads;
    // grid.x: chunks that can exist given the host's upper bound on the sequence length
    const long long tok_tiles = ((long long)batch->total_tokens + P.tok_tile - 1) / P.tok_tile;
    P.few_chunks = few_chunks_of(kFewChunksTq4, on_grid ? decode_chunks : chunk_target(tok_tiles, P.q_subgroups));
    int grid_x = P.max_chunks;
    if (batch->max_seq_len > 0) {
        const int units = (batch->max_seq_len + kUnit - 1) / kUnit + 1;
        const int bound = chunk_count(units, P.few_chunks);
        if (bound < grid_x) grid_x = bound < 1 ? 1 : bound;
    }
    // No tile has more chunks than that: the cap is lowered to it, which changes no chunk (a
    // tile's count is limited by its own units first) and keeps the partial records, and what
    // the merge kernel loads ahead of knowing the count, as small as the bound allows.
    P.max_chunks = grid_x;
    P.part_stride = grid_x;
    fill_spec_geometry(P, batch->max_seq_len);
    if (P.max_chunks > 1) {
        uint8_t* ws = reinterpret_cast<uint8_t*>((uintptr_t)ex->scratch_ptr);
        P.part_acc = reinterpret_cast<float*>(ws);
        P.part_ml = P.part_acc + (size_t)rows * P.max_chunks * kHeadDim;
    }
    const int grid_z = tiles_bound(*batch, P);
    const dim3 grid((unsigned)grid_x, (unsigned)kv_subs, (unsigned)grid_z);
    hipStream_t stream = (hipStream_t)ex->stream;
    int rc;
    // Verify batches: the keys every request has in common go through the tile kernel once, for
    // all query rows of the batch (its dequantisation is shared by 128 rows instead of 16); the
    // decode kernel takes the private rest, the merge kernel both sets of partial records.
    if (P.max_chunks > 1 && shared_prefix_applicable(batch, q_group, force_single)) {
        const int parts = shared_prefix_parts(batch->total_tokens, q_group, P.q_subgroups);
        const int stride = P.max_chunks + parts;
        const size_t need = partial_bytes(rows, stride) + sizeof(SpHeader);
        if (stride <= kMergeGroups * kMergeMaxPerGroup && need <= ex->scratch_size) {
            P.part_stride = stride;
            P.pf_split = parts;
            P.pf_slot_base = P.max_chunks;
            P.bal_tiles = tiles_per_request_bound(*batch, P);
            P.part_ml = P.part_acc + (size_t)rows * stride * kHeadDim;
            SpHeader* hdr = reinterpret_cast<SpHeader*>(P.part_ml + (size_t)rows * stride * 4);
            P.key_floor = &hdr->floor;
            hipLaunchKernelGGL(shared_prefix_probe_kernel, dim3(1), dim3(1024), 0, stream, *batch, layout->block_size, 32 / q_group, hdr);
            rc = (int)hipGetLastError();
            if (rc) return rc;
            AttnParams T = P;  // the pseudo request of the header, 128-row tiles
            T.B.num_reqs = 1;
            T.B.query_start_loc = hdr->qsl;
            T.B.seq_lens_after = &hdr->seq;
            T.B.context_lens_before = &hdr->ctx;
            T.B.max_q_len = batch->total_tokens;
            T.tok_tile = kPfRows / q_group;
            T.key_floor = nullptr;
            const int pf_tiles = (batch->total_tokens + T.tok_tile - 1) / T.tok_tile;
            rc = ensure_dynamic_lds(paged_prefill_tq4_kernel<TQ, true>, kPfSmem, true);
            if (rc) return rc;
            hipLaunchKernelGGL((paged_prefill_tq4_kernel<TQ, true>),
                               dim3((unsigned)(pf_tiles * parts), (unsigned)kv_subs, 1u), dim3(12 * 64), kPfSmem,
                               stream, T);
            rc = (int)hipGetLastError();
            if (rc) return rc;
            // More than a column tile per request: by the number of tokens, not by the bound on a request's, on which no result may depend.  (q_group
            // is a power of two, see shared_prefix_applicable: a tile holds whole tokens.)
            if ((long long)batch->total_tokens * q_group > 16ll * batch->num_reqs) {
                AttnParams W = P;
                W.tok_tile = 32 / q_group;
                W.tiles_by_request = batch->max_q_len <= W.tok_tile ? 1 : 0;
                W.bal_tiles = tiles_per_request_bound(*batch, W);
                // a chunk joins the record of the prefix's part with its number
                W.max_chunks = std::max(1, std::min(parts, chunk_target(((long long)batch->total_tokens + W.tok_tile - 1) / W.tok_tile, W.q_subgroups)));
                const int tiles = tiles_bound(*batch, W);
                rc = ensure_dynamic_lds(paged_attn_tq4_private_kernel<TQ>, smem_bytes_for(2), true);
                if (rc) return rc;
                const long long wgs = std::max((long long)grid_x * grid_z, (long long)W.max_chunks * tiles);
                hipLaunchKernelGGL(paged_attn_tq4_private_kernel<TQ>, dim3((unsigned)wgs, (unsigned)kv_subs), dim3(kTq4Waves * 64),
                                   smem_bytes_for(2), stream, P, W, (const SpHeader*)hdr, grid_x, grid_z, W.max_chunks, tiles);
            } else {
                rc = ensure_dynamic_lds(paged_attn_tq4_kernel<TQ, true>, smem_bytes_for(1), true);
                if (rc) return rc;
                hipLaunchKernelGGL((paged_attn_tq4_kernel<TQ, true>), grid, dim3(kTq4Waves * 64), smem_bytes_for(1), stream, P);
            }
            rc = (int)hipGetLastError();
            if (rc) return rc;
            return launch_split_merge<TQ, true, kHeadDim>(P, stride, kLutInvGain, stream);
        }
    }
    // Decode batches of several requests: equal shares of the batch's units per workgroup
    // instead of per-request chunks (the requests' lengths are unknown to the host and differ).
    if (plan && !on_grid) {
        P.part_acc = reinterpret_cast<float*>((uintptr_t)ex->scratch_ptr);
        P.part_ml = P.part_acc + plan_rows * kHeadDim;
        P.bal_table = reinterpret_cast<int32_t*>(P.part_ml + plan_rows * 4);
        P.max_chunks = plan_groups + 1;
        P.bal_tiles = 1;
        P.bal_cols = 16;
        P.piece_cost = kTq4PieceCost;
        P.min_upc = kMinUnitsPerChunk;
        P.bal_aligned = balanced_aligned(batch->num_reqs, plan_groups);
        P.grid_chunks = decode_chunks;
        rc = ensure_dynamic_lds(paged_attn_tq4_balanced_kernel<TQ>, smem_bytes_for(1), true);
        if (rc) return rc;
        hipLaunchKernelGGL((paged_attn_tq4_balanced_kernel<TQ>), dim3((unsigned)plan_groups, (unsigned)kv_subs),
                           dim3(kTq4Waves * 64), smem_bytes_for(1), stream, P);
        rc = (int)hipGetLastError();
        if (rc) return rc;
        return launch_balanced_merge<TQ, kHeadDim>(P, kv_subs, kLutInvGain, stream);
    }
    P.bal_tiles = tiles_per_request_bound(*batch, P);
    const auto kernel = plain_decode(P) ? paged_attn_tq4_plain_kernel<TQ> : paged_attn_tq4_kernel<TQ>;
    rc = ensure_dynamic_lds(kernel, smem_bytes_for(1), true);
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, grid, dim3(kTq4Waves * 64), smem_bytes_for(1), stream, P);
    rc = (int)hipGetLastError();
    if (rc) return rc;
    return P.max_chunks > 1 ? launch_split_merge<TQ, false, kHeadDim>(P, P.max_chunks, kLutInvGain, stream) : 0;
}

// Most tiles per request that the balanced plan takes: with more, the 128-row tile kernel or one
// workgroup per tile is the better shape.
constexpr int kBalMaxTiles = 16;
// Column tiles per workgroup (nt) and tiles per request of a balanced batch over row-format pages whose
// requests have up to q_len query tokens; no tiles: the batch is not for the plan.  Two column tiles where a
// request has more than 16 query columns; rotated 8-bit values (a second value operand: accumulator
// registers) stay with one, and head dimension 128 takes the plan with one tile per request only.
struct BalShape {
    int nt, tok_tile, tiles;
};
static BalShape rows_balanced_shape(int num_reqs, int total_tokens, int q_len, int q_group, int q_subgroups, bool vres,
                                    int head_dim) {
    const BalShape none{0, 0, 0};
    if (num_reqs < 1 || q_len < 1 || total_tokens > 65535) return none;
    BalShape s;
    s.nt = (long long)q_len * q_group > 16 && !vres && head_dim == kHeadDim ? 2 : 1;
    s.tok_tile = 16 * s.nt / q_group;
    const long long tiles = ((long long)q_len + s.tok_tile - 1) / s.tok_tile;
    if (tiles > kBalMaxTiles || (num_reqs == 1 && s.nt == 1 && tiles == 1)) return none;
    s.tiles = (int)tiles;
    if (s.nt * s.tiles > 1) {
        const long long tiles16 = ((long long)total_tokens * q_group + 15) / 16 * q_subgroups;
        if (head_dim != kHeadDim || tiles16 <= kRowsGridTiles) return none;
    } else if (head_dim != kHeadDim && num_reqs <= kRowsGridRequests128) {
        return none;
    }
    return s;
}
// rotated 8-bit value rows
static bool rows_vres(const warp34_kv_layer_layout* l) {
    return (l->v_format == WARP34_KV_FORMAT_FP8_E4M3 || l->v_format == WARP34_KV_FORMAT_Q8_0) &&
           l->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256;
}

// Balanced decode / verify over row-format pages; -1: the batch is not for it.
template <typename TQ, int KVF, bool VRES, int HD>
static int launch_rows_balanced(const warp34_exec* ex, const warp34_attention_batch* batch, AttnParams P, int kv_subs,
                                int force_single, hipStream_t stream, int* grid_chunks) {
    if (force_single || batch->sliding_window > 0 || batch->valid_token_mask != nullptr || ex->scratch_ptr == 0 ||
        (ex->scratch_ptr & 15u) != 0u)
        return -1;
    const BalShape shape =
        rows_balanced_shape(batch->num_reqs, batch->total_tokens, batch->max_q_len, P.q_group, P.q_subgroups, VRES, HD);
    const int nt = shape.nt, tiles = shape.tiles;
    if (tiles < 1) return -1;
    P.tok_tile = shape.tok_tile;
    // Fewer shares where the scratch cannot hold the records of all of them, down to three quarters or to the
    // workgroups that the chunk grid would launch; with less room the chunk grid, whose workgroups grow with the
    // batch, leaves fewer compute units idle.  8 MiB, two kv heads, Q8_0, chunk grid against plan, us: 150 decode
    // requests (102 shares) of 1000 keys 45 against 46, of 1K to 9K 194 against 140; 175 (77 shares) 46 against 61, 202 against
    // 187; 200 (52 shares) 47 against 93, 226 against 296; 235 (17 shares) 54 against 308, 262 against 1046.  40 requests x 4
    // tokens (86 shares, 80 tiles) on 1000 keys 24 against 27, on 300 to 3000 49 against 40, on 800 to 8000 112 against 67;
    // 50 x 4 (76 shares, 100 tiles) on 1000 keys 25 against 38, on 300 to 3000 50 against 51; 60 x 4 (66 shares) 54 against 64.
    const long long entries = (long long)batch->num_reqs * tiles;
    const size_t slot_bytes = partial_bytes((long long)kv_subs * 16 * nt, 1), table_bytes = (size_t)batch->total_tokens * 16;
    if (ex->scratch_size < table_bytes) return -1;
    const long long room = (long long)((ex->scratch_size - table_bytes) / slot_bytes) - entries;
    const int all_groups = balanced_groups(P.q_subgroups);
    const int groups = (int)(room < all_groups ? room : all_groups);
    const int tok16 = 16 / P.q_group, tiles16 = (batch->max_q_len + tok16 - 1) / tok16;
    if (groups < 1 || (4 * groups < 3 * all_groups &&
                       groups < (long long)batch->num_reqs * tiles16 *
                                    choose_max_chunks(ex, batch->total_tokens, P.num_q_heads, tok16, P.q_subgroups, kv_subs)))
        return -1;
    const size_t prows = (size_t)(groups + entries) * kv_subs * 16 * nt;
    P.piece_cost = kRowsPieceCost;
    if (nt * tiles > 1) P.min_upc = kMinUnitsPerWidePiece;
    P.part_acc = reinterpret_cast<float*>((uintptr_t)ex->scratch_ptr);
    P.part_ml = P.part_acc + prows * kHeadDim;
    P.bal_table = reinterpret_cast<int32_t*>(P.part_ml + prows * 4);
    P.max_chunks = groups + 1;
    P.bal_tiles = tiles;
    P.bal_cols = 16 * nt;
    P.bal_aligned = balanced_aligned(entries, groups);
    P.short_units = -1;
    if (HD == kHeadDim && nt * tiles == 1 && groups == all_groups) {
        const int chunks = decode_grid_chunks(ex, batch, P.num_q_heads, P.q_subgroups);
        if (decode_on_grid(batch, chunks, kGridUnitsRows)) {
            *grid_chunks = chunks;
            return -1;
        }
        P.grid_chunks = chunks;
    }
    if (nt == 2 || (VRES && tiles > 1 && !P.bal_aligned)) {
        if (entries <= kShortMaxEntries / 2 && (long long)batch->num_reqs * tiles16 <= std::min(groups, kShortMaxEntries)) {
            // (no entry has two pieces, on either path one workgroup does the same arithmetic: launch shape only)
            if (batch->max_seq_len > 0 && batch->max_seq_len <= kShortGridKeys) return -1;
            P.short_units = (P.bal_aligned ? kShortBytesFew : kShortBytes) / (4 * RowsLds<KVF, HD>::kHalf);
            P.short_tiles = tiles16;
            P.short_tok_tile = tok16;
        }
    }
    const auto launch = [&](auto column_tiles) -> int {
        constexpr int NT = decltype(column_tiles)::value;
        constexpr int smem = rows_smem_bytes<KVF, HD>(NT);
        // every key is read by one workgroup only when no request has two tiles: streaming loads
        const auto kernel = tiles == 1 && P.q_subgroups == 1 ? paged_attn_rows_balanced_kernel<TQ, NT, KVF, VRES, true, HD>
                                                             : paged_attn_rows_balanced_kernel<TQ, NT, KVF, VRES, false, HD>;
        int rc = ensure_dynamic_lds(kernel, smem, true);
        if (rc) return rc;
        hipLaunchKernelGGL(kernel, dim3((unsigned)groups, (unsigned)kv_subs), dim3(kKv16Waves * 64), smem, stream, P);
        rc = (int)hipGetLastError();
        if (rc) return rc;
        return launch_balanced_merge<TQ, HD>(P, kv_subs, 1.0f, stream);
    };
    if constexpr (!VRES && HD == kHeadDim) {
        if (nt == 2) return launch(std::integral_constant<int, 2>{});
    }
    return launch(std::integral_constant<int, 1>{});
}

// Groups of keys (request x kv head x chunk) of a chunk grid whose workgroups go by them (rows_by_keys), 0: in launch order, chunk by
// chunk, head by head, tile by tile.  Launch order puts the tiles of a request on one XCD where a tile's workgroups are a multiple of
// eight; else two or more XCDs fetch the same keys, and two workgroups on a CU wait for them together.  us a layer step, launch order /
// by groups, bf16 draft blocks (four kv heads), contexts from an eighth of the length up: 9 x 16 tokens (3 chunks) on 16 000 keys 82.3 /
// 65.7, 9 x 8 (7) 64.6 / 46.4, 12 x 8 (5) 85.4 / 58.5, on 6 000 42.2 / 31.8; head dimension 256, 3 x 4 (21) on 3 000 to 16 000, bf16 24.8 /
// 20.0, Q8_0 26.2 / 24.9, 1 x 4 (63) on 16 000 20.2 / 16.8.  Where launch order does as well the arithmetic costs 0.1 to 0.3 (4 x 16 on
// 2 000 keys, 8 chunks, 17.6 / 17.9), and with fewer than kKeyGroupsFrom workgroups there is nothing to gain (Q8_0, 3 x 4: 132 of them, on
// 2 900 keys, 20.1 / 20.3; 204, on 4 100, 21.2 / 21.0; 252, on 6 000, 22.9 / 22.0).
// (A batch with fewer tiles than its requests could have stays in launch order: many groups would have no tile.)
// The XCDs have to get about as much each: nearly as many groups, and each request on all of them or, from 80 groups of at least four a
// request on, many requests.  One request of 951 tokens (476 tiles of one kv head) is one group: 103 us in launch order, 694 on one XCD.
constexpr int kKeyGroupsFrom = 192;
constexpr int kKeyGroupsOfManyRequests = 80;
static int rows_key_groups(const warp34_attention_batch& B, const AttnParams& P, int kv_subs, int grid_z) {
    const int per_tile = P.max_chunks * kv_subs;
    if (P.bal_tiles < 2 || per_tile % kXcds == 0 || grid_z != (long long)B.num_reqs * P.bal_tiles) return 0;
    const long long groups = (long long)B.num_reqs * per_tile;
    const long long on_an_xcd = (groups + kXcds - 1) / kXcds;
    if (8 * kXcds * on_an_xcd > 9 * groups) return 0;
    if (per_tile < kXcds && (per_tile < kXcds / 2 || groups < kKeyGroupsOfManyRequests)) return 0;
    return groups * P.bal_tiles >= kKeyGroupsFrom && on_an_xcd <= 65535 ? (int)groups : 0;
}

// Chunk grid at head dimension 128, more workgroups than CUs but no more than two on each: the requests go by length
// (rows_longest_first); returned is how many the first round of workgroups takes, 0: in their own order.  us a layer step, bf16 draft blocks,
// mean of six sets of contexts from an eighth of the length up, one workgroup per CU / two in the requests' order / two by length:
// up to 14 000 keys 9 x 16 tokens 72.2 / 57.0 / 50.6, 12 x 16 86.2 / 74.9 / 65.5, 15 x 16 105 / 90.7 / 74.3, 13 x 8 58.0 / 55.4 / 50.0,
// 16 x 8 69.4 / 66.5 / 58.4; up to 5 000 12 x 16 45.4 / 39.9 / 37.3.  (The longest first all through: 52.2, 67.4, 80.4, 51.7, 63.2; 37.8.)
// Single sets in the requests' order were up to 18 % slower than one per CU (12 x 16, 88.9 / 105).  From kLongestFirstKeys keys a
// workgroup on: the lengths are asked for before anything else, and with shorter chunks that costs what it gains (4 x 16 up to 5 000,
// 8 chunks, 22.8 / 22.9; 4 x 8, 16 chunks, 20.1 / 20.5; 6 x 8 up to 14 000, 10 chunks, 31.6 / 30.9).
constexpr int kLongestFirstKeys = 1000;
static int rows_first_round(const warp34_attention_batch& B, const AttnParams& P, int kv_subs, int grid_z) {
    const long long per_req = (long long)P.max_chunks * kv_subs * P.bal_tiles, wgs = per_req * B.num_reqs;
    if (P.bal_tiles < 2 || B.num_reqs < 2 || B.num_reqs > 64 || grid_z != (long long)B.num_reqs * P.bal_tiles || B.sliding_window > 0 ||
        wgs <= kChipCus || wgs > 2 * kChipCus || B.max_seq_len < (long long)kLongestFirstKeys * P.max_chunks)
        return 0;
    return std::max(1, (int)(kChipCus / per_req));
}

// VRES: value rows stored rotated in an 8-bit format (residual operand, see rows_tile)
template <typename TQ, int KVF, bool VRES = false, int HD = kHeadDim>
static int launch_rows(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                       const warp34_attention_batch* batch, const void* q, void* out, int num_q_heads,
                       int force_single, const void* gate) {
    AttnParams P{};
    P.L = *layout;
    P.B = *batch;
    P.block_magic = block_magic_for(layout->block_size);
    P.q = (const uint16_t*)q;
    P.out = (uint16_t*)out;
    P.gate = (const uint16_t*)gate;
    P.num_q_heads = num_q_heads;
    P.gqa = num_q_heads / layout->local_kv_heads;
    int q_group = P.gqa;
    if (q_group > 16) {
        for (int d = 16; d >= 1; --d)
            if (P.gqa % d == 0) {
                q_group = d;
                break;
            }
    }
    P.q_group = q_group;
    P.q_group_magic = q_group_magic_for(q_group);
    P.q_subgroups = P.gqa / q_group;
    P.tok_tile = 16 / q_group;  // one N tile
    if (P.tok_tile < 1) P.tok_tile = 1;
    P.min_upc = kMinUnitsPerChunk;
    P.tiles_by_request = (batch->max_q_len > 0 && batch->max_q_len <= P.tok_tile) ? 1 : 0;
    P.rot_q = layout->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    P.rot_out = layout->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    const int grid_z = tiles_bound(*batch, P);
    const int kv_subs = layout->local_kv_heads * P.q_subgroups;
    hipStream_t stream = (hipStream_t)ex->stream;
    int rc, decode_chunks = 0;
    rc = launch_rows_balanced<TQ, KVF, VRES, HD>(ex, batch, P, kv_subs, force_single, stream, &decode_chunks);
    if (rc >= 0) return rc;
    P.max_chunks = force_single        ? 1
                   : decode_chunks > 0 ? decode_chunks
                                       : choose_max_chunks(ex, batch->total_tokens, num_q_heads, P.tok_tile, P.q_subgroups, kv_subs);
    P.part_acc = nullptr;
    P.part_ml = nullptr;
    const long long rows = (long long)batch->total_tokens * num_q_heads;
    const long long tok_tiles = ((long long)batch->total_tokens + P.tok_tile - 1) / P.tok_tile;
    P.few_chunks = few_chunks_of(kFewChunksRows, decode_chunks > 0 ? decode_chunks : chunk_target(tok_tiles, P.q_subgroups));
    int grid_x = P.max_chunks;
    if (batch->max_seq_len > 0) {
        const int units = (batch->max_seq_len + kUnit - 1) / kUnit + 1;
        const int bound = chunk_count(units, P.few_chunks);
        if (bound < grid_x) grid_x = bound < 1 ? 1 : bound;
    }
    // No tile has more chunks than that: the cap is lowered to it, which changes no chunk (a
    // tile's count is limited by its own units first) and keeps the partial records, and what
    // the merge kernel loads ahead of knowing the count, as small as the bound allows.
    P.max_chunks = grid_x;
    P.part_stride = grid_x;
    fill_spec_geometry(P, batch->max_seq_len);
    if (P.max_chunks > 1) {
        uint8_t* ws = reinterpret_cast<uint8_t*>((uintptr_t)ex->scratch_ptr);
        P.part_acc = reinterpret_cast<float*>(ws);
        P.part_ml = P.part_acc + (size_t)rows * P.max_chunks * kHeadDim;
    }
    dim3 grid((unsigned)grid_x, (unsigned)kv_subs, (unsigned)grid_z);
    P.bal_tiles = tiles_per_request_bound(*batch, P);
    P.key_groups = rows_key_groups(*batch, P, kv_subs, grid_z);
    P.first_round = HD != kHeadDim ? rows_first_round(*batch, P, kv_subs, grid_z) : 0;
    if (P.key_groups > 0) grid = dim3((unsigned)(kXcds * P.bal_tiles), (unsigned)((P.key_groups + kXcds - 1) / kXcds));
    constexpr int smem = rows_smem_bytes<KVF, HD>(1);
    auto kernel = P.key_groups > 0 || P.first_round > 0 ? paged_attn_rows_mapped_kernel<TQ, KVF, VRES, HD>
                                                        : paged_attn_rows_kernel<TQ, KVF, VRES, HD>;
    if constexpr (!VRES) {
        if (plain_rows(P)) {
            if (P.tiles_by_request == 0) kernel = paged_attn_rows_plain_kernel<TQ, KVF, HD, false>;
            else if constexpr (RowsLds<KVF, HD>::k8) kernel = paged_attn_rows_plain_kernel<TQ, KVF, HD, true>;
        }
    }
    rc = ensure_dynamic_lds(kernel, smem, true);
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, grid, dim3(kKv16Waves * 64), smem, stream, P);
    rc = (int)hipGetLastError();
    if (rc) return rc;
    return P.max_chunks > 1 ? launch_split_merge<TQ, false, HD>(P, P.max_chunks, 1.0f, stream) : 0;
}

// Chunked prefill: no split over the keys (a prefill batch has hundreds of tiles).
static bool prefill_tq4_applicable(const warp34_kv_layer_layout* layout, const warp34_attention_batch* batch,
                                   int num_q_heads) {
    const int gqa = num_q_heads / layout->local_kv_heads;
    int q_group = gqa;
    if (q_group > 16) {
        for (int d = 16; d >= 1; --d)
            if (gqa % d == 0) {
                q_group = d;
                break;
            }
    }
    return q_group > 0 && (q_group & (q_group - 1)) == 0 && batch->max_q_len > 0;
}

template <typename TQ, int KVF>
static int launch_prefill_tq4(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                              const warp34_attention_batch* batch, const void* q, void* out, int num_q_heads,
                              const void* gate, bool force_wide) {
    AttnParams P{};
    P.L = *layout;
    P.B = *batch;
    P.block_magic = block_magic_for(layout->block_size);
    P.q = (const uint16_t*)q;
    P.out = (uint16_t*)out;
    P.gate = (const uint16_t*)gate;
    P.part_acc = nullptr;
    P.part_ml = nullptr;
    P.num_q_heads = num_q_heads;
    P.gqa = num_q_heads / layout->local_kv_heads;
    int q_group = P.gqa;
    if (q_group > 16) {
        for (int d = 16; d >= 1; --d)
            if (P.gqa % d == 0) {
                q_group = d;
                break;
            }
    }
    P.q_group = q_group;
    P.q_group_magic = q_group_magic_for(q_group);
    P.q_subgroups = P.gqa / q_group;
    P.max_chunks = 1;
    P.min_upc = kMinUnitsPerChunk;
    P.rot_q = layout->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    P.rot_out = layout->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    const int kv_subs = layout->local_kv_heads * P.q_subgroups;
    if constexpr (KVF == WARP34_KV_FORMAT_TQ4) {
        // 128-row tiles on twelve waves (eight multiply, four dequantise) take 0.57 of the time of a 256-row tile, the
        // wide kernel's half tiles 0.65.  us, 128-row tiles / wide: 128 tiles of 256 rows 140 / 161, 206 303 / 301, 230 514 / 539,
        // 256 795 / 764, 318 1 287 / 1 240, 640 2 182 / 2 007, 850 3 098 / 2 813.
        const long long wide = ((long long)batch->total_tokens * q_group / pw_rows(2) + (batch->num_reqs + 1) / 2) * kv_subs;
        if (wide < kPwTq4Tiles && !force_wide) {
            P.tok_tile = kPfRows / q_group;
            const dim3 grid((unsigned)((batch->max_q_len + P.tok_tile - 1) / P.tok_tile), (unsigned)kv_subs, (unsigned)batch->num_reqs);
            const int rc = ensure_dynamic_lds(paged_prefill_tq4_kernel<TQ, false>, kPfSmem, true);
            if (rc) return rc;
            hipLaunchKernelGGL((paged_prefill_tq4_kernel<TQ, false>), grid, dim3(12 * 64), kPfSmem, (hipStream_t)ex->stream, P);
            return (int)hipGetLastError();
        }
    }
    P.tok_tile = pw_rows(2) / q_group;
    P.bal_tiles = (batch->max_q_len + P.tok_tile - 1) / P.tok_tile;
    // (the last round's cut tiles: at most kPwCus / 2 workgroups more)
    const long long wgs = (long long)P.bal_tiles * kv_subs * batch->num_reqs + kPwCus / 2;
    if (wgs > 0x7fffffffll) return (int)hipErrorNotSupported;
    const dim3 grid((unsigned)std::min<long long>(wgs, 1 << 20), (unsigned)((wgs + (1 << 20) - 1) >> 20));
    constexpr bool k8bit = KVF == WARP34_KV_FORMAT_FP8_E4M3 || KVF == WARP34_KV_FORMAT_Q8_0;
    if constexpr (k8bit) {
        if (P.rot_out) {  // rotated 8-bit value rows: codes in the value tile, block scales in the weights
            const int rc = ensure_dynamic_lds(paged_prefill_wide_kernel<TQ, KVF, true>, pw_smem<KVF>(), true);
            if (rc) return rc;
            hipLaunchKernelGGL((paged_prefill_wide_kernel<TQ, KVF, true>), grid, dim3(kPfWaves * 64), pw_smem<KVF>(),
                               (hipStream_t)ex->stream, P);
            return (int)hipGetLastError();
        }
    }
    const int rc = ensure_dynamic_lds(paged_prefill_wide_kernel<TQ, KVF, false>, pw_smem<KVF>(), true);
    if (rc) return rc;
    hipLaunchKernelGGL((paged_prefill_wide_kernel<TQ, KVF, false>), grid, dim3(kPfWaves * 64), pw_smem<KVF>(),
                       (hipStream_t)ex->stream, P);
    return (int)hipGetLastError();
}

static bool is_kv16(const warp34_kv_layer_layout* l, int format) {
    return (l->head_dim == 256 || l->head_dim == 128) && l->k_format == format && l->v_format == format &&
           l->k_transform == WARP34_KV_TRANSFORM_IDENTITY && l->v_transform == WARP34_KV_TRANSFORM_IDENTITY;
}

static bool kv16_geometry_ok(const warp34_kv_layer_layout* l, const void* q, const void* out) {
    const unsigned row_bytes = 2u * (unsigned)l->head_dim;
    return l->block_size > 0 && (l->block_size % 16) == 0 && l->k_token_stride_bytes == row_bytes &&
           l->v_token_stride_bytes == row_bytes && (l->k_base & 15u) == 0 && (l->v_base & 15u) == 0 &&
           (l->k_page_stride_bytes & 15u) == 0 && (l->k_head_stride_bytes & 15u) == 0 &&
           (l->v_page_stride_bytes & 15u) == 0 && (l->v_head_stride_bytes & 15u) == 0 &&
           (((uintptr_t)q) & 15u) == 0 && (((uintptr_t)out) & 7u) == 0;
}

// 8-bit rows: both slabs in the same format, each stored plain or rotated
static bool is_kv8(const warp34_kv_layer_layout* l, int format) {
    const auto xf_ok = [](int t) {
        return t == WARP34_KV_TRANSFORM_IDENTITY || t == WARP34_KV_TRANSFORM_RADEMACHER_WHT256;
    };
    return l->head_dim == 256 && l->k_format == format && l->v_format == format && xf_ok(l->k_transform) &&
           xf_ok(l->v_transform);
}

// 16-token runs must be contiguous and 16-byte aligned for the staging copy
static bool kv8_geometry_ok(const warp34_kv_layer_layout* l, const void* q, const void* out, unsigned row_bytes) {
    return l->block_size > 0 && (l->block_size % 16) == 0 && l->k_token_stride_bytes == row_bytes &&
           l->v_token_stride_bytes == row_bytes && (l->k_base & 15u) == 0 && (l->v_base & 15u) == 0 &&
           (l->k_page_stride_bytes & 15u) == 0 && (l->k_head_stride_bytes & 15u) == 0 &&
           (l->v_page_stride_bytes & 15u) == 0 && (l->v_head_stride_bytes & 15u) == 0 &&
           (((uintptr_t)q) & 15u) == 0 && (((uintptr_t)out) & 7u) == 0;
}

static bool is_tq4_wht(const warp34_kv_layer_layout* l) {
    return l->head_dim == 256 && l->k_format == WARP34_KV_FORMAT_TQ4 && l->v_format == WARP34_KV_FORMAT_TQ4 &&
           l->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 &&
           l->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256;
}

// TQ4 pages at head dimension 256, each slab stored rotated or plain (op_paged_attn.cu:347,570:
// the query is rotated for rotated keys, the output rotated back for rotated values)
static bool is_tq4(const warp34_kv_layer_layout* l) {
    const auto xf_ok = [](int t) {
        return t == WARP34_KV_TRANSFORM_IDENTITY || t == WARP34_KV_TRANSFORM_RADEMACHER_WHT256;
    };
    return l->head_dim == 256 && l->k_format == WARP34_KV_FORMAT_TQ4 && l->v_format == WARP34_KV_FORMAT_TQ4 &&
           xf_ok(l->k_transform) && xf_ok(l->v_transform);
}

static bool tq4_geometry_ok(const warp34_kv_layer_layout* l, const void* q) {
    // 16-token runs must be contiguous and 16-byte aligned for the staging copy
    return l->block_size > 0 && (l->block_size % 16) == 0 && l->k_token_stride_bytes == kTq4RowBytes &&
           l->v_token_stride_bytes == kTq4RowBytes && (l->k_base & 15u) == 0 && (l->v_base & 15u) == 0 &&
           (l->k_page_stride_bytes & 15u) == 0 && (l->k_head_stride_bytes & 15u) == 0 &&
           (l->v_page_stride_bytes & 15u) == 0 && (l->v_head_stride_bytes & 15u) == 0 &&
           (((uintptr_t)q) & 7u) == 0;
}

static int common_checks(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                         const warp34_attention_batch* batch, const void* q, void* out, int num_q_heads) {
    if (!ex || !layout || !batch || !q || !out) return (int)hipErrorInvalidValue;
    return 0;
}

template <typename TQ>
static int attention_entry(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                           const warp34_attention_batch* batch, const void* q, void* out, int num_q_heads,
                           int force, const void* gate = nullptr) {
    // force (the test selector): 0 = the dispatch below, 1 = the decode / verify kernel as a single
    // pass, 2 = the tile kernels (where the batch shape admits them, else as 1), 3 = as 2, TQ4 pages on the wide one
    const int force_single = force != 0 ? 1 : 0;
    const bool force_tile = force == 2 || force == 3, force_wide = force == 3;
    if (layout->local_kv_heads <= 0 || num_q_heads % layout->local_kv_heads != 0 || batch->num_reqs <= 0 ||
        !batch->query_start_loc || !batch->seq_lens_after || !batch->block_tables ||
        batch->max_blocks_per_req <= 0 || batch->sliding_window < 0 ||
        (batch->mask_mode != WARP34_ATTN_MASK_CAUSAL && batch->mask_mode != WARP34_ATTN_MASK_NONCAUSAL_WINDOW)) {
        return (int)hipErrorInvalidValue;
    }
    if (is_tq4(layout)) {
        if (!tq4_geometry_ok(layout, q) || (((uintptr_t)out) & 7u) != 0) return (int)hipErrorNotSupported;
        // Many query rows per request and enough tiles to fill the chip: the tile kernel shares
        // every dequantised key block between 256 (or 128) query rows.
        const bool many_rows = batch->max_q_len >= 32 &&
                               (long long)batch->total_tokens * num_q_heads >= 128ll * kPfRows;
        if ((force_tile || (!force && many_rows)) && prefill_tq4_applicable(layout, batch, num_q_heads))
            return launch_prefill_tq4<TQ, WARP34_KV_FORMAT_TQ4>(ex, layout, batch, q, out, num_q_heads, gate, force_wide);
        return launch_tq4<TQ>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
    }
    // 16-bit pages: the storage type must be the query type (FP16 pages with the f16 entry
    // point, BF16 pages with the bf16 one, as in the reference)
    if (is_kv16(layout, TQ::kStorageFormat)) {
        if (!kv16_geometry_ok(layout, q, out)) return (int)hipErrorNotSupported;
        // many query rows per request: the tile kernel (rows copied as stored)
        const bool many_rows = batch->max_q_len >= 32 &&
                               (long long)batch->total_tokens * num_q_heads >= 128ll * kPfRows;
        // head dimension 128 (op_kv_cache.cu:1227): the decode / verify kernel serves every batch shape
        if (layout->head_dim == 128)
            return launch_rows<TQ, TQ::kStorageFormat, false, 128>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
        if ((force_tile || (!force && many_rows)) && prefill_tq4_applicable(layout, batch, num_q_heads))
            return launch_prefill_tq4<TQ, TQ::kStorageFormat>(ex, layout, batch, q, out, num_q_heads, gate, force_wide);
        return launch_rows<TQ, TQ::kStorageFormat>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
    }
    // 8-bit pages (the tail layers of the default TQ4 policy, cache.rs:87-109)
    if (is_kv8(layout, WARP34_KV_FORMAT_FP8_E4M3)) {
        if (!kv8_geometry_ok(layout, q, out, 264)) return (int)hipErrorNotSupported;
        // many query rows per request: the tile kernel (FP8 rows have the shape of TQ4 rows)
        const bool many_rows = batch->max_q_len >= 32 &&
                               (long long)batch->total_tokens * num_q_heads >= 128ll * kPfRows;
        if ((force_tile || (!force && many_rows)) && prefill_tq4_applicable(layout, batch, num_q_heads))
            return launch_prefill_tq4<TQ, WARP34_KV_FORMAT_FP8_E4M3>(ex, layout, batch, q, out, num_q_heads, gate, force_wide);
        if (rows_vres(layout))
            return launch_rows<TQ, WARP34_KV_FORMAT_FP8_E4M3, true>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
        return launch_rows<TQ, WARP34_KV_FORMAT_FP8_E4M3>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
    }
    if (is_kv8(layout, WARP34_KV_FORMAT_Q8_0)) {
        if (!kv8_geometry_ok(layout, q, out, 272)) return (int)hipErrorNotSupported;
        const bool many_rows = batch->max_q_len >= 32 &&
                               (long long)batch->total_tokens * num_q_heads >= 128ll * kPfRows;
        if ((force_tile || (!force && many_rows)) && prefill_tq4_applicable(layout, batch, num_q_heads))
            return launch_prefill_tq4<TQ, WARP34_KV_FORMAT_Q8_0>(ex, layout, batch, q, out, num_q_heads, gate, force_wide);
        if (rows_vres(layout))
            return launch_rows<TQ, WARP34_KV_FORMAT_Q8_0, true>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
        return launch_rows<TQ, WARP34_KV_FORMAT_Q8_0>(ex, layout, batch, q, out, num_q_heads, force_single, gate);
    }
    return (int)hipErrorNotSupported;
}

// QSA sparse paged attention (op_qsa.cu:1446-1571).  Argument checks and error codes follow the
// reference's launcher; the split count is this kernel's own (enough workgroups to fill the chip,
// at least one unit per wave and split, scratch permitting).
static int launch_qsa_sparse(const warp34_exec* ex, const void* q, const void* gate,
                             const warp34_kv_layer_layout* layout, const int32_t* selected_phys_blocks,
                             const int32_t* selected_logical_blocks, const int32_t* num_selected_blocks,
                             const int32_t* token_seq_pos, const uint8_t* valid_token_mask, void* out,
                             int num_tokens, int local_q_heads, int select_k_blocks, float sm_scale, int had64) {
    if (!ex || !q || !layout || !selected_phys_blocks || !selected_logical_blocks || !num_selected_blocks ||
        !token_seq_pos || !out || num_tokens < 0 || local_q_heads <= 0 || layout->local_kv_heads <= 0 ||
        (local_q_heads % layout->local_kv_heads) != 0 || layout->head_dim != 256 || select_k_blocks < 0) {
        return (int)hipErrorInvalidValue;
    }
    if (num_tokens == 0) return 0;
    // page formats: rotated TQ4, FP16, FP8-E4M3 and Q8_0 (plain or rotated); anything else
    // (mixed K / V formats, BF16 pages) is reported as unsupported, never computed some other way
    constexpr int kFormTq4 = 1000;  // not a WARP34_KV_FORMAT_* value (FP16 is 0)
    int form = -1;  // kFormTq4, else the row format
    if (is_tq4_wht(layout)) {
        if (!tq4_geometry_ok(layout, q) || (((uintptr_t)out) & 7u) != 0) return (int)hipErrorNotSupported;
        form = kFormTq4;
    } else if (is_kv16(layout, WARP34_KV_FORMAT_FP16)) {
        if (!kv16_geometry_ok(layout, q, out)) return (int)hipErrorNotSupported;
        form = WARP34_KV_FORMAT_FP16;
    } else if (is_kv8(layout, WARP34_KV_FORMAT_FP8_E4M3)) {
        if (!kv8_geometry_ok(layout, q, out, 264)) return (int)hipErrorNotSupported;
        form = WARP34_KV_FORMAT_FP8_E4M3;
    } else if (is_kv8(layout, WARP34_KV_FORMAT_Q8_0)) {
        if (!kv8_geometry_ok(layout, q, out, 272)) return (int)hipErrorNotSupported;
        form = WARP34_KV_FORMAT_Q8_0;
    } else {
        return (int)hipErrorNotSupported;
    }
    if (gate != nullptr && (((uintptr_t)gate) & 7u) != 0) return (int)hipErrorNotSupported;
    QsaParams P{};
    P.L = *layout;
    P.gate = (const uint16_t*)gate;
    P.out = (uint16_t*)out;
    P.valid_token_mask = valid_token_mask;
    const int gqa = local_q_heads / layout->local_kv_heads;
    int q_group = gqa;
    if (q_group > 16) {
        for (int d = 16; d >= 1; --d)
            if (gqa % d == 0) {
                q_group = d;
                break;
            }
    }
    const int q_subgroups = gqa / q_group;
    P.groups_per_page = layout->block_size / 4;
    P.gpp_shift = -1;
    for (int k = 0; k < 30; ++k)
        if ((1 << k) == P.groups_per_page) P.gpp_shift = k;
    P.sm_scale = sm_scale;
    P.had64 = had64;
    P.out_scale = form == kFormTq4 ? kLutInvGain : 1.0f;
    P.rot_q = layout->k_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    P.rot_out = layout->v_transform == WARP34_KV_TRANSFORM_RADEMACHER_WHT256 ? 1 : 0;
    const int kv_subs = layout->local_kv_heads * q_subgroups;
    // work items of a token: 32-key units (TQ4) or 16-key halves (row formats), one per wave and turn
    const int max_units = form == kFormTq4 ? (select_k_blocks + 7) / 8 : (select_k_blocks + 3) / 4;
    long long want = 256ll / ((long long)num_tokens * kv_subs);
    if (want > kQsaMaxSplits) want = kQsaMaxSplits;
    const int by_units = (max_units + kQsaWaves - 1) / kQsaWaves;
    if (want > by_units) want = by_units;
    if (want < 1) want = 1;
    const size_t rows = (size_t)num_tokens * local_q_heads;
    const size_t need = rows * (size_t)want * (kHeadDim + 4) * sizeof(float);
    const int n_splits = (want > 1 && ex->scratch_ptr != 0 && (ex->scratch_ptr & 15u) == 0u && ex->scratch_size >= need) ? (int)want : 1;
    if (n_splits > 1) {
        P.part_acc = reinterpret_cast<float*>((uintptr_t)ex->scratch_ptr);
        P.part_ml = P.part_acc + rows * n_splits * kHeadDim;
    }
    const uint32_t shape = QsaShape::pack(q_group, n_splits, q_subgroups);
    const int guess = (max_units + n_splits - 1) / n_splits;
    hipStream_t stream = (hipStream_t)ex->stream;
    const dim3 grid((unsigned)num_tokens, (unsigned)kv_subs, (unsigned)n_splits);
    int rc;
    auto launch_rows_form = [&](auto kernel) {
        const int smem = kv16_smem_bytes(1);
        int r = ensure_dynamic_lds(kernel, smem);
        if (r) return r;
        hipLaunchKernelGGL(kernel, grid, dim3(kKv16Waves * 64), smem, stream, selected_phys_blocks, selected_logical_blocks,
                           num_selected_blocks, token_seq_pos, (const uint16_t*)q, select_k_blocks, guess, shape, local_q_heads, P);
        return (int)hipGetLastError();
    };
    if (form == kFormTq4) {
        rc = ensure_dynamic_lds(qsa_sparse_tq4_kernel, kQsaSmem, true);
        if (rc) return rc;
        hipLaunchKernelGGL(qsa_sparse_tq4_kernel, grid, dim3(kQsaWaves * 64), kQsaSmem, stream, selected_phys_blocks,
                           selected_logical_blocks, num_selected_blocks, token_seq_pos, (const uint16_t*)q, select_k_blocks, guess, shape,
                           local_q_heads, P);
        rc = (int)hipGetLastError();
    } else if (form == WARP34_KV_FORMAT_FP16) {
        rc = launch_rows_form(qsa_sparse_rows_kernel<WARP34_KV_FORMAT_FP16>);
    } else if (form == WARP34_KV_FORMAT_FP8_E4M3) {
        rc = P.rot_out ? launch_rows_form(qsa_sparse_rows_kernel<WARP34_KV_FORMAT_FP8_E4M3, true>)
                       : launch_rows_form(qsa_sparse_rows_kernel<WARP34_KV_FORMAT_FP8_E4M3, false>);
    } else {
        rc = P.rot_out ? launch_rows_form(qsa_sparse_rows_kernel<WARP34_KV_FORMAT_Q8_0, true>)
                       : launch_rows_form(qsa_sparse_rows_kernel<WARP34_KV_FORMAT_Q8_0, false>);
    }
    if (rc) return rc;
    if (n_splits > 1) {
        hipLaunchKernelGGL(qsa_sparse_merge_kernel, dim3((unsigned)rows), dim3(64), 0, stream, P.part_ml, P.part_acc, P.gate, P.out, n_splits,
                           P.rot_out, P.had64, P.out_scale);
        rc = (int)hipGetLastError();
    }
    return rc;
}

}  // namespace w34

using namespace w34;

// op_paged_attn.cu:1266-1448
extern "C" int warp34_paged_attention_f16(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                                          const warp34_attention_batch* batch, const void* q_in,
                                          void* attn_out, int num_q_heads) {
    const int rc = common_checks(ex, layout, batch, q_in, attn_out, num_q_heads);
    if (rc) return rc;
    if (layout->k_format == WARP34_KV_FORMAT_FP8_E4M3 || layout->v_format == WARP34_KV_FORMAT_FP8_E4M3) {
        // the reference also asks the device generation here (op_paged_attn.cu:1259); gfx950 has FP8
        if (layout->head_dim != 256) return (int)hipErrorInvalidValue;
    }
    if (batch->total_tokens <= 0 || num_q_heads <= 0) return 0;
    return attention_entry<F16>(ex, layout, batch, q_in, attn_out, num_q_heads, 0);
}

// warp34_paged_attention_f16 with the output gate of the gated full-attention layers applied as
// the rows leave the kernels (no counterpart in the reference, which calls
// warp34_apply_attn_output_gate_f16 afterwards, model/forward.rs:1192-1211): attn_out receives the
// bits of that sequence, the ungated output never goes to memory.  gate: fp16
// [total_tokens, num_q_heads, 256], 8-byte aligned; rows the attention leaves untouched (masked
// tokens and requests) stay untouched.
extern "C" int warp34_paged_attention_gated_f16(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                                                const warp34_attention_batch* batch, const void* q_in,
                                                const void* gate, void* attn_out, int num_q_heads) {
    const int rc = common_checks(ex, layout, batch, q_in, attn_out, num_q_heads);
    if (rc) return rc;
    if (gate == nullptr) return (int)hipErrorInvalidValue;
    if (layout->k_format == WARP34_KV_FORMAT_FP8_E4M3 || layout->v_format == WARP34_KV_FORMAT_FP8_E4M3) {
        if (layout->head_dim != 256) return (int)hipErrorInvalidValue;
    }
    if (batch->total_tokens <= 0 || num_q_heads <= 0) return 0;
    if ((((uintptr_t)gate) & 7u) != 0) return (int)hipErrorNotSupported;
    return attention_entry<F16>(ex, layout, batch, q_in, attn_out, num_q_heads, 0, gate);
}

// op_kv_cache.cu:1192-1241
extern "C" int warp34_paged_attention_bf16(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                                           const warp34_attention_batch* batch, const void* q_in,
                                           void* attn_out, int num_q_heads) {
    const int rc = common_checks(ex, layout, batch, q_in, attn_out, num_q_heads);
    if (rc) return rc;
    if (num_q_heads <= 0 || batch->total_tokens < 0) return (int)hipErrorInvalidValue;
    if (!batch->total_tokens) return 0;
    return attention_entry<BF16>(ex, layout, batch, q_in, attn_out, num_q_heads, 0);
}

// op_paged_attn.cu:1451-1519
extern "C" int warp34_paged_attention_f16_force_kernel_for_test(
    const warp34_exec* ex, const warp34_kv_layer_layout* layout, const warp34_attention_batch* batch,
    const void* q_in, void* attn_out, int num_q_heads, int use_64q) {
    const int rc = common_checks(ex, layout, batch, q_in, attn_out, num_q_heads);
    if (rc) return rc;
    if (batch->total_tokens <= 0 || num_q_heads <= 0) return 0;
    // the reference's selector picks the 16-row kernel (0) or one of its 64 / 128-row prefill kernels;
    // here: the decode / verify kernel as a single pass, the tile kernels, or (2) the 256-row one for TQ4 pages too
    return attention_entry<F16>(ex, layout, batch, q_in, attn_out, num_q_heads, use_64q == 0 ? 1 : use_64q == 2 ? 3 : 2);
}

// Scratch that lets a batch split fully, computed the way the launchers compute it.
// q_group / q_subgroups as in launch_tq4 / launch_rows; layout null: not known, take the largest need over
// all layouts with this many q heads.  num_reqs < 0: not known, as many as tokens.
static size_t scratch_bytes_for(const warp34_kv_layer_layout* layout, int total_tokens, int num_reqs, int num_q_heads,
                                int max_seq_len) {
    if (total_tokens <= 0 || num_q_heads <= 0) return 0;
    int q_group = 1, q_subgroups = 1, kv_subs = num_q_heads;  // the bound when the layout is unknown
    int tok_tile = 16;
    const int few = layout && is_tq4(layout) ? kFewChunksTq4 : kFewChunksRows;  // (the larger one when the layout is unknown)
    if (layout && layout->local_kv_heads > 0 && num_q_heads % layout->local_kv_heads == 0) {
        const int gqa = num_q_heads / layout->local_kv_heads;
        q_group = gqa;
        if (q_group > 16) {
            for (int d = 16; d >= 1; --d)
                if (gqa % d == 0) {
                    q_group = d;
                    break;
                }
        }
        q_subgroups = gqa / q_group;
        kv_subs = layout->local_kv_heads * q_subgroups;
        tok_tile = 16 / q_group < 1 ? 1 : 16 / q_group;
    }
    const int tiles = (int)(((long long)total_tokens + tok_tile - 1) / tok_tile);
    const int full = chunk_target(tiles, q_subgroups);
    int want = full;
    if (max_seq_len > 0) {
        const int units = (max_seq_len + kUnit - 1) / kUnit + 1;
        want = std::min(want, chunk_count(units, few_chunks_of(few, full)));
        // (the first of full, full / 2, ... that is enough is at most 2 want - 1)
        if (!layout) want = std::min(full, 2 * want - 1);
        else if (want > one_round(tiles, kv_subs)) {
            int halved = full;
            while (halved / 2 >= want) halved /= 2;
            want = halved;
        }
    }
    size_t bytes = want >= 2 ? partial_bytes((long long)total_tokens * num_q_heads, want) : 0;
    // TQ4 verify batches over long contexts may take the shared-prefix pass: its partial slots sit
    // behind the split-K ones, and a header behind the records
    if ((!layout || is_tq4(layout)) && want >= 2 && total_tokens >= 16 && (num_reqs < 0 || num_reqs >= 4) &&
        max_seq_len >= 8 * kSpMinTokens && (q_group & (q_group - 1)) == 0) {
        const int parts = shared_prefix_parts(total_tokens, q_group, q_subgroups);
        if (want + parts <= kMergeGroups * kMergeMaxPerGroup)
            bytes = partial_bytes((long long)total_tokens * num_q_heads, want + parts) + sizeof(SpHeader);
    }
    // The balanced plan: (shares + entries) partial slots of 16 columns per column tile and (kv head, q
    // subgroup), and the per-token table.
    const auto plan = [&](long long entries, int nt) {
        const size_t slots = (size_t)(balanced_groups(q_subgroups) + entries) * kv_subs * 16 * nt;
        const size_t need = partial_bytes((long long)slots, 1) + (size_t)total_tokens * 16;
        if (need > bytes) bytes = need;
    };
    if (num_reqs < 0 || num_reqs > total_tokens) num_reqs = total_tokens;
    if (layout && (is_kv16(layout, WARP34_KV_FORMAT_FP16) || is_kv16(layout, WARP34_KV_FORMAT_BF16) ||
                   is_kv8(layout, WARP34_KV_FORMAT_FP8_E4M3) || is_kv8(layout, WARP34_KV_FORMAT_Q8_0))) {
        // row formats: as launch_rows_balanced (the tokens taken as spread evenly over the requests)
        const int q_len = num_reqs > 0 ? (int)(((long long)total_tokens + num_reqs - 1) / num_reqs) : 0;
        const BalShape shape = rows_balanced_shape(num_reqs, total_tokens, q_len, q_group, q_subgroups, rows_vres(layout),
                                                   layout->head_dim);
        if (shape.tiles > 0) plan((long long)num_reqs * shape.tiles, shape.nt);
        return bytes;
    }
    // one tile per request (decode steps; not with more tokens than that many tiles hold)
    if (num_reqs >= 2 && total_tokens <= 65535 && total_tokens <= (long long)num_reqs * tok_tile) plan(num_reqs, 1);
    // layout not known, one q head per kv head: two column tiles from 17 tokens per request on, at most an entry
    // per 16 tokens
    if (!layout && total_tokens > 16 * kRowsGridTiles && total_tokens <= 65535) plan(total_tokens / 16, 2);
    return bytes;
}

extern "C" size_t warp34_paged_attention_scratch_bytes(int total_tokens, int num_q_heads, int max_seq_len) {
    return scratch_bytes_for(nullptr, total_tokens, -1, num_q_heads, max_seq_len);
}

extern "C" size_t warp34_paged_attention_scratch_bytes_for_layout(const warp34_kv_layer_layout* layout,
                                                                  int total_tokens, int num_reqs, int num_q_heads,
                                                                  int max_seq_len) {
    if (!layout) return 0;
    return scratch_bytes_for(layout, total_tokens, num_reqs, num_q_heads, max_seq_len);
}

// op_qsa.cu:1711-1730
extern "C" int warp34_qsa_sparse_paged_attn_f16(const warp34_exec* ex, const void* q, const void* gate,
                                                const warp34_kv_layer_layout* kv_layout,
                                                const int32_t* selected_phys_blocks,
                                                const int32_t* selected_logical_blocks,
                                                const int32_t* num_selected_blocks, const int32_t* token_seq_pos,
                                                const uint8_t* valid_token_mask, void* out, int num_tokens,
                                                int local_q_heads, int select_k_blocks, float sm_scale) {
    return launch_qsa_sparse(ex, q, gate, kv_layout, selected_phys_blocks, selected_logical_blocks,
                             num_selected_blocks, token_seq_pos, valid_token_mask, out, num_tokens, local_q_heads,
                             select_k_blocks, sm_scale, 0);
}

// op_qsa.cu:1732-1751
extern "C" int warp34_qsa_sparse_paged_attn_hadamard_f16(
    const warp34_exec* ex, const void* q, const void* gate, const warp34_kv_layer_layout* kv_layout,
    const int32_t* selected_phys_blocks, const int32_t* selected_logical_blocks,
    const int32_t* num_selected_blocks, const int32_t* token_seq_pos, const uint8_t* valid_token_mask, void* out,
    int num_tokens, int local_q_heads, int select_k_blocks, float sm_scale) {
    return launch_qsa_sparse(ex, q, gate, kv_layout, selected_phys_blocks, selected_logical_blocks,
                             num_selected_blocks, token_seq_pos, valid_token_mask, out, num_tokens, local_q_heads,
                             select_k_blocks, sm_scale, 1);
}

// ---- an entry point that allocates nothing -----------------------------------------------------
// warp34_paged_attention_bf16 with the split-K scratch in a file-scope device array instead of
// ex->scratch_ptr, for callers that cannot provide (or allocate) a workspace.  Every device the
// library runs on holds its own copy of the array at its own address; the address is looked up
// once per device, with that device current, and kept.  The array's NAME is a host-side stand-in
// and is never passed to a kernel or a runtime call: only the looked-up address is.
namespace w34 {
constexpr size_t kStaticScratchBytes = WARP34_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char g_static_scratch[kStaticScratchBytes];
constexpr int kStaticScratchDevices = 64;
static std::atomic<uintptr_t> g_static_scratch_addr[kStaticScratchDevices];

static int static_scratch_address(uintptr_t* out) {
    int dev = 0;
    hipError_t rc = hipGetDevice(&dev);
    if (rc != hipSuccess) return (int)rc;
    if (dev < 0 || dev >= kStaticScratchDevices) return (int)hipErrorInvalidDevice;
    uintptr_t addr = g_static_scratch_addr[dev].load(std::memory_order_acquire);
    if (addr == 0) {
        void* sym = nullptr;
        rc = hipGetSymbolAddress(&sym, HIP_SYMBOL(g_static_scratch));
        if (rc != hipSuccess) return (int)rc;
        if (sym == nullptr || ((uintptr_t)sym & 15u) != 0u) return (int)hipErrorInvalidSymbol;
        addr = (uintptr_t)sym;
        g_static_scratch_addr[dev].store(addr, std::memory_order_release);
    }
    *out = addr;
    return 0;
}
}  // namespace w34

extern "C" int warp34_paged_attention_bf16_static_scratch(const warp34_exec* ex, const warp34_kv_layer_layout* layout,
                                                          const warp34_attention_batch* batch, const void* q_in,
                                                          void* attn_out, int num_q_heads) {
    const int rc = common_checks(ex, layout, batch, q_in, attn_out, num_q_heads);
    if (rc) return rc;
    if (num_q_heads <= 0 || batch->total_tokens < 0) return (int)hipErrorInvalidValue;
    if (!batch->total_tokens) return 0;
    // The array serves every batch the way an 8 MiB ex->scratch would: the launchers take fewer
    // chunks, or leave a pass out, when the records of the full split do not fit.  Refused are only
    // batches too large for the array to be of any use: not even two records per query row fit.
    const long long rows = (long long)batch->total_tokens * num_q_heads;
    if (partial_bytes(rows, 2) > kStaticScratchBytes) return (int)hipErrorOutOfMemory;
    uintptr_t addr = 0;
    const int arc = static_scratch_address(&addr);
    if (arc) return arc;
    warp34_exec own = *ex;
    own.scratch_ptr = addr;
    own.scratch_size = kStaticScratchBytes;
    return attention_entry<BF16>(&own, layout, batch, q_in, attn_out, num_q_heads, 0);
}
