// Attention of several query rows per request over packed pages, on MFMA
// tiles (gfx950, wave64), for head dims 96 and 128, anchor and adjacent mode.
//
// The decode kernel scores one query row per workgroup with integer dot
// products on the packed codes, so n rows of one request stream the
// request's pages n times.  Here one workgroup takes a tile of up to 32 rows
// of one (request, head) and a split of its history, streams each page once,
// and dequantizes every 32-token tile into LDS as FP16 K and BF16 V (both
// row-major; V is read transposed by ds_read_b64_tr_b16), so that the tile's
// rows share it through MFMA:
//   S^T = K Q'^T     (32 tokens x 32 rows, D / 16 v_mfma_f32_32x32x16_f16)
//   O^T += V^T P^T   (D channels x 32 rows, D / 16 v_mfma_f32_32x32x16_bf16)
// The scores take FP16 operands (11-bit significands; each row of q' is
// scaled by a power of two into [-1, 1], which the scores take back), since
// BF16 operands there put the outlier channels' score error near the
// 1e-3 mean bar on short histories.  P stays in the accumulator registers
// (the token order of each P.V step is permuted to match the accumulator
// layout, and V^T is read with the same permutation).  Each of the four
// waves takes every fourth tile with its own online softmax; the waves meet
// once in LDS at the end.  The query prologue (q . R_k) runs on MFMA as well.
// The workgroup whose split of a (request, head, row tile) ends last (the
// others have written one partial (m, l, O) per row) merges the splits,
// applies R_v^T (on MFMA), adds the live tokens and writes the output.
//
// Calls whose requests average 16 rows or fewer take 16-row tiles instead:
// the same pages and dequantization, with the tile's products on
// v_mfma_f32_16x16x32 (S^T: 2 token halves x D / 32 steps; O^T: D / 16
// channel blocks, one 32-token step each), which halves the matrix work and
// the softmax's per-lane scores of a tile that would otherwise be half empty.
//
// A lane dequantizes one token's 32-channel quarter of a 16-token unit
// (lane = token x quarter); at D = 96 the fourth quarter's lanes load a copy
// of the first quarter's bytes and store nothing.
//
// Semantics (reference: attention/compute.cuh:397-505 keys, :28-107 values,
// :120-197 and :506-623 the adjacent-mode chain, prepare.cuh:13-54 and
// :203-229 live score and mean shift, merge.cuh:8-84, output.cuh:9-31):
//   anchor mode: keys alpha_L (c.s+o + bf16(mu_A))_A + (c.s+o)_L with the
//     current loop's mean as a per-row shift, values alpha_L (c.s+o)_A +
//     (c.s+o)_L (the reference rounds each restore step to BF16; one
//     rounding here, within the attention tolerance) (AnchorDecoder);
//   adjacent mode past loop 0: keys and values the BF16 restore chain over
//     records 0..L, the key chain adding bf16(mu_r) to every record but the
//     current loop's (rq_chain.h; ChainDecoder);
// P in BF16.
//
// Lane layouts of v_mfma_f32_32x32x16_bf16 (checked on gfx950): A row l % 32,
// k 8 (l / 32) + e; B column l % 32, k 8 (l / 32) + e; C register r holds row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.  Of v_mfma_f32_16x16x32:
// A row l % 16, k 8 (l / 16) + e; B column l % 16, k 8 (l / 16) + e; C
// register r holds row 4 (l / 16) + r, column l % 16.
#include "rq_multirow.h"

namespace rq {

namespace {

// The O^T accumulator tiles of one lane: D / 32 of 32 x 32 (32-row tiles) or
// D / 16 of 16 x 16 (16-row tiles).
template <int TR>
struct OutTile {
    typedef F32x16 Type;
};
template <>
struct OutTile<16> {
    typedef F32x4 Type;
};

// The head of a stream workgroup (stream_grid).
__device__ __forceinline__ int stream_head(const MultiRowParams& p) {
    return p.items > 0 ? (int)(blockIdx.x % (unsigned)p.heads) : (int)blockIdx.y;
}

template <int D, int PT, int TR, class Decoder>
__device__ __forceinline__ void multirow_stream(const MultiRowParams& p, Decoder& dec, uint8_t* lds,
                                                int* split_blocks) {
    using G = Geometry<D, TR>;
    constexpr int KS = G::KS;
    constexpr int QRS = G::QRS;
    const int head = stream_head(p);
    const PlanItem item = multirow_plan<true>(p, (int)(blockIdx.x / (unsigned)p.heads), blockIdx.x,
                                               (int)blockIdx.z / p.splits, (int)blockIdx.z % p.splits);
    const int request = __builtin_amdgcn_readfirstlane(item.request);
    const int first = __builtin_amdgcn_readfirstlane(item.first), n = __builtin_amdgcn_readfirstlane(item.rows);
    const int row0 = TR * __builtin_amdgcn_readfirstlane(item.index);
    if (request < 0 || row0 >= n) return;  // uniform over the workgroup, before any barrier
    const int split = item.split;
    const int history = __builtin_amdgcn_readfirstlane(item.tokens);
    const int tile_begin = __builtin_amdgcn_readfirstlane(split_begin(item.length, split, item.splits));
    const int tile_end = __builtin_amdgcn_readfirstlane(split_begin(item.length, split + 1, item.splits));

    // The row tile's arrival word lies in the two unused floats of its first
    // row's entry of split 0.
    float* tile_entries = p.partials + ((int64_t)head * p.entries + item.entry + row0 * item.splits) * kMultiRowEntry;
    uint64_t* arrivals = reinterpret_cast<uint64_t*>(tile_entries + 2);
    const uint64_t arrivals_seen = item.splits > 1 ? peek_arrivals(arrivals) : 0;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // provably wave-uniform
    const int lane = tid & 63;
    const int column = lane & 31;
    const int half = lane >> 5;

    // ---------------------------------------------------------------- q'
    // q' = (q . R_k) * log2(e) / sqrt(D) for the tile's rows, held as FP16
    // q' 2^-e with 2^e the row's power-of-two scale, and the row dots
    // q'.bf16(mu_A) (added per token times alpha_L) and q'.mu_L (the shift of
    // the history scores against the live ones).  The prologue always
    // prepares 32 rows from row0; a 16-row tile uses the first 16.
    uint16_t* q16 = reinterpret_cast<uint16_t*>(lds + G::kQ16Offset);
    uint16_t* r_k = reinterpret_cast<uint16_t*>(lds + G::kRkOffset);
    float* q_raw = reinterpret_cast<float*>(lds + G::kQrawOffset);
    uint16_t* q_p = reinterpret_cast<uint16_t*>(lds + G::kQpOffset);
    float* q_mu = reinterpret_cast<float*>(lds + G::kQmuOffset);  // [0..31] q'.bf16(mu_A), [32..63] q'.mu_L
    float* q_scale = q_mu + 64;                                    // [32] 2^e per row
    float* q_unscale = q_mu + 96;                                  // [32] 2^f per row (the input's scale)
    {
        const int r = tid >> 3, part = tid & 7;  // row, 16-channel part
        const bool part_active = part < G::Parts;
        const int row = row0 + r;
        uint32_t words[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        if (row < n && part_active) {
            const uint2* src = reinterpret_cast<const uint2*>(
                p.query + (int64_t)(first + row) * p.query_stride + head * D + 16 * part);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint2 v = src[i];
                words[2 * i] = v.x;
                words[2 * i + 1] = v.y;
            }
        }
        float x[16];
        float magnitude = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[2 * i] = bf16_f32(words[i] & 0xffffu);
            x[2 * i + 1] = bf16_f32(words[i] >> 16);
            magnitude = fmaxf(magnitude, fmaxf(fabsf(x[2 * i]), fabsf(x[2 * i + 1])));
        }
        if (p.key_rotation) {
            // The row scaled by a power of two 2^-f into [-1, 1]: exact in FP16
            // (a BF16 significand fits), so q.R_k runs on FP16 MFMAs and the
            // product takes 2^f back.
            magnitude = fmaxf(magnitude, __shfl_xor(magnitude, 1));
            magnitude = fmaxf(magnitude, __shfl_xor(magnitude, 2));
            magnitude = fmaxf(magnitude, __shfl_xor(magnitude, 4));
            // (f at most 127, so 2^f stays finite; the scaled row is then within 2.)
            const int f = magnitude > 0.f ? min(__builtin_amdgcn_frexp_expf(magnitude), 127) : 0;
            const float down = ldexpf(1.0f, -f);
            uint32_t h[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                h[i] = f16_bits(x[2 * i] * down) | (f16_bits(x[2 * i + 1] * down) << 16);
            if (part_active) {
                uint4* dst = reinterpret_cast<uint4*>(&q16[r * KS + 16 * part]);
                dst[0] = make_uint4(h[0], h[1], h[2], h[3]);
                dst[1] = make_uint4(h[4], h[5], h[6], h[7]);
            }
            if (part == 0) q_unscale[r] = ldexpf(1.0f, f);
            // R_k [D][D] FP16 into rows of KS halves, 16 bytes per copy.
            constexpr int kChunks = D / 8;
            const uint4* src = reinterpret_cast<const uint4*>(p.key_rotation + (int64_t)head * D * D);
#pragma unroll
            for (int i = tid; i < D * kChunks; i += kThreads)
                *reinterpret_cast<uint4*>(&r_k[(i / kChunks) * KS + 8 * (i % kChunks)]) = src[i];
        } else if (part_active) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4*>(&q_raw[r * QRS + 16 * part + 4 * i]) =
                    make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
        }
    }
    __syncthreads();
    if (item.splits > 1 && tid == 0) tag_arrivals(arrivals, p.call_tag, arrivals_seen);
    if (p.key_rotation && wave < G::Quarters) {
        // q.R_k on the matrix cores: wave w takes columns 32 w .. 32 w + 31.
        // A: lane l reads scaled row l % 32 at k = 16 m + 8 (l / 32) .. + 7.
        // B: R_k[k][c] for column 32 w + l % 32 and the same k, read
        // transposed from the row-major R_k tile (ds_read_b64_tr_b16: output
        // lane o of 16 gets element o % 4 of the 8 bytes addressed by lanes
        // o / 4 + 4 p, so lane q of a 16-lane group addresses row
        // k0 + q / 4 at columns c0 + 4 (q % 4) .. + 3 and receives column
        // c0 + q of rows k0 .. k0 + 3).
        const int group = lane >> 4, q16_lane = lane & 15;
        const int c0 = 32 * wave + 16 * (group & 1);
        const int k_half = 8 * (group >> 1);
        F32x16 c;
#pragma unroll
        for (int e = 0; e < 16; ++e) c[e] = 0.f;
#pragma unroll
        for (int m = 0; m < G::Parts; ++m) {
            const F16x8 a = *reinterpret_cast<const F16x8*>(&q16[column * KS + 16 * m + 8 * half]);
            const int k0 = 16 * m + k_half;
            const Short4 lo = read_transposed(&r_k[(k0 + (q16_lane >> 2)) * KS + c0 + 4 * (q16_lane & 3)]);
            const Short4 hi = read_transposed(&r_k[(k0 + 4 + (q16_lane >> 2)) * KS + c0 + 4 * (q16_lane & 3)]);
            const F16x8 b = __builtin_bit_cast(F16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            c = mfma(a, b, c);
        }
        // Register e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4, column 32 w + l % 32.
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int rr = 8 * (e >> 2) + 4 * half + (e & 3);
            q_raw[rr * QRS + 32 * wave + column] = c[e] * q_unscale[rr];
        }
    }
    __syncthreads();
    {
        const int cb = tid & 31, rb = tid >> 5;  // columns 4 cb .. 4 cb + 3, rows 4 rb .. 4 rb + 3
        const bool cb_active = 4 * cb < D;
        float acc[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = cb_active ? *reinterpret_cast<const float4*>(&q_raw[(4 * rb + i) * QRS + 4 * cb])
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
            acc[i][0] = v.x;
            acc[i][1] = v.y;
            acc[i][2] = v.z;
            acc[i][3] = v.w;
        }
        const float scale = kScoreScale<D>;
        float mu_a[4] = {0.f, 0.f, 0.f, 0.f}, mu_l[4] = {0.f, 0.f, 0.f, 0.f};
        if (Decoder::kAnchorMeanTerm && p.key_mean_anchor && cb_active) {
#pragma unroll
            for (int j = 0; j < 4; ++j) mu_a[j] = round_bf16(p.key_mean_anchor[head * D + 4 * cb + j]);
        }
        if (p.key_mean_loop && cb_active) {
#pragma unroll
            for (int j = 0; j < 4; ++j) mu_l[j] = p.key_mean_loop[head * D + 4 * cb + j];
        }
        // Row maxima over the 32 lanes of this half-wave (the same four rows)
        // give each row's power-of-two scale.
        float row_max[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            row_max[i] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[i][j] *= scale;
                row_max[i] = fmaxf(row_max[i], fabsf(acc[i][j]));
            }
        }
#pragma unroll
        for (int d = 16; d; d >>= 1)
#pragma unroll
            for (int i = 0; i < 4; ++i) row_max[i] = fmaxf(row_max[i], __shfl_xor(row_max[i], d));
        float dot_a[4], dot_l[4], row_scale[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // 2^e >= row_max (e from the exponent field; 1 for an all-zero row)
            const int e = row_max[i] > 0.f ? __builtin_amdgcn_frexp_expf(row_max[i]) : 0;
            row_scale[i] = ldexpf(1.0f, e);
            const float inverse = ldexpf(1.0f, -e);
            uint32_t bits[4];
            dot_a[i] = 0.f;
            dot_l[i] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const _Float16 h = (_Float16)(acc[i][j] * inverse);
                bits[j] = __builtin_bit_cast(uint16_t, h);
                const float q = (float)h * row_scale[i];
                dot_a[i] = fmaf(q, mu_a[j], dot_a[i]);
                dot_l[i] = fmaf(q, mu_l[j], dot_l[i]);
            }
            if (cb_active)
                *reinterpret_cast<uint2*>(&q_p[(4 * rb + i) * KS + 4 * cb]) =
                    make_uint2(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16));
        }
        // Sum over the 32 lanes of this half-wave (the same four rows).
#pragma unroll
        for (int d = 16; d; d >>= 1)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dot_a[i] += __shfl_xor(dot_a[i], d);
                dot_l[i] += __shfl_xor(dot_l[i], d);
            }
        if (cb == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                q_mu[4 * rb + i] = dot_a[i];
                q_mu[32 + 4 * rb + i] = dot_l[i];
                q_scale[4 * rb + i] = row_scale[i];
            }
        }
    }
    __syncthreads();
    // Q'^T operand (B of S^T = K Q'^T) for the lane's row of the tile,
    // tile_row: chunk m holds channels 16 m + 8 half + e (32-row tiles:
    // tile_row = l % 32, k_group = l / 32) or 32 m + 8 k_group + e (16-row
    // tiles: tile_row = l % 16, k_group = l / 16).
    constexpr int kQChunks = TR == 32 ? G::Parts : D / 32;
    const int tile_row = lane & (TR - 1);
    const int k_group = TR == 32 ? half : lane >> 4;
    F16x8 q_operand[kQChunks];
#pragma unroll
    for (int m = 0; m < kQChunks; ++m)
        q_operand[m] = *reinterpret_cast<const F16x8*>(&q_p[tile_row * KS + (TR == 32 ? 16 : 32) * m + 8 * k_group]);
    const float q_mu_anchor = q_mu[tile_row];
    const float row_scale = q_scale[tile_row];
    const float row_shift = q_mu[32 + (tid >> 3)];  // q'.mu_L of the finish thread's row
    __syncthreads();  // the scratch becomes the tiles

    // ---------------------------------------------------------------- history
    uint16_t* k_tile = reinterpret_cast<uint16_t*>(lds + wave * G::kWaveBytes);
    uint16_t* v_tile = k_tile + kTile * KS;  // [token][VROW] BF16
    float* alpha_tile = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(v_tile) + G::kVBytes);
    // V^T operand reads (ds_read_b64_tr_b16).  32-row tiles: lane 16 g + 4 a
    // + b (g = 2 half + g') addresses token 4 half + a of an 8-token block,
    // channels 32 t + 16 g' + 4 b..+3, and receives channel 32 t + column of
    // tokens 4 half..+3; with the D = 128 swizzle, the 32-channel chunk t
    // sits at position t ^ a.  16-row tiles: lane 16 g + 4 a + b addresses
    // token 4 g + a (and 16 + 4 g + a), channels 16 t + 4 b..+3, and receives
    // channel 16 t + l % 16 of tokens 4 g..+3 (16 + 4 g..+3); with the
    // swizzle, the 16-channel unit t sits at position t ^ (token % 8).
    const int tr_a = (lane >> 2) & 3, tr_b = lane & 3, tr_g = (lane >> 4) & 1;
    const int tr_token = TR == 32 ? 4 * half + tr_a : 4 * k_group + tr_a;
    const int v_lane = TR == 32 ? (G::kSwizzleV ? D * tr_token + 32 * tr_a + 16 * tr_g + 4 * tr_b
                                                : G::VROW * tr_token + 16 * tr_g + 4 * tr_b)
                                : (G::kSwizzleV ? D * tr_token + 16 * (tr_token & 7) + 4 * tr_b
                                                : G::VROW * tr_token + 4 * tr_b);
    auto v_read = [&](int t) __attribute__((always_inline)) {
        constexpr int kStep = TR == 32 ? 32 : 16;
        return G::kSwizzleV ? v_lane ^ (kStep * t) : v_lane + kStep * t;
    };
    const int unit_token = lane >> 2;  // token within a 16-token unit
    const int quarter = lane & 3;      // 32-channel quarter
    const bool quarter_active = quarter < G::Quarters;
    const uint32_t page_bytes = (uint32_t)(PT * p.page_width);
    const int pages = (history + PT - 1) / PT;
    const bool mean_anchor = Decoder::kAnchorMeanTerm && p.key_mean_anchor != nullptr;

    // The split's block ids, once, into LDS (-1 past the history or when invalid).
    const int first_page = tile_begin * kTile / PT;
    int split_pages = tile_end > tile_begin ? ((tile_end * kTile + PT - 1) / PT - first_page) : 0;
    if (split_pages > kMaxSplitPages) split_pages = kMaxSplitPages;  // pages past it read as zeros
    for (int i = tid; i < split_pages; i += kThreads) {
        const int page = first_page + i;
        int block = page < pages ? p.block_table[(int64_t)request * p.block_table_stride + page] : -1;
        split_blocks[i] = (block >= 0 && block < p.num_blocks) ? block : -1;
    }
    __syncthreads();

    // The page resources of one 16-token unit (empty past the history).
    auto unit_pages = [&](int unit_first) __attribute__((always_inline)) {
        const int index = unit_first / PT - first_page;
        // One unit per wave: the block id is wave-uniform, and readfirstlane
        // keeps the page resources in SGPRs (no waterfall loop per load).
        const int block = __builtin_amdgcn_readfirstlane(
            (unit_first < history && index < split_pages) ? split_blocks[index] : -1);
        const uint8_t* k_page = p.cache + ((int64_t)(block >= 0 ? block : 0) * p.heads + head) * page_bytes;
        const uint32_t bytes = block >= 0 ? page_bytes : 0u;
        return UnitPages{page_rsrc(k_page, bytes), page_rsrc(k_page + p.plane_stride, bytes),
                         unit_first % PT + unit_token};
    };

    // O^T: tile t of a 32-row tile holds channels 32 t.. (register r: channel
    // 32 t + 8 (r / 4) + 4 half + r % 4 of row tile_row), of a 16-row tile
    // channels 16 t.. (register r: channel 16 t + 4 k_group + r).
    constexpr int kOutTiles = TR == 32 ? G::Quarters : G::Parts;
    constexpr int kOutRegs = TR == 32 ? 16 : 4;
    typename OutTile<TR>::Type out[kOutTiles];
#pragma unroll
    for (int t = 0; t < kOutTiles; ++t)
#pragma unroll
        for (int r = 0; r < kOutRegs; ++r) out[t][r] = 0.f;
    float running_max = -__builtin_inff();
    float running_sum = 0.f;

    // A wave's units are the two halves of its tiles tile_begin + wave +
    // kWaves k.  The fetches carry no condition (units past the split read
    // zeros through an empty resource), which keeps the compiler's count of
    // loads in flight exact.
    const int first_tile = tile_begin + wave;
    dec.prime(unit_pages(kTile * first_tile), unit_pages(kTile * first_tile + 16));
    // The wave's priority falls as its tiles advance (StreamPriority), which
    // keeps the two workgroups of a compute unit level; it replaced a raised
    // priority over each tile's MFMAs and softmax (residual call 129.3 ->
    // 122.5 us at 16 requests x 16 rows x 8k, A/B on one box).
    const int wave_tiles = first_tile < tile_end ? (tile_end - first_tile + kWaves - 1) / kWaves : 0;
    const StreamPriority priority(wave_tiles, (int64_t)item.total * p.heads <= p.resident);
    int step = 0;
    for (int tile = first_tile; tile < tile_end; tile += kWaves, ++step) {
        priority.set(step);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int local = 16 * u + unit_token;
            const bool valid = kTile * tile + local < history;
            // Whole unit inside the history (wave-uniform): nothing to mask.
            const bool unit_valid = kTile * tile + 16 * u + 16 <= history;
            // The unit after this one, and the one after that.
            const int next_first = u == 0 ? kTile * tile + 16 : kTile * (tile + kWaves);
            const int two_on_first = kTile * (tile + kWaves) + 16 * u;
            auto store_k = [&](const float* lo, const float* hi) __attribute__((always_inline)) {
                uint32_t kw[16];
                // No mask: the scores of tokens past the history become -inf below.
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    kw[c] = pack_f16(lo[2 * c], lo[2 * c + 1]);
                    kw[8 + c] = pack_f16(hi[2 * c], hi[2 * c + 1]);
                }
                if (quarter_active) {
                    uint4* k_dst = reinterpret_cast<uint4*>(&k_tile[local * KS + 32 * quarter]);
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        k_dst[c] = make_uint4(kw[4 * c], kw[4 * c + 1], kw[4 * c + 2], kw[4 * c + 3]);
                }
            };
            auto store_v = [&](const float* lo, const float* hi) __attribute__((always_inline)) {
                uint32_t vw[16];
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    vw[c] = pack_bf16(lo[2 * c], lo[2 * c + 1]);
                    vw[8 + c] = pack_bf16(hi[2 * c], hi[2 * c + 1]);
                }
                // Slots past the history may hold any bytes (P is zero there,
                // but 0 x NaN is not): zero them in a unit that reaches past it.
                if (!unit_valid) {
                    asm volatile("");
#pragma unroll
                    for (int c = 0; c < 16; ++c) vw[c] = valid ? vw[c] : 0u;
                }
                if (quarter_active) {
                    if (TR == 16 && G::kSwizzleV) {
                        // The lane's two 16-channel units 2 quarter and
                        // 2 quarter + 1 at positions unit ^ (token % 8).
                        uint4* lo_dst = reinterpret_cast<uint4*>(&v_tile[local * G::VROW + 16 * ((2 * quarter) ^ (local & 7))]);
                        uint4* hi_dst =
                            reinterpret_cast<uint4*>(&v_tile[local * G::VROW + 16 * ((2 * quarter + 1) ^ (local & 7))]);
                        lo_dst[0] = make_uint4(vw[0], vw[1], vw[2], vw[3]);
                        lo_dst[1] = make_uint4(vw[4], vw[5], vw[6], vw[7]);
                        hi_dst[0] = make_uint4(vw[8], vw[9], vw[10], vw[11]);
                        hi_dst[1] = make_uint4(vw[12], vw[13], vw[14], vw[15]);
                    } else {
                        // Row-major V: the lane's 4 chunks of 8 channels (at D =
                        // 128 at chunk positions 4 (quarter ^ (token % 4)) + i).
                        const int chunk = G::kSwizzleV ? (quarter ^ (local & 3)) : quarter;
                        uint4* v_dst = reinterpret_cast<uint4*>(&v_tile[local * G::VROW + 32 * chunk]);
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            v_dst[c] = make_uint4(vw[4 * c], vw[4 * c + 1], vw[4 * c + 2], vw[4 * c + 3]);
                    }
                }
            };
            const float alpha_k = dec.unit(unit_pages(next_first), unit_pages(two_on_first), store_k, store_v);
            if (quarter == 0) alpha_tile[local] = alpha_k;
        }
        wave_sync();

        if constexpr (TR == 16) {
            // S^T in two 16-token halves: register r of s[h] holds token
            // 16 h + 4 k_group + r against row tile_row (the A operand's lane
            // l % 16 takes token 16 h + l % 16).
            F32x4 s[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int r = 0; r < 4; ++r) s[h][r] = 0.f;
                const uint16_t* k_row = &k_tile[(16 * h + tile_row) * KS + 8 * k_group];
#pragma unroll
                for (int m = 0; m < kQChunks; ++m)
                    s[h] = mfma(*reinterpret_cast<const F16x8*>(k_row + 32 * m), q_operand[m], s[h]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int local = 16 * h + 4 * k_group + r;
                    float x = s[h][r] * row_scale;
                    if (mean_anchor) x = fmaf(alpha_tile[local], q_mu_anchor, x);
                    s[h][r] = x;
                }
            if (kTile * tile + kTile > history) {
                asm volatile("");
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        s[h][r] = kTile * tile + 16 * h + 4 * k_group + r < history ? s[h][r] : -__builtin_inff();
            }
            // The row's scores sit in lanes l % 16 + 16 k_group.
            float tile_max = -__builtin_inff();
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) tile_max = fmaxf(tile_max, s[h][r]);
            tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16));
            tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
            const float new_max = fmaxf(running_max, tile_max);
            const float base = new_max == -__builtin_inff() ? 0.f : new_max;
            const float rescale = __builtin_amdgcn_exp2f(running_max - base);
            running_max = new_max;
            // P^T in BF16 as the B operand of O^T += V^T P^T: k-slot
            // 8 k_group + e is token 4 k_group + e (s[0][e]) for e < 4 and
            // 16 + 4 k_group + e - 4 (s[1][e - 4]) for e >= 4.
            float tile_sum = 0.f;
            Bf16x8 p_operand;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float w = __builtin_amdgcn_exp2f(s[h][r] - base);
                    p_operand[4 * h + r] = (__bf16)w;
                    tile_sum += w;
                }
            tile_sum += __shfl_xor(tile_sum, 16);
            tile_sum += __shfl_xor(tile_sum, 32);
            running_sum = running_sum * rescale + tile_sum;
            if (!__all(rescale == 1.0f)) {
#pragma unroll
                for (int t = 0; t < kOutTiles; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) out[t][r] *= rescale;
            }
#pragma unroll
            for (int t = 0; t < kOutTiles; ++t) {
                // Tokens 4 k_group + 0..3 and 16 + 4 k_group + 0..3, as P^T's k-slots.
                const Short4 lo = read_transposed(v_tile + v_read(t));
                const Short4 hi = read_transposed(v_tile + 16 * G::VROW + v_read(t));
                out[t] = mfma(__builtin_bit_cast(Bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)),
                              p_operand, out[t]);
            }
        } else {
            // S^T: register r of lane l holds token 8 (r / 4) + 4 half + r % 4 against row `column`.
            F32x16 s;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
            const uint16_t* k_row = &k_tile[column * KS + 8 * half];
#pragma unroll
            for (int m = 0; m < G::Parts; ++m)
                s = mfma(*reinterpret_cast<const F16x8*>(k_row + 16 * m), q_operand[m], s);

#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int local = 8 * (r >> 2) + 4 * half + (r & 3);
                float x = s[r] * row_scale;
                if (mean_anchor) x = fmaf(alpha_tile[local], q_mu_anchor, x);
                s[r] = x;
            }
            // Tokens past the history score -inf (only in the tile that reaches past it).
            if (kTile * tile + kTile > history) {
                asm volatile("");
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[r] = kTile * tile + 8 * (r >> 2) + 4 * half + (r & 3) < history ? s[r] : -__builtin_inff();
            }
            float tile_max = -__builtin_inff();
#pragma unroll
            for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s[r]);
            tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
            const float new_max = fmaxf(running_max, tile_max);
            const float base = new_max == -__builtin_inff() ? 0.f : new_max;
            const float rescale = __builtin_amdgcn_exp2f(running_max - base);
            running_max = new_max;
            // P^T in BF16 as the B operand of O^T += V^T P^T: step j takes
            // registers 8j..8j+7, i.e. k-slot (half, e) is token
            // 16 j + 4 half + e + (e >= 4 ? 4 : 0).
            float tile_sum = 0.f;
            Bf16x8 p_operand[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float w = __builtin_amdgcn_exp2f(s[8 * j + e] - base);
                    p_operand[j][e] = (__bf16)w;
                    tile_sum += w;
                }
            tile_sum += __shfl_xor(tile_sum, 32);
            running_sum = running_sum * rescale + tile_sum;
            if (!__all(rescale == 1.0f)) {
#pragma unroll
                for (int t = 0; t < G::Quarters; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) out[t][r] *= rescale;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint16_t* v_rows = v_tile + 16 * j * G::VROW;
#pragma unroll
                for (int t = 0; t < G::Quarters; ++t) {
                    // Tokens 4 half + 0..3 and 4 half + 8..11 of the 16, as P^T's k-slots.
                    const Short4 lo = read_transposed(v_rows + v_read(t));
                    const Short4 hi = read_transposed(v_rows + 8 * G::VROW + v_read(t));
                    out[t] = mfma(__builtin_bit_cast(Bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)),
                                  p_operand[j], out[t]);
                }
            }
        }
        wave_sync();  // the next tile overwrites this one
    }
    __builtin_amdgcn_s_setprio(0);

    // ---------------------------------------------------------------- wave merge
    __syncthreads();  // the merge buffer aliases every wave's tiles
    constexpr int MS = G::MS;
    float* merge_o = reinterpret_cast<float*>(lds);
    float* merge_ml = reinterpret_cast<float*>(lds + G::kMlOffset);
    if constexpr (TR == 16) {
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t)
            *reinterpret_cast<float4*>(&merge_o[(wave * 32 + tile_row) * MS + 16 * t + 4 * k_group]) =
                make_float4(out[t][0], out[t][1], out[t][2], out[t][3]);
    } else {
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4*>(&merge_o[(wave * 32 + column) * MS + 32 * t + 8 * g + 4 * half]) =
                    make_float4(out[t][4 * g], out[t][4 * g + 1], out[t][4 * g + 2], out[t][4 * g + 3]);
    }
    if (k_group == 0) {
        merge_ml[(wave * 32 + tile_row) * 2] = running_max;
        merge_ml[(wave * 32 + tile_row) * 2 + 1] = running_sum;
    }
    __syncthreads();
    FinishInputs<D> in;
    finish_load<D, TR>(p, head, first, row0, n, in);
    const int r = tid >> 3, chunk = tid & 7;  // row, 16-channel chunk
    const bool chunk_active = chunk < G::Parts;
    const bool valid = r < TR && row0 + r < n;
    float total_max = -__builtin_inff(), l = 0.f, o[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) o[c] = 0.f;
    if (r < TR) {
        float m_w[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            m_w[w] = merge_ml[(w * 32 + r) * 2];
            total_max = fmaxf(total_max, m_w[w]);
        }
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            if (m_w[w] == -__builtin_inff()) continue;
            const float weight = __builtin_amdgcn_exp2f(m_w[w] - total_max);
            l = fmaf(merge_ml[(w * 32 + r) * 2 + 1], weight, l);
            const float* src = &merge_o[(w * 32 + r) * MS + 16 * (chunk_active ? chunk : 0)];
#pragma unroll
            for (int c = 0; c < 16; ++c) o[c] = fmaf(src[c], weight, o[c]);
        }
    }
    if (item.splits > 1) {
        // One resource over the tile's entries (wave-uniform); the row is a lane offset.
        const int tile_rows = n - row0 < TR ? n - row0 : TR;
        const __amdgpu_buffer_rsrc_t entries =
            handoff_resource(tile_entries, (uint32_t)(tile_rows * item.splits * kMultiRowEntry * 4));
        const uint32_t row_at = (uint32_t)((valid ? r : 0) * item.splits * kMultiRowEntry * 4);
        const uint32_t at = row_at + (uint32_t)(split * kMultiRowEntry * 4);
        if (valid && chunk == 0) {
            handoff_store(entries, at, total_max);
            handoff_store(entries, at + 4, l);
        }
        if (valid && chunk_active) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                handoff_store4(entries, at + 16 + 64 * chunk + 16 * c, o[4 * c], o[4 * c + 1], o[4 * c + 2],
                               o[4 * c + 3]);
        }
        // (The flag aliases the merge buffer, which every thread has read by then.)
        if (!arrive_last_tagged(arrivals, item.splits, reinterpret_cast<int*>(lds))) return;
        finish_merge(entries, row_at, item.splits, valid, chunk_active ? chunk : 0, total_max, l, o);
    }
    __syncthreads();  // the finish's tiles alias the merge buffer
    finish_rows<D, TR>(p, head, first, row0, n, in, row_shift, total_max, l, o, lds);
}

template <int D, int PT, int TR, bool HasL, int BA, int GA, int BL, int GL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void multirow_stream_kernel(MultiRowParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[Geometry<D, TR>::kLdsBytes];
    __shared__ int split_blocks[kMaxSplitPages];  // block ids of the split's pages
    AnchorDecoder<PT, HasL, BA, GA, BL, GL> dec;
    dec.anchor = p.anchor;
    dec.residual = p.residual;
    const int quarter = threadIdx.x & 3;
    dec.lq = quarter < Geometry<D>::Quarters ? quarter : 0;
    multirow_stream<D, PT, TR>(p, dec, lds, split_blocks);
}

template <int D, int PT, int TR, int Links>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void multirow_chain_kernel(MultiRowParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[Geometry<D, TR>::kLdsBytes];
    __shared__ int split_blocks[kMaxSplitPages];  // block ids of the split's pages
    // bf16(mu_r) of records 0 .. L - 1 (the K plane's chain), FP32.
    __shared__ __attribute__((aligned(16))) float mean_lds[Links - 1][kMaxD];
    const int head = stream_head(p);
    const bool has_mean = p.key_mean_all != nullptr;
    for (int i = threadIdx.x; i < (Links - 1) * kMaxD; i += kThreads) {
        const int r = i / kMaxD, c = i % kMaxD;
        mean_lds[r][c] = (has_mean && c < D) ? bf16_f32(bf16_rn(p.key_mean_all[((int64_t)r * p.heads + head) * D + c]))
                                             : 0.f;
    }
    // (The stream's first barrier orders these stores before any read.)
    ChainDecoder<D, PT, Links> dec;
#pragma unroll
    for (int r = 0; r < Links; ++r) dec.regs[r] = p.chain[r];
    dec.mean = &mean_lds[0][0];
    dec.add_mean = has_mean;
    const int quarter = threadIdx.x & 3;
    dec.lq = quarter < Geometry<D>::Quarters ? quarter : 0;
    // The pairs (1, 0) and (0, 1) of the mean add, in registers.
    uint32_t pick_lo = 0x00003f80u, pick_hi = 0x3f800000u;
    asm("" : "+v"(pick_lo), "+v"(pick_hi));
    dec.pick_lo = pick_lo;
    dec.pick_hi = pick_hi;
    multirow_stream<D, PT, TR>(p, dec, lds, split_blocks);
}

template <int TR>
dim3 stream_grid(const MultiRowParams& p) {
    // Planned items head by head, so that the workgroups past the plan come
    // last: one that waits for a compute unit's LDS before it can exit holds
    // back every workgroup behind it (24 requests x 16 rows x 4096 tokens,
    // half of the workgroups past the plan: 146 us per residual call with
    // them in between, 121 us without).
    if (p.items > 0) return dim3((unsigned)((int64_t)p.items * p.heads));
    return dim3((unsigned)p.requests, (unsigned)p.heads, (unsigned)(p.splits * ((p.rows + TR - 1) / TR)));
}

// The launch parameters with `resident` set: the stream workgroups that the
// device holds at once.
MultiRowParams with_resident(const MultiRowParams& params, int per_cu) {
    MultiRowParams p = params;
    p.resident = (int64_t)per_cu * p.compute_units;
    return p;
}

template <int D, int PT, int TR, bool HasL, int BA, int GA, int BL, int GL>
void launch_one(const MultiRowParams& p, hipStream_t stream) {
    const auto kernel = multirow_stream_kernel<D, PT, TR, HasL, BA, GA, BL, GL>;
    static const int per_cu = resident_per_cu(reinterpret_cast<const void*>(kernel), kThreads);
    hipLaunchKernelGGL(kernel, stream_grid<TR>(p), dim3(kThreads), 0, stream, with_resident(p, per_cu));
}

template <int D, int PT, int TR, int Links>
void launch_chain(const MultiRowParams& p, hipStream_t stream) {
    const auto kernel = multirow_chain_kernel<D, PT, TR, Links>;
    static const int per_cu = resident_per_cu(reinterpret_cast<const void*>(kernel), kThreads);
    hipLaunchKernelGGL(kernel, stream_grid<TR>(p), dim3(kThreads), 0, stream, with_resident(p, per_cu));
}

template <int D, int PT, int TR, int BA, int GA, int BL>
void launch_residual_group(const MultiRowParams& p, hipStream_t stream) {
    if (p.residual.group == 32)
        launch_one<D, PT, TR, true, BA, GA, BL, 32>(p, stream);
    else
        launch_one<D, PT, TR, true, BA, GA, BL, 16>(p, stream);
}

template <int D, int PT, int TR, int BA, int GA>
void launch_anchor(const MultiRowParams& p, hipStream_t stream) {
    if (!p.has_residual)
        launch_one<D, PT, TR, false, BA, GA, 2, 32>(p, stream);
    else if (p.residual.bits == 2)
        launch_residual_group<D, PT, TR, BA, GA, 2>(p, stream);
    else
        launch_residual_group<D, PT, TR, BA, GA, 4>(p, stream);
}

template <int D, int PT, int TR, int BA>
void launch_anchor_group(const MultiRowParams& p, hipStream_t stream) {
    if (p.anchor.group == 32)
        launch_anchor<D, PT, TR, BA, 32>(p, stream);
    else
        launch_anchor<D, PT, TR, BA, 16>(p, stream);
}

template <int D, int PT, int TR>
bool launch_tr(const MultiRowParams& p, hipStream_t stream) {
    if (p.chain_length > 1) {
        switch (p.chain_length) {
            case 2: launch_chain<D, PT, TR, 2>(p, stream); return true;
            case 3: launch_chain<D, PT, TR, 3>(p, stream); return true;
            case 4: launch_chain<D, PT, TR, 4>(p, stream); return true;
            default: return false;
        }
    }
    if (p.anchor.bits == 4)
        launch_anchor_group<D, PT, TR, 4>(p, stream);
    else
        launch_anchor_group<D, PT, TR, 2>(p, stream);
    return true;
}

template <int D, int PT>
bool launch_pt(const MultiRowParams& p, hipStream_t stream) {
    return p.tile_rows == 16 ? launch_tr<D, PT, 16>(p, stream) : launch_tr<D, PT, 32>(p, stream);
}

template <int D>
bool launch_d(const MultiRowParams& p, hipStream_t stream) {
    bool launched = false;
    if (p.page_tokens == 16)
        launched = launch_pt<D, 16>(p, stream);
    else if (p.page_tokens == 32)
        launched = launch_pt<D, 32>(p, stream);
    return launched;
}

}  // namespace

// One object per head dim (RQ_HEAD_DIM), compiled side by side.
template <>
hipError_t launch_multirow<RQ_HEAD_DIM>(const MultiRowParams& p, hipStream_t stream) {
    if (p.rows == 0 || p.requests == 0) return hipSuccess;
    return launch_d<RQ_HEAD_DIM>(p, stream) ? hipGetLastError() : hipErrorInvalidValue;
}

}  // namespace rq
