// Attention of many query rows per request (a prompt chunk) over packed pages
// on MFMA tiles (gfx950, wave64), for head dims 96 and 128, anchor and
// adjacent mode.  The semantics are those of multirow.hip, whose kernels take
// the calls of few rows per request.
//
// chunk_stream_kernel: one workgroup of 8 waves takes up to 256 rows of one
// (request, head), 32 per wave, and a split of its history.  Each step
// dequantizes 128 tokens into LDS, one 16-token unit per wave (FP16 K, BF16
// V), and every wave multiplies all of them with its own rows: 16-token units
// are dequantized once per 256 rows, where multirow.hip's 32-row tiles do it
// once per 32 (dequantizing is 3/4 of their vector instructions).  The tiles
// are double-buffered with one barrier per step.  A split writes one partial
// (m, l, O) per row.  Bound: the vector work (53% of the SIMD cycles at 2
// requests of 8192 tokens x 509 rows x 16 heads) and the matrix work (31%),
// which hardly overlap on a SIMD (the two waves of a SIMD in opposite order, or
// 64 tokens per softmax in place of 32, changed nothing; row sums of the rounded
// weights by dot products were slower); where whole splits do not fill the
// compute units, those without a workgroup (12% at 4518 and 6000 tokens).
//
// chunk_finish_kernel: 32 rows of one (request, head) per workgroup of 4
// waves merge the splits, apply R_v^T, add the live tokens and write the
// output, as the last split of a tile does in multirow.hip (rq_multirow.h).
//
// Measured (2 requests of 4518 and 6000 tokens x 509 rows x 16 heads, causal,
// residual loop / anchor loop): 289 / 250 us per call on 32-row tiles with the
// live tokens on the vector units; here 104 / 97 us (stream 85 / 77).
#include "rq_multirow.h"

namespace rq {

namespace {

constexpr int kStreamThreads = 512;
constexpr int kStreamWaves = 8;
constexpr int kUnits = kChunkUnit / 16;  // units per step, one per wave
static_assert(kUnits == kStreamWaves && kChunkTileRows == 32 * kStreamWaves, "one unit and 32 rows per wave");

// Tiles of T tokens: K rows of KS halves, V rows of VROW halves whose 32-channel
// chunks sit at q ^ (token % 4) at D = 128 (see Geometry in rq_multirow.h).
template <int D, int T>
struct Tile {
    static constexpr int KS = D + 8;
    static constexpr bool kSwizzleV = D == 128;
    static constexpr int VROW = D == 128 ? D : D + 8;
    static constexpr int kKBytes = T * KS * 2;
    static constexpr int kVBytes = T * VROW * 2;
    static constexpr int kAlphaBytes = T * 4;
    static constexpr int kBytes = kKBytes + kVBytes + kAlphaBytes;
    // Lane offset (halves) of a transposed V read: lane 16 g + 4 a + b (g = 2
    // half + g') addresses token 4 half + a of an 8-token block, channels 16
    // g' + 4 b..+3 of a 32-channel chunk t (v_at), and receives channel 32 t +
    // l % 32 of tokens 4 half..+3.
    __device__ static int v_lane(int lane) {
        const int half = lane >> 5, a = (lane >> 2) & 3, b = lane & 3, g = (lane >> 4) & 1;
        return VROW * (4 * half + a) + (kSwizzleV ? 32 * a : 0) + 16 * g + 4 * b;
    }
    __device__ static int v_at(int v_lane, int t) { return kSwizzleV ? v_lane ^ (32 * t) : v_lane + 32 * t; }
    __device__ static int v_chunk(int token, int chunk) { return kSwizzleV ? chunk ^ (token & 3) : chunk; }
};

// The value of lane l and of lane l ^ 32, low half first in every lane.
__device__ __forceinline__ float2 halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_max(float v) {
    const float2 h = halves(v);
    return fmaxf(h.x, h.y);
}
__device__ __forceinline__ float halves_sum(float v) {
    const float2 h = halves(v);
    return h.x + h.y;
}

// Channel of register r of a 32 x 32 C tile t of lane half `half`.
__device__ __forceinline__ int c_channel(int t, int r, int half) { return 32 * t + 8 * (r >> 2) + 4 * half + (r & 3); }

// Rows of a request's tiles: as many tiles as kChunkTileRows needs, of equal
// rows in whole waves.
__device__ __forceinline__ int tile_step(int rows) {
    const int tiles = (rows + kChunkTileRows - 1) / kChunkTileRows;
    return 32 * (((rows + 31) / 32 + tiles - 1) / tiles);
}

// ---------------------------------------------------------------- history

template <int D, int PT, class Decoder>
__device__ __forceinline__ void chunk_stream(const MultiRowParams& p, Decoder& dec, uint8_t* lds, int* split_blocks) {
    using L = Tile<D, kChunkUnit>;
    constexpr int KS = L::KS, Quarters = D / 32, Parts = D / 16;
    const int head = (int)(blockIdx.x % (unsigned)p.heads);
    const PlanItem item = multirow_plan<false>(p, (int)(blockIdx.x / (unsigned)p.heads), 0, 0, 0);
    const int request = __builtin_amdgcn_readfirstlane(item.request);
    if (request < 0) return;
    const int first = __builtin_amdgcn_readfirstlane(item.first), n = __builtin_amdgcn_readfirstlane(item.rows);
    const int row0 = tile_step(n) * __builtin_amdgcn_readfirstlane(item.index);
    const int row_end = min(n, row0 + tile_step(n));
    if (row0 >= row_end) return;  // uniform over the workgroup, before any barrier
    const int history = __builtin_amdgcn_readfirstlane(item.tokens);
    const int step_begin = __builtin_amdgcn_readfirstlane(split_begin(item.length, item.split, item.splits));
    const int step_end = __builtin_amdgcn_readfirstlane(split_begin(item.length, item.split + 1, item.splits));

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, column = lane & 31, half = lane >> 5;
    const bool wave_active = row0 + 32 * wave < row_end;  // wave-uniform
    const int row = row0 + 32 * wave + column;
    const bool row_valid = row < row_end;
    const uint16_t* query = p.query + (int64_t)(first + (row_valid ? row : row_end - 1)) * p.query_stride + head * D;

    // The split's block ids, once, into LDS (-1 past the history or when invalid).
    const int pages = (history + PT - 1) / PT;
    const int first_page = step_begin * kChunkUnit / PT;
    int split_pages = (step_end - step_begin) * (kChunkUnit / PT);
    if (split_pages > kMaxSplitPages) split_pages = kMaxSplitPages;  // (the plan keeps them below)
    for (int i = tid; i < split_pages; i += kStreamThreads) {
        const int page = first_page + i;
        const int block = page < pages ? p.block_table[(int64_t)request * p.block_table_stride + page] : -1;
        split_blocks[i] = (block >= 0 && block < p.num_blocks) ? block : -1;
    }

    // ---------------------------------------------------------------- q'
    // q' = (q . R_k) * log2(e) / sqrt(D) of the wave's rows as the B operand
    // of S^T = K Q'^T, FP16 scaled by the row's power of two 2^-e.  The
    // product is taken as (R_k^T q^T), whose C layout puts 64 channels of row
    // l % 32 into lane l: k-slot (half, e) of step m is channel 16 m + 8 (e /
    // 4) + 4 half + e % 4, and the K tile's rows are stored in that order.
    uint16_t* r_k = reinterpret_cast<uint16_t*>(lds);  // [D][KS] FP16, aliases the tiles
    F32x16 x[Quarters];
    if (p.key_rotation) {
        constexpr int kChunks = D / 8;
        const uint4* src = reinterpret_cast<const uint4*>(p.key_rotation + (int64_t)head * D * D);
#pragma unroll
        for (int i = tid; i < D * kChunks; i += kStreamThreads)
            *reinterpret_cast<uint4*>(&r_k[(i / kChunks) * KS + 8 * (i % kChunks)]) = src[i];
        // The row scaled by a power of two into [-1, 1]: exact in FP16.
        uint2 words[Parts][2];
        float magnitude = 0.f;
#pragma unroll
        for (int m = 0; m < Parts; ++m)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                words[m][i] = *reinterpret_cast<const uint2*>(query + 16 * m + 8 * half + 4 * i);
                magnitude = fmaxf(magnitude, fmaxf(fabsf(bf16_f32(words[m][i].x & 0xffffu)), fabsf(bf16_f32(words[m][i].x >> 16))));
                magnitude = fmaxf(magnitude, fmaxf(fabsf(bf16_f32(words[m][i].y & 0xffffu)), fabsf(bf16_f32(words[m][i].y >> 16))));
            }
        magnitude = halves_max(magnitude);
        const int f = magnitude > 0.f ? min(__builtin_amdgcn_frexp_expf(magnitude), 127) : 0;
        const float down = ldexpf(1.0f, -f), up = ldexpf(1.0f, f) * kScoreScale<D>;
        F16x8 q[Parts];
#pragma unroll
        for (int m = 0; m < Parts; ++m)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                q[m][4 * i] = (_Float16)(bf16_f32(words[m][i].x & 0xffffu) * down);
                q[m][4 * i + 1] = (_Float16)(bf16_f32(words[m][i].x >> 16) * down);
                q[m][4 * i + 2] = (_Float16)(bf16_f32(words[m][i].y & 0xffffu) * down);
                q[m][4 * i + 3] = (_Float16)(bf16_f32(words[m][i].y >> 16) * down);
            }
        __syncthreads();
        // A: R_k[k][c] at c = 32 t + l % 32 and k = 16 m + 8 half + e, read
        // transposed from the row-major tile.
        const int group = lane >> 4, lane16 = lane & 15;
#pragma unroll
        for (int t = 0; t < Quarters; ++t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) x[t][r] = 0.f;
#pragma unroll
            for (int m = 0; m < Parts; ++m) {
                const int k0 = 16 * m + 8 * (group >> 1), c0 = 32 * t + 16 * (group & 1);
                const Short4 lo = read_transposed(&r_k[(k0 + (lane16 >> 2)) * KS + c0 + 4 * (lane16 & 3)]);
                const Short4 hi = read_transposed(&r_k[(k0 + 4 + (lane16 >> 2)) * KS + c0 + 4 * (lane16 & 3)]);
                const F16x8 a = __builtin_bit_cast(F16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                x[t] = mfma(a, q[m], x[t]);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) x[t][r] *= up;
        }
    } else {
#pragma unroll
        for (int t = 0; t < Quarters; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint2 w = *reinterpret_cast<const uint2*>(query + 32 * t + 8 * j + 4 * half);
                x[t][4 * j] = bf16_f32(w.x & 0xffffu) * kScoreScale<D>;
                x[t][4 * j + 1] = bf16_f32(w.x >> 16) * kScoreScale<D>;
                x[t][4 * j + 2] = bf16_f32(w.y & 0xffffu) * kScoreScale<D>;
                x[t][4 * j + 3] = bf16_f32(w.y >> 16) * kScoreScale<D>;
            }
    }
    float row_max = 0.f;
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) row_max = fmaxf(row_max, fabsf(x[t][r]));
    row_max = halves_max(row_max);
    const int exponent = row_max > 0.f ? __builtin_amdgcn_frexp_expf(row_max) : 0;
    const float row_scale = ldexpf(1.0f, exponent), inverse = ldexpf(1.0f, -exponent);
    F16x8 q_operand[Parts];
    float dot_anchor = 0.f, dot_loop = 0.f;  // q'.bf16(mu_A) 2^-e, q'.mu_L
    const bool mean_anchor = Decoder::kAnchorMeanTerm && p.key_mean_anchor != nullptr;
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int channel = head * D + c_channel(t, 4 * j, half);
            float4 mu_a = make_float4(0.f, 0.f, 0.f, 0.f), mu_l = mu_a;
            if (mean_anchor) mu_a = *reinterpret_cast<const float4*>(p.key_mean_anchor + channel);
            if (p.key_mean_loop) mu_l = *reinterpret_cast<const float4*>(p.key_mean_loop + channel);
            const float a[4] = {mu_a.x, mu_a.y, mu_a.z, mu_a.w}, l[4] = {mu_l.x, mu_l.y, mu_l.z, mu_l.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const _Float16 h = (_Float16)(x[t][4 * j + i] * inverse);
                q_operand[2 * t + (j >> 1)][4 * (j & 1) + i] = h;
                dot_anchor = fmaf((float)h, round_bf16(a[i]), dot_anchor);
                dot_loop = fmaf((float)h * row_scale, l[i], dot_loop);
            }
        }
    dot_anchor = halves_sum(dot_anchor);
    dot_loop = halves_sum(dot_loop);
    __syncthreads();  // the scratch becomes the tiles; the block ids are in LDS

    // ---------------------------------------------------------------- tiles
    const int unit_token = lane >> 2, quarter = lane & 3;
    const bool quarter_active = quarter < Quarters;
    const uint32_t page_bytes = (uint32_t)(PT * p.page_width);
    // The page resources of the wave's unit of a step (empty past the split).
    auto unit_pages = [&](int step) __attribute__((always_inline)) {
        const int unit_first = kChunkUnit * step + 16 * wave;
        const int index = unit_first / PT - first_page;
        const int block = __builtin_amdgcn_readfirstlane(
            (unit_first < history && index < split_pages) ? split_blocks[index] : -1);
        const uint8_t* k_page = p.cache + ((int64_t)(block >= 0 ? block : 0) * p.heads + head) * page_bytes;
        const uint32_t bytes = block >= 0 ? page_bytes : 0u;
        return UnitPages{page_rsrc(k_page, bytes), page_rsrc(k_page + p.plane_stride, bytes),
                         unit_first % PT + unit_token};
    };
    const int local = 16 * wave + unit_token;
    // The wave's unit of a step into the tiles of `buffer`, after the loads of
    // its unit two steps on are issued (AnchorDecoder; one step on in
    // ChainDecoder).
    auto dequantize = [&](int step, uint8_t* buffer) __attribute__((always_inline)) {
        uint16_t* k_tile = reinterpret_cast<uint16_t*>(buffer);
        uint16_t* v_tile = reinterpret_cast<uint16_t*>(buffer + L::kKBytes);
        float* alpha_tile = reinterpret_cast<float*>(buffer + L::kKBytes + L::kVBytes);
        const int unit_first = kChunkUnit * step + 16 * wave;
        const bool unit_whole = unit_first + 16 <= history;  // wave-uniform
        const bool valid = unit_first + unit_token < history;
        auto store_k = [&](const float* lo, const float* hi) __attribute__((always_inline)) {
            // 16-channel blocks in the order of the k-slots: 0-3, 8-11, 4-7, 12-15.
            constexpr int kOrder[8] = {0, 2, 8, 10, 4, 6, 12, 14};
            uint32_t w[16];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                w[c] = pack_f16(lo[kOrder[c]], lo[kOrder[c] + 1]);
                w[8 + c] = pack_f16(hi[kOrder[c]], hi[kOrder[c] + 1]);
            }
            if (quarter_active) {
                uint4* dst = reinterpret_cast<uint4*>(&k_tile[local * KS + 32 * quarter]);
#pragma unroll
                for (int c = 0; c < 4; ++c) dst[c] = make_uint4(w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]);
            }
        };
        auto store_v = [&](const float* lo, const float* hi) __attribute__((always_inline)) {
            uint32_t w[16];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                w[c] = pack_bf16(lo[2 * c], lo[2 * c + 1]);
                w[8 + c] = pack_bf16(hi[2 * c], hi[2 * c + 1]);
            }
            // Slots past the history may hold any bytes (P is zero there, but
            // 0 x NaN is not): zero them in a unit that reaches past it.
            if (!unit_whole) {
                asm volatile("");
#pragma unroll
                for (int c = 0; c < 16; ++c) w[c] = valid ? w[c] : 0u;
            }
            if (quarter_active) {
                uint4* dst = reinterpret_cast<uint4*>(&v_tile[local * L::VROW + 32 * L::v_chunk(local, quarter)]);
#pragma unroll
                for (int c = 0; c < 4; ++c) dst[c] = make_uint4(w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]);
            }
        };
        const float alpha = dec.unit(unit_pages(step + 1), unit_pages(step + 2), store_k, store_v);
        if (quarter == 0) alpha_tile[local] = alpha;
    };

    F32x16 out[Quarters];
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[t][r] = 0.f;
    float running_max = -__builtin_inff(), running_sum = 0.f;  // log2 units; this half's tokens
    const int v_lane = L::v_lane(lane);
    // The wave's rows against the 128 tokens of `buffer`.
    auto multiply = [&](int step, const uint8_t* buffer) __attribute__((always_inline)) {
        if (!wave_active) return;
        const uint16_t* k_tile = reinterpret_cast<const uint16_t*>(buffer);
        const uint16_t* v_tile = reinterpret_cast<const uint16_t*>(buffer + L::kKBytes);
        const float* alpha_tile = reinterpret_cast<const float*>(buffer + L::kKBytes + L::kVBytes);
#pragma unroll 1
        for (int pair = 0; pair < kChunkUnit / 64; ++pair) {
            const int token0 = kChunkUnit * step + 64 * pair;
            if (token0 >= history) return;
            // S^T of two 32-token tiles: their chains of MFMAs are independent.
            F32x16 s[2];
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[sub][r] = 0.f;
            const uint16_t* k_row = &k_tile[(64 * pair + column) * KS + 8 * half];
#pragma unroll
            for (int m = 0; m < Parts; ++m)
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
                    s[sub] = mfma(*reinterpret_cast<const F16x8*>(k_row + 32 * sub * KS + 16 * m), q_operand[m], s[sub]);
            // Raw scores: 2^e (row_scale) is positive and joins the exponent's fma.
            if (mean_anchor) {
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float4 a =
                            *reinterpret_cast<const float4*>(&alpha_tile[64 * pair + 32 * sub + 8 * j + 4 * half]);
                        s[sub][4 * j] = fmaf(a.x, dot_anchor, s[sub][4 * j]);
                        s[sub][4 * j + 1] = fmaf(a.y, dot_anchor, s[sub][4 * j + 1]);
                        s[sub][4 * j + 2] = fmaf(a.z, dot_anchor, s[sub][4 * j + 2]);
                        s[sub][4 * j + 3] = fmaf(a.w, dot_anchor, s[sub][4 * j + 3]);
                    }
            }
            if (token0 + 64 > history) {
                asm volatile("");
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        s[sub][r] = token0 + 32 * sub + 8 * (r >> 2) + 4 * half + (r & 3) < history
                                        ? s[sub][r]
                                        : -__builtin_inff();
            }
            float tile_max = -__builtin_inff();
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s[sub][r]);
            tile_max = halves_max(tile_max) * row_scale;
            // (A row's maximum is kept exact: its own weight is then 1, which
            // BF16 holds.  Rescaling only when it grows by 2^8 raised the
            // error against float64 from 1.9e-3 to 2.3e-3.)
            const float new_max = fmaxf(running_max, tile_max);
            const float base = new_max == -__builtin_inff() ? 0.f : new_max;
            const float rescale = __builtin_amdgcn_exp2f(running_max - base);
            running_max = new_max;
            if (!__all(rescale == 1.0f)) {
#pragma unroll
                for (int t = 0; t < Quarters; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) out[t][r] *= rescale;
            }
            float tile_sum = 0.f;
            Bf16x8 probs[2][2];
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float w = __builtin_amdgcn_exp2f(fmaf(s[sub][8 * j + e], row_scale, -base));
                        probs[sub][j][e] = (__bf16)w;
                        tile_sum += w;
                    }
            running_sum = running_sum * rescale + tile_sum;
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint16_t* v_rows = v_tile + (64 * pair + 32 * sub + 16 * j) * L::VROW;
#pragma unroll
                    for (int t = 0; t < Quarters; ++t) {
                        // Tokens 4 half + 0..3 and 4 half + 8..11 of the 16, as P^T's k-slots.
                        const Short4 lo = read_transposed(v_rows + L::v_at(v_lane, t));
                        const Short4 hi = read_transposed(v_rows + 8 * L::VROW + L::v_at(v_lane, t));
                        out[t] = mfma(
                            __builtin_bit_cast(Bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)),
                            probs[sub][j], out[t]);
                    }
                }
        }
    };

    // Step s multiplies buffer s & 1 while step s + 1 fills the other, which
    // every wave finished reading before the barrier that ended step s - 1.
    auto buffer_of = [&](int step) { return lds + (step & 1) * L::kBytes; };
    if (step_begin < step_end) {
        dec.prime(unit_pages(step_begin), unit_pages(step_begin + 1));
        dequantize(step_begin, buffer_of(step_begin));
    }
    lds_barrier();
    for (int step = step_begin; step < step_end; ++step) {
        if (step + 1 < step_end) dequantize(step + 1, buffer_of(step + 1));
        multiply(step, buffer_of(step));
        lds_barrier();
    }

    // ---------------------------------------------------------------- partial
    running_sum = halves_sum(running_sum);
    if (!row_valid) return;
    float* entry = p.partials +
                   ((int64_t)head * p.entries + item.entry + row * item.splits + item.split) * kMultiRowEntry;
    if (half == 0) *reinterpret_cast<float4*>(entry) = make_float4(running_max, running_sum, dot_loop, 0.f);
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<float4*>(entry + 4 + c_channel(t, 4 * j, half)) =
                make_float4(out[t][4 * j], out[t][4 * j + 1], out[t][4 * j + 2], out[t][4 * j + 3]);
}

template <int D, int PT, bool HasL, int BA, int GA, int BL, int GL>
__global__ __launch_bounds__(kStreamThreads) __attribute__((amdgpu_waves_per_eu(2)))
void chunk_stream_kernel(MultiRowParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * Tile<D, kChunkUnit>::kBytes];
    __shared__ int split_blocks[kMaxSplitPages];  // block ids of the split's pages
    AnchorDecoder<PT, HasL, BA, GA, BL, GL> dec;
    dec.anchor = p.anchor;
    dec.residual = p.residual;
    const int quarter = threadIdx.x & 3;
    dec.lq = quarter < D / 32 ? quarter : 0;
    chunk_stream<D, PT>(p, dec, lds, split_blocks);
}

template <int D, int PT, int Links>
__global__ __launch_bounds__(kStreamThreads) __attribute__((amdgpu_waves_per_eu(2)))
void chunk_chain_kernel(MultiRowParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * Tile<D, kChunkUnit>::kBytes];
    __shared__ int split_blocks[kMaxSplitPages];  // block ids of the split's pages
    // bf16(mu_r) of records 0 .. L - 1 (the K plane's chain), FP32.
    __shared__ __attribute__((aligned(16))) float mean_lds[Links - 1][kMaxD];
    const int head = (int)(blockIdx.x % (unsigned)p.heads);
    const bool has_mean = p.key_mean_all != nullptr;
    for (int i = threadIdx.x; i < (Links - 1) * kMaxD; i += kStreamThreads) {
        const int r = i / kMaxD, c = i % kMaxD;
        mean_lds[r][c] = (has_mean && c < D) ? round_bf16(p.key_mean_all[((int64_t)r * p.heads + head) * D + c]) : 0.f;
    }
    // (The stream's first barrier orders these stores before any read.)
    ChainDecoder<D, PT, Links> dec;
#pragma unroll
    for (int r = 0; r < Links; ++r) dec.regs[r] = p.chain[r];
    dec.mean = &mean_lds[0][0];
    dec.add_mean = has_mean;
    const int quarter = threadIdx.x & 3;
    dec.lq = quarter < D / 32 ? quarter : 0;
    // The pairs (1, 0) and (0, 1) of the mean add, in registers.
    uint32_t pick_lo = 0x00003f80u, pick_hi = 0x3f800000u;
    asm("" : "+v"(pick_lo), "+v"(pick_hi));
    dec.pick_lo = pick_lo;
    dec.pick_hi = pick_hi;
    chunk_stream<D, PT>(p, dec, lds, split_blocks);
}

// ---------------------------------------------------------------- finish

// The 32-row tile of rank `key` among the call's row tiles, the deepest first:
// the last rows, which see the most live tokens, start first, and the
// workgroups past the tiles come last.  (Each holds its LDS until it exits: a
// grid of every tile that each request could have, the empty ones first, took
// 175 us per residual call of 64 requests of 500 tokens x 48 rows x 16 heads,
// this one 147 us; 2 requests x 509 rows 98.3 and 96.6 us.)
struct FinishTile {
    int request, tile;  // request -1: past the last tile
};

__device__ __forceinline__ FinishTile finish_tile(int64_t requests, const PlanEntry& own, int key) {
    const int lane = threadIdx.x & 63;
    const int tiles = (own.rows + 31) / 32;
    if (requests == 1) {
        const int tile = __builtin_amdgcn_readfirstlane(tiles) - 1 - key;
        return FinishTile{tile >= 0 ? 0 : -1, tile};
    }
    // Tiles of index `depth` and deeper.
    auto from = [&](int depth) __attribute__((always_inline)) {
        return (int)__builtin_amdgcn_readlane(wave_scan((uint32_t)max(tiles - depth, 0), lane), 63);
    };
    if (key >= from(0)) return FinishTile{-1, 0};
    int low = 0, high = (int)wave_max_u32((uint32_t)tiles);  // from(low) > key >= from(high)
    while (high - low > 1) {
        const int middle = (low + high) / 2;
        if (from(middle) > key) low = middle;
        else high = middle;
    }
    const bool has = tiles > low;
    // (Every lane takes part in the scans.)
    const int order = (int)wave_scan(has ? 1u : 0u, lane), wanted = key - from(high) + 1;
    return FinishTile{__builtin_ctzll(__ballot(has && order == wanted)), low};
}

// 32 rows of one (request, head) per workgroup: finish_merge and finish_rows
// (rq_multirow.h).
template <int D>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void chunk_finish_kernel(MultiRowParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[Geometry<D, 32>::kLdsBytes];
    const int head = (int)(blockIdx.x % (unsigned)p.heads);
    const PlanEntry own = multirow_entry(p);
    const FinishTile at = finish_tile(p.requests, own, (int)(blockIdx.x / (unsigned)p.heads));
    if (at.request < 0) return;  // uniform over the workgroup, before any barrier
    const int request = __builtin_amdgcn_readfirstlane(at.request);
    const int row0 = 32 * __builtin_amdgcn_readfirstlane(at.tile);
    const int first = __builtin_amdgcn_readlane(own.first, request), n = __builtin_amdgcn_readlane(own.rows, request);
    FinishInputs<D> in;
    finish_load<D, 32>(p, head, first, row0, n, in);
    const PlanRequest plan = plan_request(request, multirow_sizes<false>(p), own);
    const int tid = threadIdx.x, r = tid >> 3, part = tid & 7;
    const bool valid = row0 + r < n;
    const float* tile_entries =
        p.partials + ((int64_t)head * p.entries + plan.entry + row0 * plan.splits) * kMultiRowEntry;
    const int tile_rows = n - row0 < 32 ? n - row0 : 32;
    const __amdgpu_buffer_rsrc_t entries =
        handoff_resource(tile_entries, (uint32_t)(tile_rows * plan.splits * kMultiRowEntry * 4));
    const uint32_t row_at = (uint32_t)((valid ? r : 0) * plan.splits * kMultiRowEntry * 4);
    const float shift = tile_entries[(valid ? r : 0) * plan.splits * kMultiRowEntry + 2];
    float m, l, acc[16];
    finish_merge(entries, row_at, plan.splits, valid, part < D / 16 ? part : 0, m, l, acc);
    finish_rows<D, 32>(p, head, first, row0, n, in, shift, m, l, acc, lds);
}

// ---------------------------------------------------------------- launch

template <int D, int PT, bool HasL, int BA, int GA, int BL, int GL>
void launch_one(const MultiRowParams& p, hipStream_t stream) {
    hipLaunchKernelGGL((chunk_stream_kernel<D, PT, HasL, BA, GA, BL, GL>), dim3((unsigned)((int64_t)p.items * p.heads)),
                       dim3(kStreamThreads), 0, stream, p);
}

template <int D, int PT, int Links>
void launch_links(const MultiRowParams& p, hipStream_t stream) {
    hipLaunchKernelGGL((chunk_chain_kernel<D, PT, Links>), dim3((unsigned)((int64_t)p.items * p.heads)),
                       dim3(kStreamThreads), 0, stream, p);
}

template <int D, int PT, int BA, int GA>
void launch_anchor(const MultiRowParams& p, hipStream_t stream) {
    if (!p.has_residual)
        launch_one<D, PT, false, BA, GA, 2, 32>(p, stream);
    else if (p.residual.bits == 2 && p.residual.group == 32)
        launch_one<D, PT, true, BA, GA, 2, 32>(p, stream);
    else if (p.residual.bits == 2)
        launch_one<D, PT, true, BA, GA, 2, 16>(p, stream);
    else if (p.residual.group == 32)
        launch_one<D, PT, true, BA, GA, 4, 32>(p, stream);
    else
        launch_one<D, PT, true, BA, GA, 4, 16>(p, stream);
}

template <int D, int PT>
bool launch_pt(const MultiRowParams& p, hipStream_t stream) {
    switch (p.chain_length) {
        case 0: break;
        case 2: launch_links<D, PT, 2>(p, stream); return true;
        case 3: launch_links<D, PT, 3>(p, stream); return true;
        case 4: launch_links<D, PT, 4>(p, stream); return true;
        default: return false;
    }
    if (p.anchor.bits == 4 && p.anchor.group == 32)
        launch_anchor<D, PT, 4, 32>(p, stream);
    else if (p.anchor.bits == 4)
        launch_anchor<D, PT, 4, 16>(p, stream);
    else if (p.anchor.group == 32)
        launch_anchor<D, PT, 2, 32>(p, stream);
    else
        launch_anchor<D, PT, 2, 16>(p, stream);
    return true;
}

template <int D>
bool launch_d(const MultiRowParams& p, hipStream_t stream) {
    const bool launched = p.page_tokens == 16 ? launch_pt<D, 16>(p, stream)
                                              : p.page_tokens == 32 && launch_pt<D, 32>(p, stream);
    if (!launched) return false;
    const int64_t tiles = p.rows / 32 + p.requests;  // at most, over all requests
    hipLaunchKernelGGL(chunk_finish_kernel<D>, dim3((unsigned)(tiles * p.heads)), dim3(kThreads), 0, stream, p);
    return true;
}

}  // namespace

// One object per head dim (RQ_HEAD_DIM), compiled side by side.
template <>
hipError_t launch_chunk<RQ_HEAD_DIM>(const MultiRowParams& p, hipStream_t stream) {
    if (p.rows == 0 || p.requests == 0) return hipSuccess;
    return launch_d<RQ_HEAD_DIM>(p, stream) ? hipGetLastError() : hipErrorInvalidValue;
}

}  // namespace rq
