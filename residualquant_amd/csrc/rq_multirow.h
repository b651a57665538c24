// What the several-rows kernels (multirow.hip, chunk.hip) share: the plan of a
// call over its requests' histories, the page loads and the dequantization of
// 16-token units, MFMA wrappers.
#pragma once

#include "rq_chain.h"
#include "rq_device.h"
#include "rq_kernels.h"
#include "rq_plan.h"

namespace rq {

namespace {

typedef __bf16 Bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 F16x8 __attribute__((ext_vector_type(8)));
typedef float F32x16 __attribute__((ext_vector_type(16)));
typedef float F32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 32;  // tokens per MFMA tile (two 16-token units)
constexpr int kMaxD = 128;

constexpr float kLog2e = 1.4426950408889634f;
// Pages of one history split at most (its block ids are staged in LDS); the
// host sizes splits so that a split never holds more.
constexpr int kMaxSplitPages = kMultiRowMaxSplitPages;

__device__ __forceinline__ F32x16 mfma(Bf16x8 a, Bf16x8 b, F32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ F32x16 mfma(F16x8 a, F16x8 b, F32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ F32x4 mfma(Bf16x8 a, Bf16x8 b, F32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ F32x4 mfma(F16x8 a, F16x8 b, F32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t f16_bits(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }

__device__ __forceinline__ float f16_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// Round to BF16 (nearest even) and back to FP32.
__device__ __forceinline__ float round_bf16(float x) { return bf16_f32(bf16_rn(x)); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t page_rsrc(const uint8_t* page, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(page), (short)0, (int)bytes, 0x00020000);
}

// One record's bytes for the lane's token and 32-channel quarter: 16 code
// bytes (INT4) or 8 (INT2), the FP8 scale and offset byte(s) (one for group
// 32, two for group 16) and, for residual records, the BF16 alpha.
template <int Bits>
struct RecordBytes {
    uint32_t w[Bits];
    uint32_t scale, offset, alpha;
};

template <int Bits, int G>
__device__ __forceinline__ void load_record(__amdgpu_buffer_rsrc_t page, const RecordRegion& r, int page_tokens,
                                            int row, int quarter, bool alpha, RecordBytes<Bits>& out) {
    // A 32-channel quarter holds 4 x Bits code bytes and 32 / G groups.
    const uint32_t codes = (uint32_t)(r.offset + row * r.code_bytes + quarter * 4 * Bits);
    if constexpr (Bits == 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(page, codes, 0, kStreamPolicy);
        out.w[0] = v[0]; out.w[1] = v[1]; out.w[2] = v[2]; out.w[3] = v[3];
    } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(page, codes, 0, kStreamPolicy);
        out.w[0] = v[0]; out.w[1] = v[1];
    }
    // The lane's FP8 scale and offset bytes (one group of 32 channels, or two
    // of 16) through the aligned dword holding them, shifted down: the same
    // loads for either group size, so no branch sits between the unit's
    // loads (a conditional load makes the compiler wait for every load in
    // flight, the next unit's included).  Pages are multiples of 16 bytes,
    // so the dword never crosses the page end.
    const uint32_t scales = (uint32_t)(r.offset + page_tokens * r.code_bytes + row * r.groups + quarter * (32 / G));
    const uint32_t offsets = scales + (uint32_t)(page_tokens * r.groups);
    const uint32_t shift = 8u * (scales & 3u);  // offsets sit page_tokens x groups (a multiple of 4) bytes later
    out.scale = __builtin_amdgcn_raw_buffer_load_b32(page, scales & ~3u, 0, 0) >> shift;
    out.offset = __builtin_amdgcn_raw_buffer_load_b32(page, offsets & ~3u, 0, 0) >> shift;
    out.alpha = alpha ? __builtin_amdgcn_raw_buffer_load_b16(
                            page, (uint32_t)(r.offset + page_tokens * (r.code_bytes + 2 * r.groups) + 2 * row), 0, 0)
                      : 0u;
}

// The lane's 32 codes of one record as FP32 code * 2^-9: a code held in a
// byte is that FP8 E4M3 value, so v_cvt_pk_f32_fp8 converts two per
// instruction (the scales carry the 2^9 back).
template <int Bits>
__device__ __forceinline__ void record_codes(const RecordBytes<Bits>& r, float (&c)[32]) {
    if constexpr (Bits == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int lo = (int)(r.w[i] & 0x0f0f0f0fu);         // channels 8i + 0, 2, 4, 6
            const int hi = (int)((r.w[i] >> 4) & 0x0f0f0f0fu);  // channels 8i + 1, 3, 5, 7
            const auto l01 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, false);
            const auto l23 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, true);
            const auto h01 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false);
            const auto h23 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
            float* a = c + 8 * i;
            a[0] = l01[0]; a[2] = l01[1]; a[4] = l23[0]; a[6] = l23[1];
            a[1] = h01[0]; a[3] = h01[1]; a[5] = h23[0]; a[7] = h23[1];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float* a = c + 16 * i;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                // byte j of part holds channel 4j + k
                const int part = (int)((r.w[i] >> (2 * k)) & 0x03030303u);
                const auto c01 = __builtin_amdgcn_cvt_pk_f32_fp8(part, false);
                const auto c23 = __builtin_amdgcn_cvt_pk_f32_fp8(part, true);
                a[k] = c01[0]; a[4 + k] = c01[1]; a[8 + k] = c23[0]; a[12 + k] = c23[1];
            }
        }
    }
}

// Scale (times 2^9) and offset of the lane's two 16-channel blocks.
template <int G>
__device__ __forceinline__ void record_coefficients(uint32_t scale, uint32_t offset, float (&s)[2], float (&o)[2]) {
    s[0] = __builtin_amdgcn_cvt_f32_fp8((int)scale, 0) * 512.0f;
    o[0] = __builtin_amdgcn_cvt_f32_fp8((int)offset, 0);
    s[1] = G == 32 ? s[0] : __builtin_amdgcn_cvt_f32_fp8((int)scale, 1) * 512.0f;
    o[1] = G == 32 ? o[0] : __builtin_amdgcn_cvt_f32_fp8((int)offset, 1);
}

// One plane's values for the lane's 32 channels in FP32: alpha (c.s+o)_A +
// (c.s+o)_L, evaluated per 16-channel block as c_A (alpha s_A) + (c_L s_L +
// (alpha o_A + o_L)) (two fmas per channel), or (c.s+o)_A without a loop
// record.
template <int BA, int GA, int BL, int GL, bool HasL>
__device__ __forceinline__ void plane_values(const RecordBytes<BA>& a_rec, const RecordBytes<BL>& l_rec, float alpha,
                                             float (&x)[32]) {
    float sa[2], oa[2];
    record_coefficients<GA>(a_rec.scale, a_rec.offset, sa, oa);
    float ca[32];
    record_codes<BA>(a_rec, ca);
    if constexpr (HasL) {
        float sl[2], ol[2];
        record_coefficients<GL>(l_rec.scale, l_rec.offset, sl, ol);
        float cl[32];
        record_codes<BL>(l_rec, cl);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float a = alpha * sa[b], c = fmaf(alpha, oa[b], ol[b]);
#pragma unroll
            for (int i = 16 * b; i < 16 * b + 16; ++i) x[i] = fmaf(ca[i], a, fmaf(cl[i], sl[b], c));
        }
    } else {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 16 * b; i < 16 * b + 16; ++i) x[i] = fmaf(ca[i], sa[b], oa[b]);
    }
}

typedef float F32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 F16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 Bf16x2 __attribute__((ext_vector_type(2)));
typedef short Short4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) Short4 LdsShort4;

// Two FP32 values rounded (nearest even) to a packed FP16 / BF16 pair, low first.
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(F32x2{a, b}, F16x2));
}
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(F32x2{a, b}, Bf16x2));
}

// ds_read_b64_tr_b16 (gfx950, checked on the device): within each 16 lanes,
// output lane o gets element o % 4 of the 8 bytes addressed by lanes
// o / 4 + 4 p, p = 0..3.
__device__ __forceinline__ Short4 read_transposed(const uint16_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4*)p);
}

// The page resources of one 16-token unit (wave-uniform) and the lane's row in the page.
struct UnitPages {
    __amdgpu_buffer_rsrc_t k, v;
    int row;
};

// Anchor mode: K and V of the anchor record and, for a residual loop, the
// loop's record (BA/GA and BL/GL their bits and groups).  Units stream two
// ahead: the loads of the unit two places on are issued before a unit is
// dequantized, so about two units' bytes per wave are in flight while units
// dequantize and the tiles' MFMAs run.
template <int PT, bool HasL, int BA, int GA, int BL, int GL>
struct AnchorDecoder {
    static constexpr bool kAnchorMeanTerm = HasL;  // scores add alpha_K q'.bf16(mu_A)
    struct Bytes {
        RecordBytes<BA> ka, va;
        RecordBytes<BL> kl, vl;
    };
    RecordRegion anchor, residual;
    int lq;
    Bytes ahead1, ahead2;

    __device__ __forceinline__ void fetch(const UnitPages& u, Bytes& b) const {
        load_record<BA, GA>(u.k, anchor, PT, u.row, lq, false, b.ka);
        load_record<BA, GA>(u.v, anchor, PT, u.row, lq, false, b.va);
        if constexpr (HasL) {
            load_record<BL, GL>(u.k, residual, PT, u.row, lq, true, b.kl);
            load_record<BL, GL>(u.v, residual, PT, u.row, lq, true, b.vl);
        }
    }
    __device__ __forceinline__ void prime(const UnitPages& first, const UnitPages& second) {
        fetch(first, ahead1);
        fetch(second, ahead2);
    }
    // Dequantizes the current unit (K, then V, so that only one plane's
    // values are live at a time) after issuing the loads of `two_on`;
    // store_k / store_v take the lane's 32 channels in two halves of 16.
    // Returns the token's K alpha (1 without a loop record).
    template <class StoreK, class StoreV>
    __device__ __forceinline__ float unit(const UnitPages& /*next*/, const UnitPages& two_on, StoreK store_k,
                                          StoreV store_v) {
        const Bytes cur = ahead1;
        ahead1 = ahead2;
        fetch(two_on, ahead2);
        const float alpha_k = HasL ? bf16_f32(cur.kl.alpha) : 1.f;
        {
            float k[32];
            plane_values<BA, GA, BL, GL, HasL>(cur.ka, cur.kl, alpha_k, k);
            store_k(k, k + 16);
        }
        {
            float v[32];
            plane_values<BA, GA, BL, GL, HasL>(cur.va, cur.vl, HasL ? bf16_f32(cur.vl.alpha) : 1.f, v);
            store_v(v, v + 16);
        }
        return alpha_k;
    }
};

// Adjacent mode past loop 0: K and V are the BF16 restore chain over the
// Links records 0..L (rq_chain.h), K adding bf16(mu_r) of records r < L
// (FP32 copies in LDS, `mean`: [Links - 1][kMaxD], or null).  A unit's raw
// bytes of all its records take ~6 registers per record and plane, so units
// stream one ahead: a plane's registers take the next unit's bytes as soon as
// this unit's chain of that plane is built.  Keys are rounded to BF16 (the
// chain's last link) before the FP16 tile takes them, which is exact.
template <int D, int PT, int Links>
struct ChainDecoder {
    static constexpr bool kAnchorMeanTerm = false;
    RecordRegion regs[Links];
    const float* mean;  // [Links - 1][kMaxD] in LDS (zeros without means)
    bool add_mean;
    int lq;
    uint32_t pick_lo, pick_hi;
    ChainRaw k[Links], v[Links];

    __device__ __forceinline__ void fetch_plane(__amdgpu_buffer_rsrc_t page, int row, ChainRaw (&raw)[Links]) const {
#pragma unroll
        for (int r = 0; r < Links; ++r) chain_load<PT, kStreamPolicy, 0>(page, regs[r], row, lq, r > 0, raw[r]);
    }
    __device__ __forceinline__ void prime(const UnitPages& first, const UnitPages& /*second*/) {
        fetch_plane(first.k, first.row, k);
        fetch_plane(first.v, first.row, v);
    }
    // bf16(mu_r) of channel i of the 16 channels from `base` (record r's copy kMaxD floats on).
    __device__ __forceinline__ static auto mean_of(const float* base) {
        return [base](int r, int i) __attribute__((always_inline)) { return base[r * kMaxD + i]; };
    }
    template <class StoreK, class StoreV>
    __device__ __forceinline__ float unit(const UnitPages& next, const UnitPages& /*two_on*/, StoreK store_k,
                                          StoreV store_v) {
        const float* m = mean + 32 * lq;
        float lo[16], hi[16];
        chain_build<0, Links>(k, regs, add_mean, mean_of(m), true, pick_lo, pick_hi, lo);
        chain_build<1, Links>(k, regs, add_mean, mean_of(m + 16), true, pick_lo, pick_hi, hi);
        // The last link's BF16 rounding, one pack per channel pair.
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const uint32_t a = bf16_pack(lo[i], lo[i + 1]), b = bf16_pack(hi[i], hi[i + 1]);
            lo[i] = __uint_as_float(a << 16);
            lo[i + 1] = __uint_as_float(a & 0xffff0000u);
            hi[i] = __uint_as_float(b << 16);
            hi[i + 1] = __uint_as_float(b & 0xffff0000u);
        }
        fetch_plane(next.k, next.row, k);
        store_k(lo, hi);
        chain_build<0, Links>(v, regs, false, mean_of(m), true, pick_lo, pick_hi, lo);
        chain_build<1, Links>(v, regs, false, mean_of(m), true, pick_lo, pick_hi, hi);
        fetch_plane(next.v, next.row, v);
        store_v(lo, hi);
        return 1.f;
    }
};

// Whether rows of a BF16 tensor at `base` with row stride `stride`
// (elements) start on 16-byte boundaries.  The boundary guarantees 8 bytes
// for queries and keys and 2 bytes for values and outputs.
__device__ __forceinline__ bool aligned_rows(const void* base, int64_t stride) {
    return (reinterpret_cast<uintptr_t>(base) & 15u) == 0 && (stride & 7) == 0;
}

// 16 consecutive BF16 values at `src` (a 32-byte aligned offset of an
// aligned_rows tensor when `vec`) as two 16-byte words.
__device__ __forceinline__ void load_halves16(const uint16_t* src, bool vec, uint4 (&w)[2]) {
    if (vec) {
        w[0] = reinterpret_cast<const uint4*>(src)[0];
        w[1] = reinterpret_cast<const uint4*>(src)[1];
    } else {
        uint32_t x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = (uint32_t)src[2 * i] | ((uint32_t)src[2 * i + 1] << 16);
        w[0] = make_uint4(x[0], x[1], x[2], x[3]);
        w[1] = make_uint4(x[4], x[5], x[6], x[7]);
    }
}

// log2(e) / sqrt(D)
template <int D>
constexpr float kScoreScale = D == 128 ? 1.4426950408889634f * 0.08838834764831845f
                                       : 1.4426950408889634f * 0.10206207261596575f;

constexpr int kThreads = 256;
constexpr int kWaves = 4;

// LDS geometry of the stream kernel for head dim D and TR-row tiles.
template <int D, int TR = 32>
struct Geometry {
    static constexpr int Quarters = D / 32;  // 32-channel quarters a token's lanes cover
    static constexpr int Parts = D / 16;     // 16-channel parts (MFMA k steps of the scores)
    static constexpr int KS = D + 8;         // K tile row stride (halves)
    // V tile [token][VROW] BF16.  At D = 128 the row is unpadded and
    // swizzled by token, which keeps the transposed reads free of bank
    // conflicts: for 32-row tiles (a half-wave reads 4 tokens x 32 channels)
    // its four 32-channel chunks sit at positions q ^ (token % 4), for 16-row
    // tiles (8 tokens x 16 channels) its eight 16-channel units at positions
    // u ^ (token % 8).  At D = 96 the rows are padded instead, to 104 halves
    // (32-row tiles) or 112 (16-row tiles: a stride of 56 banks puts 8
    // consecutive tokens on distinct 8-bank groups); rows stay 16-byte
    // aligned for the stores and 8-byte aligned for the reads.
    static constexpr bool kSwizzleV = D == 128;
    static constexpr int VROW = D == 128 ? D : (TR == 32 ? D + 8 : D + 16);
    static constexpr int kVBytes = D == 128 ? D * (kTile + 8) * 2 : kTile * VROW * 2;
    static constexpr int kWaveBytes = kTile * KS * 2 + kVBytes + kTile * 4;  // K (FP16), V (BF16), alpha_K
    static constexpr int kLdsBytes = kWaves * kWaveBytes;
    // Prologue scratch (aliases the tiles): q scaled into FP16 [32][KS], R_k
    // FP16 [D][KS], q.R_k FP32 [32][QRS], q' FP16 [32][KS], mean dots, row
    // scales and the rows' input exponents.
    static constexpr int QRS = D + 4;
    static constexpr int kQ16Offset = 0;
    static constexpr int kRkOffset = kQ16Offset + 32 * KS * 2;
    static constexpr int kQrawOffset = kRkOffset + D * KS * 2;
    static constexpr int kQpOffset = kQrawOffset + 32 * QRS * 4;
    static constexpr int kQmuOffset = kQpOffset + 32 * KS * 2;
    // Wave merge (aliases the tiles): O [wave][row][MS] FP32 and (m, l) per wave and row.
    static constexpr int MS = D + 4;
    static constexpr int kMlOffset = kWaves * 32 * MS * 4;
    static_assert(kTile * VROW * 2 <= kVBytes, "the row-major V tile fits its region");
    static_assert(kQmuOffset + 128 * 4 <= kLdsBytes, "prologue scratch fits in the tile LDS");
    static_assert(kMlOffset + kWaves * 32 * 2 * 4 <= kLdsBytes, "merge buffer fits in the tile LDS");
};
// The LDS writes of a wave before reads of other lanes of the same wave.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------- finish

// Row strides of the finish's tiles for head dim D: FP16 rows (halves) and the
// rotated history [row][channel] (FP32).  Region A holds the merged rows'
// FP16 parts for the rotation, region B the rotated history.
template <int D>
struct FinishGeometry {
    static constexpr int Parts = D / 16;
    static constexpr int FS = D + 8;
    static constexpr int OS = D + 4;
    static constexpr int kRegionABytes = 2 * 32 * FS * 2;  // high and low FP16 parts
    static constexpr int kRegionBFloats = 32 * OS;
    static_assert(kRegionABytes % 16 == 0 && kRegionABytes + 4 * kRegionBFloats <= Geometry<D>::kLdsBytes,
                  "the finish fits in the tile LDS");
};

__device__ __forceinline__ float row8_sum(float x) {
    x += __shfl_xor(x, 1);
    x += __shfl_xor(x, 2);
    return x + __shfl_xor(x, 4);
}

// Eight BF16 values of a 16-byte word as FP32.
__device__ __forceinline__ void widen_bf16(uint4 w, float* x) {
    const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[2 * i] = bf16_f32(v[i] & 0xffffu);
        x[2 * i + 1] = bf16_f32(v[i] >> 16);
    }
}

// The finish of one (request, head) and its rows row0 .. row0 + TR - 1, by the
// stream workgroup (256 threads) whose split of them ends last.  Thread t
// takes row t / 8 of the tile and part p = t % 8 of it: the 16 channels
// 16p..16p+15 of the merge, the query-key dots, the live values and the
// output (parts p < D / 16).  The eight threads of a row are adjacent lanes of one wave.
//   1. (finish_merge, only with several splits) merge the splits' partials
//      (m, l, O) of each row (log2 units);
//   2. rotate the tile's merged rows by R_v^T on the matrix cores (wave w
//      computes output channels 32 w .. 32 w + 31);
//   3. add the live tokens: in decode semantics the row's own token; in
//      causal semantics the request's new tokens j <= row (live_tokens);
//   4. write O / l in BF16.
// A finish launch of its own read every partial back, one split or several,
// and looked the plan up again: 2 requests of 4096 tokens x 8 rows took 26.5
// us per residual call with it and 24.6 us without, 40 requests of 50..1500
// tokens x 3 rows 54.0 and 43.8 us.

// Loads that depend on the tile alone, issued before the split's arrival:
// R_v as the B operand of the rotation MFMAs (wave w computes output channels
// 32 w .. 32 w + 31, lane l takes row 32 w + l % 32 of R_v at features 16 m +
// 8 (l / 32) .. + 7), the row's query and, in decode semantics, its own key
// and value.
template <int D>
struct FinishInputs {
    F16x8 rv[D / 16];
    uint4 qw[2], kw[2], vw[2];
};

template <int D, int TR>
__device__ __forceinline__ void finish_load(const MultiRowParams& p, int head, int first, int row0, int n,
                                            FinishInputs<D>& in) {
    const int tid = threadIdx.x;
    const int r = tid >> 3, part = tid & 7;
    const bool part_active = part < D / 16;
    const int wave = tid >> 6, lane = tid & 63;
    if (p.value_rotation != nullptr && wave < D / 32) {
        const uint16_t* src = p.value_rotation + ((int64_t)head * D + 32 * wave + (lane & 31)) * D + 8 * (lane >> 5);
#pragma unroll
        for (int m = 0; m < D / 16; ++m) in.rv[m] = *reinterpret_cast<const F16x8*>(src + 16 * m);
    }
    const int64_t row = (int64_t)first + row0 + (r < TR && row0 + r < n ? r : 0);
    // The part's 16 channels of a token row (part 0's for an inactive part,
    // whose values are never used).
    const int64_t channels = (int64_t)head * D + 16 * (part_active ? part : 0);
    load_halves16(p.query + row * p.query_stride + channels, aligned_rows(p.query, p.query_stride), in.qw);
    if (!part_active) in.qw[0] = in.qw[1] = make_uint4(0u, 0u, 0u, 0u);  // no share of the row's dots
    if (!p.causal) {
        load_halves16(p.key + row * p.key_stride + channels, aligned_rows(p.key, p.key_stride), in.kw);
        load_halves16(p.value + row * p.value_stride + channels, aligned_rows(p.value, p.value_stride), in.vw);
    }
}

// Merges the splits' partials of the thread's row and part online, four at a
// time: every load of a batch is issued before any of its arithmetic (split
// indices past the last are clamped and weighted zero, so no load sits behind
// a branch).  Rows past the tile merge nothing.  `row_at` is the offset of the
// row's split 0 in the tile's entries.
__device__ __forceinline__ void finish_merge(__amdgpu_buffer_rsrc_t entries, uint32_t row_at, int splits, bool valid,
                                             int part, float& m, float& l, float (&acc)[16]) {
    m = -__builtin_inff();
    l = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    for (int s0 = 0; s0 < splits; s0 += 4) {
        float2 ml[4];
        float4 ox[4][4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int s = s0 + b < splits ? s0 + b : splits - 1;
            const uint32_t at = row_at + (uint32_t)(s * kMultiRowEntry * 4);
            ml[b] = handoff_load2(entries, at);
#pragma unroll
            for (int c = 0; c < 4; ++c) ox[b][c] = handoff_load4(entries, at + 16 + 64 * part + 16 * c);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float ms = (valid && s0 + b < splits) ? ml[b].x : -__builtin_inff();
            const float new_max = fmaxf(m, ms);
            const float base = new_max == -__builtin_inff() ? 0.f : new_max;
            const float keep = __builtin_amdgcn_exp2f(m - base), w = __builtin_amdgcn_exp2f(ms - base);
            m = new_max;
            l = fmaf(l, keep, ml[b].y * w);
            const float x[16] = {ox[b][0].x, ox[b][0].y, ox[b][0].z, ox[b][0].w, ox[b][1].x, ox[b][1].y,
                                 ox[b][1].z, ox[b][1].w, ox[b][2].x, ox[b][2].y, ox[b][2].z, ox[b][2].w,
                                 ox[b][3].x, ox[b][3].y, ox[b][3].z, ox[b][3].w};
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = fmaf(acc[i], keep, x[i] * w);
        }
    }
}

// The causal live tokens of the thread's row (tid / 8) one by one, every product
// in FP32 (live_tokens, where its sums are not finite).
template <int D, int TR>
__device__ __forceinline__ void live_tokens_fp32(const MultiRowParams& p, int head, int first, int row0, int n,
                                                 float shift, float& m, float& l, float (&acc)[16]) {
    // (Opaque: addresses shared with the path of finite sums would stay in registers over it.)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int r = tid >> 3, part = tid & 7;
    const bool part_active = part < D / 16;
    const int row = r < TR && row0 + r < n ? row0 + r : -1;  // (sees no token)
    const int64_t channels = (int64_t)head * D + 16 * (part_active ? part : 0);
    const bool q_vec = aligned_rows(p.query, p.query_stride), k_vec = aligned_rows(p.key, p.key_stride),
               v_vec = aligned_rows(p.value, p.value_stride);
    uint4 w[2];
    float q[16];
    load_halves16(p.query + ((int64_t)first + max(row, 0)) * p.query_stride + channels, q_vec, w);
    widen_bf16(w[0], q);
    widen_bf16(w[1], q + 8);
    const int live_end = min(n, row0 + TR);
    for (int j = 0; j < live_end; ++j) {
        float k[16], v[16];
        load_halves16(p.key + ((int64_t)first + j) * p.key_stride + channels, k_vec, w);
        widen_bf16(w[0], k);
        widen_bf16(w[1], k + 8);
        load_halves16(p.value + ((int64_t)first + j) * p.value_stride + channels, v_vec, w);
        widen_bf16(w[0], v);
        widen_bf16(w[1], v + 8);
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) dot = fmaf(q[i], k[i], dot);
        const float score = row8_sum(part_active ? dot : 0.f) * kScoreScale<D> - shift;
        if (j > row) continue;
        const float new_max = fmaxf(m, score);
        const float keep = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m - new_max);
        const float weight = __builtin_amdgcn_exp2f(score - new_max);
        m = new_max;
        l = fmaf(l, keep, weight);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = fmaf(weight, v[i], acc[i] * keep);
    }
}

// Causal live tokens on MFMA, by the four waves of the tile's workgroup: the
// request's new tokens j <= row for the rows row0 .. row0 + TR - 1.  Wave w
// takes the 32-key tiles w, w + 4, ..: raw BF16 K and V into its own LDS tile,
// S^T = K Q^T and O^T += V^T P^T as in the stream, with the probabilities as
// three BF16 parts (8 significant bits each, so all 24 of the FP32 value
// multiply V, whose BF16 values and products with a part are exact in FP32; a
// third part instead of two takes 1.6 us more of a 100 us call).  The waves'
// (m, l, O) and the thread's history (m, l, acc; row tid / 8, channels
// 16 (tid % 8)..+15) then meet in LDS.  `shift` is the mean shift of that row.
// On the vector units (scores and values in FP32, 32 keys per step for the
// whole workgroup) the finish of 2 requests x 509 rows x 16 heads took 124 us,
// here 27 us.
// A part may be zero or of the other sign, and the tokens that a row does not
// see take part as 0 x V: a V that is not finite makes sums NaN that hold an
// infinity or do not hold that V.  A wave with such a sum in its eight rows
// takes their tokens again (live_tokens_fp32).
template <int D, int TR>
__device__ __forceinline__ void live_tokens(const MultiRowParams& p, int head, int first, int row0, int n, float shift,
                                            float& m, float& l, float (&acc)[16], uint8_t* lds) {
    using G = Geometry<D, 32>;
    constexpr int KS = G::KS, Quarters = G::Quarters, Parts = G::Parts, MS = G::MS;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, column = lane & 31, half = lane >> 5;
    uint16_t* k_tile = reinterpret_cast<uint16_t*>(lds + wave * G::kWaveBytes);
    uint16_t* v_tile = k_tile + kTile * KS;
    float* shifts = reinterpret_cast<float*>(lds + kWaves * G::kWaveBytes - 128);  // the last wave's alpha tile
    if ((tid & 7) == 0) shifts[tid >> 3] = shift;
    const int live_end = min(n, row0 + TR);
    const int row = row0 + column;
    const bool k_vec = aligned_rows(p.key, p.key_stride), v_vec = aligned_rows(p.value, p.value_stride);
    // Lane l stages 16 channels (part l % 8) of keys l / 8 + 8 i.
    const int part = lane & 7;
    const bool part_active = part < Parts;
    const int64_t channels = (int64_t)head * D + 16 * (part_active ? part : 0);
    uint4 kw[4][2], vw[4][2];
    auto fetch = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t at = (int64_t)first + min(c0 + (lane >> 3) + 8 * i, n - 1);  // (masked below)
            load_halves16(p.key + at * p.key_stride + channels, k_vec, kw[i]);
            load_halves16(p.value + at * p.value_stride + channels, v_vec, vw[i]);
        }
    };
    Bf16x8 q[Parts];
    {
        const uint16_t* query = p.query + ((int64_t)first + min(row, n - 1)) * p.query_stride + head * D + 8 * half;
#pragma unroll
        for (int i = 0; i < Parts; ++i) {
            const uint2 a = *reinterpret_cast<const uint2*>(query + 16 * i);
            const uint2 b = *reinterpret_cast<const uint2*>(query + 16 * i + 4);
            q[i] = __builtin_bit_cast(Bf16x8, make_uint4(a.x, a.y, b.x, b.y));
        }
    }
    __syncthreads();  // the shifts
    const float row_shift = shifts[column];
    F32x16 out[Quarters];
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) out[t][e] = 0.f;
    float running_max = -__builtin_inff(), running_sum = 0.f;
    // Transposed V reads as in the 32-row stream tiles.
    const int tr_a = (lane >> 2) & 3, tr_b = lane & 3, tr_g = (lane >> 4) & 1;
    const int v_lane = G::VROW * (4 * half + tr_a) + (G::kSwizzleV ? 32 * tr_a : 0) + 16 * tr_g + 4 * tr_b;
    for (int c0 = kTile * wave; c0 < live_end; c0 += kTile * kWaves) {
        fetch(c0);
        if (part_active) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = (lane >> 3) + 8 * i;
                uint4* kd = reinterpret_cast<uint4*>(&k_tile[j * KS + 16 * part]);
                kd[0] = kw[i][0];
                kd[1] = kw[i][1];
                const int chunk = G::kSwizzleV ? (part >> 1) ^ (j & 3) : part >> 1;
                uint4* vd = reinterpret_cast<uint4*>(&v_tile[j * G::VROW + 32 * chunk + 16 * (part & 1)]);
                vd[0] = vw[i][0];
                vd[1] = vw[i][1];
            }
        }
        wave_sync();
        F32x16 s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.f;
        const uint16_t* k_row = &k_tile[column * KS + 8 * half];
#pragma unroll
        for (int i = 0; i < Parts; ++i) s = mfma(*reinterpret_cast<const Bf16x8*>(k_row + 16 * i), q[i], s);
        float tile_max = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int j = c0 + 8 * (e >> 2) + 4 * half + (e & 3);
            s[e] = j <= row && j < n ? s[e] * kScoreScale<D> - row_shift : -__builtin_inff();
            tile_max = fmaxf(tile_max, s[e]);
        }
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
        const float new_max = fmaxf(running_max, tile_max);
        const float base = new_max == -__builtin_inff() ? 0.f : new_max;
        const float rescale = __builtin_amdgcn_exp2f(running_max - base);
        running_max = new_max;
        float tile_sum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[e] = __builtin_amdgcn_exp2f(s[e] - base);
            tile_sum += s[e];
        }
        running_sum = running_sum * rescale + tile_sum + __shfl_xor(tile_sum, 32);
        if (!__all(rescale == 1.0f)) {
#pragma unroll
            for (int t = 0; t < Quarters; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) out[t][e] *= rescale;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            Bf16x8 high, middle, low;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float w = s[8 * j + e];
                high[e] = (__bf16)w;
                const float rest = w - (float)high[e];
                middle[e] = (__bf16)rest;
                low[e] = (__bf16)(rest - (float)middle[e]);
            }
            const uint16_t* v_rows = v_tile + 16 * j * G::VROW;
#pragma unroll
            for (int t = 0; t < Quarters; ++t) {
                const int at = G::kSwizzleV ? v_lane ^ (32 * t) : v_lane + 32 * t;
                const Short4 lo = read_transposed(v_rows + at);
                const Short4 hi = read_transposed(v_rows + 8 * G::VROW + at);
                const Bf16x8 a = __builtin_bit_cast(Bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                out[t] = mfma(a, high, out[t]);
                out[t] = mfma(a, middle, out[t]);
                out[t] = mfma(a, low, out[t]);
            }
        }
        wave_sync();  // the next tile overwrites this one
    }
    __syncthreads();  // the merge buffer aliases every wave's tiles
    static_assert(G::kMlOffset + kWaves * 32 * 2 * 4 <= kWaves * G::kWaveBytes - 128, "the shifts stay");
    float* merge_o = reinterpret_cast<float*>(lds);
    float* merge_ml = reinterpret_cast<float*>(lds + G::kMlOffset);
#pragma unroll
    for (int t = 0; t < Quarters; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(&merge_o[(wave * 32 + column) * MS + 32 * t + 8 * g + 4 * half]) =
                make_float4(out[t][4 * g], out[t][4 * g + 1], out[t][4 * g + 2], out[t][4 * g + 3]);
    if (half == 0) {
        merge_ml[(wave * 32 + column) * 2] = running_max;
        merge_ml[(wave * 32 + column) * 2 + 1] = running_sum;
    }
    __syncthreads();
    const int r = tid >> 3, chunk = (tid & 7) < Parts ? tid & 7 : 0;
    float m_w[kWaves], total_max = m;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        m_w[w] = merge_ml[(w * 32 + r) * 2];
        total_max = fmaxf(total_max, m_w[w]);
    }
    const float keep = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m - total_max);
    float total = l * keep, sums[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[i] = acc[i] * keep;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const float weight = m_w[w] == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m_w[w] - total_max);
        total = fmaf(merge_ml[(w * 32 + r) * 2 + 1], weight, total);
        const float* src = &merge_o[(w * 32 + r) * MS + 16 * chunk];
#pragma unroll
        for (int i = 0; i < 16; ++i) sums[i] = fmaf(src[i], weight, sums[i]);
    }
    float zero = 0.f;  // stays 0 over finite sums, else NaN
#pragma unroll
    for (int i = 0; i < 16; ++i) zero = fmaf(sums[i], 0.f, zero);
    if (__any(r < TR && row0 + r < n && !(zero == 0.f))) {
        // (The merge buffer ends before the shifts.)
        live_tokens_fp32<D, TR>(p, head, first, row0, n, shifts[r], m, l, acc);
        return;
    }
    m = total_max;
    l = total;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = sums[i];
}

template <int D, int TR>
__device__ __forceinline__ void finish_rows(const MultiRowParams& p, int head, int first, int row0, int n,
                                            const FinishInputs<D>& in, float shift, float m, float l, float (&acc)[16],
                                            uint8_t* lds) {
    using G = FinishGeometry<D>;
    constexpr int FS = G::FS;
    constexpr int OS = G::OS;
    uint8_t* region_a = lds;
    float* hist_rot = reinterpret_cast<float*>(lds + G::kRegionABytes);
    const int tid = threadIdx.x;
    const int r = tid >> 3, part = tid & 7;
    const bool part_active = part < G::Parts;
    const bool rotate = p.value_rotation != nullptr;
    const int wave = tid >> 6, lane = tid & 63;
    const bool rotation_wave = wave < D / 32;
    const bool valid = r < TR && row0 + r < n;
    const int64_t row = (int64_t)first + row0 + (valid ? r : 0);
    const float scale = kScoreScale<D>;  // log2(e) / sqrt(D)
    const int64_t channels = (int64_t)head * D + 16 * (part_active ? part : 0);

    // 2. hist . R_v^T for the tile's rows on the matrix cores: the merged
    // rows divided by their sums (convex combinations of values, within the
    // FP16 range) as FP16 high and low parts (~22 significant bits), times
    // R_v (FP16), FP32 accumulation; the sums are multiplied back.
    if (rotate) {
        uint16_t* high = reinterpret_cast<uint16_t*>(region_a);  // [row][FS]
        uint16_t* low = high + 32 * FS;
        const float inverse = l > 0.f ? 1.0f / l : 0.f;
        uint32_t hw[8], lw[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float x0 = acc[2 * i] * inverse, x1 = acc[2 * i + 1] * inverse;
            const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
            const _Float16 r0 = (_Float16)(x0 - (float)h0), r1 = (_Float16)(x1 - (float)h1);
            hw[i] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
            lw[i] = (uint32_t)__builtin_bit_cast(uint16_t, r0) | ((uint32_t)__builtin_bit_cast(uint16_t, r1) << 16);
        }
        if (part_active) {
            uint4* hd = reinterpret_cast<uint4*>(&high[r * FS + 16 * part]);
            uint4* ld = reinterpret_cast<uint4*>(&low[r * FS + 16 * part]);
            hd[0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            hd[1] = make_uint4(hw[4], hw[5], hw[6], hw[7]);
            ld[0] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
            ld[1] = make_uint4(lw[4], lw[5], lw[6], lw[7]);
        }
        __syncthreads();
        if (rotation_wave) {
            // A operand: lane l takes merged row l % 32 at features 16 m + 8 (l / 32) .. + 7.
            F32x16 rotated;
#pragma unroll
            for (int e = 0; e < 16; ++e) rotated[e] = 0.f;
            const int a_offset = (lane & 31) * FS + 8 * (lane >> 5);
#pragma unroll
            for (int mm = 0; mm < G::Parts; ++mm) {
                rotated = mfma(*reinterpret_cast<const F16x8*>(&high[a_offset + 16 * mm]), in.rv[mm], rotated);
                rotated = mfma(*reinterpret_cast<const F16x8*>(&low[a_offset + 16 * mm]), in.rv[mm], rotated);
            }
            // Register e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4, channel 32 w + l % 32.
#pragma unroll
            for (int e = 0; e < 16; ++e)
                hist_rot[(8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)) * OS + 32 * wave + (lane & 31)] = rotated[e];
        }
        __syncthreads();
        if (part_active) {
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) {
                const float4 x = *reinterpret_cast<const float4*>(&hist_rot[r * OS + 16 * part + 4 * c4]);
                acc[4 * c4] = x.x * l;
                acc[4 * c4 + 1] = x.y * l;
                acc[4 * c4 + 2] = x.z * l;
                acc[4 * c4 + 3] = x.w * l;
            }
        }
    }

    // 3. Live tokens.
    float q[16];
    widen_bf16(in.qw[0], q);
    widen_bf16(in.qw[1], q + 8);
    if (!p.causal) {
        // The row's own token.
        float k[16], v[16];
        widen_bf16(in.kw[0], k);
        widen_bf16(in.kw[1], k + 8);
        widen_bf16(in.vw[0], v);
        widen_bf16(in.vw[1], v + 8);
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) dot = fmaf(q[i], k[i], dot);
        const float score = row8_sum(dot) * scale - shift;
        const float total_max = fmaxf(m, score);
        const float hist_weight = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m - total_max);
        const float live = __builtin_amdgcn_exp2f(score - total_max);
        l = fmaf(l, hist_weight, live);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = fmaf(live, v[i], acc[i] * hist_weight);
    } else {
        __syncthreads();  // the rotation's reads of the region are done
        live_tokens<D, TR>(p, head, first, row0, n, r < TR ? shift : 0.f, m, l, acc, lds);
    }

    // 4. Output.
    if (valid && part_active) {
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = bf16_rn(acc[2 * i] / l) | (bf16_rn(acc[2 * i + 1] / l) << 16);
        uint16_t* out = p.output + row * p.output_stride + channels;
        if (aligned_rows(p.output, p.output_stride)) {
            reinterpret_cast<uint4*>(out)[0] = make_uint4(w[0], w[1], w[2], w[3]);
            reinterpret_cast<uint4*>(out)[1] = make_uint4(w[4], w[5], w[6], w[7]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                out[2 * i] = (uint16_t)(w[i] & 0xffffu);
                out[2 * i + 1] = (uint16_t)(w[i] >> 16);
            }
        }
    }
}

// One request's rows and history.
struct RequestRows {
    int first, rows, history;
};

__device__ __forceinline__ RequestRows request_rows(const MultiRowParams& p, int request) {
    RequestRows r;
    r.first = p.query_start_loc[request];
    const int n = p.query_start_loc[request + 1] - r.first;
    const int new_tokens = p.causal ? n : 1;
    // Rows past the query tensor are not read or written.
    r.rows = r.first < 0 || r.first >= p.rows ? 0 : (int)min((int64_t)max(n, 0), p.rows - r.first);
    const int seq = p.seq_lens[request];
    // Tokens past the page table are never read.
    r.history = (int)min((int64_t)(seq > new_tokens ? seq - new_tokens : 0), p.max_pages * p.page_tokens);
    return r;
}

// (Whole false: the chunk kernels, which take no whole_length; a branch that they
// never take cost their four-record chain 2%.)
template <bool Whole>
__host__ __device__ __forceinline__ PlanSizes multirow_sizes(const MultiRowParams& p) {
    return PlanSizes{p.plan_target, p.splits, p.plan_min, p.plan_max, p.plan_max_splits, 0, 1, p.plan_unit == kTile ? 13 : 9,
                     Whole ? p.plan_whole : 0};
}

// The share of request `lane` of the call's plan.
__device__ __forceinline__ PlanEntry multirow_entry(const MultiRowParams& p) {
    const int b = threadIdx.x & 63, requests = (int)p.requests;
    const RequestRows q = request_rows(p, b < requests ? b : requests - 1);
    const int rows = b < requests ? q.rows : 0;
    return PlanEntry{(rows + p.tile_rows - 1) / p.tile_rows, (q.history + p.plan_unit - 1) / p.plan_unit, q.first,
                     q.history, rows};
}

// Item `key` of the call's plan, or, with more requests than the plan covers,
// split `split` of the call's `splits` of row tile `tile` of `request`.
// PlanItem: length in units of plan_unit tokens, tokens the history.
template <bool Whole>
__device__ __forceinline__ PlanItem multirow_plan(const MultiRowParams& p, int key, int request, int tile, int split) {
    if (p.items > 0) return plan_find((int)p.requests, key, multirow_sizes<Whole>(p), multirow_entry(p));
    const RequestRows q = request_rows(p, request);
    // About requests x the average request's row tiles x splits of the items have work.
    const int64_t tiles = max(p.rows / (p.requests * p.tile_rows), (int64_t)1);
    return PlanItem{request, tile, split, p.splits, (q.history + p.plan_unit - 1) / p.plan_unit, q.first, q.history,
                    q.rows, 0, q.first * p.splits, (int)min(p.requests * tiles * p.splits, (int64_t)INT_MAX)};
}

}  // namespace

}  // namespace rq
