// Panel tile: the multi-token product (f16 activations) with the weights
// dequantised straight into MFMA B fragments and only the activations, and the
// raw weight bytes, in LDS. Compiled once per encoding (PANEL_ENC).
//
// out[t][r] = sum_c W[r][c] * x[t][c]: A = activations (tokens x K), B = W^T,
// D = tokens x rows, F32 accumulate on v_mfma_f32_32x32x16_f16. A workgroup
// takes BM = 32 TG tokens x BN = 32 RG WR rows; WR waves split the rows, so
// each weight is decoded once per token tile, by the lane that feeds it to the
// matrix core, and WK sets of waves split K and meet in LDS at the end.
//
// Why this layout (MI355X, Q4_K 17408 x 5120; the 256 x 256 tile below it in
// gemm.hip stages f16 weights through LDS for all eight of its waves):
//  - raw bytes by LDS copies of whole 256-column row units. Fragments loaded
//    per lane (32 rows, 32 bytes each, per 64 columns) touch every cache line
//    four to five times: 774 us at 4096 tokens, against 710 with the copies
//    (and 598 when all lanes read one row's lines).
//  - activations XOR-swizzled in 16-byte chunks over row pairs: no bank
//    conflicts on fragment reads (two-way before: 44 M conflict cycles of
//    96 M, 710 -> 702 us).
//  - scales unpacked once per unit, codes into f16 by one masking operation per
//    pair and one v_fma_mix a weight: 1.6 VALU operations a weight; and the
//    hand-over to the next slab (wait, barrier, copies, first fragment reads)
//    under the last sub-step's products: 702 -> 683 us.
// At 4096 tokens the card is power-limited (1.5-1.6 GHz at 60 % MFMA
// occupancy against 1.8 GHz at 53 % in the LDS-staged tile), so fewer VALU and
// LDS operations per product count more than fewer stalls. 4096 tokens: 748 ->
// 671-676 us; 512: 134-140 -> 111-114; 128: 71 -> 41; 77: 70 -> 34; 5120 x
// 17408 Q6_K at 8 tokens 38 -> 28 us (the register verify tile).
#include <algorithm>

#include "formats.h"
#include "kernels.h"
#include "panel.h"

namespace nuq {


typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void_t;

// (t & M) | o as one v_and_or_b32 (the compiler splits it in two for a
// literal mask).
template <uint32_t M>
__device__ __forceinline__ uint32_t and_or(uint32_t t, uint32_t o) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(t), "s"(M), "v"(o));
    return r;
}

// The weights are the CPU decoders' values rounded to f16, also where a block's
// scale is infinite: +-Inf by the code's sign, NaN for a zero code. Unsigned
// codes (Q4_K, Q5_K) are read as f16 subnormals, code 2^-24, by one and (or one
// byte permute) per pair, with 2^24 in the scale.
template <uint32_t M>
__device__ __forceinline__ half2v subnormal(uint32_t t) {
    return __builtin_bit_cast(half2v, opaque_and<M>(t));
}
// from bytes I and I + 2 of t
template <uint32_t I>
__device__ __forceinline__ half2v subnormal_bytes(uint32_t t) {
    return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0u, t, 0x0c020c00u + 0x00010001u * I));
}
// Signed codes of Q6_K and IQ4_XS carry a bias: two f16 values 1024 + byte (the
// byte goes into the mantissa of 1024.0, whose ulp is 1), whose bias the F32
// addend takes out. The addend is exact (the scale has at most 18 bits, the
// bias 6), but infinite with the scale: infinite scales are replaced
// (overflowing) before, and Q6_K rows with a NaN weight found after the loop.
constexpr uint32_t F16_1024 = 0x64006400u;
template <uint32_t M>
__device__ __forceinline__ half2v biased(uint32_t t) {
    return __builtin_bit_cast(half2v, and_or<M>(t, F16_1024));
}
// from bytes I and I + 2 of t
template <uint32_t I>
__device__ __forceinline__ half2v biased_bytes(uint32_t t) {
    return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(F16_1024 | 0x00640064u, t, 0x04020400u + 0x00010001u * I));
}
// A finite value of v's sign in the place of +-Inf, whose products with codes
// other than zero overflow f16 to +-Inf again.
__device__ __forceinline__ float overflowing(float v) {
    return fabsf(v) == INFINITY ? copysignf(0x1p100f, v) : v;
}

// f16(v * mul + add), one F32 rounding before it (v_fma_mix): the value of the
// CPU decoders' product-sum.
__device__ __forceinline__ _Float16 mix(_Float16 v, float mul, float add) { return (_Float16)fmaf((float)v, mul, add); }

// Four weights of one code word: `even` holds the codes of bytes 0 and 2,
// `odd` of bytes 1 and 3.
__device__ __forceinline__ void four(half8 &f, int at, half2v even, half2v odd, float mul, float add) {
    f[at] = mix(even[0], mul, add);
    f[at + 1] = mix(odd[0], mul, add);
    f[at + 2] = mix(even[1], mul, add);
    f[at + 3] = mix(odd[1], mul, add);
}
// Four weights from the signed bytes of t. `zero` is an f16 zero the compiler
// cannot see through: with it the product and its rounding are one v_fma_mix
// (a plain product is rounded by a second instruction). One conversion a code
// takes the place of the biased form's masks, so Q8_0 needs no bias: 17408 x
// 5120 at 4096 tokens 735-737 us against 730-737.
__device__ __forceinline__ void four_signed(half8 &f, int at, uint32_t t, float mul, _Float16 zero) {
    f[at] = (_Float16)fmaf(sbyte_f<0>(t), mul, (float)zero);
    f[at + 1] = (_Float16)fmaf(sbyte_f<1>(t), mul, (float)zero);
    f[at + 2] = (_Float16)fmaf(sbyte_f<2>(t), mul, (float)zero);
    f[at + 3] = (_Float16)fmaf(sbyte_f<3>(t), mul, (float)zero);
}
__device__ __forceinline__ _Float16 opaque_zero() {
    uint32_t z = 0;
    asm("" : "+s"(z));
    return __builtin_bit_cast(half2v, z)[0];
}

// The eight 6-bit scales and minima of a Q4_K / Q5_K header as bytes (groups
// 0-3, 4-7; quant/decode.zig:155-158), d and -dmin.
__device__ __forceinline__ void open_k(u32x4 hdr, uint32_t (&sc)[2], uint32_t (&mn)[2], float &d, float &ndmin) {
    d = half_bits(hdr.x & 0xffffu);
    ndmin = -half_bits(hdr.x >> 16);
    sc[0] = opaque_and<0x3f3f3f3fu>(hdr.y);
    mn[0] = opaque_and<0x3f3f3f3fu>(hdr.z);
    sc[1] = and_or<0x30303030u>(hdr.y >> 2, opaque_and<0x0f0f0f0fu>(hdr.w));
    mn[1] = and_or<0x30303030u>(hdr.z >> 2, opaque_and<0x0f0f0f0fu>(hdr.w >> 4));
}

// A weight row's raw bytes reach LDS in units of SLABS K slabs (64 columns
// each): NCH chunks of 16 bytes, chunk c from byte src(c) of the unit, so
// every field is 16-byte aligned in LDS whatever its alignment in the file.
// A lane (row, part p) then holds the bytes of its half of every slab in
// registers: chunk<P, C>() is the f16 B fragment of MFMA sub-step C of slab
// P, and slab chunk chunk_of(C, p) the activations (8 columns) that meet it.
// read() issues the LDS reads of a lane; `unit` is the row's image, `dwords`
// its NX dwords (from byte src_dword(j)). LDS holds UNITS units of a row.
template <uint32_t ENC>
struct PanelRaw;

template <>
struct PanelRaw<12> {
    static constexpr uint32_t SLABS = 4, BYTES = 144, NCH = 9, NX = 0, UNITS = 1;
    u32x4 hdr, qs[4];
    uint32_t sc[2], mn[2];
    float d24, d20, ndmin, mul0, add0, mul1, add1;
    __device__ static uint32_t src(uint32_t c) { return 16 * c; }
    __device__ static uint32_t chunk_of(uint32_t c, uint32_t part) { return (c & 1) * 4 + part * 2 + (c >> 1); }
    __device__ __forceinline__ void read(const uint8_t *unit, const uint8_t *, uint32_t part) {
        hdr = *(const u32x4 *)unit;
#pragma unroll
        for (int p = 0; p < 4; ++p) qs[p] = *(const u32x4 *)(unit + part * 16 + 16 + 32 * p);
    }
    __device__ __forceinline__ void open() {
        float d;
        open_k(hdr, sc, mn, d, ndmin);
        d24 = d * 0x1p24f;
        d20 = d * 0x1p20f;  // high nibbles stay in place (16 q)
    }
    template <int P>
    __device__ __forceinline__ void setup(uint32_t) {
        constexpr int E = 2 * (P & 1);
        mul0 = d24 * ubyte_f<E>(sc[P >> 1]);
        mul1 = d20 * ubyte_f<E + 1>(sc[P >> 1]);
        add0 = ndmin * ubyte_f<E>(mn[P >> 1]);
        add1 = ndmin * ubyte_f<E + 1>(mn[P >> 1]);
    }
    template <int P, int C>
    __device__ __forceinline__ half8 chunk() const {
        half8 f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t t = qs[P][2 * (C >> 1) + k];
            if constexpr ((C & 1) == 0)
                four(f, 4 * k, subnormal<0x000f000fu>(t), subnormal<0x000f000fu>(t >> 8), mul0, add0);
            else
                four(f, 4 * k, subnormal<0x00f000f0u>(t), subnormal<0x00f000f0u>(t >> 8), mul1, add1);
        }
        return f;
    }
};

template <>
struct PanelRaw<13> {
    static constexpr uint32_t SLABS = 4, BYTES = 176, NCH = 11, NX = 0, UNITS = 1;
    u32x4 hdr, qh, qs[4];
    uint32_t sc[2], mn[2];
    float d24, ndmin, mul0, add0, mul1, add1;
    __device__ static uint32_t src(uint32_t c) { return 16 * c; }
    __device__ static uint32_t chunk_of(uint32_t c, uint32_t part) { return (c & 1) * 4 + part * 2 + (c >> 1); }
    __device__ __forceinline__ void read(const uint8_t *unit, const uint8_t *, uint32_t part) {
        hdr = *(const u32x4 *)unit;
        qh = *(const u32x4 *)(unit + part * 16 + 16);
#pragma unroll
        for (int p = 0; p < 4; ++p) qs[p] = *(const u32x4 *)(unit + part * 16 + 48 + 32 * p);
    }
    __device__ __forceinline__ void open() {
        float d;
        open_k(hdr, sc, mn, d, ndmin);
        d24 = d * 0x1p24f;
    }
    template <int P>
    __device__ __forceinline__ void setup(uint32_t) {
        constexpr int E = 2 * (P & 1);
        mul0 = d24 * ubyte_f<E>(sc[P >> 1]);
        mul1 = d24 * ubyte_f<E + 1>(sc[P >> 1]);
        add0 = ndmin * ubyte_f<E>(mn[P >> 1]);
        add1 = ndmin * ubyte_f<E + 1>(mn[P >> 1]);
    }
    template <int P, int C>
    __device__ __forceinline__ half8 chunk() const {
        half8 f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t t = qs[P][2 * (C >> 1) + k], h = qh[2 * (C >> 1) + k];
            if constexpr ((C & 1) == 0) {
                // bit 2P of every high byte to bit 4
                const uint32_t b = 2 * P <= 4 ? h << (4 - 2 * P) : h >> (2 * P - 4);
                const uint32_t u = and_or<0x10101010u>(b, opaque_and<0x0f0f0f0fu>(t));
                four(f, 4 * k, subnormal_bytes<0>(u), subnormal_bytes<1>(u), mul0, add0);
            } else {
                // bit 2P + 1 to bit 4
                const uint32_t b = 2 * P + 1 <= 4 ? h << (3 - 2 * P) : h >> (2 * P - 3);
                const uint32_t u = and_or<0x10101010u>(b, opaque_and<0x0f0f0f0fu>(t >> 4));
                four(f, 4 * k, subnormal_bytes<0>(u), subnormal_bytes<1>(u), mul1, add1);
            }
        }
        return f;
    }
};

// Q6_K slab P: quarters P & 1 and (P & 1) + 2 of half P >> 1, whose codes
// share their ql and qh bytes (see slab_chunk). The last chunk is moved back
// to end at the block's end.
template <>
struct PanelRaw<14> {
    static constexpr uint32_t SLABS = 4, BYTES = 210, NCH = 14, NX = 0, UNITS = 1;
    u32x4 ql[4], qh[2], sc;
    uint32_t d16;
    float d, mul0, add0, mul1, add1;
    uint64_t inf = 0;  // lanes that met an infinite d
    __device__ __forceinline__ void open() {
        d = half_bits(d16);
        inf |= __builtin_amdgcn_ballot_w64(fabsf(d) == INFINITY);
        d = overflowing(d);
    }
    __device__ static uint32_t src(uint32_t c) { return c < 13 ? 16 * c : 194; }
    __device__ static uint32_t chunk_of(uint32_t c, uint32_t part) { return (c & 1) * 4 + part * 2 + (c >> 1); }
    __device__ __forceinline__ void read(const uint8_t *unit, const uint8_t *, uint32_t part) {
#pragma unroll
        for (int p = 0; p < 4; ++p) ql[p] = *(const u32x4 *)(unit + part * 16 + 32 * p);
#pragma unroll
        for (int h = 0; h < 2; ++h) qh[h] = *(const u32x4 *)(unit + part * 16 + 128 + 32 * h);
        sc = *(const u32x4 *)(unit + 192);
        d16 = *(const uint16_t *)(unit + 13 * 16 + 14);
    }
    template <int P>
    __device__ __forceinline__ void setup(uint32_t part) {
        // scales of values 16 part.. of the two quarters: bytes 8 (P >> 1) + 2 (P & 1) + part and + 4
        const uint32_t lo = sc[2 * (P >> 1)], hi = sc[2 * (P >> 1) + 1], sh = 16 * (P & 1) + 8 * part;
        mul0 = d * (float)(int8_t)((lo >> sh) & 0xffu);
        add0 = mul0 * -1056.f;
        mul1 = d * (float)(int8_t)((hi >> sh) & 0xffu);
        add1 = mul1 * -1056.f;
    }
    template <int P, int C>
    __device__ __forceinline__ half8 chunk() const {
        constexpr int S0 = 2 * (P & 1);  // high bits of the low quarter; + 4: of the high quarter
        half8 f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t t = ql[P][2 * (C >> 1) + k], h = qh[P >> 1][2 * (C >> 1) + k];
            const uint32_t l = (C & 1) == 0 ? t : t >> 4;
            const uint32_t b = (C & 1) == 0 ? h << (4 - S0) : h >> S0;  // to bits 4, 5
            const uint32_t u = and_or<0x30303030u>(b, opaque_and<0x0f0f0f0fu>(l));
            four(f, 4 * k, biased_bytes<0>(u), biased_bytes<1>(u), (C & 1) == 0 ? mul0 : mul1,
                 (C & 1) == 0 ? add0 : add1);
        }
        return f;
    }
    // Whether a weight of the row's blocks [b0, b1) is NaN: an infinite d times
    // a zero code or scale.
    __device__ static bool nan_weight(const uint8_t *row, uint32_t b0, uint32_t b1) {
        bool nan = false;
#pragma unroll 1
        for (uint32_t b = b0; b < b1; ++b) {
            const uint8_t *blk = row + (uint64_t)b * BYTES;
            if ((load_u16_bytes(blk + 208) & 0x7fffu) != 0x7c00u) continue;
#pragma unroll 1
            for (uint32_t k = 0; k < 128; ++k) {
                const uint32_t l = blk[k], h = blk[128 + (k >> 6) * 32 + (k & 31)] >> (2 * ((k >> 5) & 1));
                nan = nan || ((l & 15u) | (h & 3u) << 4) == 32u || (l >> 4 | ((h >> 4) & 3u) << 4) == 32u ||
                      blk[192 + (k & 15)] == 0;
            }
        }
        return nan;
    }
};

// IQ4_XS: chunk 0 is the header (and the first codes again), chunk 1 + g group g
template <>
struct PanelRaw<23> {
    static constexpr uint32_t SLABS = 4, BYTES = 136, NCH = 9, NX = 0, UNITS = 1;
    u32x2 hdr;
    u32x4 qs[4];
    float mul, add;
    __device__ __forceinline__ void open() {}
    __device__ static uint32_t src(uint32_t c) { return c ? 16 * c - 8 : 0; }
    __device__ static uint32_t chunk_of(uint32_t c, uint32_t part) { return part * 4 + (c & 1) * 2 + (c >> 1); }
    __device__ __forceinline__ void read(const uint8_t *unit, const uint8_t *, uint32_t part) {
        hdr = *(const u32x2 *)unit;
#pragma unroll
        for (int p = 0; p < 4; ++p) qs[p] = *(const u32x4 *)(unit + part * 16 + 16 + 32 * p);
    }
    template <int P>
    __device__ __forceinline__ void setup(uint32_t part) {
        const uint32_t low = (hdr.y >> (8 * P + 4 * part)) & 15u;
        const int sc = (int)(low | (((hdr.x >> (16 + 4 * P + 2 * part)) & 3u) << 4)) - 32;
        mul = overflowing(half_bits(hdr.x & 0xffffu) * (float)sc);  // no code is zero; Inf x 0 stays NaN
        add = mul * -1152.f;
    }
    template <int P, int C>
    __device__ __forceinline__ half8 chunk() const {
        half8 f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t t = qs[P][2 * (C >> 1) + k];
            const uint32_t v = iq4_lookup<0x80808080u>(((C & 1) == 0 ? t : t >> 4) & 0x0f0f0f0fu);  // + 128
            four(f, 4 * k, biased<0x00ff00ffu>(v), biased<0x00ff00ffu>(v >> 8), mul, add);
        }
        return f;
    }
};

// Q8_0: units of 128 columns, block q's codes in chunks 2q and 2q + 1, its
// scale (and two codes) in dword q after them. Two units are kept in LDS, so
// a unit's copies have more than its own two slabs to land.
template <>
struct PanelRaw<8> {
    static constexpr uint32_t SLABS = 2, BYTES = 136, NCH = 8, NX = 4, UNITS = 2;
    u32x4 qa[2], qb[2];
    uint32_t d16[2];
    float mul;
    __device__ __forceinline__ void open() {}
    __device__ static uint32_t src(uint32_t c) { return c / 2 * 34 + 2 + c % 2 * 16; }
    __device__ static uint32_t src_dword(uint32_t q) { return 34 * q; }
    __device__ static uint32_t chunk_of(uint32_t c, uint32_t part) { return part * 4 + c; }
    __device__ __forceinline__ void read(const uint8_t *unit, const uint8_t *dwords, uint32_t part) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint8_t *blk = unit + part * 32 + 64 * p;
            qa[p] = *(const u32x4 *)blk;
            qb[p] = *(const u32x4 *)(blk + 16);
            d16[p] = *(const uint32_t *)(dwords + part * 4 + 8 * p);
        }
    }
    template <int P>
    __device__ __forceinline__ void setup(uint32_t) {
        mul = half_bits(d16[P] & 0xffffu);
    }
    template <int P, int C>
    __device__ __forceinline__ half8 chunk() const {
        half8 f;
#pragma unroll
        for (int k = 0; k < 2; ++k)
            four_signed(f, 4 * k, (C >> 1) == 0 ? qa[P][2 * (C & 1) + k] : qb[P][2 * (C & 1) + k], mul, opaque_zero());
        return f;
    }
};

// First column of slab ks and the column offset of its chunk c (8 columns):
// 64 consecutive columns, except Q6_K, whose slab is the quarters qa and
// qa + 2 of one half (they share their code bytes).
template <uint32_t ENC>
__device__ __forceinline__ uint32_t slab_col0(uint32_t ks) {
    return ENC == 14 ? (ks >> 2) * 256 + ((ks & 3) >> 1) * 128 + (ks & 1) * 32 : ks * 64;
}
template <uint32_t ENC>
__device__ __forceinline__ uint32_t slab_chunk(uint32_t c) {
    return ENC == 14 && c >= 4 ? 64 + 8 * (c - 4) : 8 * c;
}

// One copy global -> LDS of BYTES (16 or 4) a lane as a buffer load: uniform
// base and offset, lane offset voff, the lane's bytes at lds + BYTES lane.
template <int BYTES>
__device__ __forceinline__ void panel_copy(const void *base, uint8_t *lds, uint32_t voff, uint32_t soff) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 0xffffffff, 0x00020000);
    if constexpr (BYTES == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t *)lds, 16, voff, soff, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t *)lds, 4, voff, soff, 0, 0);
}


// Vector memory operations a wave may leave in flight at the hand-over from
// slab j to j + 1. Each hand-over issues the XI copies of slab j + DEPTH and,
// where a raw unit starts (j % U == 0), the RAW copies of the unit UNITS
// ahead. Slab j + 1's copies went out DEPTH - 1 hand-overs ago; where a unit
// ends the next unit's, issued (UNITS - 1) U + U - 1 hand-overs ago, must have
// landed too.
template <uint32_t DEPTH, uint32_t XI, uint32_t U, uint32_t RAW, uint32_t UNITS>
constexpr int pn_younger(uint32_t j) {
    uint32_t n = (DEPTH - 2) * XI;
    for (uint32_t k = 1; k < DEPTH; ++k) n += (j + 8 - k) % U == 0 ? RAW : 0;
    const uint32_t unit = (UNITS * U - 2) * XI + (UNITS - 1) * RAW;
    return (int)(j % U == U - 1 && unit < n ? unit : n);
}

template <uint32_t ENC, int TG, int RG, int WR, int WK, int DEPTH>
constexpr size_t panel_lds() {
    using Raw = PanelRaw<ENC>;
    const size_t loop = (size_t)DEPTH * WK * TG * 4096 + (size_t)32 * RG * WR * WK * Raw::UNITS * (Raw::NCH * 16 + Raw::NX * 4);
    const size_t sums = WK > 1 ? (size_t)WR * WK * TG * RG * 4096 : 0;
    return loop > sums ? loop : sums;
}
// Waves per SIMD the registers have to allow: one workgroup of four waves per
// CU where the accumulators (over 128 registers) or the LDS leave no second.
template <uint32_t ENC, int TG, int RG, int WR, int WK, int DEPTH>
constexpr int panel_waves() {
    return TG * RG > 8 || (WR * WK == 4 && panel_lds<ENC, TG, RG, WR, WK, DEPTH>() > 80 * 1024) ? 1 : 2;
}

template <uint32_t ENC, int TG, int RG, int WR, int WK, int DEPTH>
__global__ void __launch_bounds__(64 * WR * WK, (panel_waves<ENC, TG, RG, WR, WK, DEPTH>()))
    panel_kernel(const uint8_t *__restrict__ w, uint64_t stride, uint32_t rows, uint32_t columns,
                 const _Float16 *__restrict__ x, uint64_t in_stride, float *__restrict__ y, uint64_t out_stride,
                 uint32_t tokens, uint32_t full, uint32_t tail, uint32_t splits, uint32_t group,
                 float *__restrict__ work) {
    using Raw = PanelRaw<ENC>;
    constexpr uint32_t BM = 32 * TG, BN = 32 * RG * WR, SLOT = BM * 128, XI = 4 * TG / WR;
    constexpr uint32_t U = Raw::SLABS, ROWB = Raw::NCH * 16, CHUNKS = 32 * RG * Raw::NCH, COPIES = (CHUNKS + 63) / 64;
    constexpr uint32_t DCOPIES = RG * Raw::NX / 2, RAWI = COPIES + DCOPIES, REGION = 32 * RG * (ROWB + 4 * Raw::NX);
    // Each sub-step is scheduled on its own: a twentieth of the compile time
    // and within 1 % (IQ4_XS 7 % faster); without it where IQ4_XS would spill.
    constexpr bool FENCE = !(ENC == 23 && RG == 1);
    extern __shared__ __attribute__((aligned(16))) uint8_t pn_smem[];
    const uint32_t tm = (tokens + BM - 1) / BM, tn = (rows + BN - 1) / BN;
    uint32_t tile = blockIdx.x, split = 0, ks0 = 0, ks1 = columns / 64;
    const bool split_k = tile >= full;
    if (split_k) {
        tile = full + (blockIdx.x - full) % tail;
        split = (blockIdx.x - full) / tail;
        const uint32_t nb = columns / 256;
        ks0 = __builtin_amdgcn_readfirstlane(split * nb / splits * 4);
        ks1 = __builtin_amdgcn_readfirstlane((split + 1) * nb / splits * 4);
    }
    const uint32_t lane = threadIdx.x & 63, part = lane >> 5, l32 = lane & 31;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave % WR, wk = wave / WR;
    // K ranges of the workgroup's WK wave sets; a shorter range only joins
    // the barriers of the longest one's last steps
    uint32_t idle = 0;
    if constexpr (WK > 1) {
        const uint32_t nb = (ks1 - ks0) / 4, b0 = wk * nb / WK, b1 = (wk + 1) * nb / WK;
        idle = (nb + WK - 1) / WK - (b1 - b0);
        ks1 = ks0 + 4 * b1;
        ks0 += 4 * b0;
    }
    uint32_t pm, pn;
    panel_coords(tile, tm, tn, group, &pm, &pn);
    // (the divisions leave uniform values in vector registers)
    const uint32_t m_base = __builtin_amdgcn_readfirstlane(pm * BM), n_base = __builtin_amdgcn_readfirstlane(pn * BN);

    // the wave's raw image: lane i of copy t moves chunk 64 t + i of its rows
    const uint8_t *wt = w + (uint64_t)n_base * stride;
    uint8_t *xslots = pn_smem + wk * SLOT, *region = pn_smem + DEPTH * WK * SLOT + wave * (Raw::UNITS * REGION);
    const uint8_t *image = region + l32 * ROWB, *dwords = region + 32 * RG * ROWB + l32 * (4 * Raw::NX);
    uint32_t woff[COPIES], doff[DCOPIES + 1];
#pragma unroll
    for (uint32_t t = 0; t < COPIES; ++t) {
        const uint32_t id = min(64 * t + lane, CHUNKS - 1), r = id / Raw::NCH;
        woff[t] = min(wr * (32 * RG) + r, rows - 1 - n_base) * (uint32_t)stride + Raw::src(id % Raw::NCH);
    }
    if constexpr (DCOPIES > 0)
#pragma unroll
        for (uint32_t t = 0; t < DCOPIES; ++t) {
            const uint32_t id = 64 * t + lane, r = id / Raw::NX;
            doff[t] = min(wr * (32 * RG) + r, rows - 1 - n_base) * (uint32_t)stride + Raw::src_dword(id % Raw::NX);
        }
    // lane i of copy q fills 16-byte slot i % 8 of tile row m = 8 q + i / 8
    // with slab chunk (i % 8) ^ (m / 2 % 8), so the 16 rows that one cycle of a
    // fragment read takes lie in different banks; rows past the tokens re-read
    // the last one
    uint32_t xoff[XI], aoff[4];
#pragma unroll
    for (uint32_t t = 0; t < XI; ++t)
        xoff[t] = (uint32_t)((uint64_t)min(8 * (wr + WR * t) + (lane >> 3), tokens - 1 - m_base) * in_stride +
                             slab_chunk<ENC>((lane & 7) ^ (((wr + WR * t) * 4 + (lane >> 4)) & 7))) * 2;
#pragma unroll
    for (int c = 0; c < 4; ++c) aoff[c] = l32 * 128 + ((Raw::chunk_of(c, part) ^ ((lane >> 1) & 7)) << 4);
    const _Float16 *xt = x + (uint64_t)m_base * in_stride;

    floatx16 acc[TG][RG];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][g][r] = 0.f;

    const uint32_t last = ks1 - 1;
#define PN_COPY(KS, S)                                                                                         \
    {                                                                                                          \
        const uint32_t soff = slab_col0<ENC>(min((KS), last)) * 2;                                             \
        _Pragma("unroll") for (uint32_t t = 0; t < XI; ++t)                                                    \
            panel_copy<16>(xt, xslots + (S) * (WK * SLOT) + (wr + WR * t) * 1024, xoff[t], soff);               \
    }
#define PN_RAW(KS, S)                                                                                          \
    {                                                                                                          \
        const uint32_t soff = min((KS), last) / U * Raw::BYTES;                                                \
        _Pragma("unroll") for (uint32_t t = 0; t < COPIES; ++t)                                                \
            if (64 * t + 64 <= CHUNKS || lane < CHUNKS % 64)                                                   \
                panel_copy<16>(wt, region + (S) * REGION + t * 1024, woff[t], soff);                           \
        _Pragma("unroll") for (uint32_t t = 0; t < DCOPIES; ++t)                                               \
            panel_copy<4>(wt, region + (S) * REGION + 32 * RG * ROWB + t * 256, doff[t], soff);                \
    }
#define PN_READ(S)                                                                                             \
    _Pragma("unroll") for (int g = 0; g < RG; ++g)                                                             \
        raw[g].read(image + (S) * REGION + g * 32 * ROWB, dwords + (S) * REGION + g * 32 * 4 * Raw::NX, part);
#define PN_FRAGS(B, S, C)                                                                                      \
    _Pragma("unroll") for (int t = 0; t < TG; ++t) fa[B][t] =                                                  \
        *(const half8 *)(xslots + (S) * (WK * SLOT) + aoff[C] + t * 4096);
    Raw raw[RG];
    half8 fa[2][TG], fb[2][RG];
#pragma unroll
    for (uint32_t u = 0; u < Raw::UNITS; ++u) PN_RAW(ks0 + u * U, u)
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) PN_COPY(ks0 + s, s)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    PN_FRAGS(0, 0, 0)
    PN_READ(0)
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        raw[g].open();
        raw[g].template setup<0>(part);
        fb[0][g] = raw[g].template chunk<0, 0>();
    }

    // One slab: J = slab index mod 4 (ranges start at a multiple of 4). Its
    // last sub-step's products cover the hand-over to the next slab: the wait
    // for that slab's copies, the barrier after which every wave has read
    // this slab's activations, the copies into their slot, and the next
    // slab's first fragment reads.
#define PN_STEP(J)                                                                                             \
    {                                                                                                          \
        PN_SUB(J, 0)                                                                                           \
        PN_SUB(J, 1)                                                                                           \
        PN_SUB(J, 2)                                                                                           \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(pn_younger<DEPTH, XI, U, RAWI, Raw::UNITS>(J)) : "memory");    \
        __builtin_amdgcn_s_barrier();                                                                          \
        asm volatile("" ::: "memory");                                                                         \
        PN_FRAGS(0, ((J + 1) % DEPTH), 0)                                                                      \
        if constexpr (J % U == U - 1) {                                                                        \
            PN_READ(((J + 1) / U) % Raw::UNITS)                                                                \
        }                                                                                                      \
        PN_COPY(ks + J + DEPTH, J % DEPTH)                                                                     \
        if constexpr (J % U == 0) PN_RAW(ks + J + U * Raw::UNITS, (J / U) % Raw::UNITS)                                                        \
        PN_SUB(J, 3)                                                                                           \
    }
#define PN_SUB(J, C)                                                                                           \
    {                                                                                                          \
        if constexpr (C < 3) {                                                                                 \
            PN_FRAGS((C + 1) & 1, J % DEPTH, (C + 1) & 3)                                                      \
            _Pragma("unroll") for (int g = 0; g < RG; ++g) fb[(C + 1) & 1][g] =                                \
                raw[g].template chunk<J % U, (C + 1) & 3>();                                                   \
        } else {                                                                                               \
            _Pragma("unroll") for (int g = 0; g < RG; ++g) {                                                   \
                if constexpr ((J + 1) % U == 0) raw[g].open();                                                 \
                raw[g].template setup<(J + 1) % U>(part);                                                      \
                fb[0][g] = raw[g].template chunk<(J + 1) % U, 0>();                                            \
            }                                                                                                  \
        }                                                                                                      \
        _Pragma("unroll") for (int t = 0; t < TG; ++t) _Pragma("unroll") for (int g = 0; g < RG; ++g)          \
            acc[t][g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[C & 1][t], fb[C & 1][g], acc[t][g], 0, 0, 0);  \
        _Pragma("unroll") for (int q = 0; q < TG * RG; ++q) {                                                  \
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                 \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                                                 \
            __builtin_amdgcn_sched_group_barrier(0x002, (20 * RG + TG * RG - 1) / (TG * RG), 0);               \
        }                                                                                                      \
        if constexpr (FENCE) __builtin_amdgcn_sched_barrier(0);                                                \
    }
    for (uint32_t ks = ks0; ks < ks1; ks += 4) {
        PN_STEP(0)
        PN_STEP(1)
        PN_STEP(2)
        PN_STEP(3)
    }
#undef PN_SUB
#undef PN_STEP
#undef PN_FRAGS
#undef PN_COPY
#undef PN_RAW
#undef PN_READ
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no copy into LDS outlives the workgroup

    // Infinite Q6_K scales took part as values that overflow, with which a zero
    // code or scale gives 0: rows that have one there are NaN. (A scan of those
    // rows after the loop: a branch in it costs 1 % at 8 tokens.)
    if constexpr (ENC == 14) {
#pragma unroll
        for (int g = 0; g < RG; ++g)
            if (raw[g].inf >> lane & 1) {
                const uint32_t r = min(wr * (32 * RG) + g * 32 + l32, rows - 1 - n_base);
                if (Raw::nan_weight(wt + (uint64_t)r * stride, ks0 / 4, ks1 / 4))
#pragma unroll
                    for (int t = 0; t < TG; ++t)
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[t][g][q] = NAN;
            }
    }

    // D layout: lane l32 holds weight row n; register r token 8 (r / 4) + 4 part + r % 4
    float *mine = split_k ? work + (uint64_t)((tile - full) * splits + split) * (BM * BN) : nullptr;
#define PN_STORE(T, G, R, V)                                                                                   \
    {                                                                                                          \
        const uint32_t n = wr * (32 * RG) + (G) * 32 + l32, m = (T) * 32 + 8 * ((R) >> 2) + 4 * part + ((R) & 3); \
        if (m_base + m < tokens && n_base + n < rows) {                                                        \
            if (split_k) mine[m * BN + n] = (V);                                                               \
            else y[(uint64_t)(m_base + m) * out_stride + n_base + n] = (V);                                    \
        }                                                                                                      \
    }
    if constexpr (WK == 1) {
#pragma unroll
        for (int t = 0; t < TG; ++t)
#pragma unroll
            for (int g = 0; g < RG; ++g)
#pragma unroll
                for (int r = 0; r < 16; ++r) PN_STORE(t, g, r, acc[t][g][r])
    } else {
        // the wave sets' sums meet in LDS and are added in set order; set k
        // stores every WK-th quad of registers
        for (uint32_t i = 0; i < 4 * idle; ++i) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        constexpr uint32_t QUADS = TG * RG * 4;
        float4 *sums = (float4 *)pn_smem;
#pragma unroll
        for (int t = 0; t < TG; ++t)
#pragma unroll
            for (int g = 0; g < RG; ++g)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sums[(wave * QUADS + (t * RG + g) * 4 + q) * 64 + lane] =
                        make_float4(acc[t][g][4 * q], acc[t][g][4 * q + 1], acc[t][g][4 * q + 2], acc[t][g][4 * q + 3]);
        __syncthreads();
        for (uint32_t u = wk; u < QUADS; u += WK) {
            float4 v = sums[(wr * QUADS + u) * 64 + lane];
#pragma unroll
            for (uint32_t k = 1; k < WK; ++k) {
                const float4 o = sums[((k * WR + wr) * QUADS + u) * 64 + lane];
                v.x += o.x;
                v.y += o.y;
                v.z += o.z;
                v.w += o.w;
            }
            const uint32_t t = u / 4 / RG, g = u / 4 % RG, r = 4 * (u & 3);
            PN_STORE(t, g, r, v.x)
            PN_STORE(t, g, r + 1, v.y)
            PN_STORE(t, g, r + 2, v.z)
            PN_STORE(t, g, r + 3, v.w)
        }
    }
#undef PN_STORE
}

template <uint32_t ENC, int TG, int RG, int WR, int WK, int DEPTH>
static hipError_t launch_shape(hipStream_t s, const PanelArgs &a, const PanelPlan &p, float *work) {
    constexpr size_t lds = panel_lds<ENC, TG, RG, WR, WK, DEPTH>();
    static_assert(lds <= 160 * 1024, "LDS");
    hipLaunchKernelGGL((panel_kernel<ENC, TG, RG, WR, WK, DEPTH>), dim3(p.full + p.tail * p.splits),
                       dim3(64 * WR * WK), lds, s, a.w, a.stride, a.rows, a.columns, a.x, a.in_stride, a.y,
                       a.out_stride, a.tokens, p.full, p.tail, p.splits, PANEL_GROUP, work);
    return hipGetLastError();
}

template <>
hipError_t launch_panel_enc<PANEL_ENC>(hipStream_t s, const PanelArgs &a, const PanelPlan &p, float *work) {
    switch (p.shape) {
#define NUQ_PANEL_CASE(I, T, R, W, K, D)                                                                            \
    case I: return launch_shape<PANEL_ENC, T, R, W, K, D>(s, a, p, work);
        NUQ_PANEL_SHAPES(NUQ_PANEL_CASE)
#undef NUQ_PANEL_CASE
    }
    return hipErrorInvalidValue;
}

}  // namespace nuq
