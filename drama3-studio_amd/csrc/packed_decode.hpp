// Weight decode of the packed-integer banks (modes 0-3) into MFMA operand
// registers, shared by the small-call, column-group and tiled kernels.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace dmoe {

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    const v2bf p = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, p);
}

__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    return (uint32_t)f32_to_f16(a) | ((uint32_t)f32_to_f16(b) << 16);
}

// E4M3 byte -> fp32 (hardware decode of one byte).
__device__ __forceinline__ float e4m3(uint32_t byte) { return fp8x2_to_f32(byte & 0xFFu, false)[0]; }

using h2v = _Float16 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int8_t q8(float level, float rel) {
    const float v = fminf(fmaxf(__builtin_rintf(level * rel), -127.0f), 127.0f);
    return (int8_t)(int)v;
}

// Dequantized operand registers of one weight row for one 128-K block.
struct PackedRow {
    v4i r[4];  // mode 0: 4 x (8 bf16 / fp16); modes 1-3: r[0], r[1] = 2 x 16 int8
};

// Zero-point word of banks without qzeros (zero point 8 in every nibble), so
// the mode-0 fetch loads a word either way.
static __device__ int32_t g_zero_point8 = (int32_t)0x88888888u;

// The bytes a lane loads for one weight row's 128-K block (its 32 K values),
// kept apart from the dequantization so loads can be issued early.
struct PackedRaw {
    v4i a;       // mode 0: 4 code words; mode 1: int8 bytes 0..15; modes 2, 3: low-nibble words
    v4i b;       // mode 1: int8 bytes 16..31; mode 2: b[0], b[1] = 2-bit high planes
    uint32_t x;  // mode 0: fp16 scale bits; modes 2, 3: the two e4m3 rel bytes
    uint32_t z;  // mode 0: qzeros word (0x88888888: zero point 8)
};

template <int MODE>
__device__ __forceinline__ PackedRaw fetch_wrow(const QuantProjArgs& a, int e, int n, int kb, int grp) {
    const uint8_t* w = a.w + (int64_t)e * a.w_se + (int64_t)n * a.w_sn;
    const uint8_t* sc = a.s + (int64_t)e * a.s_se + (int64_t)n * a.s_sn;
    PackedRaw r{};
    if constexpr (MODE == 0) {
        r.a = *(const v4i*)(w + kb * 64 + grp * 16);
        r.x = *(const uint16_t*)(sc + kb * 2);
        const int32_t* zw = a.z ? a.z + (int64_t)e * a.z_se + (int64_t)kb * (a.N / 8) + n / 8 : &g_zero_point8;
        r.z = (uint32_t)*zw;
    } else if constexpr (MODE == 1) {
        r.a = *(const v4i*)(w + kb * 128 + grp * 32);
        r.b = *(const v4i*)(w + kb * 128 + grp * 32 + 16);
    } else {
        // 32 codes: low nibbles (16 bytes), mode 2 also 2-bit high parts (8 bytes)
        r.a = *(const v4i*)(w + kb * 64 + grp * 16);
        if constexpr (MODE == 2) {
            const uint2 high = *(const uint2*)(w + a.K / 2 + kb * 32 + grp * 8);
            r.b[0] = (int)high.x;
            r.b[1] = (int)high.y;
        }
        r.x = *(const uint16_t*)(sc + kb * 8 + grp * 2);
    }
    return r;
}

template <int MODE, bool F16>
__device__ __forceinline__ void decode_wrow(const PackedRaw& raw, int n, const float* book, PackedRow& out) {
    if constexpr (MODE == 0) {
        const float scale = f16_to_f32((uint16_t)raw.x);
        const int zp = (int)((raw.z >> (4 * (n % 8))) & 15u);
        const float bias = -(float)zp * scale;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t u = (uint32_t)raw.a[t];
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = fmaf((float)((u >> (4 * i)) & 15u), scale, bias);  // exact
#pragma unroll
            for (int i = 0; i < 4; ++i)
                out.r[t][i] = (int)(F16 ? pack_f16(v[2 * i], v[2 * i + 1]) : pack_bf16(v[2 * i], v[2 * i + 1]));
        }
    } else if constexpr (MODE == 1) {
        out.r[0] = raw.a;
        out.r[1] = raw.b;
    } else if constexpr (MODE == 2) {
        // Two codes per packed fp16 pair: code c as the fp16 64 + c (0x5400 |
        // c << 4: the low nibble tops the half's low byte, the 2-bit high part
        // ends its high byte, so byte permutes assemble the pairs); level * rel
        // = (64 + c) * rel - 96 * rel in one fma, exact (6 + 4 significant
        // bits, 96 * 448 in range); clamping to [-127, 127] before the
        // rounding equals clamping after it (integer bounds); + 1536 then
        // rounds to the nearest even integer r and leaves r's two's-complement
        // byte as the low byte of the half -- q8(level, rel) for every code and
        // E4M3 byte.
#pragma unroll
        for (int j = 0; j < 2; ++j) {  // 16 codes = K [32 g + 16 j, +16): one rel group
            const _Float16 rh = (_Float16)e4m3(raw.x >> (8 * j));  // exact
            const h2v rel2 = {rh, rh}, bias2 = rel2 * h2v{-96, -96};
            const uint32_t a0 = (uint32_t)raw.a[2 * j], a1 = (uint32_t)raw.a[2 * j + 1], hw = (uint32_t)raw.b[j];
            uint32_t hi[4];  // byte b: 0x54 | high part of code k + 4 b
#pragma unroll
            for (int k = 0; k < 4; ++k) hi[k] = ((hw >> (2 * k)) & 0x03030303u) | 0x54545454u;
            // low nibbles of even / odd codes of each word, in the bytes' high halves
            const uint32_t e0 = (a0 << 4) & 0xF0F0F0F0u, d0 = a0 & 0xF0F0F0F0u;
            const uint32_t e1 = (a1 << 4) & 0xF0F0F0F0u, d1 = a1 & 0xF0F0F0F0u;
            auto quant = [&](uint32_t codes) {  // (low half, high half) -> their INT8 in the low bytes
                h2v v = __builtin_elementwise_fma(__builtin_bit_cast(h2v, codes), rel2, bias2);
                v = __builtin_elementwise_min(__builtin_elementwise_max(v, h2v{-127, -127}), h2v{127, 127});
                return __builtin_bit_cast(uint32_t, v + h2v{1536, 1536});
            };
            const uint32_t p04 = quant(__builtin_amdgcn_perm(hi[0], e0, 0x05020400u));
            const uint32_t p15 = quant(__builtin_amdgcn_perm(hi[1], d0, 0x05020400u));
            const uint32_t p26 = quant(__builtin_amdgcn_perm(hi[2], e0, 0x05030401u));
            const uint32_t p37 = quant(__builtin_amdgcn_perm(hi[3], d0, 0x05030401u));
            const uint32_t p8c = quant(__builtin_amdgcn_perm(hi[0], e1, 0x07020600u));
            const uint32_t p9d = quant(__builtin_amdgcn_perm(hi[1], d1, 0x07020600u));
            const uint32_t pae = quant(__builtin_amdgcn_perm(hi[2], e1, 0x07030601u));
            const uint32_t pbf = quant(__builtin_amdgcn_perm(hi[3], d1, 0x07030601u));
            // int q of the group: codes 4q .. 4q + 3 (low bytes of the halves)
            const uint32_t t0 = __builtin_amdgcn_perm(p15, p04, 0x06020400u), u0 = __builtin_amdgcn_perm(p37, p26, 0x06020400u);
            const uint32_t t1 = __builtin_amdgcn_perm(p9d, p8c, 0x06020400u), u1 = __builtin_amdgcn_perm(pbf, pae, 0x06020400u);
            out.r[j][0] = (int)__builtin_amdgcn_perm(u0, t0, 0x05040100u);
            out.r[j][1] = (int)__builtin_amdgcn_perm(u0, t0, 0x07060302u);
            out.r[j][2] = (int)__builtin_amdgcn_perm(u1, t1, 0x05040100u);
            out.r[j][3] = (int)__builtin_amdgcn_perm(u1, t1, 0x07060302u);
        }
    } else {
        const float rel[2] = {e4m3(raw.x), e4m3(raw.x >> 8)};
#pragma unroll
        for (int j = 0; j < 2; ++j) {  // 16 codes = K [32 g + 16 j, +16): one rel group
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // 4 codes per output int
                uint32_t packed = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int c = j * 16 + q * 4 + b;  // code index within the lane's 32
                    const uint32_t lo = ((uint32_t)raw.a[c / 8] >> (4 * (c % 8))) & 15u;
                    packed |= ((uint32_t)(uint8_t)q8(book[lo], rel[j])) << (8 * b);
                }
                out.r[j][q] = (int)packed;
            }
        }
    }
}

template <int MODE, bool F16>
__device__ __forceinline__ void load_wrow(const QuantProjArgs& a, int e, int n, int kb, int grp, const float* book,
                                          PackedRow& out) {
    decode_wrow<MODE, F16>(fetch_wrow<MODE>(a, e, n, kb, grp), n, book, out);
}

// W4A8 INT8 weights by table: tab[rel byte * 16 + code] = q8(book[code],
// e4m3(rel byte)), so the result equals decode_wrow<3>'s.  A lane's four codes
// of an output int index the 16-byte row of its group's scale byte through
// two byte permutes (codes 0-7 and 8-15) and a byte select.
__device__ __forceinline__ void decode_w4a8_tab(const PackedRaw& raw, const int8_t* tab, PackedRow& out) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // 16 codes = K [32 g + 16 j, +16): one rel group
        const v4i row = *(const v4i*)(tab + (((uint32_t)raw.x >> (8 * j)) & 0xFFu) * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // codes 16 j + 4 q .. +3: nibbles 4 (q % 2) .. +3 of word 2 j + q / 2
            uint32_t t = ((uint32_t)raw.a[2 * j + q / 2] >> (16 * (q % 2))) & 0xFFFFu;
            t = (t | (t << 8)) & 0x00FF00FFu;
            t = (t | (t << 4)) & 0x0F0F0F0Fu;  // byte b: code 4 q + b
            const uint32_t sel = t & 0x07070707u, high = ((t >> 3) & 0x01010101u) * 0xFFu;
            const uint32_t lo8 = __builtin_amdgcn_perm((uint32_t)row[1], (uint32_t)row[0], sel);
            const uint32_t hi8 = __builtin_amdgcn_perm((uint32_t)row[3], (uint32_t)row[2], sel);
            out.r[j][q] = (int)((hi8 & high) | (lo8 & ~high));
        }
    }
}

template <int MODE>
__device__ __forceinline__ float channel_scale(const QuantProjArgs& a, int e, int n) {
    const uint8_t* sc = a.s + (int64_t)e * a.s_se + (int64_t)n * a.s_sn;
    if constexpr (MODE == 1) return *(const float*)sc;
    else return *(const float*)(sc + a.K / 16);
}

}  // namespace dmoe
