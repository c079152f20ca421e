// GGUF linear for a single activation row (M = 1): a VALU matrix-vector product.
//
// With one activation row the MFMA's 16-row tile would run 1/16 full while every lane still paid
// the decode, so this path decodes straight into packed fp16 pairs and uses v_dot2_f32_f16:
//   * each lane owns one contiguous "chunk" of a weight row (64 or 128 values: a run of whole
//     32-value blocks, or part of a 256-value super-block) and loads it with 16-byte global loads
//     (only 4-byte alignment is needed); a row is covered by 16..64 lanes, a wave covers 1..4 rows,
//     and the grid has one wave per such group of rows (its loads issued before anything else);
//   * the activation row is read once per workgroup with coalesced loads and staged in LDS in a
//     swizzled order (a lane's own chunk, read with a 256-byte lane stride straight from global
//     memory, would touch a different cache line per lane and per load); each lane keeps its
//     chunk in registers as fp16 pairs permuted to match the decode order, plus fp32 sums over
//     each scale group (needed by the offsets below);
//   * 4-bit codes: nibble pairs become fp16 (1024 + q) with one v_and_or_b32 ("0x6400 | nibble");
//     the 1024 (and any format offset) is removed in fp32 through the group sums:
//         sum_k x_k * (a * q_k + b) = a * (S - 1024 * sum x) + b * sum x,  S = sum x_k (1024 + q_k);
//     IQ4_NL / IQ4_XS / Q4_0 instead read a 256-entry LDS table byte -> (value(lo), value(hi)) and
//     pair it with (x_j, x_j+16);
//   * per lane fp32 partials are reduced across the row's lanes with xor shuffles.
// Everything after the fp16 operands is fp32; no weight is rounded to fp16.
#include <utility>

#include "qlin_internal.h"
#include "gguf_exact.h"

namespace qlin {
namespace {

// Compile-time loop: f(std::integral_constant<int, I>{}) for I in [0, N).
template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

constexpr int GV_THREADS = 256;
constexpr int GV_MAX_K = 8192;

typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32a2 __attribute__((aligned(2)));

__device__ __forceinline__ f16x2 h2(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2(h2(a), h2(b), c, false);
}
// s + x.lo + x.hi for an fp16 pair x: one v_dot2_f32_f16 against (1, 1) (the products are exact)
__device__ __forceinline__ float pair_sum(uint32_t x, float s) { return dot2(x, 0x3C003C00u, s); }
// (x & 0x000F000F) | 0x64006400: fp16 pair (1024 + low nibble of byte 0, 1024 + low nibble of byte 2)
__device__ __forceinline__ uint32_t nib_pair(uint32_t w) { return (w & 0x000F000Fu) | 0x64006400u; }
// (x & 0x00F000F0) | 0x64006400: fp16 pair (1024 + 16 * high nibble of byte 0, of byte 2), exact
__device__ __forceinline__ uint32_t nib16_pair(uint32_t w) { return (w & 0x00F000F0u) | 0x64006400u; }
// bytes 0 and 2 (< 256) -> fp16 pair (1024 + b0, 1024 + b2)
__device__ __forceinline__ uint32_t byte_pair(uint32_t w) { return (w & 0x00FF00FFu) | 0x64006400u; }
// bytes 1 and 3 -> fp16 pair (1024 + b1, 1024 + b3): one v_perm against 0x64 bytes (no shift)
__device__ __forceinline__ uint32_t byte_pair_hi(uint32_t w) { return __builtin_amdgcn_perm(0x64646464u, w, 0x04030401u); }

// Interleave two fp16 pairs (a0, a1), (b0, b1) -> (a0, b0) and (a1, b1).
__device__ __forceinline__ uint32_t lo_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t hi_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

template <int N>
__device__ __forceinline__ void load_dwords(const uint8_t* p, uint32_t* r) {
    // p is 4-byte aligned; 16-byte loads need only dword alignment on gfx950.
#pragma unroll
    for (int i = 0; i + 4 <= N; i += 4) {
        const u32x4a v = *reinterpret_cast<const u32x4a*>(p + 4 * i);
        r[i] = v.x; r[i + 1] = v.y; r[i + 2] = v.z; r[i + 3] = v.w;
    }
#pragma unroll
    for (int i = (N / 4) * 4; i < N; ++i) r[i] = reinterpret_cast<const uint32_t*>(p)[i];
}

// Byte offset `off` (compile-time) of a dword array -> the dword starting there.
template <int OFF>
__device__ __forceinline__ uint32_t dw_at(const uint32_t* r) {
    if constexpr (OFF % 4 == 0) return r[OFF / 4];
    else return __builtin_amdgcn_alignbyte(r[OFF / 4 + 1], r[OFF / 4], OFF % 4);
}
template <int OFF>
__device__ __forceinline__ float half_at(const uint32_t* r) {
    const uint32_t w = (OFF % 4 == 0) ? r[OFF / 4] : (r[OFF / 4] >> 16);
    return f16_bits_to_f32((uint16_t)(w & 0xFFFFu));
}

// --------------------------------------------------------------------------------------------
// Format policies.  VC = values per lane chunk, LD = dwords loaded per chunk, CB = chunk byte
// offset inside a row for chunk c.  prep_x() turns the chunk's VC fp16 activations (natural order,
// as VC/2 pairs) into the operand order and the group sums; dot() returns the chunk's fp32 sum.
// --------------------------------------------------------------------------------------------
template <int T> struct GV;

// K-quants Q4_K / Q5_K: chunk = half super-block (sub-blocks 4h..4h+3, 128 values).
template <int T> struct GVK45 {
    static constexpr int QK = 256, TS = (T == gguf::Q4_K) ? 144 : 176, VC = 128;
    static constexpr int XP = 64;     // fp16 pairs kept per lane
    static constexpr int NG = 4;      // scale groups per chunk
    static constexpr int LD = (T == gguf::Q4_K) ? 20 : 28;
    static constexpr bool LUT = false;
    __device__ static int64_t chunk_off(int c) { return (int64_t)(c >> 1) * TS; }
    __device__ static void load(const uint8_t* row, int c, uint32_t* r) {
        const uint8_t* b = row + (int64_t)(c >> 1) * TS;
        const int h = c & 1;
        load_dwords<4>(b, r);                                  // d, dmin, scales[12]
        if constexpr (T == gguf::Q5_K) {
            load_dwords<8>(b + 16, r + 4);                     // qh[32]
            load_dwords<16>(b + 48 + 64 * h, r + 12);          // qs for sub-blocks 4h..4h+3
        } else {
            load_dwords<16>(b + 16 + 64 * h, r + 4);
        }
    }
    // natural pairs xn[v/2] = (x_v, x_v+1), v in [0,128): qs dword j (j<16) covers, for its low
    // nibbles, values v = 64*(j/8) + 4*(j%8) + t and for its high nibbles v + 32.
    __device__ static void prep_x(const uint32_t* xn, uint32_t* xp, float* xs) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int vlo = 64 * (j / 8) + 4 * (j % 8), vhi = vlo + 32;
            const uint32_t a = xn[vlo / 2], b = xn[vlo / 2 + 1], c = xn[vhi / 2], d = xn[vhi / 2 + 1];
            xp[4 * j + 0] = lo_lo(a, b);  // (x0, x2) low
            xp[4 * j + 1] = hi_hi(a, b);  // (x1, x3) low
            xp[4 * j + 2] = lo_lo(c, d);  // high
            xp[4 * j + 3] = hi_hi(c, d);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s = pair_sum(xn[16 * g + i], s);
            }
            xs[g] = s;
        }
    }
    __device__ static float dot(const uint32_t* r, int c, const uint32_t* xp, const float* xs) {
        const int h = c & 1;
        const float d = f16_bits_to_f32((uint16_t)(r[0] & 0xFFFFu)), dmin = f16_bits_to_f32((uint16_t)(r[0] >> 16));
        const uint32_t s0 = r[1], s1 = r[2], s2 = r[3];
        constexpr int QB = (T == gguf::Q4_K) ? 4 : 12;
        float S[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t w = r[QB + j];
            const int pair = j / 8;               // sub-blocks 2*pair (low), 2*pair+1 (high)
            uint32_t lo = w, hi = w >> 4;
            if constexpr (T == gguf::Q5_K) {
                const uint32_t qh = r[4 + (j % 8)];
                const int sbl = 4 * h + 2 * pair;  // sub-block of the low nibbles
                lo = (w & 0x0F0F0F0Fu) | (((qh >> sbl) & 0x01010101u) << 4);
                hi = ((w >> 4) & 0x0F0F0F0Fu) | (((qh >> (sbl + 1)) & 0x01010101u) << 4);
                S[2 * pair] = dot2(byte_pair(lo), xp[4 * j], S[2 * pair]);
                S[2 * pair] = dot2(byte_pair_hi(lo), xp[4 * j + 1], S[2 * pair]);
                S[2 * pair + 1] = dot2(byte_pair(hi), xp[4 * j + 2], S[2 * pair + 1]);
                S[2 * pair + 1] = dot2(byte_pair_hi(hi), xp[4 * j + 3], S[2 * pair + 1]);
            } else {
                // high nibbles as 1024 + 16 q (no shift): their sums carry 16x the code term
                (void)hi;
                S[2 * pair] = dot2(nib_pair(lo), xp[4 * j], S[2 * pair]);
                S[2 * pair] = dot2(nib_pair(lo >> 8), xp[4 * j + 1], S[2 * pair]);
                S[2 * pair + 1] = dot2(nib16_pair(w), xp[4 * j + 2], S[2 * pair + 1]);
                S[2 * pair + 1] = dot2(nib16_pair(w >> 8), xp[4 * j + 3], S[2 * pair + 1]);
            }
        }
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int sb = 4 * h + g;
            int sc, mn;
            if (h == 0) {
                sc = (s0 >> (8 * g)) & 63;
                mn = (s1 >> (8 * g)) & 63;
            } else {
                sc = ((s2 >> (8 * g)) & 0xF) | (((s0 >> (8 * g + 6)) & 3) << 4);
                mn = ((s2 >> (8 * g + 4)) & 0xF) | (((s1 >> (8 * g + 6)) & 3) << 4);
            }
            (void)sb;
            const float a = d * (float)sc, b = dmin * (float)mn;
            if (T == gguf::Q4_K && (g & 1)) acc += (0.0625f * a) * S[g] - (64.0f * a + b) * xs[g];
            else acc += a * S[g] - (1024.0f * a + b) * xs[g];
        }
        return acc;
    }
};
template <> struct GV<gguf::Q4_K> : GVK45<gguf::Q4_K> {};
template <> struct GV<gguf::Q5_K> : GVK45<gguf::Q5_K> {};

// Q8_0: chunk = 2 blocks (68 bytes, 64 values).
template <> struct GV<gguf::Q8_0> {
    static constexpr int VC = 64, XP = 32, NG = 2, LD = 17;
    static constexpr bool LUT = false;
    __device__ static void load(const uint8_t* row, int c, uint32_t* r) { load_dwords<17>(row + (int64_t)c * 68, r); }
    __device__ static void prep_x(const uint32_t* xn, uint32_t* xp, float* xs) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            xp[2 * j] = lo_lo(xn[2 * j], xn[2 * j + 1]);
            xp[2 * j + 1] = hi_hi(xn[2 * j], xn[2 * j + 1]);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s = pair_sum(xn[16 * g + i], s);
            }
            xs[g] = s;
        }
    }
    template <int B>
    __device__ static float block(const uint32_t* r, const uint32_t* xp, float xsum) {
        constexpr int o = 34 * B;
        const float d = half_at<o>(r);
        float S = 0.0f;
        static_for<8>([&](auto J) {
            constexpr int j = decltype(J)::value;
            const uint32_t w = dw_at<o + 2 + 4 * j>(r) ^ 0x80808080u;
            S = dot2(byte_pair(w), xp[16 * B + 2 * j], S);
            S = dot2(byte_pair_hi(w), xp[16 * B + 2 * j + 1], S);
        });
        return d * (S - 1152.0f * xsum);
    }
    __device__ static float dot(const uint32_t* r, int, const uint32_t* xp, const float* xs) {
        return block<0>(r, xp, xs[0]) + block<1>(r, xp, xs[1]);
    }
};

// Table formats: a 256-entry LDS table maps one code byte to the fp16 pair (value(lo), value(hi));
// the pair multiplies (x_j, x_j+16).
// Q4_0 / IQ4_NL: chunk = 4 blocks (72 bytes, 128 values).
template <int T> struct GVTab32 {
    static constexpr int QK = 32, TS = 18, VC = 128, XP = 64, NG = 4, LD = 18;
    static constexpr bool LUT = true;
    __device__ static void load(const uint8_t* row, int c, uint32_t* r) { load_dwords<18>(row + (int64_t)c * 72, r); }
    // block b (32 values): byte j (j<16) holds values j (lo) and j+16 (hi): pair (x_j, x_j+16)
    __device__ static void prep_x(const uint32_t* xn, uint32_t* xp, float* xs) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int j = 0; j < 16; j += 2) {
                const uint32_t lo = xn[16 * b + j / 2], hi = xn[16 * b + 8 + j / 2];
                xp[16 * b + j] = lo_lo(lo, hi);
                xp[16 * b + j + 1] = hi_hi(lo, hi);
            }
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s = pair_sum(xn[16 * b + i], s);
            }
            xs[b] = s;
        }
    }
    template <int B>
    __device__ static float block(const uint32_t* r, const uint32_t* xp, const uint32_t* tab) {
        constexpr int o = 18 * B;
        const float d = half_at<o>(r);
        float S = 0.0f;
        static_for<4>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const uint32_t w = dw_at<o + 2 + 4 * q>(r);
#pragma unroll
            for (int t = 0; t < 4; ++t) S = dot2(tab[(w >> (8 * t)) & 0xFFu], xp[16 * B + 4 * q + t], S);
        });
        return d * S;
    }
    __device__ static float dot(const uint32_t* r, int, const uint32_t* xp, const float* xs, const uint32_t* tab) {
        (void)xs;
        return block<0>(r, xp, tab) + block<1>(r, xp, tab) + block<2>(r, xp, tab) + block<3>(r, xp, tab);
    }
};
template <> struct GV<gguf::Q4_0> : GVTab32<gguf::Q4_0> {};
template <> struct GV<gguf::IQ4_NL> : GVTab32<gguf::IQ4_NL> {};

// IQ4_XS: chunk = half super-block (sub-blocks 4h..4h+3, 128 values).
template <> struct GV<gguf::IQ4_XS> {
    static constexpr int TS = 136, VC = 128, XP = 64, NG = 4, LD = 18;
    static constexpr bool LUT = true;
    __device__ static void load(const uint8_t* row, int c, uint32_t* r) {
        const uint8_t* b = row + (int64_t)(c >> 1) * TS;
        load_dwords<2>(b, r);                          // d, scales_h, scales_l
        load_dwords<16>(b + 8 + 64 * (c & 1), r + 2);  // qs of the four sub-blocks
    }
    __device__ static void prep_x(const uint32_t* xn, uint32_t* xp, float* xs) {
        GVTab32<gguf::IQ4_NL>::prep_x(xn, xp, xs);  // same (x_j, x_j+16) pairing per 32 values
    }
    __device__ static float dot(const uint32_t* r, int c, const uint32_t* xp, const float* xs, const uint32_t* tab) {
        (void)xs;
        const int h = c & 1;
        const float d = f16_bits_to_f32((uint16_t)(r[0] & 0xFFFFu));
        const uint32_t sh = r[0] >> 16, sl = r[1];
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int s = 4 * h + g;
            const int ls = ((sl >> (8 * (s >> 1) + 4 * (s & 1))) & 0xF) | (int)(((sh >> (2 * s)) & 3u) << 4);
            float S = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w = r[2 + 4 * g + q];
#pragma unroll
                for (int t = 0; t < 4; ++t) S = dot2(tab[(w >> (8 * t)) & 0xFFu], xp[16 * g + 4 * q + t], S);
            }
            acc += (d * (float)(ls - 32)) * S;
        }
        return acc;
    }
};

// Q6_K: chunk = half super-block (128 values): ql[64h..+64], qh[32h..+32], scales[8h..+8], d.
// Blocks are 210 bytes, so a block may start 2 bytes off a dword boundary; each region is loaded
// from the dword below it and realigned with v_alignbyte.
template <> struct GV<gguf::Q6_K> {
    static constexpr int TS = 210, VC = 128, XP = 64, NG = 8, LD = 17 + 9 + 3 + 1 + 1;
    static constexpr bool LUT = false;
    // raw dwords as loaded (realigned in dot(), so that no loaded value is used before the
    // activation staging); r[30] = the block's byte offset from a dword boundary (0 or 2)
    __device__ static void load(const uint8_t* row, int c, uint32_t* r) {
        const int h = c & 1;
        const uint8_t* b = row + (int64_t)(c >> 1) * TS;
        const int sh = (int)((uintptr_t)b & 3);  // 0 or 2
        const uint8_t* a = b - sh;
        // ql and qh halves end at least 14 bytes before the block end: the extra dword stays inside
        load_dwords<17>(a + 64 * h, r);            // ql half
        load_dwords<9>(a + 128 + 32 * h, r + 17);  // qh half
        // scales and d sit at the end of the block: read no byte past it.  The third scale dword
        // is needed only when sh = 2; with sh = 0 it re-reads the second (and is shifted out).
        const uint32_t* sc = reinterpret_cast<const uint32_t*>(a + 192 + 8 * h);
        r[26] = sc[0];
        r[27] = sc[1];
        r[28] = sc[sh ? 2 : 1];
        // d in the upper half of the block's last dword (2-byte aligned): a 16-bit load held across a
        // loop would be masked, and so waited for, at the loop's end
        r[29] = *reinterpret_cast<const u32a2*>(b + 206);
        r[30] = (uint32_t)sh;
    }
    // alignbyte with shift 0 returns its low operand: the same code serves both alignments
    __device__ static void realign(const uint32_t* r, uint32_t* q) {
        const uint32_t sh = r[30];
#pragma unroll
        for (int i = 0; i < 16; ++i) q[i] = __builtin_amdgcn_alignbyte(r[i + 1], r[i], sh);
#pragma unroll
        for (int i = 17; i < 25; ++i) q[i] = __builtin_amdgcn_alignbyte(r[i + 1], r[i], sh);
        q[26] = __builtin_amdgcn_alignbyte(r[27], r[26], sh);
        q[27] = __builtin_amdgcn_alignbyte(r[28], r[27], sh);
        q[29] = r[29] >> 16;
    }
    // ql dword j: low nibbles -> values 4j..4j+3, high nibbles -> 64 + 4j..; natural pairing (x0,x2),(x1,x3)
    __device__ static void prep_x(const uint32_t* xn, uint32_t* xp, float* xs) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int vlo = 4 * j, vhi = 64 + 4 * j;
            xp[4 * j + 0] = lo_lo(xn[vlo / 2], xn[vlo / 2 + 1]);
            xp[4 * j + 1] = hi_hi(xn[vlo / 2], xn[vlo / 2 + 1]);
            xp[4 * j + 2] = lo_lo(xn[vhi / 2], xn[vhi / 2 + 1]);
            xp[4 * j + 3] = hi_hi(xn[vhi / 2], xn[vhi / 2 + 1]);
        }
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                s = pair_sum(xn[8 * g + i], s);
            }
            xs[g] = s;
        }
    }
    __device__ static float dot(const uint32_t* raw, int, const uint32_t* xp, const float* xs) {
        uint32_t r[30];
        realign(raw, r);
        const float d = f16_bits_to_f32((uint16_t)(r[29] & 0xFFFFu));
        float S[8];
#pragma unroll
        for (int g = 0; g < 8; ++g) S[g] = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t ql = r[j], qh = r[17 + (j % 8)];
            const int sl = 2 * (j / 8);  // qh shift for the low-nibble values (v = 4j < 64)
            const uint32_t lo = (ql & 0x0F0F0F0Fu) | (((qh >> sl) & 0x03030303u) << 4);
            const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (sl + 4)) & 0x03030303u) << 4);
            const int glo = j / 4, ghi = 4 + j / 4;  // 16-value groups of v = 4j and 64 + 4j
            S[glo] = dot2(byte_pair(lo), xp[4 * j], S[glo]);
            S[glo] = dot2(byte_pair_hi(lo), xp[4 * j + 1], S[glo]);
            S[ghi] = dot2(byte_pair(hi), xp[4 * j + 2], S[ghi]);
            S[ghi] = dot2(byte_pair_hi(hi), xp[4 * j + 3], S[ghi]);
        }
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int sc = (int)(int8_t)(r[26 + g / 4] >> (8 * (g % 4)));
            const float a = d * (float)sc;
            acc += a * (S[g] - 1056.0f * xs[g]);
        }
        return acc;
    }
};

template <int T>
__device__ __forceinline__ uint32_t table_entry(int b) {
    // fp16 pair (value(lo nibble), value(hi nibble)) for code byte b
    float lo, hi;
    if constexpr (T == gguf::Q4_0) {
        lo = (float)((b & 0xF) - 8);
        hi = (float)((b >> 4) - 8);
    } else {
        lo = (float)gguf::iq4nl_level(b & 0xF);
        hi = (float)gguf::iq4nl_level(b >> 4);
    }
    return (uint32_t)__builtin_bit_cast(uint16_t, (f16)lo) | ((uint32_t)__builtin_bit_cast(uint16_t, (f16)hi) << 16);
}

// LPR lanes per row (a power of two <= 64); RPP = 64 / LPR rows per pass of a wave.
// Order of work: the activation row (coalesced), then each wave's weight chunks for two passes --
// so every load is in flight before the first wait -- then the LDS staging of the activations
// (and the table, for formats with one) and the prep of the activation pairs while the weights
// arrive.  No load sits behind a lane-dependent branch: rows past N re-read row N - 1 and are
// not stored.
template <int T, int LPR>
__global__ __launch_bounds__(GV_THREADS) void gguf_gemv_kernel(const f16* __restrict__ x, const int32_t* __restrict__ xexp,
                                                               const uint8_t* __restrict__ w,
                                                               int64_t row_bytes, int N, int K,
                                                               const void* __restrict__ bias, int bias_dt,
                                                               void* __restrict__ y, int y_dt) {
    using F = GV<T>;
    constexpr int VC = F::VC;
    constexpr int RPP = 64 / LPR;  // rows per pass of a wave
    constexpr int NU = VC / 8;     // 16-byte activation units per chunk
    __shared__ uint32_t tab_all[F::LUT ? GV_THREADS / 64 : 1][F::LUT ? 256 : 1];
    __shared__ __attribute__((aligned(16))) u32x4 xs_lds[GV_MAX_K / 8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane % LPR, rp = lane / LPR;

    const int waves_total = gridDim.x * (GV_THREADS / 64);
    const int gw = blockIdx.x * (GV_THREADS / 64) + wave;
    const int passes = (N + RPP - 1) / RPP;
    const int KU = K / 8;

    // 1. the activation row, with fully coalesced loads (consecutive lanes, consecutive 16 bytes).
    //    Without branches: units past the row re-read (and below re-write) its last unit.
    u32x4 xst[GV_MAX_K / 8 / GV_THREADS];
#pragma unroll
    for (int j = 0; j < GV_MAX_K / 8 / GV_THREADS; ++j)
        xst[j] = reinterpret_cast<const u32x4*>(x)[min(tid + GV_THREADS * j, KU - 1)];
    // 2. the weight chunks of this wave's first pass (rows past N re-read row N - 1)
    auto row_of = [&](int p) { return min(p * RPP + rp, N - 1); };
    int p = gw;
    uint32_t r0[F::LD];
    __builtin_amdgcn_sched_barrier(0);
    F::load(w + (int64_t)row_of(p) * row_bytes, c, r0);
    // epilogue operands, fetched now rather than after the reduction
    const int xe = xexp ? xexp[0] : 0;
    uint32_t bv0 = 0;  // raw bits (0 reads as +0 in every dtype)
    if (bias) bv0 = load_bits_rt(bias, bias_dt, row_of(p));
    __builtin_amdgcn_sched_barrier(0);
    // 3. activations into LDS: unit i of chunk c at i * LPR + (c ^ i), so that the per-lane reads
    //    below (fixed i, consecutive c) and these writes both spread over the banks.  The fences
    //    order LDS only: the weight loads stay in flight across the barrier.
#pragma unroll
    for (int j = 0; j < GV_MAX_K / 8 / GV_THREADS; ++j) {
        const int u = min(tid + GV_THREADS * j, KU - 1);
        const int cc = u / NU, i = u % NU;
        xs_lds[i * LPR + (cc ^ i)] = xst[j];
    }
    uint32_t* tab = tab_all[F::LUT ? wave : 0];
    if constexpr (F::LUT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) tab[lane + 64 * i] = table_entry<T>(lane + 64 * i);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);  // nothing that needs a weight value moves above this point
    uint32_t xn[VC / 2];
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const u32x4 v = xs_lds[i * LPR + (c ^ i)];
        xn[4 * i] = v.x; xn[4 * i + 1] = v.y; xn[4 * i + 2] = v.z; xn[4 * i + 3] = v.w;
    }
    uint32_t xp[F::XP];
    float xsum[F::NG];
    F::prep_x(xn, xp, xsum);

    auto finish = [&](const uint32_t* r, int pp, uint32_t bv) {
        const int n = pp * RPP + rp;
        float v;
        if constexpr (F::LUT) v = F::dot(r, c, xp, xsum, tab);
        else v = F::dot(r, c, xp, xsum);
#pragma unroll
        for (int m = 1; m < LPR; m <<= 1) v += __shfl_xor(v, m, 64);
        if (c == 0 && n < N) store_rt(y, y_dt, n, __builtin_ldexpf(v, xe) + bits_to_f32_rt(bv, bias_dt));
    };
    // The first pass is computed unconditionally (its store is guarded), so its loads are not
    // moved into a branch behind the barrier; the launch sizes the grid so that it is all there is.
    for (;;) {
        finish(r0, p, bv0);
        p += waves_total;
        if (p >= passes) break;
        F::load(w + (int64_t)row_of(p) * row_bytes, c, r0);
        if (bias) bv0 = load_bits_rt(bias, bias_dt, row_of(p));
    }
}

template <int T>
hipError_t launch(const GgufGemvArgs& a, hipStream_t st) {
    using F = GV<T>;
    const int lpr = a.K / F::VC;
    const int rpp = 64 / lpr;
    const int passes = (a.N + rpp - 1) / rpp;
    // One pass per wave, every wave's loads issued up front.  Two passes per wave (half the
    // waves, the second pass's loads also up front) measured 5-14% slower at K = N = 4096: with
    // eight waves per CU instead of four, one wave's decode overlaps another's loads.
    int waves = passes;
    int blocks = (waves + 3) / 4;
    if (blocks < 1) blocks = 1;
    dim3 grid((unsigned)blocks), block(GV_THREADS);
#define QLIN_GV(L)                                                                                      \
    hipLaunchKernelGGL((gguf_gemv_kernel<T, L>), grid, block, 0, st, (const f16*)a.x, a.xexp, a.w, a.row_bytes, a.N, a.K, a.bias, \
                       a.bias_dtype, a.y, a.y_dtype)
    switch (lpr) {
        case 16: QLIN_GV(16); break;
        case 32: QLIN_GV(32); break;
        case 64: QLIN_GV(64); break;
        default: return hipErrorInvalidValue;
    }
#undef QLIN_GV
    return hipGetLastError();
}


// --------------------------------------------------------------------------------------------
// Rows of any length (and bf16 / fp32 rows of every length): LPR lanes walk a row's chunks c = l,
// l + LPR, ..., with the loads of two chunks in flight per lane.  The operand order of the activations
// is made once per workgroup, in LDS, instead of once per lane in registers (a wave's chunks change),
// and bf16 / fp32 rows are normalized there, where the prologue was a launch of its own.  Bound by
// the weight stream, the decode's VALU (Q4_K: 5 operations per two weights) and, at a few MB, by the
// latency of the first bytes.  In a HIP graph over cold weights, us against the kernels that these
// rows took before (the small-M one, or the prologue and the kernel below): Q4_K K5120 N13824 bf16
// 13.0 against 30.8 (3.1 TB/s), Q6_K K13824 N5120 bf16 19.9 against 45.2, IQ4_XS K14336 N4096 bf16
// 12.8 against 23.4, Q8_0 K11264 N4096 bf16 11.9 against 20.8, Q4_K K = N = 4096 bf16 5.4 against
// 7.5.  fp16 rows keep the kernel below at its K (Q4_K 5.0, Q6_K 5.6, Q8_0 5.6 us there).
//
// LDS operand: 16-byte unit i (8 values) of chunk c at i * C + c, so that the lanes of a row read
// consecutive units.  Byte codes: each 8 values as the pairs (0,2) (1,3) (4,6) (5,7).  Table
// formats: unit 4 b + q of a chunk holds the pairs (x_j, x_j+16), j = 4 q .. + 3, of its block b.
// Codes become exact fp16 integers (1024 + q less 1024 in one packed add), so no offset term cancels
// against the sums; the K-quants' minima take sums of 32 activations, at g * C + c.
// --------------------------------------------------------------------------------------------
template <int OFF>
__device__ __forceinline__ uint32_t less(uint32_t pair) {  // an fp16 pair minus (OFF, OFF)
    return __builtin_bit_cast(uint32_t, h2(pair) - f16x2{(f16)OFF, (f16)OFF});
}
template <int T>
struct GVRow {  // Q4_K, Q5_K
    template <typename XU, typename XS>
    __device__ static float dot(const uint32_t* r, int c, XU&& xu, XS&& xs, const uint32_t*) {
        const int h = c & 1;
        const float d = f16_bits_to_f32((uint16_t)(r[0] & 0xFFFFu)), dmin = f16_bits_to_f32((uint16_t)(r[0] >> 16));
        const uint32_t s0 = r[1], s1 = r[2], s2 = r[3];
        constexpr int QB = (T == gguf::Q4_K) ? 4 : 12;
        float S[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < 2; ++p)  // sub-blocks 2p (low nibbles), 2p + 1 (high)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u32x4 xl = xu(8 * p + q), xh = xu(8 * p + 4 + q);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t w = r[QB + 8 * p + 2 * q + e];
                    const uint32_t l0 = e ? xl.z : xl.x, l1 = e ? xl.w : xl.y, h0 = e ? xh.z : xh.x, h1 = e ? xh.w : xh.y;
                    if constexpr (T == gguf::Q5_K) {
                        const uint32_t qh = r[4 + 2 * q + e];
                        const int sb = 4 * h + 2 * p;
                        const uint32_t lo = (w & 0x0F0F0F0Fu) | (((qh >> sb) & 0x01010101u) << 4);
                        const uint32_t hi = ((w >> 4) & 0x0F0F0F0Fu) | (((qh >> (sb + 1)) & 0x01010101u) << 4);
                        S[2 * p] = dot2(less<1024>(byte_pair(lo)), l0, S[2 * p]);
                        S[2 * p] = dot2(less<1024>(byte_pair_hi(lo)), l1, S[2 * p]);
                        S[2 * p + 1] = dot2(less<1024>(byte_pair(hi)), h0, S[2 * p + 1]);
                        S[2 * p + 1] = dot2(less<1024>(byte_pair_hi(hi)), h1, S[2 * p + 1]);
                    } else {  // high nibbles as 16 q (no shift)
                        S[2 * p] = dot2(less<1024>(nib_pair(w)), l0, S[2 * p]);
                        S[2 * p] = dot2(less<1024>(nib_pair(w >> 8)), l1, S[2 * p]);
                        S[2 * p + 1] = dot2(less<1024>(nib16_pair(w)), h0, S[2 * p + 1]);
                        S[2 * p + 1] = dot2(less<1024>(nib16_pair(w >> 8)), h1, S[2 * p + 1]);
                    }
                }
            }
        // the chunk's four 6-bit scales and minima as bytes, for both halves without a branch
        const uint32_t hm = 0u - (uint32_t)h;
        const uint32_t sc = (((s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)) & hm) | (s0 & 0x3F3F3F3Fu & ~hm);
        const uint32_t mn = ((((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) & hm) | (s1 & 0x3F3F3F3Fu & ~hm);
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float a = d * (float)((sc >> (8 * g)) & 0xFFu), b = dmin * (float)((mn >> (8 * g)) & 0xFFu);
            acc += (T == gguf::Q4_K && (g & 1) ? 0.0625f * a : a) * S[g] - b * xs(g);
        }
        return acc;
    }
};
template <>
struct GVRow<gguf::Q6_K> {
    template <typename XU, typename XS>
    __device__ static float dot(const uint32_t* raw, int, XU&& xu, XS&&, const uint32_t*) {
        uint32_t r[30];
        GV<gguf::Q6_K>::realign(raw, r);
        const float d = f16_bits_to_f32((uint16_t)(r[29] & 0xFFFFu));
        float S[8];
#pragma unroll
        for (int g = 0; g < 8; ++g) S[g] = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {  // values 8q .. + 7 (low nibbles), 64 + 8q .. + 7 (high)
            const u32x4 xl = xu(q), xh = xu(8 + q);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int j = 2 * q + e, sl = 2 * (j / 8), glo = j / 4, ghi = 4 + j / 4;
                const uint32_t ql = r[j], qh = r[17 + (j % 8)];
                const uint32_t lo = (ql & 0x0F0F0F0Fu) | (((qh >> sl) & 0x03030303u) << 4);
                const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (sl + 4)) & 0x03030303u) << 4);
                S[glo] = dot2(less<1056>(byte_pair(lo)), e ? xl.z : xl.x, S[glo]);
                S[glo] = dot2(less<1056>(byte_pair_hi(lo)), e ? xl.w : xl.y, S[glo]);
                S[ghi] = dot2(less<1056>(byte_pair(hi)), e ? xh.z : xh.x, S[ghi]);
                S[ghi] = dot2(less<1056>(byte_pair_hi(hi)), e ? xh.w : xh.y, S[ghi]);
            }
        }
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int sc = (int)(int8_t)(r[26 + g / 4] >> (8 * (g % 4)));
            acc += (d * (float)sc) * S[g];
        }
        return acc;
    }
};
template <>
struct GVRow<gguf::Q8_0> {
    template <typename XU, typename XS>
    __device__ static float dot(const uint32_t* r, int, XU&& xu, XS&&, const uint32_t*) {
        float acc = 0.0f;
        static_for<2>([&](auto B) {
            constexpr int b = decltype(B)::value, o = 34 * b;
            float S = 0.0f;
            static_for<4>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                const u32x4 xv = xu(4 * b + q);
                const uint32_t w0 = dw_at<o + 2 + 8 * q>(r) ^ 0x80808080u, w1 = dw_at<o + 6 + 8 * q>(r) ^ 0x80808080u;
                S = dot2(less<1152>(byte_pair(w0)), xv.x, S);
                S = dot2(less<1152>(byte_pair_hi(w0)), xv.y, S);
                S = dot2(less<1152>(byte_pair(w1)), xv.z, S);
                S = dot2(less<1152>(byte_pair_hi(w1)), xv.w, S);
            });
            acc += half_at<o>(r) * S;
        });
        return acc;
    }
};
// four bytes of codes against one unit: a table entry is the fp16 pair of a byte's two values
__device__ __forceinline__ float tab_dot(uint32_t w, const u32x4& xv, const uint32_t* tab, float S) {
    S = dot2(tab[w & 0xFFu], xv.x, S);
    S = dot2(tab[(w >> 8) & 0xFFu], xv.y, S);
    S = dot2(tab[(w >> 16) & 0xFFu], xv.z, S);
    return dot2(tab[w >> 24], xv.w, S);
}
template <int T>
struct GVRowTab32 {
    template <typename XU, typename XS>
    __device__ static float dot(const uint32_t* r, int, XU&& xu, XS&&, const uint32_t* tab) {
        float acc = 0.0f;
        static_for<4>([&](auto B) {
            constexpr int b = decltype(B)::value, o = 18 * b;
            float S = 0.0f;
            static_for<4>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                S = tab_dot(dw_at<o + 2 + 4 * q>(r), xu(4 * b + q), tab, S);
            });
            acc += half_at<o>(r) * S;
        });
        return acc;
    }
};
template <> struct GVRow<gguf::Q4_0> : GVRowTab32<gguf::Q4_0> {};
template <> struct GVRow<gguf::IQ4_NL> : GVRowTab32<gguf::IQ4_NL> {};
template <>
struct GVRow<gguf::IQ4_XS> {
    template <typename XU, typename XS>
    __device__ static float dot(const uint32_t* r, int c, XU&& xu, XS&&, const uint32_t* tab) {
        const int h = c & 1;
        const float d = f16_bits_to_f32((uint16_t)(r[0] & 0xFFFFu));
        const uint32_t sh = r[0] >> 16, sl = r[1];
        float acc = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int s = 4 * h + g;
            const int ls = ((sl >> (8 * (s >> 1) + 4 * (s & 1))) & 0xF) | (int)(((sh >> (2 * s)) & 3u) << 4);
            float S = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) S = tab_dot(r[2 + 4 * g + q], xu(4 * g + q), tab, S);
            acc += (d * (float)(ls - 32)) * S;
        }
        return acc;
    }
};

constexpr int GVR_MAX_K = 16384;  // 32 KiB of operand in LDS

// 8 raw activations as loaded (held until the weight loads are out)
template <typename TX> struct RawUnit {
    u32x4 v[sizeof(TX) / 2];
    __device__ void load(const TX* p) {
#pragma unroll
        for (int i = 0; i < (int)sizeof(TX) / 2; ++i) v[i] = reinterpret_cast<const u32x4*>(p)[i];
    }
    __device__ float get(int e) const {
        if constexpr (sizeof(TX) == 4) return __uint_as_float(v[e / 4][e % 4]);
        else return bf16_bits_to_f32((uint16_t)(v[0][e / 2] >> (16 * (e % 2))));
    }
};

template <int T, int LPR, typename TX, int NT>
__global__ __launch_bounds__(NT) void gguf_gemv_rows_kernel(const TX* x, const int32_t* xexp, const uint8_t* w,
                                                            int64_t row_bytes, int N, int K, const void* bias,
                                                            int bias_dt, void* y, int y_dt) {
    using F = GV<T>;
    constexpr bool RAW = !std::is_same<TX, f16>::value;  // fp16 rows are used as they are
    constexpr bool TAB = F::LUT;
    constexpr int NW = NT / 64, NX = GVR_MAX_K / 8 / NT;
    constexpr int VC = F::VC, RPW = 64 / LPR;
    constexpr bool MIN = T == gguf::Q4_K || T == gguf::Q5_K;  // block minima: sums of x per 32 values
    __shared__ __attribute__((aligned(16))) u32x4 xop[GVR_MAX_K / 8];
    __shared__ float xsum[MIN ? GVR_MAX_K / 32 : 1];
    __shared__ uint32_t tab_all[TAB ? NW : 1][TAB ? 256 : 1];
    __shared__ float red[NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane % LPR, KU = K / 8, C = K / VC, IT = (C + LPR - 1) / LPR;
    const int nwaves = gridDim.x * NW, groups = (N + RPW - 1) / RPW;
    int g = blockIdx.x * NW + wave;                      // this wave's row group; then g + nwaves, ...
    auto row = [&](int gg) { return min(gg * RPW + lane / LPR, N - 1); };

    // the activations' loads first (units past the row re-read its last), then two chunks' weights
    RawUnit<TX> xv[NX];
#pragma unroll
    for (int j = 0; j < NX; ++j) xv[j].load(x + 8 * min(tid + NT * j, KU - 1));
    __builtin_amdgcn_sched_barrier(0);
    uint32_t r0[F::LD], r1[F::LD];
    // Loads run two chunks ahead of the sums, across the end of a row group into the next one; they
    // are unconditional (past the last chunk they re-read it), so that the compiler's wait for the
    // older of the two does not cover the newer.
    int fg = g, fit = 0;
    const uint8_t* frow = w + (int64_t)row(g) * row_bytes;
    auto fetch = [&](uint32_t* r) {
        F::load(frow, min(l + LPR * fit, C - 1), r);
        if (++fit == IT) {
            if (fg + nwaves < groups) {
                fg += nwaves;
                fit = 0;
                frow = w + (int64_t)row(fg) * row_bytes;
            } else {
                fit = IT - 1;
            }
        }
    };
    fetch(r0);
    fetch(r1);
    const int xe = xexp ? xexp[0] : 0;
    uint32_t bv = bias ? load_bits_rt(bias, bias_dt, row(g)) : 0u;
    __builtin_amdgcn_sched_barrier(0);

    int E = xe;
    if constexpr (RAW) {  // the prologue's normalization: fp16(x 2^-E), E the exponent of max |x|
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < NX; ++j)
            if (NT * j < KU) {
#pragma unroll
                for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(xv[j].get(e)));
            }
        amax = wave_max(amax);
        if (lane == 0) red[wave] = amax;
        lds_barrier();
#pragma unroll
        for (int i = 0; i < NW; ++i) amax = fmaxf(amax, red[i]);
        E = frexp_exp(amax);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        if (NT * j >= KU) break;
        const int u = tid + NT * j;
        uint32_t h[4];  // the unit's fp16 pairs in natural order
        if constexpr (RAW) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const f16 a = (f16)__builtin_ldexpf(xv[j].get(2 * e), -E), b = (f16)__builtin_ldexpf(xv[j].get(2 * e + 1), -E);
                h[e] = (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = xv[j].v[0][e];
        }
        constexpr int UC = VC / 8;
        const int c = u / UC, i = u % UC;
        u32x4 o;
        if constexpr (TAB) {
            // lanes t and t ^ 2 hold the same 8 places of a block's two halves: the lower makes its
            // first four pairs (x_j, x_j+16), the upper its last four
            const bool up = tid & 2;
            const uint32_t s0 = up ? h[0] : h[2], s1 = up ? h[1] : h[3];
            const uint32_t t0 = __shfl_xor((int)s0, 2, 64), t1 = __shfl_xor((int)s1, 2, 64);
            const uint32_t a0 = up ? t0 : h[0], a1 = up ? t1 : h[1], b0 = up ? h[2] : t0, b1 = up ? h[3] : t1;
            o = u32x4{lo_lo(a0, b0), hi_hi(a0, b0), lo_lo(a1, b1), hi_hi(a1, b1)};
            const int k4 = i % 4;  // units 0, 2, 1, 3 of a block make pairs 0 .. 3, 4 .. 7, 8 .. 11, 12 .. 15
            if (u < KU) xop[(i - k4 + 2 * (k4 & 1) + (k4 >> 1)) * C + c] = o;
        } else {
            o = u32x4{lo_lo(h[0], h[1]), hi_hi(h[0], h[1]), lo_lo(h[2], h[3]), hi_hi(h[2], h[3])};
            if (u < KU) xop[i * C + c] = o;
            if constexpr (MIN) {
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e) s = pair_sum(h[e], s);
                s += lane_xor<1>(s);
                s += lane_xor<2>(s);
                if (u < KU && u % 4 == 0) xsum[(i / 4) * C + c] = s;
            }
        }
    }
    uint32_t* tab = tab_all[TAB ? wave : 0];
    if constexpr (TAB) {
#pragma unroll
        for (int i = 0; i < 4; ++i) tab[lane + 64 * i] = table_entry<T>(lane + 64 * i);
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);  // nothing that needs a weight value moves above this point

    float acc = 0.0f;
    int it = 0;
    auto step = [&](uint32_t* r) {
        const int cc = l + LPR * it, c = min(cc, C - 1);
        const float v = GVRow<T>::dot(r, c, [&](int i) { return xop[i * C + c]; }, [&](int i) { return xsum[i * C + c]; }, tab);
        acc += cc < C ? v : 0.0f;
        // the refill goes into the registers just used: issued before the sum is done (the empty asm
        // pins it) it would need others, and a copy, a wait for the load, at the end of the loop
        asm volatile("" : "+v"(acc));
        __builtin_amdgcn_sched_barrier(0);
        fetch(r);
        __builtin_amdgcn_sched_barrier(0);
        if (++it == IT) {
#pragma unroll
            for (int m = 1; m < LPR; m <<= 1) acc += __shfl_xor(acc, m, 64);
            const int n = g * RPW + lane / LPR;
            if (l == 0 && n < N) store_rt(y, y_dt, n, __builtin_ldexpf(acc, E) + bits_to_f32_rt(bv, bias_dt));
            g += nwaves;
            if (bias) bv = load_bits_rt(bias, bias_dt, row(g));  // past the last group: row N - 1, not used
            acc = 0.0f;
            it = 0;
        }
    };
    const int steps = g < groups ? ((groups - g + nwaves - 1) / nwaves) * IT : 0;
    for (int s = 1; s < steps; s += 2) {
        step(r0);
        step(r1);
    }
    if (steps & 1) step(r0);
}

// Lanes per row L and row groups per wave G.  The fastest grids measured have at most one workgroup per
// CU (with more on some CUs they wait for those, and each redoes the operand): W = 1024 waves in
// workgroups of 4, 2048 in workgroups of 8.  Of those, the shortest wave: G row groups of IT chunks and
// one reduction each; of equally short ones the most lanes per row, whose loads read longer pieces of
// fewer rows and which keep more waves in flight.  us for each L at its best G: Q6_K K13824 N5120 L8
// 25.0, L16 23.7, L32 21.0, L64 19.9 (L8, L32 and L64 are equally short); Q4_K there L8 17.8, L64 15.9;
// Q8_0 K6912 N5120 L8 13.2, L64 10.8.  Q4_K K5120 N13824 L8 14.0, L16 16.6, L32 19.0; Q4_K K3072 N3072
// L16 5.3, L32 5.6, L8 6.1; Q4_K K8192 N1024 L64 4.8, L32 5.6.
inline int gemv_rows_lanes(int N, int C, int W, int& G) {
    int best = 0, L = 8;
    for (int l : {8, 16, 32, 64}) {
        if (l > 8 && l / 2 >= C) break;  // half the lanes would have no chunk
        const int64_t waves = ((int64_t)N * l + 63) / 64;
        const int g = (int)((waves + W - 1) / W), cost = g * ((C + l - 1) / l + 1);
        if (!best || cost <= best) {
            best = cost;
            L = l;
            G = g;
        }
    }
    return L;
}

template <int T, typename TX, int NT>
hipError_t launch_rows_nt(const GgufGemvArgs& a, hipStream_t st) {
    int G = 1;
    const int L = gemv_rows_lanes(a.N, a.K / GV<T>::VC, 4 * NT, G);
    const int64_t rows = (int64_t)NT / L * G;
    const dim3 grid((unsigned)((a.N + rows - 1) / rows)), block(NT);
#define QLIN_GVR(LV)                                                                                                   \
    hipLaunchKernelGGL((gguf_gemv_rows_kernel<T, LV, TX, NT>), grid, block, 0, st, (const TX*)a.x, a.xexp, a.w, a.row_bytes, \
                       a.N, a.K, a.bias, a.bias_dtype, a.y, a.y_dtype)
    switch (L) {
        case 8: QLIN_GVR(8); break;
        case 16: QLIN_GVR(16); break;
        case 32: QLIN_GVR(32); break;
        default: QLIN_GVR(64); break;
    }
#undef QLIN_GVR
    return hipGetLastError();
}

// Workgroups of 8 waves (twice the loads in flight per operand) for large Q4_K tensors: K5120 N13824 14.3
// -> 13.0 us, K13824 N5120 16.4 -> 15.2, K4096 N14336 11.7 -> 11.2, K16384 N8192 21.5 -> 20.4; below 50
// million weights the longer start loses (K5120 N8192 8.6 against 10.0).  Q5_K goes either way there (K4096 N14336
// 14.0 -> 13.3, K16384 N8192 25.3 -> 24.5, but K8192 N16384 24.5 -> 24.8, K3584 N18944 16.9 -> 17.3, K13824 N5120 18.7
// -> 19.6), Q6_K lost where it was measured (K13824 N5120 19.9 -> 21.1); both and the types not measured keep 4 waves.
template <int T, typename TX>
hipError_t launch_rows(const GgufGemvArgs& a, hipStream_t st) {
    if constexpr (T == gguf::Q4_K) {
        if ((int64_t)a.N * a.K >= 50000000) return launch_rows_nt<T, TX, 512>(a, st);
    }
    return launch_rows_nt<T, TX, 256>(a, st);
}

template <typename Fn>
bool dispatch_gemv(int t, Fn&& f) {
    switch (t) {
        case gguf::Q4_0: f.template operator()<gguf::Q4_0>(); return true;
        case gguf::Q8_0: f.template operator()<gguf::Q8_0>(); return true;
        case gguf::Q4_K: f.template operator()<gguf::Q4_K>(); return true;
        case gguf::Q5_K: f.template operator()<gguf::Q5_K>(); return true;
        case gguf::Q6_K: f.template operator()<gguf::Q6_K>(); return true;
        case gguf::IQ4_NL: f.template operator()<gguf::IQ4_NL>(); return true;
        case gguf::IQ4_XS: f.template operator()<gguf::IQ4_XS>(); return true;
        default: return false;
    }
}

}  // namespace

bool gguf_gemv_rows_supported(int type, int64_t K, int64_t row_bytes, const void* w, const void* x) {
    // The kernel's loads are clamped to a row's last chunk, so a row has one: K = 0 is not taken.  Q6_K rows
    // of an odd number of blocks start 2 bytes off a dword, which its loads realign.
    if (K < 1 || K > GVR_MAX_K || (uintptr_t)w % 4 || (uintptr_t)x % 16 || row_bytes % (type == gguf::Q6_K ? 2 : 4)) return false;
    bool ok = false;
    dispatch_gemv(type, [&]<int T>() { ok = K % GV<T>::VC == 0; });
    return ok;
}

// Short fp16 rows over few weights stay with the 16-row MFMA kernel: neither launches a prologue for them, and what
// counts is the time to the first bytes, which here waits for the operand's trip through LDS.  us, 16-row kernel and
// GEMV: Q5_K K256 N64 2.6, 3.3, N8192 3.4, 3.8, N16384 5.2, 5.4; Q4_K K256 N4096 2.9, 3.3, N12288 4.8, 4.9, N16384 5.1,
// 5.0; K768 N64 2.7, 3.1, N3072 3.3, 3.4, N8192 4.0, 3.7; K512 N1024 3.1, 3.15, N4096 3.5, 3.4.  Q4_0 and Q5_K also at
// the other lengths: Q4_0 K512 N4096 3.4, 3.6; K1024 N256 3.2, 3.3, N2048 3.60, 3.65; K1536 N64 3.2, 3.3, N1024 3.7,
// 3.65; K2304 N64 4.1, 3.5.  Q6_K and Q8_0 gain at every length (Q6_K K256 N64 19.8, 3.5; Q8_0 K256 2.8, 2.65).
bool gguf_short_row(int type, int64_t N, int64_t K) {
    if (K < 1 || K % 256 || K >= 2048 || type == gguf::Q6_K || type == gguf::Q8_0) return false;
    if (K == 256 || K == 768) return N * K <= 3 << 20;
    return (type == gguf::Q4_0 || type == gguf::Q5_K) && N * K <= 2 << 20;
}

hipError_t run_gguf_gemv_rows(const GgufGemvArgs& a, hipStream_t st) {
    if (!gguf_gemv_rows_supported(a.type, a.K, a.row_bytes, a.w, a.x)) return hipErrorInvalidValue;
    if (a.y_dtype != DT_F32 && a.y_dtype != DT_F16 && a.y_dtype != DT_BF16) return hipErrorInvalidValue;
    hipError_t err = hipErrorInvalidValue;
    dispatch_gemv(a.type, [&]<int T>() {
        if (a.x_dtype == DT_F16) err = launch_rows<T, f16>(a, st);
        else if (a.x_dtype == DT_BF16) err = launch_rows<T, bf16_t>(a, st);
        else if (a.x_dtype == DT_F32) err = launch_rows<T, float>(a, st);
    });
    return err;
}

bool gguf_gemv_supported(int type, int64_t M, int64_t K, int64_t row_bytes, const void* w, const void* x) {
    if (M != 1 || K > GV_MAX_K || (uintptr_t)w % 4 || (uintptr_t)x % 16 || row_bytes % 4) return false;
    bool ok = false;
    dispatch_gemv(type, [&]<int T>() {
        const int64_t vc = GV<T>::VC;
        if (K % vc) return;
        const int64_t lpr = K / vc;
        ok = (lpr == 16 || lpr == 32 || lpr == 64);
    });
    return ok;
}

hipError_t run_gguf_gemv(const GgufGemvArgs& a, hipStream_t st) {
    if (a.y_dtype != DT_F32 && a.y_dtype != DT_F16 && a.y_dtype != DT_BF16) return hipErrorInvalidValue;
    hipError_t err = hipErrorInvalidValue;
    bool ok = dispatch_gemv(a.type, [&]<int T>() { err = launch<T>(a, st); });
    return ok ? err : hipErrorInvalidValue;
}

}  // namespace qlin
