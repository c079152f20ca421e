// Main loops of the 256 x 256 tile GEMMs: two groups of four waves take turns on the matrix cores.
//
// A k-tile is 128 bytes of every activation row (64 fp16 or 128 int8 values).  Wave w = 4 wm + wn owns
// rows 128 wm .. and columns 64 wn .. of the tile (8 x 4 sub-tiles of 16 x 16) and works through a
// k-tile in four steps of 16 MFMAs, one quadrant (64 rows x 32 columns, the whole k-tile) each:
//     step 0: rows' half 0, columns' half 0     (reads the fragments of A0)
//     step 1: half 0, half 1                    (B1)
//     step 2: half 1, half 1                    (A1)
//     step 3: half 1, half 0                    (the next k-tile's B0)
// A step is a memory phase (fragment reads, the issue of one half-tile's LDS DMA) and a compute phase,
// each ended by a barrier.  Waves 4 .. 7 run one phase behind waves 0 .. 3, and wave w
// shares a SIMD with wave w + 4: while one computes the other reads, so the matrix cores meet neither
// an LDS round trip nor the barrier's skew.
//
// LDS holds two k-tiles, each operand in two half-tiles of 128 rows that are refilled on their own: a
// half-tile is free from the step after its last read, and its successor is requested then.  Step n
// reads what was requested in step n - 7 or before, so a request has six steps (about 3000 cycles) to
// land; before the barrier that ends the memory phase of step n - 1 every wave waits for its own part
// of it.  Both groups have read a half-tile, and waited for the reads, at least one barrier before any
// wave's request overwrites it.
//
// What bounds it: the loop keeps the matrix cores 95% busy (2048 of 2160 cycles a k-tile) and the card
// then lowers its clock to 1.5 - 1.6 GHz, so power decides.  16 x 16 sub-tiles draw less than 32 x 32
// (fragments held, no DMA: 1.95 against 1.66 GHz): 8192 x 8192 x 4096 fp16 1431 against 1253 TFLOP/s.
// DMAs issued between the MFMAs instead of in the memory phase: 1385; ahead of the fragment reads, with
// 32 x 32 sub-tiles: 1092 against 1253 (the reads then wait behind them).  PingPong takes both operands as
// the MFMAs do.  int8 weights against fp16 activations have a loop of their own, PingPongW8 below: widened
// between these MFMAs of 16 cycles (40 VALU operations a step, in either phase) they took 3082 - 3448 cycles a
// k-tile, 1206 - 1262 TFLOP/s.
#pragma once
#include <type_traits>

#include "qlin_internal.h"

namespace qlin {


template <bool I8>  // int8 x int8 into int32, or fp16 x fp16 into fp32
struct PingPong {
    static constexpr int AH = 128 * 128;                       // bytes of a half-tile: 128 rows of 128 bytes
    static constexpr int LDS = 8 * AH;                         // [2 k-tiles][A0 A1], then [2][B0 B1]
    static constexpr int KEEP = 12;                            // DMA instructions of six steps
    using Acc = std::conditional_t<I8, i32x4, f32x4>;

    // a, b: the tile's first rows (m0 .., n0 ..) at k = 0; lda, ldb: row strides in bytes; rows past arows /
    // brows re-read the last one.  ktiles whole k-tiles, at least 1.
    // acc[i][j], lane l, element r: row 128 wm + 16 i + 4 (l / 16) + r, column 64 wn + 16 j + l % 16.
    __device__ static __forceinline__ void run(uint8_t* smem, const uint8_t* a, int64_t lda, int arows, const uint8_t* b,
                                               int64_t ldb, int brows, int ktiles, int tid, Acc (&acc)[8][4]) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wm = wave >> 2, wn = wave & 3, r16 = lane & 15, g = lane >> 4;
        // DMA instruction i of a half-tile fills its 16-byte chunks u = 512 i + tid.  Row hr of half x of
        // the activations is tile row 128 (hr / 64) + 64 x + hr % 64, of the weights 64 (hr / 32) + 32 x +
        // hr % 32; logical chunk c of a row sits at c ^ (hr / 2) % 8, so that the 16 rows a 16-lane group
        // reads at one logical chunk fall in 16 distinct bank groups.
        uint32_t ao[2][2], bo[2][2];
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int u = 512 * i + tid, hr = u / 8, c = 16 * ((u % 8) ^ ((hr / 2) % 8));
                ao[half][i] = (uint32_t)(min(128 * (hr / 64) + 64 * half + hr % 64, arows - 1) * lda) + c;
                bo[half][i] = (uint32_t)(min(64 * (hr / 32) + 32 * half + hr % 32, brows - 1) * ldb) + c;
            }
        // half x of k-tile kt into buffer kt % 2 = buf; past the end: re-reads the last k-tile
        auto dma = [&](const uint8_t* base, const uint32_t (&off)[2], int kt, uint8_t* dst) {
            const uint8_t* src = base + (int64_t)min(kt, ktiles - 1) * 128;
#pragma unroll
            for (int i = 0; i < 2; ++i) lds_dma16(src + off[i], dst + 16 * (512 * i + 64 * wave));
        };
        auto dma_a = [&](int kt, int x, int buf) { dma(a, ao[x], kt, smem + (2 * buf + x) * AH); };
        auto dma_b = [&](int kt, int x, int buf) { dma(b, bo[x], kt, smem + (4 + 2 * buf + x) * AH); };

        // fragments of 16 bytes: lane l holds row (column) l % 16 of a 16 x 16 sub-tile and one of four
        // chunks of a 64-byte step e: chunk 4 e + l / 16 in both operands
        u32x4 fa[4][2], fb[3][2][2];  // fb: B0 of even and odd k-tiles, B1
        const uint8_t* ard = smem + (64 * wm + r16) * 128;
        const uint8_t* brd = smem + 4 * AH + (32 * wn + r16) * 128;
        const int sw = (r16 / 2) % 8;
        auto read_a = [&](int x, int buf) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    fa[i][e] = *reinterpret_cast<const u32x4*>(ard + (2 * buf + x) * AH + 2048 * i +
                                                               16 * ((4 * e + g) ^ sw));
        };
        auto read_b = [&](int x, int buf, u32x4 (&f)[2][2]) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    f[j][e] = *reinterpret_cast<const u32x4*>(brd + (2 * buf + x) * AH + 2048 * j + 16 * ((4 * e + g) ^ sw));
        };
        auto compute = [&](int x, int y, const u32x4 (&f)[2][2]) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        Acc& c = acc[4 * x + i][2 * y + j];
                        if constexpr (I8)
                            c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, fa[i][e]), __builtin_bit_cast(i32x4, f[j][e]), c, 0, 0, 0);
                        else
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, fa[i][e]), __builtin_bit_cast(f16x8, f[j][e]), c, 0, 0, 0);
                    }
        };
        // a barrier that orders this wave's LDS reads (waited for before it) and DMAs (waited for by
        // count) at the compiler's level too
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto mem_end = [&]() {
            wait_lgkmcnt0();
            wait_vmcnt<KEEP>();
            barrier();
        };
        auto tile = [&](int t, auto par) {
            constexpr int P = decltype(par)::value;
            read_a(0, P);
            dma_b(t + 2, 0, P);
            mem_end();
            compute(0, 0, fb[P]);
            barrier();
            read_b(1, P, fb[2]);
            dma_a(t + 2, 0, P);
            mem_end();
            compute(0, 1, fb[2]);
            barrier();
            read_a(1, P);
            dma_b(t + 2, 1, P);
            mem_end();
            compute(1, 1, fb[2]);
            barrier();
            read_b(0, P ^ 1, fb[P ^ 1]);
            dma_a(t + 2, 1, P);
            mem_end();
            compute(1, 0, fb[P]);
            barrier();
        };

#pragma unroll
        for (int t = 0; t < 2; ++t) {  // the requests of steps -8 .. -1
            dma_b(t, 0, t);
            dma_a(t, 0, t);
            dma_b(t, 1, t);
            dma_a(t, 1, t);
        }
        wait_vmcnt<KEEP>();  // B0 and A0 of the first k-tile
        barrier();
        read_b(0, 0, fb[0]);
        wait_lgkmcnt0();
        barrier();
        if (wm) barrier();  // waves 4 .. 7: one phase behind
        int t = 0;
        for (; t + 1 < ktiles; t += 2) {
            tile(t, std::integral_constant<int, 0>{});
            tile(t + 1, std::integral_constant<int, 1>{});
        }
        if (t < ktiles) tile(t, std::integral_constant<int, 0>{});
        if (!wm) barrier();
        wait_vmcnt<0>();
    }
};

// The same two groups and quadrants for fp16 activations against int8 weights, which are widened to fp16
// after the LDS read (exactly: fp16 bits 0x6400 | (q + 128), minus 1152).  Sub-tiles are 32 x 32 here, 8
// MFMAs a step: the other wave's widening (40 VALU operations in steps 1 and 3) finds issue slots
// between MFMAs of 32 cycles, not between those of 16 cycles.  The DMAs go between the MFMAs of the
// compute phase, since the memory phases are the longer ones here.
//
// A weight half-tile of 128 rows x 128 bytes holds two k-tiles (64-byte rows touch twice the cache lines
// a DMA instruction); it is read raw in steps 0 (B1) and 2 (B0 of the next k-tile), beside the
// activations, widened in the next step, and refilled by one instruction in each of four even steps.
// Steps read requests of six steps before or earlier.
struct PingPongW8 {
    static constexpr int AH = 128 * 128, LDS = 8 * AH;         // [2 k-tiles][A0 A1], then [2 pairs][B0 B1]
    static constexpr int KEEP = 6;                             // DMA instructions of four steps
    using Acc = f32x16;

    // As PingPong::run; ktiles is the number of 64-value k-tiles, even.  acc[i][j], lane l, element r: row
    // 128 wm + 32 i + 8 (r / 4) + 4 (l / 32) + r % 4, column 64 wn + 32 j + l % 32.
    __device__ static __forceinline__ void run(uint8_t* smem, const uint8_t* a, int64_t lda, int arows, const uint8_t* b,
                                               int64_t ldb, int brows, int ktiles, int tid, Acc (&acc)[4][2]) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wm = wave >> 2, wn = wave & 3, r32 = lane & 31, h = lane >> 5;
        uint32_t ao[2][2], bo[2][2];
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int u = 512 * i + tid, hr = u / 8, c = 16 * ((u % 8) ^ ((hr / 2) % 8));
                ao[half][i] = (uint32_t)(min(128 * (hr / 64) + 64 * half + hr % 64, arows - 1) * lda) + c;
                bo[half][i] = (uint32_t)(min(64 * (hr / 32) + 32 * half + hr % 32, brows - 1) * ldb) + c;
            }
        auto dma_a = [&](int kt, int x, int buf, int i) {
            lds_dma16(a + (int64_t)min(kt, ktiles - 1) * 128 + ao[x][i], smem + (2 * buf + x) * AH + 16 * (512 * i + 64 * wave));
        };
        auto dma_b1 = [&](int pair, int x, int buf, int i) {
            lds_dma16(b + (int64_t)min(pair, ktiles / 2 - 1) * 128 + bo[x][i], smem + (4 + 2 * buf + x) * AH + 16 * (512 * i + 64 * wave));
        };
        // the weight DMA of step 0 (i = 0) or 2 (i = 1) of k-tile t, t % 4 = Q: B1 of pair t / 2 + 1 in an even
        // k-tile, B0 of pair (t + 3) / 2 in an odd one
        auto dma_b = [&](int t, int i, auto q) {
            constexpr int Q = decltype(q)::value;
            dma_b1((t + 2 + Q % 2) / 2, 1 - Q % 2, ((Q + 2 + Q % 2) / 2) % 2, i);
        };
        // fragments: activations 16 bytes of row l % 32, chunk 4 p + 2 h + e for piece s = 2 p + e; one 16-byte
        // weight read (chunk 2 p + h of the k-tile's four) serves pieces 2 p and 2 p + 1
        u32x4 fa[2][4], fb[3][4], wq[2];  // fb: B0 of even and odd k-tiles, B1
        const uint8_t* ard = smem + (64 * wm + r32) * 128;
        const uint8_t* brd = smem + 4 * AH + (32 * wn + r32) * 128;
        const int sw = (r32 / 2) % 8;
        auto read_a = [&](int x, int buf) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    fa[i][s] = *reinterpret_cast<const u32x4*>(ard + (2 * buf + x) * AH + 4096 * i +
                                                               16 * ((4 * (s / 2) + 2 * h + s % 2) ^ sw));
        };
        auto read_b = [&](int x, auto q) {  // of a k-tile with t % 4 = Q
            constexpr int Q = decltype(q)::value % 4;
#pragma unroll
            for (int p = 0; p < 2; ++p)
                wq[p] = *reinterpret_cast<const u32x4*>(brd + (2 * (Q / 2) + x) * AH + 16 * ((4 * (Q % 2) + 2 * p + h) ^ sw));
        };
        auto widen = [&](u32x4 (&f)[4]) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const uint32_t u = wq[s / 2][2 * (s % 2) + d] ^ 0x80808080u;
                    const f16x2 off = {(f16)-1152.0f, (f16)-1152.0f};
                    f[s][2 * d] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + off);
                    f[s][2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + off);
                }
        };
        // the step's DMAs (i = 0, 1) after the second and the fifth MFMA
        auto compute = [&](int x, int y, const u32x4 (&f)[4], auto&& dma) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    Acc& c = acc[2 * x + i][y];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[i][s]), __builtin_bit_cast(f16x8, f[s]), c, 0, 0, 0);
                    if (2 * s + i == 1 || 2 * s + i == 4) {
                        __builtin_amdgcn_sched_barrier(0);
                        dma(2 * s + i == 4);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
        };
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto tile = [&](int t, auto q) {
            constexpr int Q = decltype(q)::value, P = Q % 2;
            read_a(0, P);
            read_b(1, q);
            wait_lgkmcnt0();
            barrier();
            compute(0, 0, fb[P], [&](int i) { if (!i) dma_b(t, 0, q); });
            barrier();
            widen(fb[2]);
            wait_vmcnt<KEEP>();
            barrier();
            compute(0, 1, fb[2], [&](int i) { dma_a(t + 2, 0, P, i); });
            barrier();
            read_a(1, P);
            read_b(0, std::integral_constant<int, Q + 1>{});
            wait_lgkmcnt0();
            barrier();
            compute(1, 1, fb[2], [&](int i) { if (!i) dma_b(t, 1, q); });
            barrier();
            widen(fb[P ^ 1]);
            wait_vmcnt<KEEP>();
            barrier();
            compute(1, 0, fb[P], [&](int i) { dma_a(t + 2, 1, P, i); });
            barrier();
        };

        constexpr std::integral_constant<int, 0> q0{};
        constexpr std::integral_constant<int, 1> q1{};
        constexpr std::integral_constant<int, 2> q2{};
        constexpr std::integral_constant<int, 3> q3{};
        // the first B0, then the requests of steps -8 .. -1
        dma_b1(0, 0, 0, 0);
        dma_b1(0, 0, 0, 1);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            dma_b(-2, x, q2);
            dma_a(0, x, 0, 0);
            dma_a(0, x, 0, 1);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            dma_b(-1, x, q3);
            dma_a(1, x, 1, 0);
            dma_a(1, x, 1, 1);
        }
        wait_vmcnt<KEEP>();  // all but the last two of B0 and the whole second k-tile's A
        barrier();
        read_b(0, q0);
        wait_lgkmcnt0();
        widen(fb[0]);
        barrier();
        if (wm) barrier();  // waves 4 .. 7: one phase behind
        int t = 0;
        for (; t + 3 < ktiles; t += 4) {
            tile(t, q0);
            tile(t + 1, q1);
            tile(t + 2, q2);
            tile(t + 3, q3);
        }
        if (t < ktiles) {
            tile(t, q0);
            tile(t + 1, q1);
        }
        if (!wm) barrier();
        wait_vmcnt<0>();
    }
};

}  // namespace qlin
