// Input gradient of the frozen-weight packed linears (roblennon/mac-kernels-public:
// int8_linear_grad_input, bench/bench_int8_backward.py:15, 52; the backward of
// int8_linear_trainable / w4a8_linear_trainable, train/train_lora.py:187-188, 210, 221).
//
// The weight in the original basis is W[n, :] = s[n] q[n, :] H (q the stored int8 codes or the
// W4A8 int8 grid, s the per-row scale, H the block Hadamard of the ConvRot group, H = H^T = H^-1),
// so  dx = dy W = ((dy diag(s)) q) H.
//   bwd_rows_kernel: a[m, n] = fp16((dy[m, n] s[n]) 2^-E[m]), E[m] the exponent of the row's
//     max |dy s| (one rounding, no overflow or underflow of the row's large values), rows
//     zero-padded to a multiple of 128;
//   bwd_gemm_kernel, bwd_gemm_pair_kernel: c = a q over n with fp16 MFMA (the int8 codes are exact fp16), one
//     workgroup per 128 rows x 256 columns of dx; the weight tile goes to LDS as stored (rows
//     of n, k contiguous) and each MFMA fragment (8 consecutive n of one column) is one
//     transposing 8-byte LDS read, widened in registers; the epilogue scales rows by 2^E[m],
//     applies H to each 16-lane run of the row and rounds once to dx's dtype.
#include <type_traits>

#include "qlin_internal.h"
#include "hadamard.h"

namespace qlin {

namespace {

constexpr int BW_BM = 128, BW_BK = 256, BW_BN = 64;
// weight tile in LDS as stored, [64 n][256 k] int8, row r's 16-byte chunk c at chunk c ^ 2 (r % 8):
// the transposing fragment reads (8 rows x 2 chunk halves per 16 lanes, even and odd chunks in the two
// groups of a 32-lane half) fall on distinct banks
constexpr int BW_ASZ = BW_BM * BW_BN * 2, BW_BUF = BW_ASZ + BW_BN * BW_BK;  // bytes of a stage: a tile, weight tile
__device__ __forceinline__ int bw_chunk(int row, int c) { return c ^ (2 * (row & 7)); }
constexpr int BW_OW = BW_BK + BW_BK / 4;  // epilogue row stride in floats: 4 pad floats per 16

// a[m, :] = fp16(dy[m, :] * s * 2^-E[m]), zero past N up to lda; e[m] = E[m].  8 consecutive
// values per thread and step, 16-byte loads and stores when the rows allow.
template <typename T>
__device__ __forceinline__ void load8_row(const T* row, int64_t n, int64_t N, bool vec, float* v) {
    if (vec && n + 8 <= N) {
        if constexpr (sizeof(T) == 2) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(row + n);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                T lo, hi;
                const uint16_t l16 = (uint16_t)(w[i] & 0xFFFFu), h16 = (uint16_t)(w[i] >> 16);
                __builtin_memcpy(&lo, &l16, 2);
                __builtin_memcpy(&hi, &h16, 2);
                v[2 * i] = dtype_traits<T>::to_f32(lo);
                v[2 * i + 1] = dtype_traits<T>::to_f32(hi);
            }
        } else {
            const f32x4 a = *reinterpret_cast<const f32x4*>(row + n), b = *reinterpret_cast<const f32x4*>(row + n + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = a[i];
                v[4 + i] = b[i];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = n + i < N ? dtype_traits<T>::to_f32(row[n + i]) : 0.f;
    }
}

// 8 scale values from n (stride 0: one value for every row of the weight)
template <typename TS>
__device__ __forceinline__ void load8_scale(const TS* s, int64_t n, int64_t N, int64_t stride, float* v) {
    if (stride == 0) {
        const float c = dtype_traits<TS>::to_f32(s[0]);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = c;
    } else if (sizeof(TS) == 4 && n + 8 <= N && (uintptr_t)(s + n) % 16 == 0) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(s + n), b = *reinterpret_cast<const f32x4*>(s + n + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = a[i];
            v[4 + i] = b[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = n + i < N ? dtype_traits<TS>::to_f32(s[n + i]) : 0.f;
    }
}

template <typename T, typename TS>
__global__ __launch_bounds__(256) void bwd_rows_kernel(const T* __restrict__ dy, int64_t ldd, int64_t N,
                                                       const TS* __restrict__ s, int64_t s_stride,
                                                       f16* __restrict__ a, int64_t lda, int32_t* __restrict__ e) {
    __shared__ float red[4];
    const int64_t m = blockIdx.x;
    const int tid = threadIdx.x;
    const T* row = dy + m * ldd;
    const bool vec = ldd % 8 == 0 && (uintptr_t)dy % 16 == 0;
    float amax = 0.f;
    for (int64_t n = 8 * tid; n < N; n += 2048) {
        float v[8], sv[8];
        load8_row(row, n, N, vec, v);
        load8_scale(s, n, N, s_stride, sv);
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i] * sv[i]));  // zeros past N
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int E = frexp_exp(amax);
    f16* out = a + m * lda;
    for (int64_t n = 8 * tid; n < lda; n += 2048) {  // lda is a multiple of 128: whole 8-value pieces
        float v[8], sv[8];
        load8_row(row, n, N, vec, v);
        load8_scale(s, n, N, s_stride, sv);
        f16x8 hv;
#pragma unroll
        for (int i = 0; i < 8; ++i) hv[i] = (f16)__builtin_ldexpf(v[i] * sv[i], -E);  // 0 past N
        *reinterpret_cast<f16x8*>(out + n) = hv;
    }
    if (tid == 0) e[m] = E;
}

// 8 int8 (two dwords, in order) -> 8 exact fp16: bits 0x6400 | (q + 128) = 1152 + q, minus 1152.
__device__ __forceinline__ f16x8 i8x8_to_f16(uint32_t w0, uint32_t w1) {
    const f16x2 off = {(f16)-1152.0f, (f16)-1152.0f};
    const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
    const f16x2 h0 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u)) + off;
    const f16x2 h1 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u)) + off;
    const f16x2 h2 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u)) + off;
    const f16x2 h3 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)) + off;
    return f16x8{h0[0], h0[1], h1[0], h1[1], h2[0], h2[1], h3[0], h3[1]};
}

typedef int v2i __attribute__((ext_vector_type(2)));

// The output of a tile, four passes of 32 rows through LDS (the pipeline buffers are no longer read; the caller has
// synchronized): element (row, c) at row * BW_OW + c + 4 (c / 16).
template <int G>
__device__ __forceinline__ void bwd_store(const BwdGemmArgs& p, const f32x16 (&acc)[2][2], uint8_t* smem, int64_t m0, int64_t k0,
                                          int tid) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32 = lane & 31, h = lane >> 5, wm = wave >> 2, wk = wave & 3;
    float* ot = reinterpret_cast<float*>(smem);
    const bool vec = (p.ldo % 8 == 0) && ((uintptr_t)p.out % 16 == 0);
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {  // unrolled: acc[pass % 2] must stay in registers
        if (pass) __syncthreads();
        // C layout: lane l, register e holds row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32
        if (wm == pass / 2) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = 8 * (e / 4) + 4 * h + e % 4, c = 64 * wk + 32 * j + r32;
                    ot[row * BW_OW + c + 4 * (c >> 4)] = acc[pass % 2][j][e];
                }
        }
        __syncthreads();
        const int row = 4 * wave + (lane >> 4), run = lane & 15;
        const float* src = ot + row * BW_OW + 20 * run;
        float v[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(src + 4 * q);
            v[4 * q] = t.x; v[4 * q + 1] = t.y; v[4 * q + 2] = t.z; v[4 * q + 3] = t.w;
        }
        const int64_t m = m0 + 32 * pass + row, k = k0 + 16 * run;
        const int E = p.e[min(m, p.M - 1)];
        if constexpr (G > 0) {
            hadamard16<G>(v, lane);
            const float nrm = hadamard_norm<G>();
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] *= nrm;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = __builtin_ldexpf(v[i], E);
        if (m < p.M && k < p.K) {
            store8_rt(p.out, p.out_dt, m * p.ldo + k, v, 8, vec);
            store8_rt(p.out, p.out_dt, m * p.ldo + k + 8, v + 8, 8, vec);
        }
    }
}

// dx tile: rows m0 .. m0 + 127, columns k0 .. k0 + 255.  Wave w = 4 wm + wk owns rows 64 wm .. + 63 and
// columns 64 wk .. + 63 of the tile (2 x 2 sub-tiles of 32 x 32).  A stage is 64 values of n: a tile
// [128][64] fp16 and weight tile [64][256] int8, both brought in by LDS DMA as they lie in memory; the
// weight fragments (8 consecutive n of one column) are transposing LDS reads, widened to fp16 in registers.
//
// The two groups of four waves take turns on the matrix cores, as in gemm_pp.h: stage t is a memory phase
// (reads of the a fragments of stage t and the raw weights of stage t + 1, the requests of stage t + 3's
// a tile and stage t + 4's weight tile) and a compute phase (16 MFMAs, stage t + 1's weights widened
// between them), each ended by a barrier, and waves 4 .. 7 run one phase behind waves 0 .. 3, with which they share
// their SIMDs.  LDS holds four stages.  With the memory phase of stage t of waves 0 .. 3 as phase 2t:
//   the a tile of stage t is last read in phase 2t + 1 (waves 4 .. 7), the weight tile of stage t in phase
//   2t - 1; their buffers are refilled from phase 2t + 2 and 2t on: in stage t + 1 and stage t;
//   a wave's requests of stage t - 2 (a tile t + 1, weight tile t + 2) have landed before the barrier that
//   ends its memory phase t: 8 younger ones may be outstanding.  Their first reads are in phase 2t + 2.
// Against the same tile through registers with all waves in phase (bwd_gemm_pair_kernel below; matrix cores about a
// third busy), M1056 K6144 N16384: 311 -> 214 us, 992 TFLOP/s; 216 of 256 CUs have a tile there and 8% of the tile rows are padding.
template <int G>
__global__ __launch_bounds__(512) void bwd_gemm_kernel(BwdGemmArgs p) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[4 * BW_BUF];
    static_assert(32 * BW_OW * 4 <= 4 * BW_BUF, "output staging must fit");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32 = lane & 31, h = lane >> 5, wm = wave >> 2, wk = wave & 3;
    const int64_t m0 = (int64_t)blockIdx.y * BW_BM, k0 = (int64_t)blockIdx.x * BW_BK;
    const int nst = (int)(p.lda / BW_BN);  // lda is N rounded up to 128: even; a is zero past N
    // DMA instruction i of a tile fills its 16-byte chunks u = 512 i + tid: a tile row u / 8, logical chunk
    // (u % 8) ^ (row / 2) % 8; weight row u / 16, logical chunk bw_chunk(row, u % 16)
    const f16* asrc[2];
    const int8_t* bsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int u = 512 * i + tid, ar = u / 8, br = u / 16;
        asrc[i] = p.a + min(m0 + ar, p.M - 1) * p.lda + 8 * ((u % 8) ^ ((ar / 2) % 8));
        // columns past K re-read (never stored)
        bsrc[i] = p.b + min<int64_t>(br, p.N - 1) * p.ldb + min(k0 + 16 * bw_chunk(br, u % 16), p.K - 16);
    }
    auto dma_a = [&](int t, int buf) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            lds_dma16(asrc[i] + (int64_t)BW_BN * min(t, nst - 1), smem + buf * BW_BUF + 16 * (512 * i + 64 * wave));
    };
    // called for t = 0, 1, ..: a row's pointer moves on while the next row is one of the weight's, and stays
    // from then on (rows past N meet a = 0)
    auto dma_b = [&](int t, int buf) {
        const int64_t left = p.N - (int64_t)BW_BN * (t + 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            lds_dma16(bsrc[i], smem + buf * BW_BUF + BW_ASZ + 16 * (512 * i + 64 * wave));
            bsrc[i] += 32 * i + tid / 16 < left ? BW_BN * p.ldb : 0;
        }
    };
    // a fragments of stage t; raw weights of stage t + 1; widened weights of even and odd stages
    f16x8 af[2][4], bf[2][2][4];
    v2i raw[2][4];
    auto read_a = [&](int buf) {
        const uint8_t* src = smem + buf * BW_BUF + (64 * wm + r32) * 128;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                af[i][st] = *reinterpret_cast<const f16x8*>(src + 4096 * i + 16 * ((2 * st + h) ^ ((r32 / 2) % 8)));
    };
    // transposing fragment reads: in each 16-lane group, lane i names row nb + i / 2 at column
    // kc + 8 (i % 2) and receives column kc + i of rows nb .. nb + 7.  As one asm block that waits for
    // them: ahead of the builtin the compiler waits for every DMA in flight.
    const int gi = lane & 15, g = lane >> 4, brow = 8 * (g >> 1) + (gi >> 1);
    uint32_t bad[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        bad[j] = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem + BW_ASZ + brow * BW_BK +
                 16 * bw_chunk(brow, (64 * wk + 32 * j + 16 * (g & 1)) >> 4) + 8 * (gi & 1);
    auto read_b = [&](int buf) {
        asm volatile(
            "ds_read_b64_tr_b8 %0, %8\n"
            "ds_read_b64_tr_b8 %1, %9\n"
            "ds_read_b64_tr_b8 %2, %8 offset:4096\n"
            "ds_read_b64_tr_b8 %3, %9 offset:4096\n"
            "ds_read_b64_tr_b8 %4, %8 offset:8192\n"
            "ds_read_b64_tr_b8 %5, %9 offset:8192\n"
            "ds_read_b64_tr_b8 %6, %8 offset:12288\n"
            "ds_read_b64_tr_b8 %7, %9 offset:12288\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(raw[0][0]), "=&v"(raw[1][0]), "=&v"(raw[0][1]), "=&v"(raw[1][1]), "=&v"(raw[0][2]),
              "=&v"(raw[1][2]), "=&v"(raw[0][3]), "=&v"(raw[1][3])
            : "v"(bad[0] + buf * BW_BUF), "v"(bad[1] + buf * BW_BUF)
            : "memory");
    };
    auto widen = [&](int j, int st) { return i8x8_to_f16((uint32_t)raw[j][st].x, (uint32_t)raw[j][st].y); };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](int t, auto q) {
        constexpr int Q = decltype(q)::value;  // t % 4
        read_a(Q);
        __builtin_amdgcn_sched_barrier(0);
        read_b((Q + 1) % 4);
        __builtin_amdgcn_sched_barrier(0);
        dma_a(t + 3, (Q + 3) % 4);
        dma_b(t + 4, Q);
        wait_lgkmcnt0();
        wait_vmcnt<8>();
        barrier();
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bf[(Q + 1) % 2][j][st] = widen(j, st);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i][st], bf[Q % 2][j][st], acc[i][j], 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < 16; ++i) {  // an MFMA, then five of the 80 widening operations
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
        }
        barrier();
    };
    // the requests of stages -4 .. -1, in their order
    dma_b(0, 0);
    dma_a(0, 0);
    dma_b(1, 1);
    dma_a(1, 1);
    dma_b(2, 2);
    dma_a(2, 2);
    dma_b(3, 3);
    wait_vmcnt<8>();  // weight tiles 0 and 1, a tile 0
    barrier();
    read_b(0);
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int j = 0; j < 2; ++j) bf[0][j][st] = widen(j, st);
    barrier();
    if (wm) barrier();  // waves 4 .. 7: one phase behind
    constexpr std::integral_constant<int, 0> q0{};
    constexpr std::integral_constant<int, 1> q1{};
    constexpr std::integral_constant<int, 2> q2{};
    constexpr std::integral_constant<int, 3> q3{};
    int t = 0;
    for (; t + 3 < nst; t += 4) {
        stage(t, q0);
        stage(t + 1, q1);
        stage(t + 2, q2);
        stage(t + 3, q3);
    }
    if (t < nst) {
        stage(t, q0);
        stage(t + 1, q1);
    }
    if (!wm) barrier();
    wait_vmcnt<0>();
    __syncthreads();  // every wave is past the main loop, its DMAs included
    bwd_store<G>(p, acc, smem, m0, k0, tid);
}

struct BwdRegs {
    u32x4 a[2];  // 16 halves of one row of the a tile
    u32x4 b[2];  // 16 int8 of each of two weight rows
};

// The same tile and fragments with all waves in phase, for short sums, mostly on grids of more than one round (run_bwd_gemm):
// through registers into two LDS buffers of 34 KiB, and at most 128 registers (a few spilled), so that two workgroups
// share a CU and one's start and output overlap the other's sum.  A stage's loads are issued two stages before it is
// computed; loads past the last stage re-read it and are never computed.  A tile LDS row has 8 halves of padding.
template <int G>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 8))) void bwd_gemm_pair_kernel(BwdGemmArgs p) {
    constexpr int LS = BW_BN + 8, ASZ = BW_BM * LS * 2, BUF = ASZ + BW_BN * BW_BK;
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * BUF];
    static_assert(32 * BW_OW * 4 <= 2 * BUF, "output staging must fit");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r32 = lane & 31, h = lane >> 5, wm = wave >> 2, wk = wave & 3;
    const int64_t m0 = (int64_t)blockIdx.y * BW_BM, k0 = (int64_t)blockIdx.x * BW_BK;
    // global load assignment: a row tid / 4, 16 halves at 16 (tid % 4); weight rows tid / 16 and 32 + tid / 16 of the
    // stage, 16 bytes at column 16 (tid % 16) of the tile
    const f16* ap = p.a + min(m0 + tid / 4, p.M - 1) * p.lda + 16 * (tid & 3);
    const int brow = tid >> 4, bc = tid & 15;
    const int8_t* bp = p.b + min(k0 + 16 * bc, p.K - 16);  // columns past K re-read (never stored)
    const int last = (int)(p.lda / BW_BN) - 1;             // an odd number: lda is N rounded up to 128
    auto load = [&](int s, BwdRegs& r) {
        const u32x4* pa = reinterpret_cast<const u32x4*>(ap + (int64_t)BW_BN * s);
        r.a[0] = pa[0];
        r.a[1] = pa[1];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int64_t n = min((int64_t)BW_BN * s + 32 * i + brow, p.N - 1);  // rows past N meet a = 0
            r.b[i] = *reinterpret_cast<const u32x4*>(bp + n * p.ldb);
        }
    };
    auto store = [&](const BwdRegs& r, int buf) {
        f16* ad = reinterpret_cast<f16*>(smem + buf * BUF) + (tid >> 2) * LS + 16 * (tid & 3);
        uint8_t* bs = smem + buf * BUF + ASZ;
        *reinterpret_cast<u32x4*>(ad) = r.a[0];
        *reinterpret_cast<u32x4*>(ad + 8) = r.a[1];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = 32 * i + brow;
            *reinterpret_cast<u32x4*>(bs + row * BW_BK + 16 * bw_chunk(row, bc)) = r.b[i];
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const int gi = lane & 15, g = lane >> 4;  // the transposing reads of bwd_gemm_kernel
    auto compute = [&](int buf) {
        const f16* as = reinterpret_cast<const f16*>(smem + buf * BUF);
        const uint8_t* bs = smem + buf * BUF + ASZ;
#pragma unroll
        for (int st = 0; st < BW_BN / 16; ++st) {
            f16x8 af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                af[i] = *reinterpret_cast<const f16x8*>(as + (64 * wm + 32 * i + r32) * LS + 16 * st + 8 * h);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = 16 * st + 8 * (g >> 1) + (gi >> 1), kc = 64 * wk + 32 * j + 16 * (g & 1);
                const uint8_t* src = bs + row * BW_BK + 16 * bw_chunk(row, kc >> 4) + 8 * (gi & 1);
                const v2i w = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)src);
                bf[j] = i8x8_to_f16((uint32_t)w.x, (uint32_t)w.y);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    };
    // stage s lives in register set s % 2 and LDS buffer s % 2
    BwdRegs r0, r1;
    load(0, r0);
    load(1, r1);
    store(r0, 0);
    __syncthreads();
    for (int s = 0; s < last; s += 2) {
        load(min(s + 2, last), r0);
        compute(0);
        store(r1, 1);
        __syncthreads();
        load(min(s + 3, last), r1);
        compute(1);
        store(r0, 0);
        __syncthreads();
    }
    bwd_store<G>(p, acc, smem, m0, k0, tid);
}

}  // namespace

hipError_t run_bwd_rows(const void* dy, int dy_dt, int64_t ldd, int64_t M, int64_t N, const void* s, int s_dt,
                        int64_t s_stride, f16* a, int64_t lda, int32_t* e, hipStream_t st) {
    if (M == 0) return hipSuccess;
    if (lda < N || lda % (2 * BW_BN)) return hipErrorInvalidValue;
    bool ok = false;
    auto go = [&](auto dy_tag, auto s_tag) {
        using T = decltype(dy_tag);
        using TS = decltype(s_tag);
        hipLaunchKernelGGL((bwd_rows_kernel<T, TS>), dim3((unsigned)M), dim3(256), 0, st, (const T*)dy, ldd, N,
                           (const TS*)s, s_stride, a, lda, e);
        ok = true;
    };
    auto by_s = [&](auto dy_tag) {
        if (s_dt == DT_F32) go(dy_tag, float{});
        else if (s_dt == DT_F16) go(dy_tag, f16{});
        else if (s_dt == DT_BF16) go(dy_tag, bf16_t{});
    };
    if (dy_dt == DT_F32) by_s(float{});
    else if (dy_dt == DT_F16) by_s(f16{});
    else if (dy_dt == DT_BF16) by_s(bf16_t{});
    if (!ok) return hipErrorInvalidValue;
    return hipGetLastError();
}

// Short sums on more than one round of the 256 CUs: the kernel that two workgroups share a CU with.  In the other
// one's four stages of loads and its output overlap nothing, and the more rounds, the longer a sum has to be to win
// that back.  us for gradient rows and GEMM, bf16, G 256, two-group and pair kernel:
//   288 tiles (M2200 K4096): N512 44.2, 40.0; N1280 61.7, 61.2; N1536 67.2, 66.5; N1792 72.7, 73.1; N2048 78.3, 80.3
//   504 tiles (M2600 K6144): N512 47.6, 43.5; N1536 76.6, 73.4; N2048 90.5, 89.2; N2304 98.7, 98.7; N2560 105.5, 106.2
//   2016 tiles (M4600 K14336): N512 154, 123; N1024 205, 179; N2048 316, 304; N2304 344, 336; N2560 372, 368
//   4800 tiles (M9504 K16384): N2304 792, 781; N2560 854, 869
// and sums of two stages on any grid (M64 K4096 N128 16.4, 16.1; N256 17.7, 17.8; N512 19.8, 21.2).
bool bwd_gemm_pair(int64_t tiles, int64_t stages) {
    return stages <= (tiles > 512 ? 36 : tiles > 416 ? 32 : tiles > 256 ? 26 : 2);
}

hipError_t run_bwd_gemm(const BwdGemmArgs& p, hipStream_t st) {
    if (p.M == 0 || p.K == 0) return hipSuccess;
    // the kernels' loads assume: K a multiple of 16 (16-byte weight loads from clamped columns),
    // 16-byte aligned weight rows, lda a multiple of 128 covering N, N >= 1
    if (p.K % 16 || p.ldb % 16 || (uintptr_t)p.b % 16 || p.lda % (2 * BW_BN) || p.lda < p.N || p.N < 1 ||
        (uintptr_t)p.a % 16)
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)((p.K + BW_BK - 1) / BW_BK), (unsigned)((p.M + BW_BM - 1) / BW_BM));
    const bool pair = bwd_gemm_pair((int64_t)grid.x * grid.y, p.lda / BW_BN);
    bool ok = false;
    auto go = [&]<int G>() {
        if (pair) hipLaunchKernelGGL((bwd_gemm_pair_kernel<G>), grid, dim3(512), 0, st, p);
        else hipLaunchKernelGGL((bwd_gemm_kernel<G>), grid, dim3(512), 0, st, p);
        ok = true;
    };
    if (!dispatch_group(p.G, go) || !ok) return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace qlin
