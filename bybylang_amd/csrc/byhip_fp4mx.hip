// byhip_fp4mx.hip - fp32 activations on FP4-KM weights with an E2M1 / E8M0 decode table (gfx950).
//
// y[M, N] = x[M, K] . W^T, W = lut[code] * lut[16 + scale byte] with E2M1's values and the scales 2^(b - 127).
// Such weights are exact in bf16 over the table's whole range (v_cvt_scalef32_pk_bf16_fp4, subnormals
// included), and an fp32 activation is the sum of three bf16 terms, so three v_mfma_f32_16x16x32_bf16 with
// fp32 accumulation hold every bit of both. Two fp16 terms, two MFMAs, hold as much only while
// a row's activations lie within fp16's range of each other.
//   What three terms cannot form as the reference does is computed again in fp32 arithmetic, tile by tile: scale
//   bytes from 253 on (products that may not be finite) and activations that are not finite or so large
//   that their second term overflows.
//
// Block: 16 FM rows x 128 columns, eight waves, two per SIMD. Waves w, w + 2, .. (p = w % 2) form K group p, which
// takes every other 128-value step of the block. The group's four waves split the columns, 32 each, over all
// rows; at 64 rows into two halves of rows and of columns (32 x 64), so that each activation is split
// into its terms by two waves rather than four: the splitting bounds the kernel.
//
// Activations stay fp32 on the way: a step's 512 bytes per row, whole lines, move into LDS by direct loads (chunk
// k of row r at slot k ^ (r % 16): the 16 rows of a fragment read hit distinct banks), two buffers per group,
// and each wave splits its fragments in registers. Lane (c, g) = (lane % 16, lane / 16) takes the step's 32-value
// group g: 16 bytes of weights per column, dword q of them multiplied in quarter q of the step. Its bytes'
// low nibbles are elements 4 q .. 4 q + 3 of the group, the high ones 16 + 4 q ..: chunks 8 g + q and
// 8 g + 4 + q of the row. One barrier per step, before its last quarter, frees the step's buffer and
// publishes the next one's; weights run two steps ahead.
//
// What bounds it: at few rows a launch's fixed costs and the splits' sum, with more the splitting and the matrix
// pipe, which overlap in part: at M = 512, K = N = 4096 MFMAs fill 36 % of the SIMDs' cycles and other VALU
// work 37 %, and waves wait for data or the barrier for 35 % of theirs. us, against the exact fp32 GEMM, which took
// such tables before, and two fp16 planes with scales checked in the kernel: M = 16, K = N = 4096 10.1 (16.4,
// 12.8); M = 47 17.9 (34.8, 18.1); M = 128, K = 4096, N = 6144 37.0 (149, 28.6); M = 512, K = N = 4096 59.3
// (243, 42.6; 414 with one zero-filled group per tile, whose scale byte 0 sent the tile to fp32 arithmetic).
// Error against 64 bits there 1.1e-7 (planes 3.6e-7). Order of MFMAs and VALU left to the compiler: fixed
// by scheduling groups 66.4.
#include <algorithm>

#include "byhip_gemm.h"
#include "byhip_internal.h"
#include "byhip_kernels.h"

namespace byhip {
namespace {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kBN = 128;
constexpr int kStep = 128;                 // K values per step
constexpr int kPitch = kBN + 4;            // floats per row of a staged partial tile
constexpr uint32_t kPast = 0x80000000u;    // added to an offset: every resource here rejects it
constexpr uint32_t kByteMax = 252u;        // the largest scale byte whose products are all finite

template <int FM>
struct MxTile {
    static constexpr int kBM = 16 * FM;
    static constexpr int kXBuf = kBM * kStep * 4;        // one step's activations
    static constexpr int kLdsX = 2 * 2 * kXBuf;          // two K groups x two buffers
    static constexpr int kLdsRed = 2 * kBM * kPitch * 4; // two partial tiles
    static constexpr int kLds = kLdsX > kLdsRed ? kLdsX : kLdsRed;
};

// The block's tile in fp32 arithmetic, each weight lut[code] * lut[16 + scale byte] as the
// reference forms it, x in fp32, v_mfma_f32_16x16x4_f32: wave w computes columns 16 w .. + 15 over
// 32-value groups g0 .. g1 - 1 and leaves its sums in `red`.
template <int FM>
__device__ __forceinline__ void fp4_tile_exact(const GemmArgs& a, int m0, int n0, int g0, int g1,
                                               float* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int n = n0 + 16 * wid + c;
    const float* const x = static_cast<const float*>(a.x);
    const float* const lut = a.lut;
    f4 acc[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[i] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    for (int G = g0; G < g1; ++G) {
        uint32_t w = 0;
        float s = 0.0f;
        if (n < a.N) {
            w = *reinterpret_cast<const uint32_t*>(a.blob + (size_t)n * (a.K >> 1) + 16 * (size_t)G + 4 * g);
            s = lut[16 + a.blob[a.scale_base + (size_t)n * (a.K >> 5) + G]];
        }
        float wl[4], wh[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            wl[j] = n < a.N ? lut[(w >> (8 * j)) & 15u] * s : 0.0f;
            wh[j] = n < a.N ? lut[(w >> (8 * j + 4)) & 15u] * s : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int m = m0 + 16 * i + c;
            float4 xl = make_float4(0.0f, 0.0f, 0.0f, 0.0f), xh = xl;
            if (m < a.M) {
                const float* r = x + (size_t)m * a.K + 32 * (size_t)G + 4 * g;
                xl = *reinterpret_cast<const float4*>(r);
                xh = *reinterpret_cast<const float4*>(r + 16);
            }
            const float al[4] = {xl.x, xl.y, xl.z, xl.w}, ah[4] = {xh.x, xh.y, xh.z, xh.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(al[j], wl[j], acc[i], 0, 0, 0);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[j], wh[j], acc[i], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = (16 * i + 4 * g + r) * kPitch + 16 * wid + c;
            red[at] = acc[i][r];
            red[16 * FM * kPitch + at] = 0.0f;  // the second K group's partial tile
        }
}

// Eight fp32 values, xl[i] and xh[i] in turn, as three bf16 terms each, cut off rather than rounded: 8 + 8 + 8
// bits, all of a value's 24. v_dot2_f32_bf16 with -1 on one side of a pair leaves that side's remainder, exactly,
// also among subnormals (minus[l]: -1 for side l; in registers the compiler cannot see through, since it
// would make the low one an inline constant, which the instruction takes as an fp32 pattern). The second
// and third terms come 2^16 times as large, which keeps the last bits of values near and below 2^-126 within
// bf16's subnormals. An infinity or a NaN makes them NaN, a value past 2^119 may make them infinite.
__device__ __forceinline__ void bf16_terms(const f4& xl, const f4& xh, const uint32_t (&minus)[2], bf8 (&t)[3]) {
    auto rest = [&](uint32_t pair, int l, float v) __attribute__((always_inline)) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), __builtin_bit_cast(bf16x2_t, minus[l]), v, false);
    };
    auto high = [](float l, float h) __attribute__((always_inline)) {  // the high halves of a pair
        return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l), 0x07060302u);
    };
    uint32_t u[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        u[0][e] = high(xl[e], xh[e]);
        const float l1 = rest(u[0][e], 0, xl[e]) * 65536.0f, h1 = rest(u[0][e], 1, xh[e]) * 65536.0f;
        u[1][e] = high(l1, h1);
        u[2][e] = high(rest(u[1][e], 0, l1), rest(u[1][e], 1, h1));
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) t[i] = __builtin_bit_cast(bf8, u[i]);
}

template <int FM, int YT>
__global__ __launch_bounds__(512, FM == 1 ? 4 : 2) void gemm_fp4_mx(GemmArgs a) {
    if (a.gate && *a.gate != a.gate_want) return;  // another route was chosen (whole grid)
    using S = MxTile<FM>;
    constexpr int RH = FM == 4 ? 2 : 1;            // halves of rows
    constexpr int FR = FM / RH, FN = 2 * RH;       // a wave's fragments of rows and columns
    constexpr int BM = S::kBM, kXBuf = S::kXBuf, kXLoads = 2 * FM;
    // One LDS array for everything, the eight waves' `bad` words at its end: beside a second one the
    // compiler does not tell the direct loads from the fragment reads apart and waits for every load.
    __shared__ __attribute__((aligned(16))) uint8_t lds[S::kLds + 32];

    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = wid & 1, h = wid >> 1, ch = RH == 2 ? h & 1 : h, rh = RH == 2 ? h >> 1 : 0;
    const int c = lane & 15, g = lane >> 4;
    int bx = blockIdx.x, by = blockIdx.y;
    {
        // the wide tile's XCD-grouped tile order
        const int gx = gridDim.x, gy = gridDim.y, tiles = gx * gy, id = bx + gx * by;
        const int j = tiles % 8 == 0 ? (id % 8) * (tiles / 8) + id / 8 : id;
        const int grp = j / (4 * gx), rows = min(4, gy - 4 * grp), r = j % (4 * gx);
        by = 4 * grp + r % rows;
        bx = r / rows;
    }
    const int n0 = bx * kBN, m0 = by * BM, K = a.K;
    // the block's steps; a K group's step q is step p + 2 q of them, zeros past the last
    const int step0 = a.part ? (int)blockIdx.z * a.split_steps : 0;
    const int steps = a.part ? min(a.split_steps, K / kStep - step0) : K / kStep;
    const int nq = (steps + 1) / 2;

    // Rows past M and columns past N read zeros through the range checks.
    const rsrc_t xr = make_rsrc(a.x, (uint32_t)((size_t)a.M * K * 4));
    const rsrc_t wr = make_rsrc(a.blob, (uint32_t)((size_t)a.N * (K >> 1)));
    const rsrc_t sr = make_rsrc(a.blob + a.scale_base, (uint32_t)((size_t)a.N * (K >> 5)));
    // Direct load i (0 .. 2 FM - 1) of wave h: rows 2 h + 8 i and the next one; the swizzle of lane l's
    // slot l % 32 depends on i only through its parity.
    const int r0 = 2 * h + (lane >> 5);
    const uint32_t xo[2] = {(uint32_t)(m0 + r0) * (uint32_t)K * 4u + 16u * (uint32_t)((lane & 31) ^ r0),
                            (uint32_t)(m0 + r0) * (uint32_t)K * 4u + 16u * (uint32_t)((lane & 31) ^ (r0 + 8))};
    const int n = n0 + 16 * FN * ch + c;
    const uint32_t wo = (uint32_t)n * (uint32_t)(K >> 1) + 16u * (uint32_t)g;
    const uint32_t so = (uint32_t)n * (uint32_t)(K >> 5) + 8u * (uint32_t)g;
    uint8_t* const xgrp = lds + p * 2 * kXBuf;
    const int rd = 512 * (16 * FR * rh + c) + 16 * ((8 * g) ^ c);

    auto load_x = [&](int q, int buf) __attribute__((always_inline)) {
        const int s = p + 2 * q;
        const uint32_t off = s < steps ? 512u * (uint32_t)(step0 + s) : kPast;
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) lds_dma16(xr, xgrp + buf * kXBuf + 1024 * (h + 4 * i), xo[i & 1] + (uint32_t)(32 * i) * (uint32_t)K, off);
    };
    v4u wv[2][FN];
    auto load_w = [&](v4u (&w)[FN], int q) __attribute__((always_inline)) {
        const int s = p + 2 * q;
        const uint32_t off = s < steps ? 64u * (uint32_t)(step0 + s) : kPast;
#pragma unroll
        for (int j = 0; j < FN; ++j) w[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, wo + (uint32_t)(8 * j) * (uint32_t)K, off, 0);
    };
    // Scale bytes: the dword of lane (c, i) holds the four bytes (groups 0 .. 3) of column c in the group's step
    // 4 v + i, so one load per column and four steps; lane (c, g) fetches byte g of the step's dword
    // from lane (c, q % 4). The scale 2^(b - 127) is b << 23, byte 0 as the conversion takes it.
    uint32_t sb[FN], sbn[FN], ss[FN];
    bool bad = false;
    auto load_sb = [&](uint32_t (&d)[FN], int v) __attribute__((always_inline)) {
        const int s0 = p + 8 * v;  // step of lane group 0; the lane's own is s0 + 2 g
        const uint32_t past = s0 + 2 * g >= steps ? kPast : 0u;
#pragma unroll
        for (int j = 0; j < FN; ++j)
            d[j] = __builtin_amdgcn_raw_buffer_load_b32(sr, (so + (uint32_t)(j * (K >> 1))) | past, 4u * (uint32_t)(step0 + s0), 0);
    };
    auto scale_of = [&](const uint32_t (&d)[FN], int q, uint32_t (&s)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const uint32_t b = ((uint32_t)__builtin_amdgcn_ds_bpermute(4 * (16 * (q & 3) + c), (int)d[j]) >> (8 * g)) & 255u;
            bad = bad || b > kByteMax;
            s[j] = b << 23;
        }
    };
    auto decode = [&](const v4u (&w)[FN], int q, bf8 (&b)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const uint32_t d = w[j][q];
            const float s = __builtin_bit_cast(float, ss[j]);
            const bf16x2_t v[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 0), __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 1),
                                   __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 2), __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, s, 3)};
            b[j] = __builtin_bit_cast(bf8, v);
        }
    };
    auto read_x = [&](int buf, int q, f4 (&x)[FR][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int l = 0; l < 2; ++l) x[i][l] = *reinterpret_cast<const f4*>(xgrp + buf * kXBuf + (rd ^ (16 * q + 64 * l)) + 8192 * i);
    };

    uint32_t minus[2];
    asm volatile("s_mov_b32 %0, 0x0000bf80" : "=s"(minus[0]));
    asm volatile("s_mov_b32 %0, 0xbf800000" : "=s"(minus[1]));
    // The second and third terms have sums of their own, 2^16 times as large.
    f4 acc[FR][FN], low[FR][FN];
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = low[i][j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto mfmas = [&](const f4 (&x)[FR][2], const bf8 (&b)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FR; ++i) {
            bf8 t[3];
            bf16_terms(x[i][0], x[i][1], minus, t);
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t[0], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < FN; ++j) low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t[1], b[j], low[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < FN; ++j) low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t[2], b[j], low[i][j], 0, 0, 0);
        }
    };
    f4 xa[FR][2], xb[FR][2];
    bf8 wa[FN], wb[FN];
    load_sb(sb, 0);
    load_w(wv[0], 0);
    load_x(0, 0);
    __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
    load_x(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    load_w(wv[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<kXLoads + FN>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    scale_of(sb, 0, ss);
    read_x(0, 0, xa);
    decode(wv[0], 0, wa);

    // Step q = base + k. The wait before the last quarter leaves only the weights issued behind step q + 1's
    // activations in flight.
    auto step = [&](int q, auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        __builtin_amdgcn_sched_barrier(0);
        mfmas(xa, wa);
        read_x(k, 1, xb);
        decode(wv[k], 1, wb);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(xb, wb);
        read_x(k, 2, xa);
        decode(wv[k], 2, wa);
        __builtin_amdgcn_sched_barrier(0);
        if ((q & 3) == 3) {
#pragma unroll
            for (int j = 0; j < FN; ++j) sb[j] = sbn[j];
        }
        mfmas(xa, wa);
        read_x(k, 3, xb);
        decode(wv[k], 3, wb);
        scale_of(sb, q + 1, ss);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<FN>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if ((q & 3) == 0) load_sb(sbn, (q >> 2) + 1);
        load_x(q + 2, k);
        __builtin_amdgcn_sched_barrier(0);
        load_w(wv[k], q + 2);
        mfmas(xb, wb);
        read_x(k ^ 1, 0, xa);
        decode(wv[k ^ 1], 0, wa);
        __builtin_amdgcn_sched_barrier(0);
    };
    // left in the middle of a round rather than guarded there: the compiler would wait for the newest weights
    // at the head of the loop, as if they could be the ones needed
    for (int q = 0;;) {
        step(q, std::integral_constant<int, 0>{});
        if (++q >= nq) break;
        step(q, std::integral_constant<int, 1>{});
        if (++q >= nq) break;
    }

    // Partial tiles -> LDS, once every wave's loads have landed and every wave is done with the
    // buffers -> the two groups' sums -> y or the split-K partials.
    wait_vmcnt<0>();
    uint32_t* const bads = reinterpret_cast<uint32_t*>(lds + S::kLds);
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) bad = bad || !__builtin_isfinite(low[i][j][r]);
    const bool any = __any(bad);
    if (lane == 0) bads[wid] = any ? 1u : 0u;
    __syncthreads();
    const uint4 b0 = reinterpret_cast<const uint4*>(bads)[0], b1 = reinterpret_cast<const uint4*>(bads)[1];
    const bool redo = (b0.x | b0.y | b0.z | b0.w | b1.x | b1.y | b1.z | b1.w) != 0u;
    float* red = reinterpret_cast<float*>(lds);  // [2 groups][BM rows][kPitch]
    if (redo) {
        fp4_tile_exact<FM>(a, m0, n0, 4 * step0, 4 * (step0 + steps), red);
    } else {
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[(p * BM + 16 * (FR * rh + i) + 4 * g + r) * kPitch + 16 * FN * ch + 16 * j + c] = fmaf(low[i][j][r], 0x1p-16f, acc[i][j][r]);
    }
    __syncthreads();
    float* part = a.part ? a.part + (size_t)blockIdx.z * splitk_stride(a.M, a.N) : nullptr;
    const bool vec = out8_vector_ok<YT>(a, part);
    for (int u = tid; u < BM * 16; u += 512) {  // chunk of 8 outputs: row u / 16, columns 8 (u % 16)
        const int row = u >> 4, col = (u & 15) * 8, m = m0 + row;
        if (m >= a.M) continue;
        const float* src = red + row * kPitch + col;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const float4 s0 = *reinterpret_cast<const float4*>(src + e);
            const float4 s1 = *reinterpret_cast<const float4*>(src + BM * kPitch + e);
            v[e] = s0.x + s1.x; v[e + 1] = s0.y + s1.y; v[e + 2] = s0.z + s1.z; v[e + 3] = s0.w + s1.w;
        }
        store_out8<YT>(a, part, vec, m, n0 + col, v);
    }
}

template <int FM>
void launch_mx_fm(const GemmArgs& a, int splits) {
    const dim3 grid((a.N + kBN - 1) / kBN, (a.M + 16 * FM - 1) / (16 * FM), splits);
    switch (a.y_dtype) {
    case BYHIP_F32: launch("gemm_fp4_mx", (gemm_fp4_mx<FM, BYHIP_F32>), grid, dim3(512), 0, a); break;
    case BYHIP_F16: launch("gemm_fp4_mx", (gemm_fp4_mx<FM, BYHIP_F16>), grid, dim3(512), 0, a); break;
    default: launch("gemm_fp4_mx", (gemm_fp4_mx<FM, BYHIP_BF16>), grid, dim3(512), 0, a); break;
    }
    BYHIP_LAUNCHED("gemm_fp4_mx");
}

// K splits: the count that minimises rounds of blocks x (steps per split + 4) (4 for a block's first loads
// and epilogue), plus 4 steps for the sum's launch and a quarter per split for what it reads; at least two steps
// per split. (us, forced splits: M = 48, K = 1024, N = 4096 1 / 2 / 4 / 8 17.7 / 14.4 / 12.5 / 14.5;
// M = 16, K = N = 4096 4 / 6 / 8 11.9 / 11.0 / 10.0; M = 24, K = 4096, N = 14336 1 / 2 / 4 39.5 / 26.0 / 29.5;
// M = 300, K = 14336, N = 2048 2 / 3 / 4 104 / 76 / 112.)
int mx_splits(long tiles, int steps) {
    const long cus = compute_units();
    int best = 1;
    double best_t = 1e300;
    for (int s = 1; s <= std::max(1, steps / 2); ++s) {
        const int per = (steps + s - 1) / s;
        if ((steps + per - 1) / per != s) continue;  // the same split as a smaller s
        const double t = (double)((tiles * s + cus - 1) / cus) * (per + 4) + (s > 1 ? 4.0 + 0.25 * s : 0.0);
        if (t < 0.97 * best_t) best = s, best_t = t;
    }
    return best;
}

}  // namespace

bool fp4_mx_ok(const GemmArgs& a) {
    return a.x_dtype == BYHIP_F32 && reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && a.K % kStep == 0 && (uint64_t)a.K * 4 * 128 < kPast &&
           reinterpret_cast<uintptr_t>(a.blob) % 16 == 0 && a.scale_base % 4 == 0 && (uint64_t)(a.N + kBN) * (a.K / 2) < kPast;
}

void launch_fp4_mx(const GemmArgs& a0) {
    // Row blocks whose offsets stay below 2^31, with the rows a tile reaches past them.
    const size_t rows = std::min<size_t>((kPast / ((size_t)a0.K * 4) - 64) / 64 * 64, 65535 * 16);
    for (size_t m = 0; m < (size_t)a0.M; m += rows) {
        GemmArgs a = a0;
        a.M = (int)std::min<size_t>(rows, (size_t)a0.M - m);
        a.x = static_cast<const float*>(a0.x) + m * a0.K;
        a.y = static_cast<uint8_t*>(a0.y) + m * a0.N * dtype_bytes(a0.y_dtype);
        // the fewest tiles of up to 64 rows, cut to the rows there are
        const int row_tiles = (a.M + 63) / 64, fm = (a.M + 16 * row_tiles - 1) / (16 * row_tiles);
        const long tiles = (long)((a.N + kBN - 1) / kBN) * ((a.M + 16 * fm - 1) / (16 * fm));
        const int forced = env_int("BYHIP_Q4_SPLIT", 0);
        const int splits = choose_split(a, tiles, a.K / kStep, 1, forced > 0 ? forced : mx_splits(tiles, a.K / kStep), 1);
        if (splits == 1) a.part = nullptr;
        switch (fm) {
        case 1: launch_mx_fm<1>(a, splits); break;
        case 2: launch_mx_fm<2>(a, splits); break;
        case 3: launch_mx_fm<3>(a, splits); break;
        default: launch_mx_fm<4>(a, splits); break;
        }
        if (a.part) launch_splitk_sum(a, splits);
    }
}

}  // namespace byhip
