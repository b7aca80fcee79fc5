// byhip_planes.hip - fp32 activations as two fp16 planes against quantized or half weights (gfx950).
//
// y[M, N] = x[M, K] . W^T. Each row of x is brought onto fp16's range by an exact power of two
// (undone on the output) and split into hi = fp16(x) and lo = fp16(x - hi), about 23 bits of x
// (split_planes); hi . w + lo . w in v_mfma_f32_16x16x32_f16 with fp32 accumulation then keeps
// them, for weights that are exact in fp16:
//   FP4-KM with E2M1 values and scales whose products with them are all halves
//   F16    (gemm_planes_half, below, where both operands go through LDS)
//   Q4     on the prefill copy: the codes less their zero (whole numbers) go through the MFMAs, and each
//          32-value group's sums are scaled in fp32. Two MFMAs per product where weights as two fp16
//          terms (the wide tile on fp32 activations) take three.
//
// gemm_planes. Block: 16 FM rows x 128 columns, eight waves, two per SIMD. Waves w, w + 2, .. (p = w % 2) form K
// group p, which takes every other 128-value step of the block; wave h = w / 2 of the group owns
// columns 32 h .. 32 h + 31 (2 fragments) and all rows: each decoded weight fragment feeds 2 FM
// MFMAs (hi and lo), and each activation fragment read from LDS 2. Two K groups rather than four
// (the wide tile) halve the LDS the activations need, so two planes of 64 rows fit four buffers.
//
// A 128-value step is two sub-steps of 64 values (one 128-byte line of each plane row); the group's
// slice of both planes moves straight into LDS by direct loads, 16-byte chunk k of row r at slot
// k ^ x_swizzle(r), four buffers, loads three sub-steps ahead. Lane (c, g) = (lane % 16, lane / 16)
// multiplies chunks 2 g and 2 g + 1 of the slice with its weights of column c:
//   Q4      chunks g and 4 + g instead: MFMA kk then covers one 32-value group, positions 32 kk + 8 g ..
//           + 7 per lane, one dword of the prefill copy (a fragment's 64 dwords are 256 contiguous
//           bytes). Its sums wait in registers of their own and are scaled and added during the next K
//           half's MFMAs, which start from zero.
//   FP4-KM  the four lane groups hold the step's four 32-value groups, one 16-byte load per column
//           and step: bytes 4 q .. 4 q + 3 of the group are elements 4 q .. 4 q + 3 (low nibbles)
//           and 16 + 4 q .. (high); sub-step e multiplies q = 2 e and 2 e + 1. split_planes writes the
//           planes in that order, chunk 8 (q / 2) + 2 g + q % 2 of a 128-value block holding elements
//           4 q, 16 + 4 q, 4 q + 1, .. of group g. One lane then needs one scale per step.
// Sub-steps run in two halves around one block barrier, as in the wide tile (byhip_gemm.hip).
#include <algorithm>

#include "byhip_gemm.h"
#include "byhip_internal.h"
#include "byhip_kernels.h"

namespace byhip {
namespace {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kBN = 128;
constexpr int kSub = 64;              // K values per sub-step
constexpr int kDepth = 4;             // activation buffers per K group
constexpr int kSets = 4;              // weight register sets
constexpr int kUnroll = 8;            // sub-steps per loop iteration
constexpr int kPitch = kBN + 4;       // floats per row of a staged partial tile
constexpr uint32_t kPast = 0x80000000u;    // added to an offset: every resource here rejects it

template <int FM>
struct PlaneShape {
    static constexpr int kBM = 16 * FM;
    static constexpr int kXBuf = 2 * kBM * kSub * 2;     // one buffer: both planes' slices
    static constexpr int kLdsX = 2 * kDepth * kXBuf;     // two K groups
    static constexpr int kLdsRed = 2 * kBM * kPitch * 4; // two partial tiles
    static constexpr int kLds = kLdsX > kLdsRed ? kLdsX : kLdsRed;
};

template <BFormat F, int FM, int YT, bool ZG = false>
__global__ __launch_bounds__(512, FM == 1 || (FM == 2 && F == BFormat::Fp4Km) ? 4 : 2) void gemm_planes(GemmArgs a) {
    if (a.gate && *a.gate != a.gate_want) return;  // another route was chosen (whole grid)
    constexpr bool FP4 = F == BFormat::Fp4Km, Q4 = F == BFormat::Q4Fast;
    constexpr int FN = 2;
    constexpr int WV = 2;  // weight registers of a set, in 16-byte units
    using S = PlaneShape<FM>;
    constexpr int BM = S::kBM, kXBuf = S::kXBuf;
    // One LDS array for everything: beside a second one (a table, or the one inside __syncthreads_or) the
    // compiler no longer told the direct loads from the fragment reads apart and waited for every load
    // in flight before each read: 47 us instead of 43 at M = 512, K = N = 4096.
    __shared__ __attribute__((aligned(16))) uint8_t lds[S::kLds];

    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = wid & 1, h = wid >> 1;
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
    const int n0 = bx * kBN, m0 = by * BM;
    const int K = a.K;
    // the block's 128-value steps (the last one half empty when K / 64 is odd) and 64-value slices
    const int step0 = a.part ? (int)blockIdx.z * a.split_steps : 0;
    const int steps_all = (K + 127) / 128;
    const int steps = a.part ? min(a.split_steps, steps_all - step0) : steps_all;
    const int slices = min(2 * steps, K / kSub - 2 * step0);
    const int pairs_all = (steps + 1) / 2, nt_all = 2 * pairs_all;  // per K group: its steps, sub-steps

    // The scales live in registers as halves, entries 4 l .. 4 l + 3 in lane l, looked up across lanes.
    float lut_v[FP4 ? 4 : 1];
    uint32_t lut_h[FP4 ? 2 : 1];
    if constexpr (FP4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) lut_v[i] = a.lut[16 + 4 * lane + i];
    }

    const rsrc_t xr = make_rsrc(h < 2 ? a.x : a.x_lo, (uint32_t)((size_t)a.M * K * 2));
    const uint32_t nsub = (uint32_t)K / kSub;
    const uint32_t wpf_bytes = ((uint32_t)a.N + 15) / 16 * nsub * 512, spf_bytes = ((uint32_t)a.N + 63) / 64 * nsub * 256;
    const rsrc_t wr = FP4 ? make_rsrc(a.blob, (uint32_t)((size_t)a.N * (K >> 1))) : make_rsrc(a.wpf, wpf_bytes);
    const rsrc_t sr = FP4 ? make_rsrc(a.blob + a.scale_base, (uint32_t)((size_t)a.N * (K >> 5))) : make_rsrc(a.spf, spf_bytes);
    const rsrc_t zr = ZG ? make_rsrc(a.zpf, spf_bytes) : sr;
    // Direct load q (0 .. FM - 1) of wave h: stacked rows 8 FM h + 8 q + lane / 8 of the slice (the
    // high plane's BM rows, then the low plane's), LDS slot lane % 8.
    uint32_t xo[FM];
#pragma unroll
    for (int q = 0; q < FM; ++q) {
        const int r = 8 * FM * (h & 1) + 8 * q + (lane >> 3), chunk = (lane & 7) ^ x_swizzle(r);
        xo[q] = (uint32_t)(m0 + r) * (uint32_t)K * 2u + 16u * chunk;
    }
    uint32_t wo[FN], so[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n0 + 32 * h + 16 * j + c;
        wo[j] = FP4 ? (uint32_t)n * (uint32_t)(K >> 1) + 16u * g
                    : ((uint32_t)n >> 4) * nsub * 512u + 8u * c + 128u * (uint32_t)(g >> 1) + 4u * (uint32_t)(g & 1);
        so[j] = (uint32_t)n * (uint32_t)(K >> 5) + 8u * g;
    }
    // Q4 scales (and zeros): the wave's 2 fragments are fragments 2 (h % 2) and the next of their quad
    const uint32_t sq = (uint32_t)(n0 + 32 * h) / 64u * nsub * 256u + 8u * c + 4u * (uint32_t)(h & 1);
    uint8_t* const xgrp = lds + p * kDepth * kXBuf;
    const int rd0 = 128 * c + 16 * ((Q4 ? g : 2 * g) ^ x_swizzle(c));
    const int rd1 = 128 * c + 16 * ((Q4 ? 4 + g : 2 * g + 1) ^ x_swizzle(c));

    // The group's sub-step t is slice 2 p + 4 (t / 2) + t % 2 of the block; past the last it reads zeros.
    auto load_x = [&](int t, int buf) __attribute__((always_inline)) {
        const int sl = 2 * p + 4 * (t >> 1) + (t & 1);
        const uint32_t off = sl < slices ? 128u * (uint32_t)(2 * step0 + sl) : kPast;
#pragma unroll
        for (int q = 0; q < FM; ++q) lds_dma16(xr, xgrp + buf * kXBuf + 1024 * (FM * h + q), xo[q], off);
    };
    // FP4-KM: the 16 bytes per column of the group's step q (sub-steps 2 q and 2 q + 1); Q4: per MFMA
    // kk a dword per fragment, w[kk][j], the fragments' scales w[kk][2] and zeros w[kk][3].
    v4u wv[kSets][WV];
    auto load_w = [&](v4u (&w)[WV], int t) __attribute__((always_inline)) {
        if constexpr (Q4) {
            const int sl = 2 * p + 4 * (t >> 1) + (t & 1);
            const uint32_t u = (uint32_t)(2 * step0 + (sl < slices ? sl : 0)), past = sl < slices ? 0u : kPast;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int j = 0; j < FN; ++j) w[kk][j] = __builtin_amdgcn_raw_buffer_load_b32(wr, wo[j], past + 512u * u + 256u * kk, 0);
                w[kk][2] = __builtin_amdgcn_raw_buffer_load_b32(sr, sq, past + 256u * u + 128u * kk, 0);
                if constexpr (ZG) w[kk][3] = __builtin_amdgcn_raw_buffer_load_b32(zr, sq, past + 256u * u + 128u * kk, 0);
            }
        } else {
            const int s = p + 2 * t;
            const uint32_t off = s < steps ? 64u * (uint32_t)(step0 + s) : kPast;
#pragma unroll
            for (int j = 0; j < FN; ++j) w[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, wo[j], off, 0);
        }
    };
    // FP4-KM scale bytes: the dword of lane (c, i) holds the four bytes (groups 0 .. 3) of column c in
    // the group's step 4 v + i, so one load per column and four steps; lane (c, g) fetches byte g
    // of the step's dword from lane (c, q % 4).
    uint32_t sb[FP4 ? FN : 1], sbn[FP4 ? FN : 1], ss[FP4 ? FN : 1];
    auto load_sb = [&](uint32_t (&d)[FP4 ? FN : 1], int v) __attribute__((always_inline)) {
        const int s0 = p + 8 * v;  // step of lane group 0; the lane's own is s0 + 2 g
        const uint32_t past = s0 + 2 * g >= steps ? kPast : 0u;
#pragma unroll
        for (int j = 0; j < (FP4 ? FN : 0); ++j)
            d[j] = __builtin_amdgcn_raw_buffer_load_b32(sr, so[j] | past, 4u * (uint32_t)(step0 + s0), 0);
    };
    auto scale_of = [&](const uint32_t (&d)[FP4 ? FN : 1], int q, uint32_t (&s)[FP4 ? FN : 1]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < (FP4 ? FN : 0); ++j) {
            const uint32_t b = ((uint32_t)__builtin_amdgcn_ds_bpermute(4 * (16 * (q & 3) + c), (int)d[j]) >> (8 * g)) & 255u;
            const uint32_t v0 = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(b & 252u), (int)lut_h[0]);
            const uint32_t v1 = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(b & 252u), (int)lut_h[FP4 ? 1 : 0]);
            const uint32_t v = (((b & 2u) ? v1 : v0) >> (16 * (b & 1u))) & 0xFFFFu;
            s[j] = v | (v << 16);  // columns past N and steps past the last: weights of zero
        }
    };

    f4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};

    const _Float16 zlo = (_Float16)(1024.0f + a.zero_value), zhi = (_Float16)(64.0f + a.zero_value);
    uint32_t mag_lo = 0, mag_hi = 0;
    if constexpr (Q4) {
        asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(mag_lo));
        asm volatile("v_mov_b32 %0, 0x54005400" : "=v"(mag_hi));
    }
    // Weights of MFMA kk of sub-step parity e (Q4: q - zero, and the fragments' scales of its group).
    auto decode = [&](const v4u (&w)[WV], int e, int kk, h8 (&b)[FN], float (&s)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            if constexpr (Q4) {
                s[j] = (float)bits_h((uint16_t)(w[kk][2] >> (16 * j)));
                h2 z0 = {zlo, zlo}, z1 = {zhi, zhi};
                if constexpr (ZG) {
                    const _Float16 z = bits_h((uint16_t)(w[kk][3] >> (16 * j)));
                    z0 = (h2){z, z} + (h2){1024, 1024};
                    z1 = (h2){z, z} + (h2){64, 64};
                }
                const uint32_t d = w[kk][j], d8 = d >> 8;
                const uint4 u = make_uint4(h2_bits(bits_h2((d & 0x000F000Fu) | mag_lo) - z0), h2_bits(bits_h2((d & 0x00F000F0u) | mag_hi) - z1),
                                           h2_bits(bits_h2((d8 & 0x000F000Fu) | mag_lo) - z0), h2_bits(bits_h2((d8 & 0x00F000F0u) | mag_hi) - z1));
                b[j] = *reinterpret_cast<const h8*>(&u);
            } else {
                const uint32_t d = w[j][2 * e + kk];
                const h2 s2 = bits_h2(ss[j]);
                const uint4 u = make_uint4(h2_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 0) * s2),
                                           h2_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 1) * s2),
                                           h2_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 2) * s2),
                                           h2_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 3) * s2));
                b[j] = *reinterpret_cast<const h8*>(&u);
            }
        }
    };
    auto read_x = [&](int buf, int kk, h8 (&x)[2][FM]) __attribute__((always_inline)) {
        const uint8_t* src = xgrp + buf * kXBuf + (kk ? rd1 : rd0);
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
            for (int i = 0; i < FM; ++i) x[pl][i] = *reinterpret_cast<const h8*>(src + 128 * BM * pl + 2048 * i);
    };
    // Q4: the group's sums of the last K half, not yet scaled, and their scales.
    f4 sums[Q4 ? FM : 1][FN];
    float sc[FN] = {};
#pragma unroll
    for (int i = 0; i < (Q4 ? FM : 1); ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) sums[i][j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto scale_sums = [&](int i, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(sc[j], sums[i][j][r], acc[i][j][r]);
    };
    auto mfmas = [&](const h8 (&x)[2][FM], const h8 (&b)[FN], const float (&s)[FN]) __attribute__((always_inline)) {
        if constexpr (Q4) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    scale_sums(i, j);
                    sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[1][i], b[j], (f4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                }
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[0][i], b[j], sums[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < FN; ++j) sc[j] = s[j];
            return;
        }
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[pl][i], b[j], acc[i][j], 0, 0, 0);
    };

    // Loads of a sub-step at position k of the unrolled loop (weights first, then activations): the
    // activations of sub-step t + 3, the weights of t + 3 (Q4) or, on even t, of step t / 2 + 3
    // (FP4-KM, with the next four steps' scale bytes at k = 0).
    constexpr int kXLoads = FM;
    auto issued = [](int k) constexpr {
        return kXLoads + (FP4 ? ((k & 1) ? 0 : FN) + (k == 0 ? FN : 0) : 2 * (FN + 1 + ZG));
    };

    h8 ax0[2][FM], ax1[2][FM], bw0[FN], bw1[FN];
    float s0[FN] = {}, s1[FN] = {};
    if constexpr (FP4) load_sb(sb, 0);
    static_for<3>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        load_w(wv[k], k);
        load_x(k, k);
        __builtin_amdgcn_sched_barrier(0);  // the wait below counts on this order
    });
    if constexpr (FP4) {
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = h_bits((_Float16)lut_v[i]);
        lut_h[0] = b[0] | (b[1] << 16);
        lut_h[1] = b[2] | (b[3] << 16);
    }
    wait_vmcnt<2 * (kXLoads + (FP4 ? FN : 2 * (FN + 1 + ZG)))>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (FP4) scale_of(sb, 0, ss);
    read_x(0, 0, ax0);
    decode(wv[0], 0, 0, bw0, s0);

    constexpr int kMfmas = 2 * FM * FN;  // per K half
    // VALU operations beside each MFMA; Q4: the first half of the MFMAs beside the scaling
    constexpr int kValuPerMfma = FP4 ? (FN * 9 + kMfmas - 1) / kMfmas : 4;
    // Sub-step t = base + k. Its loads, in `wait` order: at the mid-step wait those of this and of the
    // previous sub-step may stay in flight, which leaves t + 1's activations landed.
    auto step = [&](int t, auto kc, auto guard) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, e = k & 1;
        constexpr int set = FP4 ? (k >> 1) % kSets : k % kSets;             // t's weights
        constexpr int set1 = FP4 ? ((k + 1) >> 1) % kSets : (k + 1) % kSets;  // t + 1's
        const bool live = !decltype(guard)::value || t < nt_all;
        uint32_t sn[FP4 ? FN : 1];
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (Q4) load_w(wv[(k + 3) % kSets], t + 3);
        if constexpr (FP4 && e == 0) load_w(wv[((k >> 1) + 3) % kSets], (t >> 1) + 3);
        if constexpr (FP4 && k == 0) load_sb(sbn, (t >> 3) + 1);
        load_x(t + 3, (k + 3) % kDepth);
        if (live) {
            mfmas(ax0, bw0, s0);
            read_x(k % kDepth, 1, ax1);
            decode(wv[set], e, 1, bw1, s1);
            if constexpr (FP4 && e == 1) scale_of(k == 7 ? sbn : sb, (t >> 1) + 1, sn);
#pragma unroll
            for (int m = 0; m < kMfmas; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);                   // one MFMA
                if (m < 2 * FM) __builtin_amdgcn_sched_group_barrier(0x0100, 1, 0);   // a fragment read
                if (m < issued(k)) __builtin_amdgcn_sched_group_barrier(0x0010, 1, 0);  // a load
                __builtin_amdgcn_sched_group_barrier(0x0002, kValuPerMfma, 0);        // its share of the VALU
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<issued((k + 7) % 8) + issued(k)>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (live) {
            if constexpr (FP4 && e == 1) {
#pragma unroll
                for (int j = 0; j < FN; ++j) ss[j] = sn[j];
            }
            mfmas(ax1, bw1, s1);
            read_x((k + 1) % kDepth, 0, ax0);
            decode(wv[set1], e ^ 1, 0, bw0, s0);
#pragma unroll
            for (int m = 0; m < kMfmas; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x0008, 1, 0);                  // one MFMA
                if (m < 2 * FM) __builtin_amdgcn_sched_group_barrier(0x0100, 1, 0);  // a fragment read
                __builtin_amdgcn_sched_group_barrier(0x0002, kValuPerMfma, 0);       // its share of the VALU
            }
        }
        if constexpr (FP4 && k == 7) {
#pragma unroll
            for (int j = 0; j < FN; ++j) sb[j] = sbn[j];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int t = 0;
    for (; t + kUnroll <= nt_all; t += kUnroll)
        static_for<kUnroll>([&](auto kc) { step(t + decltype(kc)::value, kc, std::false_type{}); });
    if (t < nt_all)
        static_for<kUnroll>([&](auto kc) { step(t + decltype(kc)::value, kc, std::true_type{}); });

    if constexpr (Q4) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) scale_sums(i, j);
    }
    // Partial tiles -> LDS, once every wave's loads have landed and every wave is done with the
    // buffers -> the two groups' sums -> y or the split-K partials.
    wait_vmcnt<0>();
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);  // [2 groups][BM rows][kPitch]
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[(p * BM + 16 * i + 4 * g + r) * kPitch + 32 * h + 16 * j + c] = acc[i][j][r];
    __syncthreads();
    float* part = a.part ? a.part + (size_t)blockIdx.z * splitk_stride(a.M, a.N) : nullptr;
    const bool vec = out8_vector_ok<YT>(a, part);
#pragma unroll
    for (int k = 0; k < (BM * 16 + 511) / 512; ++k) {
        const int u = tid + 512 * k;  // chunk of 8 outputs: row u / 16, columns 8 (u % 16)
        if (u >= BM * 16) break;
        const int row = u >> 4, col = (u & 15) * 8;
        const int m = m0 + row;
        if (m >= a.M) continue;
        const float* src = red + row * kPitch + col;
        const int sh = a.row_shift[m];
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const float4 s0 = *reinterpret_cast<const float4*>(src + e);
            const float4 s1 = *reinterpret_cast<const float4*>(src + BM * kPitch + e);
            v[e] = __builtin_amdgcn_ldexpf(s0.x + s1.x, -sh);
            v[e + 1] = __builtin_amdgcn_ldexpf(s0.y + s1.y, -sh);
            v[e + 2] = __builtin_amdgcn_ldexpf(s0.z + s1.z, -sh);
            v[e + 3] = __builtin_amdgcn_ldexpf(s0.w + s1.w, -sh);
        }
        store_out8<YT>(a, part, vec, m, n0 + col, v);
    }
}

// gemm_planes_half: half weights, both operands through LDS. A fragment's 16 rows x 64 bytes of half
// weights loaded straight into registers touch half a line per row, which costs the load unit as
// much as whole lines: that alone took 18 of 42 us at M = 130, K = 4096, N = 6144. Here the weights'
// 128 lines per 64-value sub-step go into LDS by direct loads beside the planes', and both are read as
// fragments; one K group, so the buffers hold them.
//   Block: 16 RP FR rows x 128 columns, RP x CP waves; wave w owns 128 / CP columns from part w % CP and
//   16 FR rows from part w / CP. Loads run kDepth - 1 sub-steps ahead, each sub-step in two halves
//   around one barrier as above. LDS bounds it: per sub-step a 64-row tile of 8 waves reads 96 KB of
//   fragments and takes in 32 KB for 512 clocks of MFMAs per SIMD. A 128-row tile's waves (32 x 64
//   outputs) read 2/3 of that per MFMA; four waves of that shape on 64 rows do too, but one wave
//   per SIMD hides less: 39 us for 29 below.
//   Time with split_planes and the splits' sum, against weights in registers:
//     M = 130, K = 4096, N = 6144: 42.1 -> 29.2 us     M = 512, K = N = 4096: 48.7 -> 39.0
//     M = 256, K = 4096, N = 14336: 86 (64 rows), 66 (128 rows)
//     M = 16, K = 4096, N = 6144: 16.4 -> 15.2         M = 1: 15.3 -> 14.1
template <int RP, int FR, int CP>
struct HalfShape {
    static constexpr int kWaves = RP * CP, kFN = kBN / 16 / CP, kBM = 16 * RP * FR;
    static constexpr int kRows = 2 * kBM + kBN;                 // lines per buffer: planes, then weights
    static constexpr int kBuf = kRows * 128, kDepth = kBM == 64 ? 4 : 3;
    static constexpr int kLoads = kRows / 8 / kWaves;           // per wave and sub-step
    static constexpr int kPlane = kBM / 8 / kWaves;             // of them a plane's
    static constexpr int kRed = kBM * kPitch * 4;
    static constexpr int kLds = kDepth * kBuf > kRed ? kDepth * kBuf : kRed;
};

template <int RP, int FR, int CP, int YT>
__global__ __launch_bounds__(64 * RP * CP, RP * FR == 2 ? 4 : 2) void gemm_planes_half(GemmArgs a) {
    using S = HalfShape<RP, FR, CP>;
    constexpr int BM = S::kBM, D = S::kDepth, FN = S::kFN, NW = S::kWaves;
    __shared__ __attribute__((aligned(16))) uint8_t lds[S::kLds];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = wid % CP, rh = wid / CP, c = lane & 15, g = lane >> 4;
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
    const int s_all = K / kSub, s_first = a.part ? (int)blockIdx.z * a.split_steps : 0;
    const int nt = a.part ? min(a.split_steps, s_all - s_first) : s_all;

    // Line groups NW i .. are one operand's each, except that 32 rows have both planes in the first NW.
    const uint32_t plane = (uint32_t)((size_t)a.M * K * 2);
    const rsrc_t xr = make_rsrc(S::kPlane == 0 && wid >= NW / 2 ? a.x_lo : a.x, plane), xlr = make_rsrc(a.x_lo, plane);
    const rsrc_t wr = make_rsrc(a.w16, (uint32_t)((size_t)a.N * K * 2));
    // Direct load i of wave w: line group w + NW i, rows 8 (w + NW i) + lane / 8 of the buffer (high plane,
    // low plane, weights); rows past M or N read zeros.
    uint32_t off[S::kLoads];
#pragma unroll
    for (int i = 0; i < S::kLoads; ++i) {
        const int r = 8 * (wid + NW * i) + (lane >> 3);
        const uint32_t row = r >= 2 * BM ? (uint32_t)(n0 + r - 2 * BM) : (uint32_t)(m0 + (r >= BM ? r - BM : r));
        off[i] = row * (uint32_t)K * 2u + 16u * (uint32_t)((lane & 7) ^ x_swizzle(r & 15));
    }
    auto load = [&](int t, int buf) __attribute__((always_inline)) {
        const uint32_t o = t < nt ? 128u * (uint32_t)(s_first + t) : kPast;
        static_for<S::kLoads>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            uint8_t* const to = lds + buf * S::kBuf + 1024 * (wid + NW * i);
            if constexpr (i >= (S::kPlane ? 2 * S::kPlane : 1)) lds_dma16(wr, to, off[i], o);
            else if constexpr (S::kPlane && i >= S::kPlane) lds_dma16(xlr, to, off[i], o);
            else lds_dma16(xr, to, off[i], o);
        });
    };
    const int rd[2] = {128 * c + 16 * ((2 * g) ^ x_swizzle(c)), 128 * c + 16 * ((2 * g + 1) ^ x_swizzle(c))};

    // Sums of their own for each plane and K half of a sub-step, added up at the end: in one chain of
    // roundings the error against 64 bits was 5.8e-7 (M = 130, K = 4096), so it is 2.9e-7.
    f4 acc[2][2][FR][FN];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[s >> 1][s & 1][i][j] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto read = [&](int buf, int kk, h8 (&x)[2][FR], h8 (&b)[FN]) __attribute__((always_inline)) {
        const uint8_t* const s = lds + buf * S::kBuf + rd[kk];
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j] = *reinterpret_cast<const h8*>(s + 128 * (2 * BM + 16 * FN * h + 16 * j));
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
            for (int i = 0; i < FR; ++i) x[pl][i] = *reinterpret_cast<const h8*>(s + 128 * (BM * pl + 16 * FR * rh + 16 * i));
    };
    auto mfmas = [&](const h8 (&x)[2][FR], const h8 (&b)[FN], f4 (&s)[2][FR][FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
            for (int i = 0; i < FR; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    s[pl][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[pl][i], b[j], s[pl][i][j], 0, 0, 0);
    };

    h8 x0[2][FR], x1[2][FR], b0[FN], b1[FN];
    static_for<D - 1>([&](auto kc) {
        load(decltype(kc)::value, decltype(kc)::value);
        __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
    });
    wait_vmcnt<(D - 2) * S::kLoads>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    read(0, 0, x0, b0);
    auto step = [&](int t, auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        __builtin_amdgcn_sched_barrier(0);
        load(t + D - 1, (k + D - 1) % D);
        mfmas(x0, b0, acc[0]);
        read(k, 1, x1, b1);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<(D - 2) * S::kLoads>();  // t + 1's lines have landed
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        mfmas(x1, b1, acc[1]);
        read((k + 1) % D, 0, x0, b0);
        __builtin_amdgcn_sched_barrier(0);
    };
    int t = 0;
    for (; t + D <= nt; t += D) static_for<D>([&](auto kc) { step(t + decltype(kc)::value, kc); });
    static_for<D - 1>([&](auto kc) {
        if (t + decltype(kc)::value < nt) step(t + decltype(kc)::value, kc);
    });

    // tiles -> LDS, once every load has landed and every wave is done with the buffers -> y or partials
    wait_vmcnt<0>();
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[(16 * FR * rh + 16 * i + 4 * g + r) * kPitch + 16 * FN * h + 16 * j + c] =
                    (acc[0][0][i][j][r] + acc[1][0][i][j][r]) + (acc[0][1][i][j][r] + acc[1][1][i][j][r]);
    __syncthreads();
    float* part = a.part ? a.part + (size_t)blockIdx.z * splitk_stride(a.M, a.N) : nullptr;
    const bool vec = out8_vector_ok<YT>(a, part);
#pragma unroll
    for (int k = 0; k < BM * 16 / (64 * NW); ++k) {
        const int u = tid + 64 * NW * k, row = u >> 4, col = (u & 15) * 8, m = m0 + row;
        if (m >= a.M) continue;
        const float* src = red + row * kPitch + col;
        const int sh = a.row_shift[m];
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const float4 q = *reinterpret_cast<const float4*>(src + e);
            v[e] = __builtin_amdgcn_ldexpf(q.x, -sh);
            v[e + 1] = __builtin_amdgcn_ldexpf(q.y, -sh);
            v[e + 2] = __builtin_amdgcn_ldexpf(q.z, -sh);
            v[e + 3] = __builtin_amdgcn_ldexpf(q.w, -sh);
        }
        store_out8<YT>(a, part, vec, m, n0 + col, v);
    }
}

// Rows of fp32 activations as two fp16 planes (one block per row): the row's power-of-two shift t
// brings its largest magnitude into [2^14, 2^15); hi = fp16(x 2^t), lo = fp16(x 2^t - hi), and an
// infinite x gives an infinite hi and lo = 0. A thread makes 16-byte chunks of 8 values: elements
// 8 i .. 8 i + 7 (natural order), or for FP4-KM (FP4) elements 4 q .. and 16 + 4 q .. of a 32-value
// group interleaved, chunk i = 4 G + q of the row at 16 (G / 4) + 8 (q / 2) + 2 (G % 4) + q % 2. The
// first kHeld chunks of a thread stay in registers between the maximum and the split.
constexpr int kHeld = 4;
template <bool FP4>
__device__ __forceinline__ void split_row(const float* __restrict__ x, int K, bool planes, int* __restrict__ shifts,
                                          uint4* __restrict__ hi, uint4* __restrict__ lo) {
    __shared__ float part[4];
    const size_t row = (size_t)blockIdx.x * K;
    const float4* r = reinterpret_cast<const float4*>(x + row);
    const int nc = K / 8;
    auto first = [](int i) { return FP4 ? 8 * (i >> 2) + (i & 3) : 2 * i; };  // float4 index of a chunk
    constexpr int second = FP4 ? 4 : 1;
    float4 ha[kHeld], hb[kHeld];
    float mx = 0.0f;
    auto most = [&](const float4& v) {
        mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int i = (int)threadIdx.x + 256 * u;
        ha[u] = i < nc ? r[first(i)] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        hb[u] = i < nc ? r[first(i) + second] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        most(ha[u]);
        most(hb[u]);
    }
    for (int i = (int)threadIdx.x + 256 * kHeld; i < nc; i += 256) {
        most(r[first(i)]);
        most(r[first(i) + second]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
    __syncthreads();
    const int t = fp16_range_shift(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
    if (threadIdx.x == 0) shifts[blockIdx.x] = t;
    if (!planes) return;
    auto split = [&](int i, const float4& va, const float4& vb) {
        const float s[8] = {va.x, FP4 ? vb.x : va.y, FP4 ? va.y : va.z, FP4 ? vb.y : va.w,
                            FP4 ? va.z : vb.x, FP4 ? vb.z : vb.y, FP4 ? va.w : vb.z, vb.w};
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint16_t hh[2], ll[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const float v = __builtin_amdgcn_ldexpf(s[2 * e + d], t);
                const _Float16 he = (_Float16)v;
                const float rest = __builtin_isinf(v) ? 0.0f : v - (float)he;
                hh[d] = h_bits(he);
                ll[d] = h_bits((_Float16)rest);
            }
            hw[e] = hh[0] | ((uint32_t)hh[1] << 16);
            lw[e] = ll[0] | ((uint32_t)ll[1] << 16);
        }
        const size_t at = row / 8 + (FP4 ? 16 * (i >> 4) + 8 * ((i & 3) >> 1) + 2 * ((i >> 2) & 3) + (i & 1) : i);
        hi[at] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        lo[at] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int i = (int)threadIdx.x + 256 * u;
        if (i < nc) split(i, ha[u], hb[u]);
    }
    for (int i = (int)threadIdx.x + 256 * kHeld; i < nc; i += 256) split(i, r[first(i)], r[first(i) + second]);
}

// GATE: FP4-KM calls with a gate; without one its loads would stand before the row's (0.3 us).
template <bool FP4, bool GATE = false>
__global__ __launch_bounds__(256) void split_planes(const float* __restrict__ x, int K, int* __restrict__ shifts,
                                                   uint4* __restrict__ hi, uint4* __restrict__ lo, const int* gate, int gate_want) {
    if (GATE && *gate != gate_want) return;  // another route was chosen (whole grid)
    split_row<FP4>(x, K, true, shifts, hi, lo);
}

// Calls whose route the device chooses (recorded ones, tables without a host copy): each block classifies the
// decode table (thread b: scale entry b), the first one writes the class to *flag, and each then brings its
// row of x (null: none) into the form that the class's kernel takes: planes, or the shift alone. One launch
// for the three that would take, as the routes' split-K sums share one (launch_route_sums): a launch that
// does nothing still costs 1.5 to 2 us. Recorded, us, each of ten launches by itself / these six: K = N = 4096,
// M = 16 E8M0 26.5 / 19.2, E2M1 on halves 26.9 / 19.5, other halves 39.4 / 30.9, any values 32.5 / 25.3; K = 4096,
// N = 6144, M = 47 39.6 / 32.5, 34.0 / 26.6, 52.0 / 43.1, 78.4 / 71.1.
__global__ __launch_bounds__(256) void fp4km_prepare(const float* __restrict__ t, int mx, int e2m1, int* flag, const float* __restrict__ x,
                                                     int K, int* __restrict__ shifts, uint4* __restrict__ hi, uint4* __restrict__ lo) {
    constexpr uint32_t bits[16] = {0u, 0x3F000000u, 0x3F800000u, 0x3FC00000u, 0x40000000u, 0x40400000u, 0x40800000u,
                                   0x40C00000u, 0x80000000u, 0xBF000000u, 0xBF800000u, 0xBFC00000u, 0xC0000000u,
                                   0xC0400000u, 0xC0800000u, 0xC0C00000u};
    const uint32_t b = threadIdx.x;
    const float s = t[16 + b];
    bool halves = true, same = true;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float p = t[i] * s;
        halves = halves && __builtin_isfinite(p) && (float)(_Float16)p == p;
        same = same && __builtin_bit_cast(uint32_t, t[i]) == bits[i];
    }
    halves = __syncthreads_and(halves);
    const bool e8m0 = __syncthreads_and(b >= 253u || __builtin_bit_cast(uint32_t, s) == (b ? b << 23 : 0x00400000u));
    const int cls = same && e8m0 && mx ? kTableMx : !halves ? kTableAny : same && e2m1 ? kTableE2m1 : kTableHalves;
    if (b == 0 && blockIdx.x == 0) *flag = cls;
    if (x && (cls == kTableE2m1 || cls == kTableHalves)) split_row<true>(x, K, cls == kTableE2m1, shifts, hi, lo);
}

template <BFormat F, int FM, bool ZG>
void launch_planes_y(const GemmArgs& a, int splits) {
    const dim3 grid((a.N + kBN - 1) / kBN, (a.M + 16 * FM - 1) / (16 * FM), splits);
    switch (a.y_dtype) {
    case BYHIP_F32: launch("gemm_planes", (gemm_planes<F, FM, BYHIP_F32, ZG>), grid, dim3(512), 0, a); break;
    case BYHIP_F16: launch("gemm_planes", (gemm_planes<F, FM, BYHIP_F16, ZG>), grid, dim3(512), 0, a); break;
    default: launch("gemm_planes", (gemm_planes<F, FM, BYHIP_BF16, ZG>), grid, dim3(512), 0, a); break;
    }
    BYHIP_LAUNCHED("gemm_planes");
}

template <BFormat F, bool ZG = false>
void launch_planes_fm(const GemmArgs& a, int fm, int splits) {
    switch (fm) {
    case 1: launch_planes_y<F, 1, ZG>(a, splits); break;
    case 2: launch_planes_y<F, 2, ZG>(a, splits); break;
    case 3: launch_planes_y<F, 3, ZG>(a, splits); break;
    default: launch_planes_y<F, 4, ZG>(a, splits); break;
    }
}

// FP4-KM: row fragments per tile, the fewest tiles of up to 64 rows, cut to the rows there are.
int planes_fm(int M) {
    const int row_tiles = (M + 63) / 64;
    return (M + 16 * row_tiles - 1) / (16 * row_tiles);
}

long planes_tiles(int M, int N) {
    const int rows = 16 * planes_fm(M);
    return (long)((N + kBN - 1) / kBN) * ((M + rows - 1) / rows);
}

// A number of K splits and the time a pass is expected to take, in steps.
struct Pass {
    int splits;
    double time;
};

// FP4-KM: K splits, in 128-value steps: the count that minimises rounds of blocks x (steps per split + 12)
// (12 for a block's fixed cost: first loads, epilogue), plus 6 steps for the sum's launch.
Pass planes_pass(int K, long tiles) {
    const int steps = (K + 127) / 128;
    const long cus = compute_units();
    Pass best = {1, 1e300};
    for (int s = 1; s <= std::max(1, steps / 4); ++s) {
        const int per = (steps + s - 1) / s;
        if ((steps + per - 1) / per != s) continue;  // the same split as a smaller s
        const double t = (double)((tiles * s + cus - 1) / cus) * (per + 12) + (s > 1 ? 6.0 : 0.0);
        if (t < 0.97 * best.time) best = {s, t};
    }
    return best;
}

// Q4: row fragments per tile and K splits together, by the time of their rounds of blocks in us. A block of 2 / 3 / 4
// fragments takes 5.9 / 6.7 / 7.7 us and 0.75 / 0.72 / 0.86 per 128-value step, a sum 3.1 us and 1.6 per 1e6 partial
// values. Fitted to 112 calls of M = 49 .. 1082, K = 128 .. 14336, N = 1088 .. 14336 at every height with 1 to 6
// splits: the choice is on average 0.2% from the fastest of those, the fewest 64-row tiles were 7.6%; it is never
// the slower of the two. us, fewest tiles / this: M = 496, K = 1920, N = 1984 25.9 (64 rows, 2 splits) / 19.6 (32 rows);
// M = 343, K = 1792, N = 5632 40.6 / 30.9 (32); M = 198, K = 3264, N = 4224 33.6 / 26.2 (32); M = 391, K = 6144, N = 10240 149 / 126
// (48); M = 567, K = 3712, N = 8128 106 / 93 (48); M = 509, K = 4096, N = 14336 147 either way (64).
struct Q4Tile {
    int fm;
    Pass pass;
};
Q4Tile q4_tile(int M, int K, int N, size_t room) {  // room: scratch for the partials
    const int steps = (K + 127) / 128;
    const int most = std::max(1, std::min<int>(steps / 4, (int)(room / (splitk_stride(M, N) * sizeof(float)))));
    const long cus = compute_units(), cols = (N + kBN - 1) / kBN;
    if (M <= 16) return {1, planes_pass(K, cols)};
    constexpr double kBlock[3] = {5.9, 6.7, 7.7}, kStepUs[3] = {0.75, 0.72, 0.86};
    Q4Tile best = {4, {1, 1e300}};
    for (int fm = 4; fm >= 2; --fm) {
        if (16 * fm >= M + 16) continue;  // a fragment of rows past M
        const long tiles = cols * ((M + 16 * fm - 1) / (16 * fm));
        for (int s = 1; s <= most; ++s) {
            const int per = (steps + s - 1) / s;
            if ((steps + per - 1) / per != s) continue;  // the same split as a smaller s
            const double t = (double)((tiles * s + cus - 1) / cus) * (kBlock[fm - 2] + per * kStepUs[fm - 2]) +
                             (s > 1 ? 3.1 + 1.6e-6 * M * N * s : 0.0);
            if (t < best.pass.time) best = {fm, {s, t}};
        }
    }
    return best;
}

// The same for gemm_planes_half, in 64-value steps: 16 for a block's fixed cost, 12 for the sum's launch and
// 1.5 per split for what it reads (M = 32, K = 4096, N = 6144: 4 splits 16.3 us, 6 splits,
// a second block on some of the CUs, 17.9, 1 split 24.5).
Pass half_pass(long tiles, int steps) {
    const long cus = compute_units();
    Pass best = {1, 1e300};
    for (int s = 1; s <= std::max(1, steps / 8); ++s) {
        const int per = (steps + s - 1) / s;
        if ((steps + per - 1) / per != s) continue;
        const double t = (double)((tiles * s + cus - 1) / cus) * (per + 16) + (s > 1 ? 12.0 + 1.5 * s : 0.0);
        if (t < 0.97 * best.time) best = {s, t};
    }
    return best;
}

template <int RP, int FR, int CP>
void launch_half_y(const GemmArgs& a, int splits) {
    using S = HalfShape<RP, FR, CP>;
    const dim3 grid((a.N + kBN - 1) / kBN, (a.M + S::kBM - 1) / S::kBM, splits), block(64 * S::kWaves);
    switch (a.y_dtype) {
    case BYHIP_F32: launch("gemm_planes_half", (gemm_planes_half<RP, FR, CP, BYHIP_F32>), grid, block, 0, a); break;
    case BYHIP_F16: launch("gemm_planes_half", (gemm_planes_half<RP, FR, CP, BYHIP_F16>), grid, block, 0, a); break;
    default: launch("gemm_planes_half", (gemm_planes_half<RP, FR, CP, BYHIP_BF16>), grid, block, 0, a); break;
    }
    BYHIP_LAUNCHED("gemm_planes_half");
}

// Rows per tile: 32, two blocks per CU, for up to 32 rows (M = 8, K = N = 4096: 12.6 us, 64 rows
// 13.1); else 64, or 128 where its rounds of blocks, each 1.6 times as long, take less time (M = 256, K =
// 4096, N = 14336: one round for two, 66 us for 86; M = 512, K = N = 4096: one round either way, 45 for 39).
struct HalfTiles {
    int rows;
    long tiles;
};
HalfTiles half_tiles(int M, int K, int N) {
    const int cus = compute_units();
    const long cols = (N + kBN - 1) / kBN, t64 = cols * ((M + 63) / 64), t128 = cols * ((M + 127) / 128);
    if (M <= 32) return {32, cols};
    if ((uint64_t)K * 256 < kPast / 2 && 8 * ((t128 + cus - 1) / cus) < 5 * ((t64 + cus - 1) / cus)) return {128, t128};
    return {64, t64};
}

void launch_half_rows(const GemmArgs& a0) {
    GemmArgs a = a0;
    const HalfTiles h = half_tiles(a.M, a.K, a.N);
    const int steps = a.K / kSub, forced = env_int("BYHIP_Q4_SPLIT", 0);
    const int splits = choose_split(a, h.tiles, steps, 1, forced > 0 ? forced : half_pass(h.tiles, steps).splits, 1);
    if (splits == 1) a.part = nullptr;
    if (h.rows == 32) launch_half_y<2, 1, 4>(a, splits);
    else if (h.rows == 128) launch_half_y<4, 2, 2>(a, splits);
    else launch_half_y<2, 2, 4>(a, splits);
    if (a.part) launch_splitk_sum(a, splits);
}

template <BFormat F>
void launch_planes_rows(const GemmArgs& a0) {
    GemmArgs a = a0;
    Q4Tile tile = {planes_fm(a.M), {}};
    if constexpr (F == BFormat::Q4Fast) tile = q4_tile(a.M, a.K, a.N, a.work_bytes);
    else tile.pass = planes_pass(a.K, planes_tiles(a.M, a.N));
    const int fm = tile.fm, forced = env_int("BYHIP_Q4_SPLIT", 0);
    const long tiles = (long)((a.N + kBN - 1) / kBN) * ((a.M + 16 * fm - 1) / (16 * fm));
    const int splits = choose_split(a, tiles, (a.K + 127) / 128, 1, forced > 0 ? forced : tile.pass.splits, 1);
    if (splits == 1) a.part = nullptr;
    if constexpr (F == BFormat::Q4Fast) {
        if (a.zeros) launch_planes_fm<F, true>(a, fm, splits);
        else launch_planes_fm<F>(a, fm, splits);
    } else {
        launch_planes_fm<F>(a, fm, splits);
    }
    if (a.part) launch_splitk_sum(a, splits);
}

// The row shifts and both planes.
size_t plane_bytes(int M, int K) {
    return ((size_t)M * sizeof(int) + 255) / 256 * 256 + 2 * (((size_t)M * K * 2 + 255) / 256 * 256);
}

// Rows whose planes fit half the scratch (the rest holds split-K partials) and whose offsets stay below 2^31.
size_t plane_rows(const GemmArgs& a) {
    const size_t work_bytes = a.work ? a.work_bytes : kWorkspaceBytes;
    return std::min<size_t>({work_bytes / 2 / ((size_t)a.K * 4 + sizeof(int)), ((size_t)kPast / 2) / ((size_t)a.K * 2), 65535 * 16});
}

// The time of passes of `rows` rows each and one of what is left.
double passes_time(BFormat fmt, const GemmArgs& a, int rows) {
    auto pass = [&](int m) {
        if (m == 0) return 0.0;
        if (fmt == BFormat::Q4Fast) return q4_tile(m, a.K, a.N, (a.work ? a.work_bytes : kWorkspaceBytes) - plane_bytes(m, a.K)).pass.time;
        if (fmt == BFormat::Fp4Km) return planes_pass(a.K, planes_tiles(m, a.N)).time;
        const HalfTiles h = half_tiles(m, a.K, a.N);
        return half_pass(h.tiles, a.K / kSub).time * (h.rows == 128 ? 1.6 : 1.0);
    };
    return (double)(a.M / rows) * pass(rows) + pass(a.M % rows);
}

// Rows of a pass over the weights: all of them up to the whole 64-row tiles that fit the scratch. Past that, all
// of them where they fit, those whole tiles, or even shares of them, by the time of the passes' rounds of blocks
// (us, K = N = 4096, M = 970: all 85, 960 + 10 94; M = 1024: 960 + 64 rows 105, 2 x 512 92; M = 2048: 2 x 960 + 128 185, 3 x 704
// 227; K = 14336, N = 4096, M = 300: 256 + 44 100, 192 + 108 113; K = 11328, N = 6016, M = 361: all 147, 320 + 41 130).
int planes_pass_rows(BFormat fmt, const GemmArgs& a) {
    const int most = (int)plane_rows(a), full = most / 64 * 64;
    if (a.M <= std::max(full, std::min(most, 63))) return a.M;
    if (full == 0) return most;
    const int blocks = (a.M + full - 1) / full, even = (a.M + 64 * blocks - 1) / (64 * blocks) * 64;
    int best = full;
    double best_t = passes_time(fmt, a, full);
    for (const int rows : {even, a.M <= most ? a.M : even}) {
        const double t = passes_time(fmt, a, rows);
        if (t < (rows == a.M ? 1.03 : 0.97) * best_t) best = rows, best_t = t;
    }
    return best;
}

}  // namespace

bool gemm_planes_one_pass(BFormat fmt, const GemmArgs& a) { return planes_pass_rows(fmt, a) >= a.M; }

double gemm_planes_q4_us(const GemmArgs& a) { return passes_time(BFormat::Q4Fast, a, planes_pass_rows(BFormat::Q4Fast, a)); }

bool gemm_planes_ok(BFormat fmt, const GemmArgs& a) {
    constexpr uint64_t kLim = kPast;  // offsets stay below 2^31 (loads past the end)
    if (a.x_dtype != BYHIP_F32 || reinterpret_cast<uintptr_t>(a.x) % 16 != 0) return false;
    if ((uint64_t)(a.K) * 2 * 128 >= kLim || plane_rows(a) == 0) return false;
    if (fmt == BFormat::Fp4Km)
        return a.K % 128 == 0 && reinterpret_cast<uintptr_t>(a.blob) % 16 == 0 && a.scale_base % 4 == 0 &&
               (uint64_t)(a.N + kBN) * (a.K / 2) < kLim;
    if (fmt == BFormat::Q4Fast)
        return a.wpf && a.spf && (!a.zeros || a.zpf) && a.scale_f16 && a.K % kSub == 0 && (uint64_t)(a.N + kBN) * a.K / 2 < kLim;
    if (fmt == BFormat::F16)
        return a.K % kSub == 0 && reinterpret_cast<uintptr_t>(a.w16) % 16 == 0 && (uint64_t)(a.N + kBN) * a.K * 2 < kLim;
    return false;
}

namespace {

// Where the row shifts and planes of M rows go, and what of the scratch is left.
struct PlaneScratch {
    int* shifts;
    uint8_t *hi, *lo, *rest;
    size_t rest_bytes;
};

PlaneScratch plane_scratch(const GemmArgs& a) {
    uint8_t* const work = static_cast<uint8_t*>(a.work ? a.work : workspace());
    const size_t bytes = a.work ? a.work_bytes : kWorkspaceBytes;
    const size_t shift_bytes = ((size_t)a.M * sizeof(int) + 255) / 256 * 256, plane = ((size_t)a.M * a.K * 2 + 255) / 256 * 256;
    const size_t used = plane_bytes(a.M, a.K);
    return {reinterpret_cast<int*>(work), work + shift_bytes, work + shift_bytes + plane, work + used, bytes - used};
}

}  // namespace

bool launch_fp4km_prepare(const GemmArgs& a, bool mx, bool e2m1, int* flag) {
    const bool f32 = a.x_dtype == BYHIP_F32, fits = !f32 || (size_t)a.M <= plane_rows(a);
    PlaneScratch p = {};
    if (f32 && fits) p = plane_scratch(a);
    launch("fp4km_prepare", fp4km_prepare, dim3(f32 && fits ? (unsigned)a.M : 1u), dim3(256), 0, a.lut, (int)mx, (int)e2m1, flag,
           f32 && fits ? static_cast<const float*>(a.x) : nullptr, a.K, p.shifts, reinterpret_cast<uint4*>(p.hi), reinterpret_cast<uint4*>(p.lo));
    BYHIP_LAUNCHED("fp4km_prepare");
    return fits;
}

void launch_gemm_planes(BFormat fmt, const GemmArgs& a0) {
    const size_t rows = (size_t)(a0.prepared ? a0.M : planes_pass_rows(fmt, a0));
    for (size_t m = 0; m < (size_t)a0.M; m += rows) {
        GemmArgs a = a0;
        a.M = (int)std::min<size_t>(rows, (size_t)a0.M - m);
        const float* const x = static_cast<const float*>(a0.x) + m * a0.K;
        a.y = static_cast<uint8_t*>(a0.y) + m * a0.N * dtype_bytes(a0.y_dtype);
        const PlaneScratch p = plane_scratch(a);
        if (!a.prepared) {
            launch("split_planes", fmt != BFormat::Fp4Km ? split_planes<false> : a.gate ? split_planes<true, true> : split_planes<true>, dim3((unsigned)a.M), dim3(256), 0, x, a.K,
                   p.shifts, reinterpret_cast<uint4*>(p.hi), reinterpret_cast<uint4*>(p.lo), a.gate, a.gate_want);
            BYHIP_LAUNCHED("split_planes");
        }
        a.x = p.hi;
        a.x_lo = p.lo;
        a.row_shift = p.shifts;
        a.work = p.rest;
        a.work_bytes = p.rest_bytes;
        if (fmt == BFormat::Fp4Km) launch_planes_rows<BFormat::Fp4Km>(a);
        else if (fmt == BFormat::Q4Fast) launch_planes_rows<BFormat::Q4Fast>(a);
        else launch_half_rows(a);
    }
}

}  // namespace byhip
