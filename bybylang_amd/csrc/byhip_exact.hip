// byhip_exact.hip - the exact fp32 GEMM for the quantized weight formats (gfx950).
//
// y[M, N] = x[M, K] . W^T where every weight is formed in fp32 exactly as the reference forms it:
//   Q4      ((float)q - zero) * scale, any scales, zeros and group size (cpu_vm.c:467-470,
//           cpu_kernels_impl.inc:309-314)
//   FP4-KM  lut[nibble] * lut[16 + scale byte] (cpu_vm.c:611-618)
//   F16     the half widened (cpu_vm.c:571-575)
// Activations are used in fp32 (fp16 ones widened exactly); products and sums are fp32, in
// v_mfma_f32_16x16x4_f32. This is the route for data the fp16 MFMA kernels cannot hold exactly:
// Q4 weights outside fp16's range, the micro-VM's Q4 ops (fp32 arithmetic in the reference) above two
// rows, and FP4-KM tables above one row that are neither E2M1 with E8M0 scales nor all halves in their
// products. Q4 rows with fp32 scales take gemm_f32_q4 (below), the pipelined form, where it fits. It differs
// from the reference only in the order of the fp32 additions.
//
// Block: BM x 64 outputs, 4 waves; wave w owns columns 16w .. 16w+15 and all BM rows (BM / 16
// fragments). K steps of 64: each thread stages BM / 4 activations and 16 weights of one column
// (formed in fp32) into LDS, then each wave issues 16 MFMAs per fragment.
// Operand layout of v_mfma_f32_16x16x4_f32: lane l supplies A[l % 16][g] and B[g][l % 16] for its
// lane group g = l / 16; the result lane l holds C[4g + i][l % 16], i = 0..3. In MFMA kk (0..15) of a
// step, lane group g supplies K position 16g + kk, so one 16-byte LDS read gives a lane four MFMAs'
// worth of an operand; both operands use that order, so every product pairs the same k.
// Split-K: when the tiles leave CUs idle, block z covers K steps [z * split_steps, ...) and writes
// fp32 partials that splitk_sum adds in slice order.
#include <algorithm>

#include "byhip_gemm.h"
#include "byhip_internal.h"
#include "byhip_kernels.h"

namespace byhip {
namespace {

constexpr int EBK = 64;        // K values per step
constexpr int ELD = EBK + 4;   // floats per LDS row: 16-byte aligned rows, 4-bank skew per row

// FX activations of row m from position k (zeros past M and K), widened to fp32.
template <bool XF32, int FX>
__device__ __forceinline__ void exact_x(const GemmArgs& a, int m, int k, float* v) {
    const bool row = m < a.M;
    const size_t base = (size_t)m * a.K;
#pragma unroll
    for (int e = 0; e < FX; ++e) {
        const bool ok = row && k + e < a.K;
        if constexpr (XF32) v[e] = ok ? static_cast<const float*>(a.x)[base + k + e] : 0.0f;
        else v[e] = ok ? (float)static_cast<const _Float16*>(a.x)[base + k + e] : 0.0f;
    }
}

// The 16 weights of column n at K positions k .. k+15 (k % 16 == 0), formed as the reference forms
// them; zeros past N and K.
template <BFormat F>
__device__ __forceinline__ void exact_w(const GemmArgs& a, int n, int k, const float* lut_s, float* w) {
#pragma unroll
    for (int e = 0; e < 16; ++e) w[e] = 0.0f;
    if (n >= a.N || k >= a.K) return;
    if constexpr (F == BFormat::Fp4Km) {
        // FP4-KM group g = k / 32: byte j holds element j (low nibble) and j + 16 (high nibble)
        const int g = k >> 5, hi = (k >> 4) & 1;
        const uint4 d = *reinterpret_cast<const uint4*>(a.blob + (size_t)n * (a.K >> 1) + (size_t)g * 16);
        const float s = lut_s[16 + a.blob[a.scale_base + (size_t)n * (a.K >> 5) + g]];
        const uint32_t dw[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t byte = (dw[j >> 2] >> (8 * (j & 3))) & 0xFFu;
            w[j] = lut_s[hi ? byte >> 4 : byte & 15u] * s;
        }
    } else if constexpr (F == BFormat::F16) {
        const _Float16* p = reinterpret_cast<const _Float16*>(a.w16) + (size_t)n * a.K + k;
#pragma unroll
        for (int e = 0; e < 16; ++e) w[e] = (float)p[e];
    } else {
        // Q4: nibble k at byte k / 2 of the row, even k in the low nibble
        const uint8_t* row = a.wq + (size_t)n * a.row_bytes;
        uint32_t b[8];
        if (a.row_bytes % 4 == 0 && reinterpret_cast<uintptr_t>(a.wq) % 4 == 0) {
            const uint32_t* r32 = reinterpret_cast<const uint32_t*>(row + (k >> 1));
            const uint32_t w0 = r32[0], w1 = (size_t)(k >> 1) + 4 < a.row_bytes ? r32[1] : 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                b[i] = (w0 >> (8 * i)) & 0xFFu;
                b[4 + i] = (w1 >> (8 * i)) & 0xFFu;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) b[i] = (size_t)(k >> 1) + i < a.row_bytes ? row[(k >> 1) + i] : 0u;
        }
        const size_t rowg = (size_t)n * a.gpr;
        int g = a.group ? k / a.group : 0;
        int next = a.group ? (g + 1) * a.group : 0x7FFFFFFF;
        auto scale_at = [&](int gg) {
            return a.scale_f16 ? (float)static_cast<const _Float16*>(a.scales)[rowg + gg]
                               : static_cast<const float*>(a.scales)[rowg + gg];
        };
        float s = scale_at(g), z = a.zeros ? a.zeros[rowg + g] : a.zero_value;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            if (k + e >= a.K) break;
            if (k + e >= next) {
                ++g;
                next += a.group;
                s = scale_at(g);
                z = a.zeros ? a.zeros[rowg + g] : a.zero_value;
            }
            const uint32_t q = (b[e >> 1] >> (4 * (e & 1))) & 15u;
            w[e] = ((float)q - z) * s;
        }
    }
}

__device__ __forceinline__ void store_any(void* y, int y_dtype, size_t idx, float v) {
    if (y_dtype == BYHIP_F32) store_y<BYHIP_F32>(y, idx, v);
    else if (y_dtype == BYHIP_F16) store_y<BYHIP_F16>(y, idx, v);
    else store_y<BYHIP_BF16>(y, idx, v);
}

template <BFormat F, bool XF32, int BM>
__global__ __launch_bounds__(256) void gemm_f32_exact(GemmArgs a) {
    if (a.gate && *a.gate != a.gate_want) return;  // the other route was chosen (whole grid)
    constexpr int FM = BM / 16;      // row fragments per wave
    constexpr int FX = BM / 4;       // activations a thread stages per step
    constexpr int XT = EBK / FX;     // threads per activation row
    __shared__ __attribute__((aligned(16))) float xs[BM * ELD];
    __shared__ __attribute__((aligned(16))) float ws[64 * ELD];
    __shared__ float lut_s[F == BFormat::Fp4Km ? 272 : 1];

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int g = lane >> 4, c = lane & 15;
    const int n0 = blockIdx.x * 64, m0 = blockIdx.y * BM;
    const int total = (a.K + EBK - 1) / EBK;
    const int s_first = a.part ? (int)blockIdx.z * a.split_steps : 0;
    const int nsteps = a.part ? min(a.split_steps, total - s_first) : total;

    if constexpr (F == BFormat::Fp4Km) {
        for (int i = tid; i < 272; i += 256) lut_s[i] = a.lut[i];
        __syncthreads();
    }

    f4 acc[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[i] = (f4){0.0f, 0.0f, 0.0f, 0.0f};

    const int xrow = tid / XT, xseg = tid % XT;  // the activation row this thread stages, FX values
    const int wcol = tid >> 2, wseg = tid & 3;   // the weight column, 16 values
    for (int s = 0; s < nsteps; ++s) {
        const int k0 = (s_first + s) * EBK;
        float xv[FX], wv[16];
        exact_x<XF32, FX>(a, m0 + xrow, k0 + xseg * FX, xv);
        exact_w<F>(a, n0 + wcol, k0 + wseg * 16, lut_s, wv);
#pragma unroll
        for (int t = 0; t < FX / 4; ++t)
            *reinterpret_cast<float4*>(&xs[xrow * ELD + xseg * FX + 4 * t]) =
                make_float4(xv[4 * t], xv[4 * t + 1], xv[4 * t + 2], xv[4 * t + 3]);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            *reinterpret_cast<float4*>(&ws[wcol * ELD + wseg * 16 + 4 * t]) =
                make_float4(wv[4 * t], wv[4 * t + 1], wv[4 * t + 2], wv[4 * t + 3]);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 b = *reinterpret_cast<const float4*>(&ws[(16 * wid + c) * ELD + 16 * g + 4 * q]);
            float4 av[FM];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                av[i] = *reinterpret_cast<const float4*>(&xs[(16 * i + c) * ELD + 16 * g + 4 * q]);
            const float bj[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const float aj[4] = {av[i].x, av[i].y, av[i].z, av[i].w};
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(aj[j], bj[j], acc[i], 0, 0, 0);
                }
        }
        __syncthreads();
    }

    float* part = a.part ? a.part + (size_t)blockIdx.z * splitk_stride(a.M, a.N) : nullptr;
    const int n = n0 + 16 * wid + c;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * g + r;
            if (m < a.M && n < a.N) {
                if (part) part[(size_t)m * a.N + n] = acc[i][r];
                else store_any(a.y, a.y_dtype, (size_t)m * a.N + n, acc[i][r]);
            }
        }
}

// The same arithmetic for Q4 weights in whole 128-value steps (groups of 32 2^j values, or one per
// row), with loads in flight beside the math: 16 FM rows x 128 columns per block, eight waves, wave w
// owning columns 16 w .. 16 w + 15 and all rows.
//   A step is 128 values: lane (c, g) = (lane % 16, lane / 16) takes the step's 32-value chunk g of
//   column c, one 16-byte load and one scale and zero, and supplies position 32 g + t in MFMA t
//   (0 .. 31). Activations move straight into LDS (2 rows of 512 bytes per load, whole lines; 16-byte
//   chunk k of row r at slot k ^ (r % 16), so the 16 rows of a fragment read hit distinct banks),
//   three buffers, loads two steps ahead, one barrier per step.
//   What bounds it: a launch's ramp and the split-K sum at few rows, the fp32 MFMAs with more.
//   Group 32, fp32 scales and zeros (us with the sum, gemm_f32_exact on one copy of the weights / here on three
//   in turn): K = N = 4096 M = 16 26.7 / 14.6, M = 64 60.0 / 29.6; K = N = 8192, M = 64 204.8 / 79.8; K = 2048,
//   N = 600, M = 33 19.5 / 13.8.
constexpr int kRStep = 128;

template <int FM>
struct RowsShape {
    static constexpr int kBM = 16 * FM, kBN = 128;
    static constexpr int kBuf = kBM * kRStep * 4;
};

template <int FM, bool ZU>
__global__ __launch_bounds__(512, FM <= 2 ? 4 : 2) void gemm_f32_q4(GemmArgs a) {
    using S = RowsShape<FM>;
    constexpr int kLoads = FM + 2 + (ZU ? 0 : 1);  // per wave and step
    __shared__ __attribute__((aligned(16))) uint8_t lds[3 * S::kBuf];
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * S::kBN, m0 = blockIdx.y * S::kBM, n = n0 + 16 * wid + c;
    const int total = a.K / kRStep;
    const int s_first = a.part ? (int)blockIdx.z * a.split_steps : 0;
    const int nt = a.part ? min(a.split_steps, total - s_first) : total;
    const int gshift = a.group ? 31 - __builtin_clz((uint32_t)a.group >> 5) : 0;  // chunks per group, log2

    // Rows past M and columns past N read zeros through the range checks.
    const rsrc_t xr = make_rsrc(a.x, (uint32_t)((size_t)a.M * a.K * 4));
    const rsrc_t wr = make_rsrc(a.wq, (uint32_t)((size_t)a.N * a.row_bytes));
    const rsrc_t sr = make_rsrc(a.scales, (uint32_t)((size_t)a.N * a.gpr * 4));
    const rsrc_t zr = make_rsrc(ZU ? a.scales : (const void*)a.zeros, ZU ? 0u : (uint32_t)((size_t)a.N * a.gpr * 4));
    // direct load q of wave w: rows 2 (FM w + q) and the next one
    uint32_t xo[FM];
#pragma unroll
    for (int q = 0; q < FM; ++q) {
        const int r = 2 * (FM * wid + q) + (lane >> 5);
        xo[q] = (uint32_t)(m0 + r) * (uint32_t)a.K * 4u + 16u * (uint32_t)((lane & 31) ^ (r & 15));
    }
    const uint32_t wo = (uint32_t)n * (uint32_t)a.row_bytes + 16u * (uint32_t)g;
    const uint32_t so = (uint32_t)n * (uint32_t)a.gpr * 4u;
    struct W {
        v4u q;
        uint32_t s, z;
    };
    auto load = [&](W& w, int t, int buf) __attribute__((always_inline)) {
        const bool ok = t < nt;
        const uint32_t u = (uint32_t)(s_first + (ok ? t : 0)), past = ok ? 0u : 0x80000000u;
        w.q = __builtin_amdgcn_raw_buffer_load_b128(wr, wo, past + 64u * u, 0);
        const uint32_t grp = a.group ? (4u * u + (uint32_t)g) >> gshift : 0u;
        w.s = __builtin_amdgcn_raw_buffer_load_b32(sr, so + 4u * grp, past, 0);
        if constexpr (!ZU) w.z = __builtin_amdgcn_raw_buffer_load_b32(zr, so + 4u * grp, past, 0);
#pragma unroll
        for (int q = 0; q < FM; ++q) lds_dma16(xr, lds + buf * S::kBuf + 1024 * (FM * wid + q), xo[q], past + 512u * u);
    };

    // Two sums per fragment, of even and odd products, added at the end: half the chain of roundings (one sum,
    // M = 23, K = 7040, N = 1792: error against 64 bits 4.0e-7, two 2.9e-7).
    f4 acc[FM], acc_odd[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[i] = acc_odd[i] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    W w[3];
    load(w[0], 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // the first wait counts on this order
    load(w[1], 1, 1);
    auto step = [&](int t, auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        wait_vmcnt<kLoads>();  // the loads of step t + 1 may stay in flight
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load(w[(k + 2) % 3], t + 2, (k + 2) % 3);
        const float s = __builtin_bit_cast(float, w[k].s), z = ZU ? a.zero_value : __builtin_bit_cast(float, w[k].z);
        const uint8_t* const x = lds + k * S::kBuf + 512 * c;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t even = w[k].q[d] & 0x0F0F0F0Fu, odd = (w[k].q[d] >> 4) & 0x0F0F0F0Fu;
            float wf[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wf[2 * e] = ((float)((even >> (8 * e)) & 255u) - z) * s;
                wf[2 * e + 1] = ((float)((odd >> (8 * e)) & 255u) - z) * s;
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                // chunks 8 g + 2 d and the next one of row 16 i + c (read as compiler vectors: before
                // HIP's float4 the compiler waits for every direct load in flight)
                const f4 x0 = *reinterpret_cast<const f4*>(x + 8192 * i + 16 * ((8 * g + 2 * d) ^ c));
                const f4 x1 = *reinterpret_cast<const f4*>(x + 8192 * i + 16 * ((8 * g + 2 * d + 1) ^ c));
                const float xv[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[e], wf[e], acc[i], 0, 0, 0);
                    acc_odd[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[e + 1], wf[e + 1], acc_odd[i], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int t = 0;
    for (; t + 3 <= nt; t += 3) static_for<3>([&](auto kc) { step(t + decltype(kc)::value, kc); });
    static_for<2>([&](auto kc) {
        if (t + decltype(kc)::value < nt) step(t + decltype(kc)::value, kc);
    });
    wait_vmcnt<0>();

    float* part = a.part ? a.part + (size_t)blockIdx.z * splitk_stride(a.M, a.N) : nullptr;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * g + r;
            const float v = acc[i][r] + acc_odd[i][r];
            if (m < a.M && n < a.N) {
                if (part) part[(size_t)m * a.N + n] = v;
                else store_any(a.y, a.y_dtype, (size_t)m * a.N + n, v);
            }
        }
}

// The same for up to 16 rows and so few columns that 128-column blocks would need K split over the grid:
// a block owns 16 columns over all of K and its eight waves split K (wave w takes steps w, w + 8, ..), each
// with two activation buffers of its own and no barrier; the partial tiles are added in wave order
// through LDS, so there is no second launch. K = N = 4096, M = 16, three copies of the weights in turn: 12.8 us
// against 14.6 with 8 K splits and their sum; the fp32 MFMAs and the weights' decoding take 5.6 of it per
// 4,096 of K.
template <bool ZU>
__global__ __launch_bounds__(512, 2) void gemm_f32_q4_cols(GemmArgs a) {
    constexpr int kBuf = 16 * kRStep * 4, kLoads = 8 + 2 + (ZU ? 0 : 1);  // per wave and step
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) uint8_t lds[8 * 2 * kBuf];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, n = n0 + c;
    const int total = a.K / kRStep, nt = total > wid ? (total - wid + 7) / 8 : 0;
    const int gshift = a.group ? 31 - __builtin_clz((uint32_t)a.group >> 5) : 0;

    const rsrc_t xr = make_rsrc(a.x, (uint32_t)((size_t)a.M * a.K * 4));
    const rsrc_t wr = make_rsrc(a.wq, (uint32_t)((size_t)a.N * a.row_bytes));
    const rsrc_t sr = make_rsrc(a.scales, (uint32_t)((size_t)a.N * a.gpr * 4));
    const rsrc_t zr = make_rsrc(ZU ? a.scales : (const void*)a.zeros, ZU ? 0u : (uint32_t)((size_t)a.N * a.gpr * 4));
    uint32_t xo[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int r = 2 * q + (lane >> 5);
        xo[q] = (uint32_t)r * (uint32_t)a.K * 4u + 16u * (uint32_t)((lane & 31) ^ r);
    }
    const uint32_t wo = (uint32_t)n * (uint32_t)a.row_bytes + 16u * (uint32_t)g;
    const uint32_t so = (uint32_t)n * (uint32_t)a.gpr * 4u;
    uint8_t* const xb = lds + wid * 2 * kBuf;
    struct W {
        v4u q;
        uint32_t s, z;
    };
    auto load = [&](W& w, int t, int buf) __attribute__((always_inline)) {
        const bool ok = t < nt;
        const uint32_t u = ok ? (uint32_t)(wid + 8 * t) : 0u, past = ok ? 0u : 0x80000000u;
        w.q = __builtin_amdgcn_raw_buffer_load_b128(wr, wo, past + 64u * u, 0);
        const uint32_t grp = a.group ? (4u * u + (uint32_t)g) >> gshift : 0u;
        w.s = __builtin_amdgcn_raw_buffer_load_b32(sr, so + 4u * grp, past, 0);
        if constexpr (!ZU) w.z = __builtin_amdgcn_raw_buffer_load_b32(zr, so + 4u * grp, past, 0);
#pragma unroll
        for (int q = 0; q < 8; ++q) lds_dma16(xr, xb + buf * kBuf + 1024 * q, xo[q], past + 512u * u);
    };
    f4 acc[2] = {(f4){0.0f, 0.0f, 0.0f, 0.0f}, (f4){0.0f, 0.0f, 0.0f, 0.0f}};
    W w[2];
    load(w[0], 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
    auto step = [&](int t, auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        // the reads of step t - 1 have returned (its MFMAs used them), so its buffer is free
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load(w[k ^ 1], t + 1, k ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<kLoads>();  // step t's loads have landed
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const float s = __builtin_bit_cast(float, w[k].s), z = ZU ? a.zero_value : __builtin_bit_cast(float, w[k].z);
        const uint8_t* const x = xb + k * kBuf + 512 * c;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t even = w[k].q[d] & 0x0F0F0F0Fu, odd = (w[k].q[d] >> 4) & 0x0F0F0F0Fu;
            const f4 x0 = *reinterpret_cast<const f4*>(x + 16 * ((8 * g + 2 * d) ^ c));
            const f4 x1 = *reinterpret_cast<const f4*>(x + 16 * ((8 * g + 2 * d + 1) ^ c));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float we = ((float)((even >> (8 * e)) & 255u) - z) * s, wq = ((float)((odd >> (8 * e)) & 255u) - z) * s;
                const float xe = e < 2 ? x0[2 * e] : x1[2 * e - 4], xq = e < 2 ? x0[2 * e + 1] : x1[2 * e - 3];
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xe, we, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xq, wq, acc[1], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int t = 0; t < nt; t += 2) {
        step(t, std::integral_constant<int, 0>{});
        if (t + 1 < nt) step(t + 1, std::integral_constant<int, 1>{});
    }
    // every wave is done with its buffers and their direct loads have landed
    wait_vmcnt<0>();
    __syncthreads();
    f4* const red = reinterpret_cast<f4*>(lds);
    red[64 * wid + lane] = acc[0] + acc[1];
    __syncthreads();
    if (threadIdx.x < 64) {
        f4 v = red[lane];
#pragma unroll
        for (int i = 1; i < 8; ++i) v += red[64 * i + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 4 * g + r;
            if (m < a.M && n < a.N) store_any(a.y, a.y_dtype, (size_t)m * a.N + n, v[r]);
        }
    }
}

template <int FM>
void launch_f32_q4_fm(const GemmArgs& a, dim3 grid) {
    if (a.zeros) launch("gemm_f32_q4", (gemm_f32_q4<FM, false>), grid, dim3(512), 0, a);
    else launch("gemm_f32_q4", (gemm_f32_q4<FM, true>), grid, dim3(512), 0, a);
    BYHIP_LAUNCHED("gemm_f32_q4");
}

// K splits: as many as leave one block per CU, each of at least two steps (K = N = 4096, M = 16, 4 / 8 /
// 16 splits: 18.3 / 13.4 / 14.6 us).
void launch_f32_q4(GemmArgs a) {
    // Up to 16 rows on at most one 16-column block per CU (us, 128-column blocks with split K / this, three
    // copies of the weights in turn: K = N = 4096, M = 16 14.6 / 12.8, M = 4 13.5 / 12.0; K = 8192, N = 4096 20.5 / 19.6;
    // K = 2048, N = 1000 9.6 / 8.4; K = 1024, N = 512 9.4 / 6.3; past it, one copy, K = 4096, N = 6144, M = 9
    // 17.4 / 18.4).
    if (a.M <= 16 && (a.N + 15) / 16 <= compute_units() && env_int("BYHIP_Q4_SPLIT", 0) == 0) {
        const dim3 grid((unsigned)((a.N + 15) / 16));
        if (a.zeros) launch("gemm_f32_q4_cols", gemm_f32_q4_cols<false>, grid, dim3(512), 0, a);
        else launch("gemm_f32_q4_cols", gemm_f32_q4_cols<true>, grid, dim3(512), 0, a);
        BYHIP_LAUNCHED("gemm_f32_q4_cols");
        return;
    }
    const int row_tiles = (a.M + 63) / 64, fm = (a.M + 16 * row_tiles - 1) / (16 * row_tiles);
    const int rows = (a.M + 16 * fm - 1) / (16 * fm);
    const long tiles = (long)((a.N + 127) / 128) * rows;
    const int steps = a.K / kRStep;
    const int forced = env_int("BYHIP_Q4_SPLIT", 0);
    const int want = (int)std::max<long>(1, std::min<long>(compute_units() / tiles, steps / 2));
    const int splits = choose_split(a, tiles, steps, 1, forced > 0 ? forced : want, 1);
    if (splits == 1) a.part = nullptr;
    const dim3 grid((unsigned)((a.N + 127) / 128), (unsigned)rows, (unsigned)splits);
    switch (fm) {
    case 1: launch_f32_q4_fm<1>(a, grid); break;
    case 2: launch_f32_q4_fm<2>(a, grid); break;
    case 3: launch_f32_q4_fm<3>(a, grid); break;
    default: launch_f32_q4_fm<4>(a, grid); break;
    }
    if (a.part) launch_splitk_sum(a, splits);
}

template <BFormat F, bool XF32>
void launch_exact_bm(const GemmArgs& a, int bm, dim3 grid) {
    switch (bm) {
    case 16: launch("gemm_f32_exact", (gemm_f32_exact<F, XF32, 16>), grid, dim3(256), 0, a); break;
    case 32: launch("gemm_f32_exact", (gemm_f32_exact<F, XF32, 32>), grid, dim3(256), 0, a); break;
    default: launch("gemm_f32_exact", (gemm_f32_exact<F, XF32, 64>), grid, dim3(256), 0, a); break;
    }
    BYHIP_LAUNCHED("gemm_f32_exact");
}

template <BFormat F>
void launch_exact_x(const GemmArgs& a, int bm, dim3 grid) {
    if (a.x_dtype == BYHIP_F32) launch_exact_bm<F, true>(a, bm, grid);
    else launch_exact_bm<F, false>(a, bm, grid);
}

}  // namespace

bool gemm_f32_q4_ok(const GemmArgs& a) {
    constexpr uint64_t kLim = 0x80000000u;
    const int chunks = a.group >> 5;
    return a.x_dtype == BYHIP_F32 && !a.scale_f16 && a.K % kRStep == 0 &&
           (a.group == 0 || (a.group % 32 == 0 && (chunks & (chunks - 1)) == 0)) &&
           reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && reinterpret_cast<uintptr_t>(a.wq) % 16 == 0 && a.row_bytes % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a.scales) % 4 == 0 && reinterpret_cast<uintptr_t>(a.zeros) % 4 == 0 &&
           (uint64_t)(a.M + 64) * a.K * 4 < kLim && (uint64_t)(a.N + 128) * a.row_bytes < kLim &&
           (uint64_t)(a.N + 128) * a.gpr * 4 < kLim;
}

void launch_gemm_exact(BFormat fmt, const GemmArgs& a0) {
    GemmArgs a = a0;
    if (a.M <= 0 || a.N <= 0 || a.K <= 0) return;
    if (fmt != BFormat::Q4Fast && fmt != BFormat::Q4Generic && a.K % 32 != 0)
        fail("byhip: internal: the exact FP4-KM / F16 GEMM needs K %% 32 == 0 (K=%d)", a.K);
    if ((fmt == BFormat::Q4Fast || fmt == BFormat::Q4Generic) && gemm_f32_q4_ok(a)) return launch_f32_q4(a);
    const int bm = a.M <= 16 ? 16 : (a.M <= 32 ? 32 : 64);
    if ((a.M + bm - 1) / bm > 65535) fail("byhip: M=%d too large for one launch", a.M);
    const long tiles = (long)((a.N + 63) / 64) * ((a.M + bm - 1) / bm);
    const int nsteps = (a.K + EBK - 1) / EBK;
    const int splits = choose_split(a, tiles, nsteps, 4, 0, 2);
    const dim3 grid((unsigned)((a.N + 63) / 64), (unsigned)((a.M + bm - 1) / bm), (unsigned)splits);
    switch (fmt) {
    case BFormat::Fp4Km: launch_exact_x<BFormat::Fp4Km>(a, bm, grid); break;
    case BFormat::F16: launch_exact_x<BFormat::F16>(a, bm, grid); break;
    default: launch_exact_x<BFormat::Q4Generic>(a, bm, grid); break;
    }
    if (a.part) launch_splitk_sum(a, splits);
}

}  // namespace byhip
