// byhip_fp4gemv.hip - the FP4-KM decode GEMV (one row of fp32 activations, gfx950).
//
// y[n] = sum_k x[k] * lut[code] * lut[16 + scale byte] for any decode table. The work is split as in the Q4
// decode GEMV (byhip_gemv.hip): a wave owns kRows weight rows,
// lane l the 32-value groups l, l + 64, .. of each (one 16-byte load and one scale byte); every load
// goes out before the first wait, activations, scale bytes, then weights.
//
// Activations stay fp32, staged once per block in LDS as the runs of four that four bytes of a group
// multiply: low nibbles x[4 t ..], high nibbles x[16 + 4 t ..]. Where the table's 16 values are E2M1's, which
// each wave sees for itself, v_cvt_scalef32_pk_f32_fp4 turns a byte into
// twice its two values, whole numbers, so products with subnormal activations stay exact too; two
// chains of fp32 FMAs sum a group, and half its scale multiplies the sum. Where that order differs from
// the reference's x * (value * scale) by more than rounding, the group is computed element by element as
// the reference does: a sum that is not finite (activations near fp32's largest, infinities, NaNs), a
// scale whose product with 6 overflows or with 0.5 is not exact. Other tables take that form throughout,
// their values looked up in LDS (11.4 us, 51 on the general GEMM; recorded calls, which had queued every route
// behind a look at the table, 7.0 us for 19.7 with E2M1 values and 10.4 for 57.9 with others).
//
// What bounds it: K = 4096, N = 14336, 31.2 MB: 6.9 us against 6.4 for the bytes at the rate of a
// large copy (8.9 us with two fp16 terms per activation and v_dot2_f32_f16, which held 23 bits of them and
// split the row in every block; 16.0 us on gemm_planes, whose 16-row tiles and second launch one row
// cannot use).
#include "byhip_gemm.h"
#include "byhip_internal.h"
#include "byhip_kernels.h"

namespace byhip {
namespace {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kRows = 2;  // rows per wave, as the Q4 GEMV at one activation row
constexpr float kScaleMax = 0x1p125f;  // products of scales up to here with 6 are finite

__device__ constexpr uint32_t e2m1_bits(int i) {  // fp32 bits of the E2M1 value of code i
    constexpr uint32_t v[8] = {0u, 0x3F000000u, 0x3F800000u, 0x3FC00000u, 0x40000000u, 0x40400000u, 0x40800000u, 0x40C00000u};
    return v[i & 7] | (i & 8 ? 0x80000000u : 0u);
}

template <int CPL, int YT>
__global__ __launch_bounds__(256) void fp4_gemv(GemmArgs a) {
    constexpr int R = kRows;
    constexpr int XC = (CPL + 1) / 2;  // half groups a thread stages: 2 G <= 128 CPL over 256 threads
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int K = a.K, N = a.N, G = K >> 5;
    // half l (0: low nibbles, 1: high) of piece t (bytes 4 t .. 4 t + 3) of group i at float4 index
    // (2 t + l) G + i; the table
    f4* const xs = reinterpret_cast<f4*>(lds);
    float* const table = reinterpret_cast<float*>(xs + 8 * G);
    const int n0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + (tid >> 6)) * R);

    const rsrc_t wr = make_rsrc(a.blob, (uint32_t)((size_t)N * (K >> 1)));
    const rsrc_t sr = make_rsrc(a.blob + a.scale_base, (uint32_t)((size_t)N * G));
    const rsrc_t xr = make_rsrc(a.x, (uint32_t)K * 4u);

    // 1. activations: thread i takes half h = i % 2 of group i / 2, values 8 h .. 8 h + 7 and 16 more on
    uint4 xv[XC][4];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int idx = (tid + 256 * i) >> 1, h = tid & 1;
        const uint32_t off = idx < G ? 128u * (uint32_t)idx + 32u * (uint32_t)h : kOutOfRange;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            xv[i][t] = buf_load16(xr, off == kOutOfRange ? off : off + 16u * (t & 1) + 64u * (t >> 1));
    }
    const float lut_v = a.lut[16 + tid], lut_e = a.lut[tid & 15];
    // 2. scale bytes, 3. weights (streamed once: non-temporal); rows past N read zeros
    uint32_t sb[R][CPL];
    v4u wv[R][CPL];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
            sb[r][c] = __builtin_amdgcn_raw_buffer_load_b8(sr, (uint32_t)min(lane + 64 * c, G - 1), (uint32_t)min(n0 + r, N) * (uint32_t)G, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
            wv[r][c] = __builtin_amdgcn_raw_buffer_load_b128(wr, 16u * (uint32_t)min(lane + 64 * c, G - 1),
                                                             (uint32_t)min(n0 + r, N) * (uint32_t)(K >> 1), 2);
    __builtin_amdgcn_sched_barrier(0);  // every load is out before the first wait

    // 4. stage
    table[16 + tid] = lut_v;
    if (tid < 16) table[tid] = lut_e;
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int idx = (tid + 256 * i) >> 1, h = tid & 1;
        if (idx < G) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                xs[(2 * (2 * h + (t & 1)) + (t >> 1)) * G + idx] = __builtin_bit_cast(f4, xv[i][t]);
        }
    }
    __syncthreads();
    if (n0 >= N) return;
    const bool e2m1 = __all(__builtin_bit_cast(uint32_t, lut_e) == e2m1_bits(lane & 15));

    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ci = lane + 64 * c, cc = min(ci, G - 1);
        float pl[R], ph[R];
#pragma unroll
        for (int r = 0; r < R; ++r) pl[r] = ph[r] = 0.0f;
#pragma unroll
        for (int t = 0; t < (e2m1 ? 4 : 0); ++t) {
            const f4 xl = xs[2 * t * G + cc], xh = xs[(2 * t + 1) * G + cc];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t d = wv[r][c][t];
                const f32x2_t w[4] = {__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 2.0f, 0), __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 2.0f, 1),
                                      __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 2.0f, 2), __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 2.0f, 3)};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    pl[r] = fmaf(xl[q], w[q][0], pl[r]);
                    ph[r] = fmaf(xh[q], w[q][1], ph[r]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float s = table[16 + (sb[r][c] & 255u)], hs = 0.5f * s, p = pl[r] + ph[r];
            if (ci < G) {
                if (e2m1 && fabsf(s) <= kScaleMax && hs + hs == s && __builtin_isfinite(p)) {
                    acc[r] = fmaf(hs, p, acc[r]);
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const f4 xl = xs[2 * t * G + cc], xh = xs[(2 * t + 1) * G + cc];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const uint32_t b = wv[r][c][t] >> (8 * q);
                            acc[r] = fmaf(xl[q], table[b & 15u] * s, acc[r]);
                            acc[r] = fmaf(xh[q], table[(b >> 4) & 15u] * s, acc[r]);
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float v = wave_sum_lane63(acc[r]);
        if (lane == 63 && n0 + r < N) store_y<YT>(a.y, n0 + r, v);
    }
}

template <int CPL>
void launch_cpl(const GemmArgs& a) {
    const int G = a.K / 32;
    const size_t lds = (size_t)G * 128 + 272 * 4;
    const dim3 grid((a.N + 4 * kRows - 1) / (4 * kRows));
    switch (a.y_dtype) {
    case BYHIP_F32: launch("fp4_gemv", (fp4_gemv<CPL, BYHIP_F32>), grid, dim3(256), lds, a); break;
    case BYHIP_F16: launch("fp4_gemv", (fp4_gemv<CPL, BYHIP_F16>), grid, dim3(256), lds, a); break;
    default: launch("fp4_gemv", (fp4_gemv<CPL, BYHIP_BF16>), grid, dim3(256), lds, a); break;
    }
    BYHIP_LAUNCHED("fp4_gemv");
}

}  // namespace

// At most 8 groups per lane, and the staged row within 64 KB of LDS.
bool fp4_gemv_ok(const GemmArgs& a) {
    return a.M == 1 && a.x_dtype == BYHIP_F32 && a.K % 32 == 0 && a.K <= 15360 &&
           reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && reinterpret_cast<uintptr_t>(a.blob) % 16 == 0 &&
           (uint64_t)(a.N + 1) * (a.K / 2) < kOutOfRange;
}

void launch_fp4_gemv(const GemmArgs& a) {
    const int cpl = (a.K / 32 + 63) / 64;
    switch (cpl) {
    case 1: launch_cpl<1>(a); break;
    case 2: launch_cpl<2>(a); break;
    case 3: launch_cpl<3>(a); break;
    case 4: launch_cpl<4>(a); break;
    case 5: case 6: launch_cpl<6>(a); break;
    default: launch_cpl<8>(a); break;
    }
}

}  // namespace byhip
