// byhip_fp4gemv.hip - the FP4-KM decode GEMV (one row of fp32 activations, gfx950).
//
// y[n] = sum_k x[k] * lut[code] * lut[16 + scale byte] for tables whose 16 values are E2M1's. Work
// split and arithmetic follow the Q4 decode GEMV (byhip_gemv.hip): a wave owns kRows weight rows,
// lane l the 32-value groups l, l + 64, .. of each (one 16-byte load and one scale byte); every load
// goes out before the first wait, activations, scale bytes, then weights.
//
// Activations: each 32-value group is brought onto fp16's range by an exact power of two and split
// into fp16 hi + lo (about 23 bits of x over the whole fp32 range), staged once per block in LDS as
// the pairs (x[j], x[j + 16]) that byte j of a group multiplies. v_cvt_scalef32_pk_f16_fp4 turns a
// byte into its two values, two v_dot2_f32_f16 multiply them (exact products, fp32 sums), and the
// group's sum is scaled in fp32 by lut[16 + byte] and the power of two. A scale that is not finite
// multiplies element by element, as the reference does, so its NaNs and infinities come out alike.
//
// What bounds it: K = 4096, N = 14336, 31.2 MB: 9.0 us against 6.4 for the bytes at the rate of a
// large copy (16.0 us on gemm_planes, whose 16-row tiles and second launch one row cannot use); the
// rest is each block's staging of x and a launch's ramp, as in the Q4 GEMV.
#include "byhip_gemm.h"
#include "byhip_internal.h"
#include "byhip_kernels.h"

namespace byhip {
namespace {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kRows = 2;  // rows per wave, as the Q4 GEMV at one activation row

template <int CPL, int YT>
__global__ __launch_bounds__(256) void fp4_gemv(GemmArgs a) {
    if (a.gate && *a.gate != a.gate_want) return;  // another route was chosen (whole grid)
    constexpr int R = kRows;
    constexpr int XC = (CPL + 1) / 2;  // half groups a thread stages: 2 G <= 128 CPL over 256 threads
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int K = a.K, N = a.N, G = K >> 5;
    // piece t (bytes 4 t .. 4 t + 3's pairs) of group i at uint4 index t G + i, hi then lo; the groups'
    // back-scales; the scale table
    uint4* const xh = reinterpret_cast<uint4*>(lds);
    uint4* const xl = xh + 4 * G;
    float* const back = reinterpret_cast<float*>(xl + 4 * G);
    float* const table = back + G;
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
    const float lut_v = a.lut[16 + tid];
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

    // 4. stage: the two lanes of a group share its maximum
    table[tid] = lut_v;
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        const int idx = (tid + 256 * i) >> 1, h = tid & 1;
        if (idx < G) {
            float v[16];  // x[8 h + e] and x[16 + 8 h + e]
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v[4 * t] = __builtin_bit_cast(float, xv[i][t].x);
                v[4 * t + 1] = __builtin_bit_cast(float, xv[i][t].y);
                v[4 * t + 2] = __builtin_bit_cast(float, xv[i][t].z);
                v[4 * t + 3] = __builtin_bit_cast(float, xv[i][t].w);
            }
            float mx = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = fmaxf(mx, fabsf(v[e]));
            mx = fmaxf(mx, __shfl_xor(mx, 1, kWave));
            const int sh = fp16_range_shift(mx);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float u = __builtin_amdgcn_ldexpf(v[4 * j + q], sh), w = __builtin_amdgcn_ldexpf(v[8 + 4 * j + q], sh);
                    const _Float16 hu = (_Float16)u, hw = (_Float16)w;
                    const _Float16 lu = (_Float16)(__builtin_isinf(u) ? 0.0f : u - (float)hu);
                    const _Float16 lw = (_Float16)(__builtin_isinf(w) ? 0.0f : w - (float)hw);
                    hi[q] = (uint32_t)h_bits(hu) | ((uint32_t)h_bits(hw) << 16);
                    lo[q] = (uint32_t)h_bits(lu) | ((uint32_t)h_bits(lw) << 16);
                }
                xh[(2 * h + j) * G + idx] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                xl[(2 * h + j) * G + idx] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            }
            if (h == 0) back[idx] = __builtin_amdgcn_ldexpf(1.0f, -sh);
        }
    }
    __syncthreads();
    if (n0 >= N) return;

    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ci = lane + 64 * c, cc = min(ci, G - 1);
        float p[R];
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint4 hq = xh[t * G + cc], lq = xl[t * G + cc];
            const uint32_t hp[4] = {hq.x, hq.y, hq.z, hq.w}, lp[4] = {lq.x, lq.y, lq.z, lq.w};
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t d = wv[r][c][t];
                const h2 w[4] = {__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 0), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 1),
                                 __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 2), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.0f, 3)};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    p[r] = __builtin_amdgcn_fdot2(bits_h2(hp[q]), w[q], p[r], false);
                    p[r] = __builtin_amdgcn_fdot2(bits_h2(lp[q]), w[q], p[r], false);
                }
            }
        }
        const float b = back[cc];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float s = table[sb[r][c] & 255u];
            if (ci < G) {
                if (__builtin_isfinite(s)) {
                    acc[r] = fmaf(s, p[r] * b, acc[r]);
                } else {
                    const float* const x = static_cast<const float*>(a.x) + 32 * (size_t)ci;
#pragma unroll 1
                    for (int j = 0; j < 16; ++j) {
                        const uint32_t w4 = j < 4 ? wv[r][c][0] : j < 8 ? wv[r][c][1] : j < 12 ? wv[r][c][2] : wv[r][c][3];
                        const h2 w = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w4 >> (8 * (j & 3)), 1.0f, 0);
                        acc[r] = fmaf(x[j], (float)w[0] * s, acc[r]);
                        acc[r] = fmaf(x[j + 16], (float)w[1] * s, acc[r]);
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
    const size_t lds = (size_t)G * 128 + (size_t)G * 4 + 256 * 4;
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
