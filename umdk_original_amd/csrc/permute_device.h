// Device code shared by the permute kernels: a wavefront, or a workgroup where there are few tokens, loads one token row,
// quantises it in registers and stores it to any number of destination rows.
//
// Reference semantics (paths relative to the reference tree):
//   quant   src/cam/comm_operator/ascend_kernels/moe_dispatch_normal/op_kernel/moe_dispatch_normal.h:278-316
//           (scale = 127/(max|x| + 1e-12)), and the fused kernel's QuantToken,
//           src/cam/comm_operator/ascend_kernels/fused_deep_moe/op_kernel/fused_deep_moe/gemm/kernel/
//           grouped_matmul_slice_m_per_token_dequant_swiglu_quant_multistage_workspace.h:780-818 (no epsilon)
//   rows    moe_dispatch_normal.h:486-535 (int8 or 16-bit row, fp32 scale and (srcRank, token, k) per row)
// QUANT 3 has no counterpart in the reference: OCP FP8 E4M3 values with one power-of-two (E8M0) scale per row
// and 128 columns, as include/cam_fp8_spec.h defines them.
#ifndef CAM_PERMUTE_DEVICE_H_
#define CAM_PERMUTE_DEVICE_H_

#include "cam_device.h"
#include "cam_kernels.h"

namespace cam {

constexpr int kDispWaves = 4;         // tokens (waves) per workgroup
constexpr int kDispMaxChunks = 14;    // 16-byte chunks per lane: H <= 14 * 64 * 8 = 7168

__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d)
{
    return (uint32_t)(a & 0xff) | ((uint32_t)(b & 0xff) << 8) | ((uint32_t)(c & 0xff) << 16) |
           ((uint32_t)(d & 0xff) << 24);
}

// 16-bit activation formats.  ACT = 0: bf16 (the upper half of an fp32); ACT = 1: IEEE fp16.
template <int ACT>
__device__ __forceinline__ float act_bits_to_f32(uint32_t bits16)
{
    if (ACT == 0) {
        return bf16_bits_to_f32(bits16);
    }
    return (float)__builtin_bit_cast(_Float16, (unsigned short)bits16);  // exact
}

// One token row held by kLanes threads (a wavefront or a workgroup): thread l owns the 16-byte chunks l, l + kLanes, ...
template <int CHUNKS, int LANES>
struct TokenRow {
    static constexpr int kChunks = CHUNKS, kLanes = LANES;
    v4u raw[CHUNKS];
    v2u q[CHUNKS];
    float scale_out;
    uint32_t scale8[CHUNKS];  // QUANT 3: E8M0 scale of the 128-column block chunk j of this thread lies in
};
typedef TokenRow<kDispMaxChunks, kWave> WaveRow;
template <int NT>
using GroupRow = TokenRow<(kDispMaxChunks * kWave + NT - 1) / NT, NT>;  // a workgroup of NT threads

// The maximum over the threads that hold a row.
struct WaveMax {
    __device__ __forceinline__ float operator()(float m) const { return wave_max(m); }
};
template <int NT>
struct GroupMax {
    float *slots;  // LDS, one per wave
    __device__ __forceinline__ float operator()(float m) const
    {
        m = wave_max(m);
        __syncthreads();  // the maxima before these have been read
        if ((threadIdx.x & (kWave - 1)) == 0) {
            slots[threadIdx.x >> 6] = m;
        }
        __syncthreads();
        m = slots[0];
#pragma unroll
        for (int w = 1; w < NT / kWave; ++w) {
            m = fmaxf(m, slots[w]);
        }
        return m;
    }
};

// Exponent x of the smallest power of two 2^x with amax / 2^x <= 448 (amax = m * 2^e: e - 8, one more when
// m > 1.75), 0 for amax == 0, clamped to [-127, 127].
__device__ __forceinline__ int fp8_block_scale_exp(float amax)
{
    const uint32_t a = __float_as_uint(amax);
    if (a == 0u) {
        return 0;
    }
    int e;
    uint32_t frac;
    if ((a >> 23) == 0u) {
        const int lead = __clz(a) - 9;  // shifts that bring the leading one to bit 22
        e = -127 - lead;
        frac = (a << (lead + 1)) & 0x7fffffu;
    } else {
        e = (int)(a >> 23) - 127;
        frac = a & 0x7fffffu;
    }
    const int x = e - 8 + (frac > 0x600000u ? 1 : 0);
    return min(max(x, -127), 127);
}

__device__ __forceinline__ float exp2_int(int x)
{
    return x >= -126 ? __uint_as_float((uint32_t)(x + 127) << 23) : __uint_as_float(0x00400000u);
}

template <typename Row>
__device__ __forceinline__ void load_token_row(const uint16_t *x, int t, int H, int lane, Row &r)
{
    const int nch = H >> 3;  // 8 values per chunk
    const v4u *src = (const v4u *)(x + (long long)t * H);
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        const int c = j * Row::kLanes + lane;
        r.raw[j] = v4u{0u, 0u, 0u, 0u};
        if (c < nch) {
            r.raw[j] = __builtin_nontemporal_load(src + c);
        }
    }
}

// FP8 with one scale per 128 columns.  Chunk c = kLanes j + lane holds columns 8c .. 8c+7, so a block of 128
// columns is the 16 chunks of lanes 16 q .. 16 q + 15 at one j: its largest magnitude is a maximum over a
// quarter of the wave.  The scaled values lie within +-448, where the hardware conversion (round to nearest
// even) needs no saturation.
template <int ACT, typename Row>
__device__ __forceinline__ void quant_token_row_fp8(Row &r)
{
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        float x[8];
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[2 * i] = act_bits_to_f32<ACT>(r.raw[j][i] & 0xffffu);
            x[2 * i + 1] = act_bits_to_f32<ACT>(r.raw[j][i] >> 16);
            m = fmaxf(m, fmaxf(fabsf(x[2 * i]), fabsf(x[2 * i + 1])));
        }
        m = row_max(m);
        const int e = fp8_block_scale_exp(m);
        r.scale8[j] = (uint32_t)(e + 127);
        const float f1 = exp2_int(-(e / 2)), f2 = exp2_int(-(e - e / 2));
        int lo = 0, hi = 0;
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[0], f1), f2), __fmul_rn(__fmul_rn(x[1], f1), f2), lo,
                                             false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[2], f1), f2), __fmul_rn(__fmul_rn(x[3], f1), f2), lo,
                                             true);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[4], f1), f2), __fmul_rn(__fmul_rn(x[5], f1), f2), hi,
                                             false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[6], f1), f2), __fmul_rn(__fmul_rn(x[7], f1), f2), hi,
                                             true);
        r.q[j] = v2u{(uint32_t)lo, (uint32_t)hi};
    }
}

// QUANT 1: scale = 127 / (max|x| + 1e-12); QUANT 2: scale = 127 / max|x|, an all-zero row giving zeros and scale 0.
template <int QUANT, int ACT, typename Row, typename Max>
__device__ __forceinline__ void quant_token_row(Row &r, const Max &row_max)
{
    if (QUANT == 3) {
        quant_token_row_fp8<ACT, Row>(r);
        return;
    }
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            m = fmaxf(m, fabsf(act_bits_to_f32<ACT>(r.raw[j][i] & 0xffffu)));
            m = fmaxf(m, fabsf(act_bits_to_f32<ACT>(r.raw[j][i] >> 16)));
        }
    }
    m = row_max(m);
    // Keep the row as its 16-bit words across the two passes: left alone, the compiler holds the 112 converted
    // floats of the maximum pass for the scaling pass (a shift each to redo) and the kernel needs a third more
    // registers.
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            asm volatile("" : "+v"(r.raw[j][i]));
        }
    }
    float s;
    bool zero_row = false;
    if (QUANT == 1) {
        s = __fdiv_rn(127.0f, __fadd_rn(m, 1e-12f));
    } else {
        zero_row = (m == 0.0f);
        s = zero_row ? 0.0f : __fdiv_rn(127.0f, m);
    }
    r.scale_out = zero_row ? 0.0f : __fdiv_rn(1.0f, s);
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        int v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = (int)rintf(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] & 0xffffu), s));
            v[2 * i + 1] = (int)rintf(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] >> 16), s));
        }
        r.q[j] = v2u{pack4(v[0], v[1], v[2], v[3]), pack4(v[4], v[5], v[6], v[7])};
    }
}

// Quantisation of one COPY of a token row under a per-expert smooth scale
// (src/cam/comm_operator/ascend_kernels/moe_dispatch_shmem/op_kernel/moe_dispatch_shmem.h:693-733):
// xf = float(x) * smooth[h] (one rounded multiply), then the no-epsilon variant on xf.  r.raw is left untouched.
template <int ACT, typename Row, typename Max>
__device__ __forceinline__ void quant_token_row_smooth(Row &r, const float *__restrict__ smooth, int H, int lane,
                                                       const Max &row_max)
{
    const int nch = H >> 3;
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        const int c = j * Row::kLanes + lane;
        if (c < nch) {
            const v4f s0 = *(const v4f *)(smooth + c * 8);
            const v4f s1 = *(const v4f *)(smooth + c * 8 + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float sa = i < 2 ? s0[2 * i] : s1[2 * i - 4], sb = i < 2 ? s0[2 * i + 1] : s1[2 * i - 3];
                m = fmaxf(m, fabsf(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] & 0xffffu), sa)));
                m = fmaxf(m, fabsf(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] >> 16), sb)));
            }
        }
    }
    m = row_max(m);
    const bool zero_row = m == 0.0f;
    const float s = zero_row ? 0.0f : __fdiv_rn(127.0f, m);
    r.scale_out = zero_row ? 0.0f : __fdiv_rn(1.0f, s);
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        const int c = j * Row::kLanes + lane;
        int v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (c < nch) {
            const v4f s0 = *(const v4f *)(smooth + c * 8);
            const v4f s1 = *(const v4f *)(smooth + c * 8 + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float sa = i < 2 ? s0[2 * i] : s1[2 * i - 4], sb = i < 2 ? s0[2 * i + 1] : s1[2 * i - 3];
                v[2 * i] = (int)rintf(__fmul_rn(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] & 0xffffu), sa), s));
                v[2 * i + 1] = (int)rintf(__fmul_rn(__fmul_rn(act_bits_to_f32<ACT>(r.raw[j][i] >> 16), sb), s));
            }
        }
        r.q[j] = v2u{pack4(v[0], v[1], v[2], v[3]), pack4(v[4], v[5], v[6], v[7])};
    }
}

// QUANT 3: one E8M0 byte per 128 columns, written by the first of its sixteen threads.
template <typename Row>
__device__ __forceinline__ void store_row_scales8(const Row &r, uint8_t *scales, long long row, int H, int lane)
{
    const int nch = H >> 3;
    uint8_t *sc = scales + row * (H >> 7);
    if ((lane & 15) == 0) {
#pragma unroll
        for (int j = 0; j < Row::kChunks; ++j) {
            const int c = j * Row::kLanes + lane;
            if (c < nch) {
                sc[c >> 4] = (uint8_t)r.scale8[j];
            }
        }
    }
}

// 16 or 8 bytes of a row; PLAIN: through the L2 like any store, else non-temporal.
template <bool PLAIN, typename T>
__device__ __forceinline__ void store_piece(T v, T *dst)
{
    if constexpr (PLAIN) {
        *dst = v;
    } else {
        __builtin_nontemporal_store(v, dst);
    }
}

// The scale (of int8 rows) and the triple of output row `row`.
template <int QUANT>
__device__ __forceinline__ void store_row_origin(float scale, float *scales, int32_t *src_info, int src_rank, long long row, int t, int k)
{
    if (QUANT == 1 || QUANT == 2) {
        scales[row] = scale;
    }
    if (src_info != nullptr) {
        src_info[3 * row + 0] = src_rank;
        src_info[3 * row + 1] = t;
        src_info[3 * row + 2] = k;
    }
}

// Stores the row (quantised or raw) to output row `row`, with the scales of an FP8 row.
template <int QUANT, bool PLAIN, typename Row>
__device__ __forceinline__ void store_token_row(const Row &r, void *out, float *scales, long long row, int H, int lane)
{
    const int nch = H >> 3;
    if (QUANT != 0) {
        v2u *dst = (v2u *)((int8_t *)out + row * H);
#pragma unroll
        for (int j = 0; j < Row::kChunks; ++j) {
            const int c = j * Row::kLanes + lane;
            if (c < nch) {
                store_piece<PLAIN>(r.q[j], dst + c);
            }
        }
    } else {
        v4u *dst = (v4u *)((uint16_t *)out + row * H);
#pragma unroll
        for (int j = 0; j < Row::kChunks; ++j) {
            const int c = j * Row::kLanes + lane;
            if (c < nch) {
                store_piece<PLAIN>(r.raw[j], dst + c);
            }
        }
    }
    if (QUANT == 3) {
        store_row_scales8(r, (uint8_t *)scales, row, H, lane);
    }
}

}  // namespace cam

#endif  // CAM_PERMUTE_DEVICE_H_
