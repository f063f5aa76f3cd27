// Device-side helpers shared by the CAM kernels (gfx950, 64-wide wavefronts).
#ifndef CAM_DEVICE_H_
#define CAM_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cam {

constexpr int kWave = 64;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16)
{
    return __uint_as_float(bits16 << 16);
}

// Round-to-nearest-even fp32 -> bf16 bit pattern (NaN stays a quiet NaN).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f)
{
    const uint32_t u = __float_as_uint(f);
    const uint32_t rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    const uint32_t quiet = (u >> 16) | 0x0040u;
    return (u & 0x7fffffffu) > 0x7f800000u ? quiet : rounded;  // both sides computed: a select, no branch
}

// Two fp32 values -> two bf16 bit patterns (lo in bits 0..15) with ONE hardware conversion instruction.  Its results
// equal f32_to_bf16_bits on every one of the 2^32 inputs, NaNs included (checked exhaustively on the GPU by
// camCalibBf16Conversion and tests/test_gpu_gemm.py); it takes one vector instruction where the arithmetic form
// takes nine per value.
typedef float cam_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 cam_bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f32x2_to_bf16x2_bits(float lo, float hi)
{
    const cam_f32x2 p = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, cam_bf16x2));
}

// Round-to-nearest-even fp32 -> IEEE fp16 bit pattern (the hardware conversion; overflow gives infinity).
__device__ __forceinline__ uint32_t f32_to_fp16_bits(float f)
{
    return (uint32_t)__builtin_bit_cast(unsigned short, (_Float16)f);
}

__device__ __forceinline__ float fp16_bits_to_f32(uint32_t bits16)
{
    return (float)__builtin_bit_cast(_Float16, (unsigned short)bits16);  // exact
}

__device__ __forceinline__ int lane_id()
{
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// Reductions and scans across the lanes of a wave go through the data-parallel primitives of the vector ALU: a lane reads a
// neighbour's register in the instruction that combines the two, a few cycles a step, where a shuffle through the LDS
// crossbar takes about a hundred.  Every lane of the wave has to be active.
constexpr int kDppRowShr = 0x110;      // + n: lane i reads lane i - n of its row of sixteen
constexpr int kDppRowRor = 0x120;      // + n: rotation by n inside the row
constexpr int kDppRowBcast15 = 0x142;  // lane 15 of every row to the whole next row
constexpr int kDppRowBcast31 = 0x143;  // lane 31 to rows 2 and 3
constexpr int kDppSwapPairs = 0xb1;    // lane i reads lane i ^ 1
constexpr int kDppSwapQuads = 0x4e;    // i ^ 2
constexpr int kDppHalfMirror = 0x141;  // 7 - i of each eight
constexpr int kDppMirror = 0x140;      // 15 - i of each sixteen

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp(int none, int v)  // `none` where there is no lane to read, or the row is not in ROWS
{
    return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);
}

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp_max(float v)
{
    return fmaxf(v, __int_as_float(dpp<CTRL, ROWS>(__float_as_int(v), __float_as_int(v))));
}

// Maximum over the sixteen lanes of a row, in all of them.
__device__ __forceinline__ float row_max(float v)
{
    v = dpp_max<kDppRowRor + 8>(v);
    v = dpp_max<kDppRowRor + 4>(v);
    v = dpp_max<kDppRowRor + 2>(v);
    return dpp_max<kDppRowRor + 1>(v);
}

// Maximum over aligned groups of n lanes (a power of two, wave-uniform), in all of them.
__device__ __forceinline__ float group_max(float v, int n)
{
    v = n > 1 ? dpp_max<kDppSwapPairs>(v) : v;
    v = n > 2 ? dpp_max<kDppSwapQuads>(v) : v;
    v = n > 4 ? dpp_max<kDppHalfMirror>(v) : v;
    v = n > 8 ? dpp_max<kDppMirror>(v) : v;
    for (int off = 16; off < n; off <<= 1) {
        v = fmaxf(v, __shfl_xor(v, off, kWave));
    }
    return v;
}

__device__ __forceinline__ float wave_max(float v)
{
    v = row_max(v);
    v = dpp_max<kDppRowBcast15, 0xa>(v);
    v = dpp_max<kDppRowBcast31, 0xc>(v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), kWave - 1));
}

// Inclusive scan across the 64 lanes of a wave.
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    v += dpp<kDppRowShr + 1>(0, v);
    v += dpp<kDppRowShr + 2>(0, v);
    v += dpp<kDppRowShr + 4>(0, v);
    v += dpp<kDppRowShr + 8>(0, v);
    v += dpp<kDppRowBcast15, 0xa>(0, v);
    return v + dpp<kDppRowBcast31, 0xc>(0, v);
}

// The last lane's value of such a scan, in all of them.
__device__ __forceinline__ int wave_last(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }

__device__ __forceinline__ int wave_sum(int v) { return wave_last(wave_inclusive_scan(v)); }

}  // namespace cam

#endif  // CAM_DEVICE_H_
