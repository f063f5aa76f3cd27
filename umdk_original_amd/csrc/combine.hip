// Weighted un-permute and reduce back to token order (bandwidth-bound gather).
//
// Reference semantics (paths relative to the reference tree):
//   src/cam/comm_operator/ascend_kernels/moe_combine_normal/op_kernel/moe_combine_normal.h:303-338
//   src/cam/comm_operator/ascend_kernels/fused_deep_moe/op_kernel/fused_deep_moe/raw_distributed/
//   cam_moe_distribute_combine.h:726-780
// acc = 0 (fp32); for k ascending, skipping absent slots: acc = acc + (float(row) * w[t,k]) with the
// multiply and the add rounded separately; out = bf16 round-to-nearest-even of acc.
//
// Design.  The reference scatters every row into a per-(token,k) window slot and then reads the slots
// back; here the rows are gathered straight from the expert-major buffer.  A workgroup of 128
// threads owns 1024 contiguous columns of one token, so row indices and weights are uniform across
// the workgroup; each thread issues up to eight independent 16-byte row loads before it starts the
// ordered accumulation, then stores 16 bytes of bf16.  Every row byte is read exactly once.
//
// Rows quantised for the wire (src/cam/comm_operator/ascend_kernels/moe_combine_shmem/op_kernel/
// moe_combine_shmem.h, IsQuant): a row is H int8 values followed by H/8 bf16 scales, one per block of 8 columns.
//   quantise (:567-592):   m = max |x| over the block; s = m * (1/127); stored scale = bf16(s);
//                          q = int8_rne(fp16_rne(x / s)), with the unrounded s.
//   dequantise (:755-773): v = bf16_rne(float(q) * float(stored scale)), then the weighted sum as above.
// A thread of the gather owns exactly one block of 8 columns, so it reads 8 + 2 bytes per row instead of 16.
#include "cam_device.h"
#include "cam_kernels.h"

namespace cam {

namespace {

constexpr int kCombThreads = 128;
constexpr int kCombBatch = 8;
// Workgroups that share the columns of a token, 8 columns a thread.
constexpr int64_t column_segments(int64_t H) { return (H / 8 + kCombThreads - 1) / kCombThreads; }
constexpr int kScanRows = 1024;  // triples a workgroup looks through at most, 8 a thread

// Rows at or beyond *row_limit (the receive total, epRecvCounts[E-1] of moe_combine_normal.h:206-207) were
// never written by the dispatch that filled the buffers; whatever triple they hold is ignored.
__global__ void invert_src_info_kernel(const int32_t *src_info, long long A, const int32_t *row_limit, int T, int K,
                                       int32_t *slot_row)
{
    long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (row_limit != nullptr) {
        A = min(A, (long long)*row_limit);
    }
    if (r >= A) {
        return;
    }
    int t = src_info[3 * r + 1];
    int k = src_info[3 * r + 2];
    if (t >= 0 && t < T && k >= 0 && k < K) {
        slot_row[(long long)t * K + k] = (int32_t)r;
    }
}

// The row of slot (t,k), or -1: from the map, or, with BY_COUNTS, the way the SHMEM combine finds it
// (moe_combine_shmem.h:514-556,833-837): the rows of the experts before the slot's, plus its rank within the expert.
// Chosen at compile time, so that nothing is asked between the row loads of a gather.  (No difference in time that shows: dispatch
// + combine of 4096 tokens x 7168 take 150.7 to 151.2 us either way.)
template <bool BY_COUNTS>
__device__ __forceinline__ long long row_of_slot(const CombineArgs &a, long long slot)
{
    if (!BY_COUNTS) {
        return a.slot_row[slot];
    }
    // (no branch, so that the loads of a token's slots stay side by side)
    const int e = a.ids[slot];
    const int before = a.ep_send_counts[min(max(e - 1, 0), a.E - 1)];
    const long long row = (long long)(e > 0 ? before : 0) + a.expand_idx[slot];
    return e >= 0 && e < a.E ? row : -1;
}

// Rows of the activation type (ACT: 0 = bf16, 1 = IEEE fp16) -> wire rows, whose block scales are of that type
// too (moe_combine_shmem.h:567-592 keeps them as ExpandXType).  One thread per block of 8 columns.
template <int ACT>
__global__ __launch_bounds__(256) void comm_quant_kernel(const uint16_t *__restrict__ y, long long A, int H,
                                                         const int32_t *__restrict__ row_limit,
                                                         uint8_t *__restrict__ out)
{
    const int blocks_per_row = H / 8;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long row = i / blocks_per_row;
    const int b = (int)(i - row * blocks_per_row);
    const long long rows = row_limit == nullptr ? A : min(A, (long long)*row_limit);
    if (row >= rows) {
        return;
    }
    const v4u v = __builtin_nontemporal_load((const v4u *)(y + row * H + b * 8));
    float x[8];
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        x[2 * c] = ACT == 0 ? bf16_bits_to_f32(v[c] & 0xffffu) : fp16_bits_to_f32(v[c] & 0xffffu);
        x[2 * c + 1] = ACT == 0 ? bf16_bits_to_f32(v[c] >> 16) : fp16_bits_to_f32(v[c] >> 16);
        m = fmaxf(m, fmaxf(fabsf(x[2 * c]), fabsf(x[2 * c + 1])));
    }
    const long long pitch = (long long)H + H / 4;
    uint32_t q[2] = {0u, 0u};
    uint16_t sbits = 0;
    if (m != 0.0f) {
        const float s = __fmul_rn(m, 1.0f / 127.0f);
        sbits = (uint16_t)(ACT == 0 ? f32_to_bf16_bits(s) : f32_to_fp16_bits(s));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const _Float16 h = (_Float16)__fdiv_rn(x[j], s);  // round to nearest even
            const int qi = (int)rintf((float)h);
            q[j >> 2] |= (uint32_t)(qi & 0xff) << (8 * (j & 3));
        }
    }
    uint8_t *dst = out + row * pitch;
    *(v2u *)(dst + b * 8) = v2u{q[0], q[1]};
    *(uint16_t *)(dst + H + b * 2) = sbits;
}

// ACT: 0 = bf16 rows and output, 1 = IEEE fp16 (the layer's activation type).
template <int ACT>
__device__ __forceinline__ float comb_act_to_f32(uint32_t bits16)
{
    return ACT == 0 ? bf16_bits_to_f32(bits16) : fp16_bits_to_f32(bits16);
}

// SCAN: no map has been made; a workgroup looks through the triples for its token's rows by itself (the last of several that name the
// same slot).  It takes the place of invert_src_info_kernel where there are few of them (combine_scans).
template <bool WIRE, int ACT, bool BY_COUNTS, bool SCAN = false>
__global__ __launch_bounds__(kCombThreads) void combine_kernel(CombineArgs a, int segs)
{
    const int t = blockIdx.x / segs;
    const int seg = blockIdx.x - t * segs;
    const int col = (seg * kCombThreads + threadIdx.x) * 8;
    __shared__ int row_s[SCAN ? kMaxTopk : 1];
    if constexpr (SCAN) {
        int token[kScanRows / kCombThreads];
#pragma unroll
        for (int i = 0; i < kScanRows / kCombThreads; ++i) {  // all in one round trip
            const int r = i * kCombThreads + (int)threadIdx.x;
            token[i] = r < a.A ? a.src_info[3 * r + 1] : -1;
        }
        if (threadIdx.x < kMaxTopk) {
            row_s[threadIdx.x] = -1;
        }
        __syncthreads();
        const int limit = a.row_limit == nullptr ? (int)a.A : min((int)a.A, *a.row_limit);
#pragma unroll
        for (int i = 0; i < kScanRows / kCombThreads; ++i) {
            const int r = i * kCombThreads + (int)threadIdx.x;
            if (r < limit && token[i] == t) {
                const int k = a.src_info[3 * r + 2];
                if (k >= 0 && k < a.K) {
                    atomicMax(&row_s[k], r);
                }
            }
        }
        __syncthreads();
    }
    if (col >= a.H) {
        return;
    }
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        acc[j] = 0.0f;
    }
    const bool live = a.t_active == nullptr || t < *a.t_active;
    const long long rows = a.row_limit == nullptr ? a.A : min(a.A, (long long)*a.row_limit);
    const bool add_shared = live && a.shared != nullptr;
    v4u sh = {0u, 0u, 0u, 0u};
    if (add_shared) {  // requested with the routed rows, used after them
        sh = __builtin_nontemporal_load((const v4u *)(a.shared + (long long)t * a.H + col));
    }
    if (live) {
        for (int k0 = 0; k0 < a.K; k0 += kCombBatch) {
            v4u v[kCombBatch];  // WIRE: x, y = the 8 int8 values, z = the block's scale (bf16 bits)
            float w[kCombBatch];
            bool ok[kCombBatch];
#pragma unroll
            for (int j = 0; j < kCombBatch; ++j) {
                const int k = k0 + j;
                ok[j] = false;
                w[j] = 0.0f;
                v[j] = v4u{0u, 0u, 0u, 0u};
                if (k < a.K) {
                    const long long slot = (long long)t * a.K + k;
                    const long long row = SCAN ? row_s[k] : row_of_slot<BY_COUNTS>(a, slot);
                    bool good = row >= 0 && row < rows;
                    if (!SCAN && good && a.src_info != nullptr) {
                        // The inverse map is not pre-cleared: accept a row only if it names this slot.
                        good = a.src_info[3 * row + 1] == t && a.src_info[3 * row + 2] == k;
                    }
                    if (good) {
                        ok[j] = true;
                        w[j] = a.w[slot];
                        if (WIRE) {
                            const uint8_t *src = (const uint8_t *)a.y + row * ((long long)a.H + a.H / 4);
                            const v2u q = __builtin_nontemporal_load((const v2u *)(src + col));
                            const uint16_t sc = __builtin_nontemporal_load((const uint16_t *)(src + a.H) + (col >> 3));
                            v[j] = v4u{q[0], q[1], sc, 0u};
                        } else {
                            v[j] = __builtin_nontemporal_load((const v4u *)(a.y + row * a.H + col));
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < kCombBatch; ++j) {
                if (ok[j] && WIRE) {
                    const float sc = comb_act_to_f32<ACT>(v[j][2]);
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const int q = (int)(int8_t)((v[j][c >> 2] >> (8 * (c & 3))) & 0xffu);
                        // the row as it leaves the wire: rounded to the activation type (moe_combine_shmem.h:755-773)
                        const float p = __fmul_rn((float)q, sc);
                        const float x = ACT == 0 ? bf16_bits_to_f32(f32_to_bf16_bits(p))
                                                 : fp16_bits_to_f32(f32_to_fp16_bits(p));
                        acc[c] = __fadd_rn(acc[c], __fmul_rn(x, w[j]));
                    }
                } else if (ok[j]) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        float x0 = comb_act_to_f32<ACT>(v[j][c] & 0xffffu);
                        float x1 = comb_act_to_f32<ACT>(v[j][c] >> 16);
                        acc[2 * c] = __fadd_rn(acc[2 * c], __fmul_rn(x0, w[j]));
                        acc[2 * c + 1] = __fadd_rn(acc[2 * c + 1], __fmul_rn(x1, w[j]));
                    }
                }
            }
        }
    }
    if (add_shared) {  // the shared expert's row: un-weighted, after the routed rows
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            acc[2 * c] = __fadd_rn(acc[2 * c], comb_act_to_f32<ACT>(sh[c] & 0xffffu));
            acc[2 * c + 1] = __fadd_rn(acc[2 * c + 1], comb_act_to_f32<ACT>(sh[c] >> 16));
        }
    }
    v4u o;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        o[c] = ACT == 0 ? f32x2_to_bf16x2_bits(acc[2 * c], acc[2 * c + 1])
                        : f32_to_fp16_bits(acc[2 * c]) | (f32_to_fp16_bits(acc[2 * c + 1]) << 16);
    }
    __builtin_nontemporal_store(o, (v4u *)(a.out + (long long)t * a.H + col));
}

// Wire rows whose pitch keeps every 16-byte piece aligned (H a multiple of 64): a thread owns two blocks of 8
// columns and reads 16 + 4 bytes per row, the widths of the bf16 gather.  The arithmetic is that of
// combine_kernel<true>; the rebuilt values are rounded to bf16 two at a time by the hardware conversion
// (round to nearest even, subnormals kept), which is what keeps the kernel bound by memory rather than by the
// vector ALU (5.2 TB/s against 4.1 TB/s with 8 columns per thread and integer rounding).
constexpr int kWireBatch = 4;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <bool BY_COUNTS>
__global__ __launch_bounds__(kCombThreads) void combine_wire16_kernel(CombineArgs a, int segs)
{
    const int t = blockIdx.x / segs;
    const int seg = blockIdx.x - t * segs;
    const int col = (seg * kCombThreads + threadIdx.x) * 16;
    if (col >= a.H) {
        return;
    }
    float acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        acc[j] = 0.0f;
    }
    const bool live = a.t_active == nullptr || t < *a.t_active;
    const long long rows = a.row_limit == nullptr ? a.A : min(a.A, (long long)*a.row_limit);
    const long long pitch = (long long)a.H + a.H / 4;
    if (live) {
        for (int k0 = 0; k0 < a.K; k0 += kWireBatch) {
            v4u v[kWireBatch];
            uint32_t sc2[kWireBatch];
            float w[kWireBatch];
            bool ok[kWireBatch];
#pragma unroll
            for (int j = 0; j < kWireBatch; ++j) {
                const int k = k0 + j;
                ok[j] = false;
                w[j] = 0.0f;
                v[j] = v4u{0u, 0u, 0u, 0u};
                sc2[j] = 0u;
                if (k < a.K) {
                    const long long slot = (long long)t * a.K + k;
                    const long long row = row_of_slot<BY_COUNTS>(a, slot);
                    bool good = row >= 0 && row < rows;
                    if (good && a.src_info != nullptr) {
                        good = a.src_info[3 * row + 1] == t && a.src_info[3 * row + 2] == k;
                    }
                    if (good) {
                        ok[j] = true;
                        w[j] = a.w[slot];
                        const uint8_t *src = (const uint8_t *)a.y + row * pitch;
                        v[j] = __builtin_nontemporal_load((const v4u *)(src + col));
                        sc2[j] = __builtin_nontemporal_load((const uint32_t *)(src + a.H + (col >> 2)));
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < kWireBatch; ++j) {
                if (ok[j]) {
                    const float s_lo = __uint_as_float(sc2[j] << 16);
                    const float s_hi = __uint_as_float(sc2[j] & 0xffff0000u);
#pragma unroll
                    for (int c = 0; c < 16; c += 2) {
                        const int q0 = (int)(int8_t)((v[j][c >> 2] >> (8 * (c & 3))) & 0xffu);
                        const int q1 = (int)(int8_t)((v[j][c >> 2] >> (8 * ((c + 1) & 3))) & 0xffu);
                        const float sc = c < 8 ? s_lo : s_hi;
                        // one conversion instruction rounds both products to bf16 (nearest even)
                        const f32x2 p = {__fmul_rn((float)q0, sc), __fmul_rn((float)q1, sc)};
                        const f32x2 x = __builtin_convertvector(__builtin_convertvector(p, bf16x2), f32x2);
                        acc[c] = __fadd_rn(acc[c], __fmul_rn(x[0], w[j]));
                        acc[c + 1] = __fadd_rn(acc[c + 1], __fmul_rn(x[1], w[j]));
                    }
                }
            }
        }
    }
    if (live && a.shared != nullptr) {
        const v4u *sp = (const v4u *)(a.shared + (long long)t * a.H + col);
        const v4u s[2] = {__builtin_nontemporal_load(sp), __builtin_nontemporal_load(sp + 1)};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            acc[2 * c] = __fadd_rn(acc[2 * c], bf16_bits_to_f32(s[c >> 2][c & 3] & 0xffffu));
            acc[2 * c + 1] = __fadd_rn(acc[2 * c + 1], bf16_bits_to_f32(s[c >> 2][c & 3] >> 16));
        }
    }
    v4u o[2];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        o[c >> 2][c & 3] = f32x2_to_bf16x2_bits(acc[2 * c], acc[2 * c + 1]);
    }
    v4u *dst = (v4u *)(a.out + (long long)t * a.H + col);
    __builtin_nontemporal_store(o[0], dst);
    __builtin_nontemporal_store(o[1], dst + 1);
}

}  // namespace

hipError_t launch_invert_src_info(const int32_t *src_info, int64_t A, const int32_t *row_limit, int T, int K,
                                  int32_t *slot_row, hipStream_t stream)
{
    if (A <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(invert_src_info_kernel, dim3((unsigned)((A + 255) / 256)), dim3(256), 0, stream, src_info,
                       (long long)A, row_limit, T, K, slot_row);
    return hipGetLastError();
}

hipError_t launch_comm_quant(const uint16_t *y, int act_fp16, int64_t A, int H, const int32_t *row_limit,
                             uint8_t *out, hipStream_t stream)
{
    if (A <= 0) {
        return hipSuccess;
    }
    if (H % 8 != 0) {
        return hipErrorInvalidValue;
    }
    const long long n = (long long)A * (H / 8);
    const long long blocks = (n + 255) / 256;
    if (blocks > 0x7fffffffll) {
        return hipErrorInvalidValue;
    }
    if (act_fp16) {
        hipLaunchKernelGGL(comm_quant_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, stream, y, (long long)A, H,
                           row_limit, out);
    } else {
        hipLaunchKernelGGL(comm_quant_kernel<0>, dim3((unsigned)blocks), dim3(256), 0, stream, y, (long long)A, H,
                           row_limit, out);
    }
    return hipGetLastError();
}

template <bool BY_COUNTS>
static hipError_t launch_combine_as(const CombineArgs &a, hipStream_t stream)
{
    if (a.T <= 0) {
        return hipSuccess;
    }
    if (a.H % 8 != 0) {
        return hipErrorInvalidValue;
    }
    const int segs = (int)column_segments(a.H);
    const long long blocks = (long long)a.T * segs;
    if (blocks > 0x7fffffffll) {
        return hipErrorInvalidValue;
    }
    if (a.wire_rows && a.act_fp16) {
        hipLaunchKernelGGL((combine_kernel<true, 1, BY_COUNTS>), dim3((unsigned)blocks), dim3(kCombThreads), 0, stream, a, segs);
    } else if (a.wire_rows && a.H % 64 == 0) {
        const int segs16 = (a.H / 16 + kCombThreads - 1) / kCombThreads;
        hipLaunchKernelGGL(combine_wire16_kernel<BY_COUNTS>, dim3((unsigned)(a.T * segs16)), dim3(kCombThreads), 0, stream, a,
                           segs16);
    } else if (a.wire_rows) {
        hipLaunchKernelGGL((combine_kernel<true, 0, BY_COUNTS>), dim3((unsigned)blocks), dim3(kCombThreads), 0, stream, a, segs);
    } else if (a.act_fp16) {
        hipLaunchKernelGGL((combine_kernel<false, 1, BY_COUNTS>), dim3((unsigned)blocks), dim3(kCombThreads), 0, stream, a, segs);
    } else {
        hipLaunchKernelGGL((combine_kernel<false, 0, BY_COUNTS>), dim3((unsigned)blocks), dim3(kCombThreads), 0, stream, a, segs);
    }
    return hipGetLastError();
}

// A combine of few rows is as long as its launches.  us, layout + dispatch + combine, with the map / without: one token x 4096, top-8 34.6 /
// 30.7, 64 x 2048, top-4 31.5 / 27.8, 100 x 4096, top-6 35.1 / 31.2, 128 x 7168, top-8 50.5 / 46.8 (1024 rows), 1000 x 1024, top-1
// 32.4 / 28.9.  A thread's triples are one round trip to the L2; with more of them, each workgroup reading all, the launch that is
// saved costs less.  So it does with many workgroups that hardly do anything else: combine alone in a graph, top-1, 1024 x 1024 5.0 / 3.5,
// 1024 x 4096 6.7 / 5.9, 800 x 7168 7.8 / 7.5, 1024 x 5120 7.7 / 7.6, 1024 x 6144 8.4-8.8 / 8.6, 1024 x 7168 9.3 / 10.1; top-2, 512 x
// 7168 7.5 / 6.9.
bool combine_scans(int64_t T, int64_t K, int64_t A, int64_t H)
{
    return A > 0 && A <= kScanRows && K <= kMaxTopk && T * K <= kScanRows &&
           T * column_segments(H) * A <= 5ll * kScanRows * kScanRows;
}

hipError_t launch_combine(const CombineArgs &a, hipStream_t stream)
{
    if (a.ids == nullptr && a.slot_row == nullptr) {
        if (a.src_info == nullptr || a.wire_rows || !combine_scans(a.T, a.K, a.A, a.H) || a.H % 8 != 0) {
            return hipErrorInvalidValue;
        }
        if (a.T <= 0) {
            return hipSuccess;
        }
        const int segs = (int)column_segments(a.H);
        const dim3 grid((unsigned)(a.T * segs)), block(kCombThreads);
        if (a.act_fp16) {
            hipLaunchKernelGGL((combine_kernel<false, 1, false, true>), grid, block, 0, stream, a, segs);
        } else {
            hipLaunchKernelGGL((combine_kernel<false, 0, false, true>), grid, block, 0, stream, a, segs);
        }
        return hipGetLastError();
    }
    return a.ids != nullptr ? launch_combine_as<true>(a, stream) : launch_combine_as<false>(a, stream);
}

}  // namespace cam
