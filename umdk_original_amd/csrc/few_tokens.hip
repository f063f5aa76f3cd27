// The int8 and FP8 layers for a handful of tokens in two launches: their routing and quantisation in the gate/up GEMM, the re-quantisation
// and the weighted sum in the down GEMM.
//
// Same operands and results as the launches of dispatch.hip, stream_gemm.hip and combine.hip (the reference's stages, cited there): int8 bit
// for bit, FP8 with the fp32 sums of a column added in another order.
//
// What bounds it: the weights of the experts that the tokens name, 151 MB for one token of a layer of H 4096, I 1536, top-8, which
// take 23 us at the rate that streams reach; each of the four launches it was before (plan and permute, gate/up, down,
// combine) began and ended with several microseconds in which no weight moved.  With so few (token, k) slots every workgroup can
// find out by itself what the launches in front of it and behind it were for:
//   * gate/up: a workgroup of eight waves is 16 gate and 16 up columns of one expert.  It reads the ids (at most 32), asks for its
//     first weights as soon as it knows its expert, and quantises the expert's tokens to LDS while they are on their way.
//   * down: a workgroup of eight waves is 16 output columns of ALL slots, so the weighted sum over a token's slots needs no other
//     workgroup.  It quantises the fp32 products of every slot (192 KB at most, out of L2) while its first weights are on
//     their way.
// 16 columns, half of what the weights are packed by, because the shapes leave few workgroups otherwise: 768 and 256 in the example, whose
// launches take 20.0 and 13.0 us under the tracer (four before: 5.0 + 19.7 + 13.0 + 4.5), the layer 32.0 us (43.0).  Waves per gate/up
// workgroup and K steps in flight per wave, layer of one token / of four: 4 and 16 36.5 / 111.9 us, 4 and 8 33.5 / 103.6, 4 and 4 32.8 / 101.9, 8 and
// 8 36.1 / 110.8, 8 and 3, as built, 32.9 / 101.7: few loads to a wave, which leave room for more waves to a CU, beat many.
// The four lanes of a column then hold the four 16-byte quarters of a 64-byte K step, which is what v_mfma_i32_16x16x64_i8 takes;
// its sixteen rows are the expert's tokens (eight at most), the last of them repeated.  FP8 steps are 128 bytes of K, one block of scales:
// a lane holds 32 bytes of its column, which is what v_mfma_scale_f32_16x16x128_f8f6f4 takes.
#include <algorithm>

#include "cam_device.h"
#include "cam_kernels.h"
#include "permute_device.h"
#include "../../include/cam_expf_spec.h"

namespace cam {

namespace {

constexpr int kUpThreads = 512, kUpWaves = kUpThreads / kWave;
constexpr int kDownThreads = 512, kDownWaves = kDownThreads / kWave;
constexpr int kColumns = 16;   // of a workgroup: product columns, or output columns
constexpr int kUpRing = 3;     // 64-byte K steps in flight per wave
constexpr int kDownRing = 8;   // (12: layer of one token +0.6 us)
constexpr int kFewRowBytes = 49152;  // int8 rows in LDS
constexpr int kFewMaxI = 3072;          // products of a row in the registers of a wave

template <bool FP8>
struct Form {
    typedef v4i Weights;    // a lane's share of a step of 16 columns
    typedef v4i Sum;
    typedef int One;
    static constexpr int kStep = 64;   // K bytes
    static __device__ __forceinline__ v4i multiply(v4i w, v4i x, v4i sum, int, int)
    {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x, sum, 0, 0, 0);
    }
};
template <>
struct Form<true> {
    typedef v8i Weights;
    typedef v4f Sum;
    typedef float One;
    static constexpr int kStep = 128;
    static __device__ __forceinline__ v4f multiply(v8i w, v8i x, v4f sum, int w_scale, int x_scale)
    {
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, sum, 0, 0, 0, w_scale, 0, x_scale);
    }
};

__device__ __forceinline__ void lds_barrier()
{
    // LDS traffic of this wave is done, weight loads stay in flight (a __syncthreads would drain them)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Who goes where, found by every wave: lane i is slot i = token * K + k.  An expert has a row for every token that names it; the
// slots of a token that names it more than once share the row of the first of them.
struct Slots {
    int id;                    // the slot's expert, -1 where it has none
    unsigned long long peers;  // slots of the same expert
    int row_slot;              // the slot whose row this one's is
    unsigned long long rows;   // the slots that have a row of their own
    unsigned long long first;  // the first slot of every expert that has any

    __device__ __forceinline__ Slots(const FewTokensArgs &a, int loaded_id)
    {
        const int lane = lane_id();
        int active = a.T;
        if (a.mask != nullptr) {  // their number is the active prefix
            active = 0;
            for (int t = 0; t < a.T; ++t) {
                active += a.mask[t] != 0 ? 1 : 0;
            }
        }
        id = lane < active * a.K && loaded_id >= 0 && loaded_id < a.E ? loaded_id : -1;
        peers = 0;
        for (int i = 0; i < a.T * a.K; ++i) {
            peers |= __builtin_amdgcn_readlane(id, i) == id ? 1ull << i : 0ull;
        }
        const int token = lane / a.K;
        row_slot = __ffsll(peers & (((1ull << a.K) - 1) << (min(token, a.T - 1) * a.K))) - 1;
        rows = __ballot(id >= 0 && row_slot == lane);
        first = __ballot(id >= 0 && (peers & ((1ull << lane) - 1ull)) == 0);
    }

    static __device__ __forceinline__ int load(const FewTokensArgs &a)
    {
        const int lane = lane_id();
        return a.ids[min(lane, a.T * a.K - 1)];
    }

    __device__ __forceinline__ int experts() const { return __popcll(first); }

    // The first slot of expert number j of those that have any.
    __device__ __forceinline__ int first_slot(int j) const
    {
        unsigned long long rest = first;
        for (int i = 0; i < j; ++i) {
            rest &= rest - 1;
        }
        return __builtin_amdgcn_readfirstlane(__ffsll(rest) - 1);
    }

    __device__ __forceinline__ int expert_of(int slot) const { return __builtin_amdgcn_readlane(id, slot); }

    // The slots whose rows are those of the slot's expert, one per token.
    __device__ __forceinline__ unsigned long long rows_of(int slot) const
    {
        const unsigned lo = __builtin_amdgcn_readlane((unsigned)peers, slot);
        const unsigned hi = __builtin_amdgcn_readlane((unsigned)(peers >> 32), slot);
        return (((unsigned long long)hi << 32) | lo) & rows;
    }
};

// The slot of row n of an expert's rows; beyond them the last one's.
__device__ __forceinline__ int nth_slot(unsigned long long rows, int n)
{
    const int count = __popcll(rows);
    for (int i = 0; i < count - 1; ++i) {
        rows &= i < n ? rows - 1 : ~0ull;
    }
    return __ffsll(rows) - 1;
}

// Where 16 columns of packed weights lie: lane l of a wave takes column l % 16 and quarter l / 16 of a step of K.
template <bool FP8>
struct WeightColumns {
    const int8_t *base;  // of the 64-column group
    int lane_offset;     // this lane's first 16 bytes in a step (FP8: its other 16 lie 512 bytes on)
    int step;            // bytes from one step to the next
    // 16-column part `part` (0 .. 3) of group nw of [Kd, N]
    __device__ __forceinline__ WeightColumns(const int8_t *w, int Kd, int N, int nw, int part)
    {
        const int b8 = nw >> 3, q = lane_id() >> 4, c = (part & 1) * 16 + (lane_id() & 15);
        const int step64 = min(8, N / 64 - 8 * b8) * 4096;
        base = w + (long long)b8 * 8 * Kd * 64 + (nw & 7) * 4096;
        if (FP8) {
            lane_offset = (q >> 1) * step64 + (q & 1) * 2048 + (part >> 1) * 1024 + c * 16;
            step = 2 * step64;
        } else {
            lane_offset = (q >> 1) * 2048 + (part >> 1) * 1024 + ((q & 1) * 32 + c) * 16;
            step = step64;
        }
    }
};

// This lane's share of step t; a step that is not there fetches nothing and gives zeros.
template <bool FP8>
__device__ __forceinline__ typename Form<FP8>::Weights load_weights(const int8_t *base, int lane_offset, int at, bool there)
{
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, there ? 0x7fffffff : 0, 0x00020000);
    const v4i lo = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_offset, at, 2));
    if constexpr (FP8) {
        const v4i hi = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_offset + 512, at, 2));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
        return lo;
    }
}

template <bool FP8, int ACT>
__global__ __launch_bounds__(kUpThreads, 4) void few_tokens_up_kernel(FewTokensArgs a)
{
    typedef Form<FP8> F;
    extern __shared__ __attribute__((aligned(16))) int8_t rows_s[];  // [T][H]
    __shared__ __attribute__((aligned(16))) typename F::Sum part_s[kUpWaves][2][kWave];
    __shared__ float scale_s[kFewTokens];
    __shared__ uint8_t scale8_s[kFewTokens][kFewMaxH / 128];
    __shared__ float max_s[2][kUpWaves];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, I = a.I;
    const int blocks = I / kColumns;
    const int loaded_id = Slots::load(a);
    // A row of the expert at a time is quantised by all threads; the first kRowsAhead of them are asked for together.  (one token: its
    // row, without a look at the ids)
    constexpr int kRowsAhead = 4;
    typedef TokenRow<(kFewMaxH / 8 + kUpThreads - 1) / kUpThreads, kUpThreads> Row;
    v4u raw[kRowsAhead][Row::kChunks];
    auto load_row = [&](v4u (&dst)[Row::kChunks], int token, bool there) {
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)(a.x + (long long)token * H), 0, there ? H * 2 : 0, 0x00020000);
#pragma unroll
        for (int i = 0; i < Row::kChunks; ++i) {
            dst[i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (i * kUpThreads + tid) * 16, 0, 0));
        }
    };
    if (a.T == 1) {
        load_row(raw[0], 0, true);
    }
    const Slots slots(a, loaded_id);

    if (blockIdx.x == gridDim.x - 1) {  // tokens per expert
        __shared__ int count_s[kMaxExperts];
        for (int e = tid; e < a.E; e += kUpThreads) {
            count_s[e] = 0;
        }
        __syncthreads();
        if (wave == 0 && ((slots.first >> lane) & 1) != 0) {
            count_s[slots.id] = __popcll(slots.peers);
        }
        __syncthreads();
        for (int e = tid; e < a.E; e += kUpThreads) {
            a.tokens_per_expert[e] = count_s[e];
        }
        return;
    }

    const int j = (int)blockIdx.x / blocks;
    const int c0 = ((int)blockIdx.x - j * blocks) * kColumns;   // first product column
    if (j >= slots.experts()) {
        return;
    }
    const int lead = slots.first_slot(j);
    const int g = slots.expert_of(lead);
    const unsigned long long row_slots = slots.rows_of(lead);
    const int rows = __popcll(row_slots);   // T at most
    if (a.T > 1) {
#pragma unroll
        for (int n = 0; n < kRowsAhead; ++n) {
            load_row(raw[n], __builtin_amdgcn_readfirstlane(nth_slot(row_slots, n)) / a.K, n < rows);
        }
    }

    // a packed group holds 32 gate columns, then their 32 up columns
    const int nw = c0 >> 5, half = (c0 >> 4) & 1;
    const int8_t *w = a.per_expert ? a.list.w[g] : a.w + (long long)g * H * 2 * I;
    const float *ws = a.per_expert ? a.list.s[g] : a.w_scale + (long long)g * 2 * I;
    const WeightColumns<FP8> gate(w, H, 2 * I, nw, half), up(w, H, 2 * I, nw, 2 + half);
    const int KT = H / F::kStep;
    float gate_scale = 0.0f, up_scale = 0.0f;
    int block_scales[2] = {0, 0};   // FP8: lane kb holds those of K block kb
    if constexpr (FP8) {
        const int nblk = (2 * I) >> 7;
        const uint8_t *s8 = a.w_scale8 + ((long long)g * KT + min(lane, KT - 1)) * nblk;
        block_scales[0] = s8[c0 >> 7];
        block_scales[1] = s8[(I + c0) >> 7];
    } else {
        gate_scale = ws[c0 + (tid & 15)];
        up_scale = ws[I + c0 + (tid & 15)];
    }
    constexpr int kRing = FP8 ? (kUpRing + 1) / 2 : kUpRing;
    typename F::Weights ring[kRing][2];
    auto issue = [&](int i, int q) {
        const int t = wave + kUpWaves * q;
        ring[i][0] = load_weights<FP8>(gate.base, gate.lane_offset, t * gate.step, t < KT);
        ring[i][1] = load_weights<FP8>(gate.base, up.lane_offset, t * gate.step, t < KT);
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i) {
        issue(i, i);
    }

    struct Max {
        float *slots;
        __device__ __forceinline__ float operator()(float m) const
        {
            m = wave_max(m);
            if (lane_id() == 0) {
                slots[threadIdx.x >> 6] = m;
            }
            lds_barrier();
            m = slots[0];
#pragma unroll
            for (int w = 1; w < kUpWaves; ++w) {
                m = fmaxf(m, slots[w]);
            }
            return m;
        }
    };
    auto quantise = [&](int n, const v4u (&v)[Row::kChunks]) {
        Row r;
#pragma unroll
        for (int i = 0; i < Row::kChunks; ++i) {
            r.raw[i] = v[i];
        }
        quant_token_row<FP8 ? 3 : 2, ACT>(r, Max{max_s[n & 1]});  // (in turns: the maxima before have been read when a slot comes up again)
#pragma unroll
        for (int i = 0; i < Row::kChunks; ++i) {
            const int c = i * kUpThreads + tid;
            if (c < H >> 3) {
                *(v2u *)(rows_s + n * H + c * 8) = r.q[i];
            }
        }
        if (FP8) {
            store_row_scales8(r, scale8_s[n], 0, H, tid);
        } else if (tid == 0) {
            scale_s[n] = r.scale_out;
        }
    };
#pragma unroll
    for (int n = 0; n < kRowsAhead; ++n) {
        if (n < rows) {
            quantise(n, raw[n]);
        }
    }
    for (int n = kRowsAhead; n < rows; ++n) {
        load_row(raw[0], __builtin_amdgcn_readfirstlane(nth_slot(row_slots, n)) / a.K, true);
        quantise(n, raw[0]);
    }
    lds_barrier();

    typename F::Sum sum[2] = {typename F::Sum{}, typename F::Sum{}};
    const int row = min(lane & 15, rows - 1);
    const int8_t *mine = rows_s + row * H + (lane >> 4) * (F::kStep / 4);
    for (int q = 0; wave + kUpWaves * q < KT; q += kRing) {
#pragma unroll
        for (int i = 0; i < kRing; ++i) {
            const int t = min(wave + kUpWaves * (q + i), KT - 1);
            const typename F::Weights x = *(const typename F::Weights *)(mine + t * F::kStep);
            int sx = 0, sw[2] = {0, 0};
            if constexpr (FP8) {
                sx = scale8_s[row][t];
                sw[0] = __builtin_amdgcn_readlane(block_scales[0], t);
                sw[1] = __builtin_amdgcn_readlane(block_scales[1], t);
            }
            sum[0] = F::multiply(ring[i][0], x, sum[0], sw[0], sx);
            sum[1] = F::multiply(ring[i][1], x, sum[1], sw[1], sx);
            issue(i, q + i + kRing);
        }
    }
    part_s[wave][0][lane] = sum[0];
    part_s[wave][1][lane] = sum[1];
    lds_barrier();
    // lane l of a sum holds row l % 16 and columns 4 (l / 16) .. + 3; here a thread is row tid / 16 and column tid % 16
    const int n = tid >> 4, c = tid & 15;
    if (n >= rows) {
        return;
    }
    typename F::One sg = 0, su = 0;   // (in the order of the waves)
#pragma unroll
    for (int v = 0; v < kUpWaves; ++v) {
        sg += ((const typename F::One *)&part_s[v][0][(c >> 2) * 16 + n])[c & 3];
        su += ((const typename F::One *)&part_s[v][1][(c >> 2) * 16 + n])[c & 3];
    }
    float tg = sg, tu = su;
    if constexpr (!FP8) {  // (FP8 sums carry their scales already)
        const float xs = scale_s[n];
        tg = __fmul_rn(__fmul_rn((float)sg, gate_scale), xs);
        tu = __fmul_rn(__fmul_rn((float)su, up_scale), xs);
    }
    a.products[(long long)nth_slot(row_slots, n) * I + c0 + c] = __fmul_rn(cam_silu_spec(tg), tu);
}

// RW: slots whose products a wave quantises.
template <bool FP8, int ACT, int RW>
__global__ __launch_bounds__(kDownThreads, RW == 1 ? 4 : 2) void few_tokens_down_kernel(FewTokensArgs a)
{
    typedef Form<FP8> F;
    constexpr int kParts = FP8 ? kDownWaves : 1;   // FP8 sums are added in the order of the waves
    constexpr int kBlocks = kFewRowBytes / 128;
    extern __shared__ __attribute__((aligned(16))) int8_t rows_s[];  // [slots][I]
    __shared__ typename F::One sum_s[kParts][kFewSlots][kColumns];
    __shared__ float column_s[FP8 ? 1 : kFewSlots][kColumns];   // the scale of the slot's expert for each column
    __shared__ uint8_t x_scale8_s[FP8 ? kBlocks : 1], w_scale8_s[FP8 ? kBlocks : 1];   // [slots][I / 128], of the slot's expert
    __shared__ float scale_s[kFewSlots], weight_s[kFewSlots];
    __shared__ int row_s[kFewSlots];   // the slot whose sums are this one's, -1 where it has no expert
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, I = a.I, A = a.T * a.K;
    const int c0 = (int)blockIdx.x * kColumns;
    const int loaded_id = Slots::load(a);
    // Products of RW slots per wave at a time, whether they have an expert or not: nobody looks at what the others leave.
    constexpr int kQuads = kFewMaxI / 4 / kWave;
    v4f prod[RW][kQuads];
    auto load_products = [&](int first) {
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const int slot = min(first + wave + i * kDownWaves, A - 1);
            const __amdgpu_buffer_rsrc_t rsrc =
                __builtin_amdgcn_make_buffer_rsrc((void *)(a.products + (long long)slot * I), 0, I * 4, 0x00020000);
#pragma unroll
            for (int q = 0; q < kQuads; ++q) {
                prod[i][q] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (q * kWave + lane) * 16, 0, 0));
            }
        }
    };
    // (the arithmetic of requant_kernel and requant_fp8_kernel)
    auto quantise = [&](int first) {
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const int slot = first + wave + i * kDownWaves;
            if constexpr (FP8) {
#pragma unroll
                for (int q = 0; q < kQuads; ++q) {
                    const int c = q * kWave + lane;   // a block of 128 columns to 32 lanes
                    const v4f v = prod[i][q];
                    const float m = group_max(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))), 32);
                    const int ex = fp8_block_scale_exp(m);
                    const float f1 = exp2_int(-(ex / 2)), f2 = exp2_int(-(ex - ex / 2));
                    int w = 0;
                    w = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(v[0], f1), f2), __fmul_rn(__fmul_rn(v[1], f1), f2), w, false);
                    w = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(v[2], f1), f2), __fmul_rn(__fmul_rn(v[3], f1), f2), w, true);
                    if (slot < A && c < I >> 2) {
                        *(int *)(rows_s + slot * I + c * 4) = w;
                        if ((lane & 31) == 0) {
                            x_scale8_s[slot * (I >> 7) + (c >> 5)] = (uint8_t)(ex + 127);
                        }
                    }
                }
                continue;
            }
            float m = 0.0f;
#pragma unroll
            for (int q = 0; q < kQuads; ++q) {
                m = fmaxf(m, fmaxf(fmaxf(fabsf(prod[i][q][0]), fabsf(prod[i][q][1])), fmaxf(fabsf(prod[i][q][2]), fabsf(prod[i][q][3]))));
            }
            m = wave_max(m);
            const bool zero_row = m == 0.0f;
            const float rcp = zero_row ? 0.0f : __fdiv_rn(1.0f, m);
            if (slot < A) {
                if (lane == 0) {
                    scale_s[slot] = zero_row ? 0.0f : __fmul_rn(m, 1.0f / 127.0f);
                }
#pragma unroll
                for (int q = 0; q < kQuads; ++q) {
                    const int c = q * kWave + lane;
                    if (c < I >> 2) {
                        int b[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            b[e] = (int)rintf(__fmul_rn(__fmul_rn(prod[i][q][e], 127.0f), rcp));
                        }
                        *(uint32_t *)(rows_s + slot * I + c * 4) = pack4(b[0], b[1], b[2], b[3]);
                    }
                }
            }
        }
    };
    int batch = 0;
    load_products(batch);
    if constexpr (RW > 1) {
        for (; batch + RW * kDownWaves < A; batch += RW * kDownWaves) {
            quantise(batch);
            load_products(batch + RW * kDownWaves);
        }
    }
    const Slots slots(a, loaded_id);
    const int KT = I / F::kStep;
    float column = 0.0f, weight = 0.0f;
    int w_scale8 = 0;
    const int g = __shfl(slots.id, min(FP8 ? tid / KT : tid >> 4, kWave - 1), kWave);   // (by all lanes)
    if constexpr (FP8) {
        if (tid < A * KT && g >= 0) {
            w_scale8 = a.w_scale8[((long long)g * KT + tid % KT) * (H >> 7) + (c0 >> 7)];
        }
    } else if (tid < A * kColumns && g >= 0) {
        column = (a.per_expert ? a.list.s[g] : a.w_scale + (long long)g * H)[c0 + (tid & 15)];
    }
    for (int i = tid; i < kParts * kFewSlots * kColumns; i += kDownThreads) {
        (&sum_s[0][0][0])[i] = 0;
    }
    if (tid < A) {
        weight = a.gates[tid];
        row_s[tid] = slots.id >= 0 ? slots.row_slot : -1;
    }

    // this wave's share of the K steps of all experts, one after the other
    const int steps = slots.experts() * KT, share = (steps + kDownWaves - 1) / kDownWaves;
    const int begin = wave * share, end = min(steps, begin + share);
    constexpr int kRing = FP8 ? kDownRing / 2 : kDownRing;
    typename F::Weights ring[kRing];
    int ask_j = begin / KT, ask_t = begin - ask_j * KT;   // the next step to ask for
    const int8_t *ask_w = a.w;
    int ask_step = 0;
    const WeightColumns<FP8> none(nullptr, I, H, c0 >> 6, (c0 >> 4) & 3);
    auto ask_expert = [&](int j) {
        if (j < slots.experts()) {
            const int g = slots.expert_of(slots.first_slot(j));
            const WeightColumns<FP8> wc(a.per_expert ? a.list.w[g] : a.w + (long long)g * I * H, I, H, c0 >> 6, (c0 >> 4) & 3);
            ask_w = wc.base;
            ask_step = wc.step;
        }
    };
    ask_expert(ask_j);
    auto issue = [&](int i, int f) {
        ring[i] = load_weights<FP8>(ask_w, none.lane_offset, ask_t * ask_step, f < end);
        if (++ask_t == KT) {
            ask_t = 0;
            ask_expert(++ask_j);
        }
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i) {
        issue(i, begin + i);
    }

    if constexpr (FP8) {
        if (tid < A * KT) {
            w_scale8_s[tid] = (uint8_t)w_scale8;
        }
    } else if (tid < A * kColumns) {
        column_s[tid >> 4][tid & 15] = column;
    }
    if (tid < A) {
        weight_s[tid] = weight;
    }
    quantise(batch);
    lds_barrier();

    int j = begin / KT, t = begin - j * KT;
    int rows = 0, lead = 0, slot = 0;   // of the expert, its first slot, the slot of this lane's row
    typename F::Sum sum{};
    auto expert = [&]() {
        lead = slots.first_slot(j);
        const unsigned long long row_slots = slots.rows_of(lead);
        rows = __popcll(row_slots);
        slot = nth_slot(row_slots, lane & 15);
    };
    auto leave = [&]() {  // whole numbers: the order in which the waves add them does not matter
        if ((lane & 15) < rows) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                typename F::One *to = &sum_s[FP8 ? wave : 0][slot][(lane >> 4) * 4 + e];
                if constexpr (FP8) {
                    *to = sum[e];   // a wave has an expert's steps one after the other
                } else {
                    atomicAdd(to, sum[e]);
                }
            }
        }
        sum = typename F::Sum{};
    };
    if (begin < end) {
        expert();
    }
    for (int f = begin; f < end; f += kRing) {
#pragma unroll
        for (int i = 0; i < kRing; ++i) {
            if (f + i < end) {
                const typename F::Weights x = *(const typename F::Weights *)(rows_s + slot * I + t * F::kStep + (lane >> 4) * (F::kStep / 4));
                int sw = 0, sx = 0;
                if constexpr (FP8) {
                    sw = w_scale8_s[lead * KT + t];
                    sx = x_scale8_s[slot * KT + t];
                }
                sum = F::multiply(ring[i], x, sum, sw, sx);
                ++t;
                if (t == KT || f + i + 1 == end) {
                    leave();
                    if (f + i + 1 < end) {
                        t = 0;
                        ++j;
                        expert();
                    }
                }
                issue(i, f + i + kRing);
            }
        }
    }
    lds_barrier();

    // dequantised to the activation type, then the weighted sum in the order of k
    if (tid < a.T * kColumns) {
        const int token = tid >> 4, c = tid & 15;
        float acc = 0.0f;
        for (int k = 0; k < a.K; ++k) {
            const int s = row_s[token * a.K + k];
            if (s >= 0) {
                float v;
                if constexpr (FP8) {
                    v = sum_s[0][s][c];
#pragma unroll
                    for (int p = 1; p < kParts; ++p) {
                        v += sum_s[p][s][c];
                    }
                } else {
                    v = __fmul_rn(__fmul_rn((float)sum_s[0][s][c], column_s[s][c]), scale_s[s]);
                }
                if (ACT == 1) {
                    asm("" : "+v"(v));  // rounded to fp32 first, as in the GEMMs: the conversion must not swallow the product
                    v = fp16_bits_to_f32(f32_to_fp16_bits(v));
                } else {
                    v = bf16_bits_to_f32(f32x2_to_bf16x2_bits(v, v) & 0xffffu);
                }
                acc = __fadd_rn(acc, __fmul_rn(v, weight_s[token * a.K + k]));
            }
        }
        a.out[(long long)token * H + c0 + c] =
            (uint16_t)(ACT == 1 ? f32_to_fp16_bits(acc) : f32x2_to_bf16x2_bits(acc, acc) & 0xffffu);
    }
}

template <bool FP8, int ACT>
void launch_up(dim3 grid, dim3 block, size_t lds, hipStream_t stream, const FewTokensArgs &a)
{
    hipLaunchKernelGGL((few_tokens_up_kernel<FP8, ACT>), grid, block, lds, stream, a);
}

template <bool FP8, int ACT>
void launch_down(dim3 grid, dim3 block, size_t lds, hipStream_t stream, const FewTokensArgs &a)
{
    if (a.T * a.K <= kDownWaves) {
        hipLaunchKernelGGL((few_tokens_down_kernel<FP8, ACT, 1>), grid, block, lds, stream, a);
    } else {
        hipLaunchKernelGGL((few_tokens_down_kernel<FP8, ACT, 2>), grid, block, lds, stream, a);
    }
}

bool few_tokens_valid(const FewTokensArgs &a)
{
    return few_tokens_apply(a.T, a.K, a.E, a.H, a.I, a.w_scale8 != nullptr) &&
           (a.w_scale8 == nullptr || (a.H % 128 == 0 && a.I % 128 == 0 && !a.per_expert && !a.x_is_fp16));
}

}  // namespace

// Up to eight slots of one token always, of more tokens while their products, which each of the down launch's workgroups quantises first, are
// not too many for the output columns it has, or where there are so few experts that several slots name one; up to sixteen, and 32 of few tokens, where the down launch, whose workgroups are one for 16
// output columns, has enough of them for the length of its rows, and where the slots name different experts (a gate/up workgroup is
// one expert's, and quantises all of its tokens).  us per layer, four launches or five / these two;
// T x H, top-K of E, I: 1 x 4096, 8 of 128, 1536 43.0 / 32.0; 1 x 4096, 1 of 128, 1536 24.8 / 11.0; 1 x 7168, 8 of 64, 2048 74.6 / 62.3; 1 x 512, 8
// of 64, 3072 28.2 / 28.6; 2 x 4096, 8 of 128, 1536 68.3 / 58.1 (both tokens the same 43.6 / 35.7); 8 x 512, 1 of 4, 3072 21.8 / 17.1; 8 x 6144, 2 of
// 16, 2048 90.3 / 79.6.  Nine to sixteen slots by slots * I / H: 8 23.1 / 18.3, 12 65.7 / 58.0 and 41.1 / 39.3, 24 30.9 / 32.7 and 65.0 / 67.2
// (also 30.8 / 30.0), 48 42.8 / 54.1.  More: 4 x 4096, 8 of 128, 1536 116.5 / 102.0 (the same experts for all 65.4 / 46.2), 4 x 4096, 8 of 64, 512
// 47.1 / 43.8, 3 x 4096, 8 of 48, 2048 111.3 / 94.0; not 8 x 4096, 4 of 8, 1536 41.9 / 46.0, 4 x 2048, 8 of 64, 1024 47.5 / 51.2, 6 x 5120, 3 of 40,
// 1024 59.1 / 60.1.
// Eight slots of few output columns (replayed from a graph), I 3072: 512 1 x 8 28.4 / 29.2, 2 x 4 26.6 / 30.3, 8 x 1 25.6 / 29.1; 768 1 x 8 30.7 / 30.5, 2 x 4
// 29.2 / 30.4, 8 x 1 28.0 / 29.5; 1024 8 x 1 30.0 / 31.3; 1152 8 x 1 31.9 / 31.0; 2560: 512 8 x 1 24.8 / 26.3, 768 8 x 1 26.7 / 25.9; 2048: 512 2 x 4
// 23.4 / 22.5; six slots 2 x 3 of 512, 3072 26.0 / 25.1.
// That was 48 experts; 8 x 512, top-1, 3072 of 8 23.9 / 22.7, of 12 23.8 / 23.1, of 16 25.5 / 26.9, 2 x 512, top-4, of 8 25.6 / 24.9, of 12 25.9 / 27.2, of 16 26.4 / 27.0.
// FP8 up to sixteen slots: 1 x 4096, 8 of 128, 1536 49.2 / 34.3, 1 of 128 38.0 / 12.7, 1 x 7168, 8 of 64, 2048 82.3 / 62.8, 2 x 4096, 8 of 64, 1536 62.7 /
// 59.4 (the same 52.2 / 39.3), 2 x 7168, 8 of 64, 2048 127.8 / 124.2, 4 x 4096, 4 of 8, 1024 42.9 / 28.5, 2 x 1024, 8 of 64, 768 28.9 / 26.0, 1 x 1024, 8
// of 64, 2048 28.5 / 24.3; not 1 x 1024, 8 of 64, 3072 32.1 / 33.2, 2 x 1024, 8 of 64, 1024 28.7 / 29.7, 2 x 2048, 6 of 64, 2048 39.8 / 43.0, 5 x 4096,
// 3 of 64, 2048 69.2 / 70.5, 3 x 7168, 8 of 64, 1024 101.4 / 104.1.
// Over eight slots the down launch has one workgroup to a CU, and from 4224 to 6144 output columns 264 to 384 of them: a second round of a
// few.  Times as fast as the launches before (replayed from a graph; of 64 experts): FP8, 16 slots of 1536 4224 0.82, 5120 0.94, 6144 1.00, 12 of 2560
// 4608 0.91, 5632 0.93; little or very much to quantise gains all the same, 16 of 1024 4608 1.00 and, skewed, 1.15, 12 of 3072 5888 1.13, 6144
// 1.17.  int8, 16 slots of 2048 4224 0.91, 4608 0.97, 5120 0.98, 12 of 1536 4224 1.06; 32 of 512 4224 0.80, 5120 0.89, 6144 0.90, 24 of 1536 4608 0.95, 6144
// 1.11, of 2048 5120 1.04.
bool few_tokens_apply(int64_t T, int64_t K, int64_t E, int64_t H, int64_t I, bool fp8)
{
    const int64_t slots = T * K;
    if (T < 1 || T > kFewTokens || K < 1 || slots > kFewSlots || E < 1 || E > kMaxExperts || H < 64 || H > kFewMaxH || I < 64 || I > kFewMaxI ||
        H % 64 != 0 || I % 64 != 0 || T * H > kFewRowBytes || slots * I > kFewRowBytes) {
        return false;
    }
    const bool second_round = slots > 8 && H > 4096 && H <= 6144;
    if (fp8) {
        if (second_round && 10 * slots * I > 37 * H && slots * I < 36000) {
            return false;
        }
        return slots <= 8 ? slots * I <= 16 * H : slots <= 16 && (slots * I <= 7 * H || slots * I <= 12288);
    }
    if (slots <= 8) {
        return T == 1 || slots * I <= 12288 + 11 * H || 2 * E <= 3 * slots;
    }
    if (second_round && (slots <= 16 ? H < 4608 && slots * I > 24000 : slots * I < 40960 && (H < 5632 || I <= 512))) {
        return false;
    }
    return slots * I <= 16 * H && (slots <= 16 || (T <= 4 && H >= 4096 && E >= 2 * slots));
}

hipError_t launch_few_tokens_up(const FewTokensArgs &a, hipStream_t stream)
{
    if (!few_tokens_valid(a)) {
        return hipErrorInvalidValue;
    }
    const dim3 grid((unsigned)(a.T * a.K * (a.I / kColumns) + 1)), block(kUpThreads);
    const size_t lds = (size_t)a.T * a.H;
    if (a.w_scale8 != nullptr) {
        launch_up<true, 0>(grid, block, lds, stream, a);
    } else {
        a.x_is_fp16 ? launch_up<false, 1>(grid, block, lds, stream, a) : launch_up<false, 0>(grid, block, lds, stream, a);
    }
    return hipGetLastError();
}

hipError_t launch_few_tokens_down(const FewTokensArgs &a, hipStream_t stream)
{
    if (!few_tokens_valid(a)) {
        return hipErrorInvalidValue;
    }
    const dim3 grid((unsigned)(a.H / kColumns)), block(kDownThreads);
    const size_t lds = (size_t)a.T * a.K * a.I;
    if (a.w_scale8 != nullptr) {
        launch_down<true, 0>(grid, block, lds, stream, a);
    } else {
        a.x_is_fp16 ? launch_down<false, 1>(grid, block, lds, stream, a) : launch_down<false, 0>(grid, block, lds, stream, a);
    }
    return hipGetLastError();
}

}  // namespace cam
