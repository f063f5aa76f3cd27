// Token permutation with fused per-token int8 quantisation (bandwidth-bound).
//
// Reference semantics (paths relative to the reference tree):
//   send side   src/cam/comm_operator/ascend_kernels/moe_dispatch_normal/op_kernel/moe_dispatch_normal.h:330-396
//   quant       the same file :278-316 (scale = 127/(max|x| + 1e-12)), and the fused kernel's QuantToken,
//               src/cam/comm_operator/ascend_kernels/fused_deep_moe/op_kernel/fused_deep_moe/gemm/kernel/
//               grouped_matmul_slice_m_per_token_dequant_swiglu_quant_multistage_workspace.h:780-818 (no epsilon)
//   receive     moe_dispatch_normal.h:486-535 (rows land at recvCount[i-1] + j; triple and scale per row)
//
// Design.  The reference reads a token once per top-k copy and moves every row twice (sender ->
// window -> output).  Here one wavefront owns one token: lane l loads the 16-byte chunks l, l+64, ...
// of the row (each load instruction covers 1 KB of contiguous memory) exactly once, the row maximum
// is reduced with wave shuffles alone (no LDS, no workgroup barrier, so waves never wait for each
// other), the row is quantised in registers and each chunk's 8 result bytes are stored, again 512
// contiguous bytes per instruction, to each of the K destination rows.  HBM traffic is the
// algorithmic minimum: H*2 bytes read and K*H bytes written per token.
#include "cam_device.h"
#include "cam_kernels.h"
#include "permute_device.h"
#include "rank_device.h"

namespace cam {

namespace {

// Output row of entry (t,k), or -1.
__device__ __forceinline__ long long dispatch_row(const DispatchArgs &a, int t, int k)
{
    const long long i = (long long)t * a.K + k;
    if (a.dst_row != nullptr) {
        return a.dst_row[i];
    }
    const int e = a.idx[i];
    if (e < 0 || e >= a.E) {
        return -1;
    }
    const long long window_row = (long long)a.send_offset[e] + a.send_token_idx[i];
    const long long pre = e == 0 ? 0 : a.recv_count[e - 1];
    return pre + (window_row - a.recv_offset[e]);
}

// The output rows of a token's copies, that of copy k in lane k: all of them in one round trip, in front of the token's own row.  Asked
// for one by one, each waits for the stores of the copy before (see asks_one_by_one).  us, plan and permute replayed from a graph, one by one
// with the triples of lane 0 / this: 1999 x 4096, int8, 6 of 64 18.1 / 17.4, 2048 x 7168, 8 of 64 33.3 / 32.6, 5000 x 2048, FP8 37.3 / 35.7; 16-bit
// rows 1999 x 4096 24.0 / 23.8.
__device__ __forceinline__ long long own_row(const DispatchArgs &a, int t, int lane)
{
    const long long row = lane < a.K ? dispatch_row(a, t, lane) : -1;
    return row < a.A ? row : -1;
}

__device__ __forceinline__ long long row_of_lane(long long own, int k)
{
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)own, k), hi = __builtin_amdgcn_readlane((unsigned)((unsigned long long)own >> 32), k);
    return (long long)((unsigned long long)hi << 32 | lo);
}

// How the rows are stored.  Plain stores leave the L2 (32 MB) in a better order than the waves wrote the pieces of far apart rows in,
// and a reader that goes through the rows once finds more of them in the memory-side cache.  But what still lies in the L2 at the
// end of the launch has to be written back before the next one, which costs more than it gains while that is most of the
// output.  us, non-temporal / plain, 16-bit rows: dispatch alone, 33 MB 14.8 / 16.3, 49 MB 16.8 / 19.0, 84 MB 24.5 / 28.7, 115 MB 32.0 / 35.1, 168 MB
// 44.1 / 45.1, 210 MB 53.8 / 52.8, 420 MB 100.3 / 98.4; with a pass over the rows behind it, 84 MB 58.8 / 53.0, 115 MB 77.7 / 63.5, 168 MB
// 105.3 / 89.1, 210 MB 128.5 / 119.4, 420 MB 240 / 237; with a product of these rows 84 MB 181.0 / 177.9, 168 MB 420 / 414, 420 MB 763 / 757;
// with a gather of other rows 72 MB 37.8 / 38.3, 79 MB 40.9 / 40.1, 196 MB 89.0 / 89.3, 803 MB 346 / 341.
// 8-bit rows are there for the expert GEMMs, whose tiles read them several times over, and these are slower behind plain stores,
// although a single pass gains as above (84 MB 61.8 / 53.3): dispatch and GMM1, int8, rows of 7168 to 32 experts 88 MB 421.5 / 437.4, 105 MB
// 486.7 / 492.4, 126 MB 562.7 / 562.1, 155 MB 675.5 / 684.4, to 256 126 MB 239.1 / 254.8, of 4096 to 128 88 MB 256.0 / 266.5; with GMM2 and
// combine 657.8 / 669.7, 747.8 / 760.0, 879.6 / 876.9, 1038 / 1050, 458.8 / 481.7, 429.1 / 434.8.  FP8, 7168 to 32, 88 MB 410.7 / 423.4.
// Rows that are no whole lines of 128 bytes (no GEMM here takes 8-bit ones): the L2 puts the two halves of a line together, so they gain from
// less on, dispatch with a gather of other rows: 16-bit 34 MB 25.3 / 27.8, 50 MB 32.8 / 32.0, 90 MB 56.7 / 49.4, 96 MB 65.5 / 57.5; int8 19 MB
// 25.0 / 26.9, 56 MB 48.2 / 46.1, 172 MB 130.5 / 120.7, 235 MB 176.2 / 166.0.
bool stores_plainly(const DispatchArgs &a)
{
    const long long pitch = (long long)a.H * (a.quant == 0 ? 2 : 1), bytes = (long long)a.T * a.K * pitch;
    if (pitch % 128 != 0) {
        return bytes >= 48ll << 20;
    }
    return a.quant == 0 && bytes >= 72ll << 20;
}

// Whether a wave asks for the row of a copy behind the stores of the copy before, which spaces its stores out: very many 8-bit rows
// lie in memory faster then, although a wave takes longer, and int8 rows also where their tokens begin not to stay in the L2s.  us, plan and
// permute replayed from a graph, all at once / one by one, T x H, top-K of E:
// int8 235 MB 4096 x 7168, 8 of 256 68.1 / 64.1, 192 MB 8000 x 3000, 8 of 512 62.1 / 58.0, 172 MB 3000 x 7168, 8 of 64 50.1 / 48.3; FP8 235 MB 69.3 / 68.2;
// 16-bit rows level, 470 MB 95.4 / 95.3.  (A wait for the stores alone does not help: 68.7 in the first.)
// int8 by MiB of tokens: 28 2936 x 5000, 5 of 12 24.2 / 24.8, 4893 x 3000 28.2 / 28.6; 30 3145 x 5000, 4 of 8 27.0 / 24.1, 5242 x 3000, 6 of 64 36.1 / 33.0,
// 3145 x 5000, 8 of 256 41.6 / 38.3, but 2194 x 7168, 8 of 256 40.2 / 40.7 and 7680 x 2048, 4 of 8 29.3 / 31.3 (8 of 256 45.5 / 45.4); 40 4194 x 5000, 6
// of 64 44.4 / 39.6; 45 3291 x 7168, 4 of 8 35.6 / 32.0, 5760 x 4096 38.7 / 34.0; 47 3543 x 6904, 6 of 64 50.6 / 41.2; 60 4388 x 7168, 4 of 8 47.2 / 47.2,
// 70 5120 49.5 / 50.7; FP8 level.
bool asks_one_by_one(const DispatchArgs &a)
{
    const long long tokens = 2ll * a.T * a.H;
    const bool beyond_l2 = (a.quant == 1 || a.quant == 2) && a.H > 2048 && tokens >= 29ll << 20 && tokens < 63ll << 20;
    return a.quant != 0 && (beyond_l2 || (long long)a.T * a.K * a.H >= 152ll << 20);
}

// Four workgroups per CU (128 registers a lane) keep all 1024 workgroups of a 4096-token batch resident at once;
// the FP8 variant would spill at that size and stays at three.
template <int QUANT, int ACT, bool PLAIN>
__global__ __launch_bounds__(kDispWaves * kWave, QUANT == 3 ? 3 : 4) void dispatch_kernel(DispatchArgs a, bool one_by_one)
{
    const int t = (int)blockIdx.x * kDispWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    if (t >= a.T) {
        return;
    }
    const long long own = own_row(a, t, lane);
    WaveRow r;
    load_token_row(a.x, t, a.H, lane, r);
    if (QUANT != 0) {
        quant_token_row<QUANT, ACT>(r, WaveMax());
    }
    for (int k = 0; k < a.K; ++k) {
        const long long row = one_by_one ? dispatch_row(a, t, k) : row_of_lane(own, k);
        if (row >= 0 && row < a.A) {
            store_token_row<QUANT, PLAIN>(r, a.out, a.scales, row, a.H, lane);
        }
    }
    if (own >= 0) {
        store_row_origin<QUANT>(r.scale_out, a.scales, a.src_info, a.src_rank, own, t, lane);
    }
}

// The quantising permute with per-expert smooth scales: every copy of a token is quantised on its own, under the
// scale row of its destination expert (moe_dispatch_shmem.h:492-549,693-733).  One wave per token; the token row
// is loaded once and stays in registers across its copies.
template <int ACT, bool PLAIN>
__global__ __launch_bounds__(kDispWaves * kWave) void dispatch_smooth_kernel(DispatchArgs a)
{
    const int t = (int)blockIdx.x * kDispWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    if (t >= a.T) {
        return;
    }
    const long long own = own_row(a, t, lane);
    const int own_id = lane < a.K ? a.idx[(long long)t * a.K + lane] : -1;
    WaveRow r;
    load_token_row(a.x, t, a.H, lane, r);
    for (int k = 0; k < a.K; ++k) {
        const long long row = row_of_lane(own, k);
        const int e = __builtin_amdgcn_readlane(own_id, k);
        if (row < 0 || e < 0 || e >= a.E) {
            continue;
        }
        quant_token_row_smooth<ACT>(r, a.smooth + (long long)e * a.H, a.H, lane, WaveMax());
        store_token_row<2, PLAIN>(r, a.out, a.scales, row, a.H, lane);
        if (lane == 0) {
            store_row_origin<2>(r.scale_out, a.scales, a.src_info, a.src_rank, row, t, k);
        }
    }
}

// Plan and permute in one launch, for id sequences short enough that every workgroup can look at all of them.
// A workgroup per token.  While its row is on its way it finds where the row goes: the row of entry (t,k) is the number
// of entries that name an earlier expert plus the number of earlier entries that name the same one, so a look at all
// T * K ids (counted with ballots) gives the rows and the ranks of the K entries with no table, no scan and nothing to
// wait for from another workgroup.  Workgroup 0 counts for the per-expert outputs.  With few tokens the latency of one
// row is what the launch takes, so it is spread over sixteen waves (four from 257 tokens on) instead of one.
// The triples and scales of a token's copies are stored at once, a lane each (by one thread 128 x 7168, 8 of 256 6.40 -> 6.12, 300 x 4096 8.64 -> 8.31).
// Launches: one token x 4096 to 128 experts, top-8: 3.5 + 7.4 us -> 5.9; 64 x 4096 FP8: 6.2 + 15.6 -> 7.4; 128 x 7168 to 256
// experts: 6.1 + 9.8 -> 7.8.
// What bounds it beside the latencies is the counting, top-k times over a thread's ids, so an id is compared twice a time and with
// nothing else: what lies behind the active tokens, or behind this one, is struck out beforehand.  Replayed from a graph, us, with a look
// at the place of every id instead / this: 128 x 4096, top-8 of 128 6.44 / 5.94, 256 7.75 / 6.97, 128 x 7168, top-8 of 256 7.05 / 6.37, 341 x 4096,
// top-6 10.44 / 9.12, 170 x 2048, top-12 8.66 / 7.49.  A wave per k that looks at all ids: 7.38, 9.97, 7.38, 11.41, 10.64.
constexpr int kSmallIds = 2048;   // ids per launch (rows of at most 29 MB)
template <typename IdT, int QUANT, int ACT, bool SMOOTH, int NT>
__global__ __launch_bounds__(NT) void dispatch_small_kernel(PlanArgs p, DispatchArgs a)
{
    constexpr int kPer = kSmallIds / NT;   // ids per thread
    constexpr int kWaves = NT / kWave;
    __shared__ int counts[kWaves][kMaxTopk];  // entries before the expert's, and earlier entries of it (<< 16): per wave and k
    __shared__ int row_s[kMaxTopk];
    __shared__ float max_s[kWaves];
    __shared__ int active_s;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid >> 6;
    const IdT *__restrict__ idx = (const IdT *)p.idx;
    const int n_all = p.T * p.K;
    const int E = p.E, K = p.K;

    if (blockIdx.x == 0) {  // counts, offsets and totals
        __shared__ int hist[kMaxExperts];
        __shared__ int scan_s[kWaves];
        __shared__ int total_s;
        int id[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int j = tid + i * NT;
            id[i] = j < n_all ? load_id(idx, j, E) : -1;
        }
        const int t_active = count_active(p.mask, p.T, tid, NT, &active_s);
        for (int i = tid; i < kMaxExperts; i += NT) {
            hist[i] = 0;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (tid + i * NT < t_active * K && id[i] >= 0) {
                atomicAdd(&hist[id[i]], 1);
            }
        }
        __syncthreads();
        write_expert_outputs<NT>(p, hist, t_active, tid, scan_s, &total_s);
        clear_stream_queues(p, tid, NT);
        return;
    }

    const int t = (int)blockIdx.x - 1;
    GroupRow<NT> r;
    load_token_row(a.x, t, a.H, tid, r);
    int id[kPer];  // entries tid, tid + NT, ...; -1 where none
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int j = tid + i * NT;
        id[i] = -1;
        if (i * NT < n_all && j < n_all) {
            id[i] = load_id(idx, j, E);
        }
    }
    const int own_ids = lane < K ? load_id(idx, t * K + lane, E) : -1;  // lane k: the id of entry (t,k)
    const int t_active = count_active(p.mask, p.T, tid, NT, &active_s);
    const int n = t_active * K;
    int earlier_id[kPer];   // those of the tokens before
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int j = tid + i * NT;
        id[i] = j < n ? id[i] : -1;
        earlier_id[i] = j < t * K ? id[i] : -1;
    }
    int found = 0;   // lane k: this wave's counts for entry (t,k)
    for (int k = 0; k < K; ++k) {
        const int e = __builtin_amdgcn_readlane(own_ids, k);
        int before = 0, earlier = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (i * NT < n) {
                before += __popcll(__ballot((unsigned)id[i] < (unsigned)max(e, 0)));
                earlier += __popcll(__ballot(earlier_id[i] == e));
            }
        }
        if (wave == 0) {  // and in the token itself
            earlier += __popcll(__ballot(own_ids == e) & ((1ull << k) - 1));
        }
        found = lane == k ? before | earlier << 16 : found;
    }
    if (lane < K) {
        counts[wave][lane] = found;
    }
    if (QUANT != 0 && !SMOOTH) {
        quant_token_row<QUANT, ACT>(r, GroupMax<NT>{max_s});
    }
    __syncthreads();
    if (tid < K) {
        const int own = t * K + tid;
        int row = -1, rank = -1;
        if (own < n && own_ids >= 0) {
            int sum = 0;   // (2048 of either at most)
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                sum += counts[w][tid];
            }
            rank = sum >> 16;
            row = (sum & 0xffff) + rank;
        }
        row_s[tid] = row;
        p.pos[own] = rank;
        if (p.dst_row != nullptr) {
            p.dst_row[own] = row;
        }
    }
    __syncthreads();
    for (int k = 0; k < K; ++k) {
        const int row = row_s[k];
        if (row < 0 || row >= a.A) {
            continue;
        }
        if constexpr (SMOOTH) {
            const int e = __builtin_amdgcn_readlane(own_ids, k);
            quant_token_row_smooth<ACT>(r, a.smooth + (long long)e * a.H, a.H, tid, GroupMax<NT>{max_s});
        }
        store_token_row<QUANT, false>(r, a.out, a.scales, row, a.H, tid);
        if (SMOOTH && tid == 0) {
            store_row_origin<QUANT>(r.scale_out, a.scales, a.src_info, a.src_rank, row, t, k);
        }
    }
    if (!SMOOTH && tid < K && row_s[tid] >= 0 && row_s[tid] < a.A) {
        store_row_origin<QUANT>(r.scale_out, a.scales, a.src_info, a.src_rank, row_s[tid], t, tid);
    }
}

template <typename IdT, int QUANT, bool SMOOTH, int NT>
hipError_t launch_small_with(const PlanArgs &p, const DispatchArgs &a, hipStream_t stream)
{
    const dim3 grid((unsigned)p.T + 1), block(NT);
    if (a.x_is_fp16 && QUANT != 0) {  // (a copy does not look at the format)
        hipLaunchKernelGGL((dispatch_small_kernel<IdT, QUANT, 1, SMOOTH, NT>), grid, block, 0, stream, p, a);
    } else {
        hipLaunchKernelGGL((dispatch_small_kernel<IdT, QUANT, 0, SMOOTH, NT>), grid, block, 0, stream, p, a);
    }
    return hipGetLastError();
}

template <typename IdT, int QUANT, bool SMOOTH = false>
hipError_t launch_small_as(const PlanArgs &p, const DispatchArgs &a, hipStream_t stream)
{
    // sixteen waves per token while every token has a CU of its own
    return p.T <= 256 ? launch_small_with<IdT, QUANT, SMOOTH, 1024>(p, a, stream)
                      : launch_small_with<IdT, QUANT, SMOOTH, 256>(p, a, stream);
}

template <typename IdT>
hipError_t launch_small(const PlanArgs &p, const DispatchArgs &a, hipStream_t stream)
{
    if (a.smooth != nullptr) {
        return launch_small_as<IdT, 2, true>(p, a, stream);
    }
    switch (a.quant) {
        case 0: return launch_small_as<IdT, 0>(p, a, stream);
        case 1: return launch_small_as<IdT, 1>(p, a, stream);
        case 2: return launch_small_as<IdT, 2>(p, a, stream);
        default: return launch_small_as<IdT, 3>(p, a, stream);
    }
}

template <bool PLAIN>
void launch_dispatch_as(const DispatchArgs &a, hipStream_t stream)
{
    const dim3 grid((a.T + kDispWaves - 1) / kDispWaves), block(kDispWaves * kWave);
    const bool fp16 = a.x_is_fp16 != 0, paced = asks_one_by_one(a);
    if (a.smooth != nullptr) {
        if (fp16) {
            hipLaunchKernelGGL((dispatch_smooth_kernel<1, PLAIN>), grid, block, 0, stream, a);
        } else {
            hipLaunchKernelGGL((dispatch_smooth_kernel<0, PLAIN>), grid, block, 0, stream, a);
        }
    } else if (a.quant == 0) {
        hipLaunchKernelGGL((dispatch_kernel<0, 0, PLAIN>), grid, block, 0, stream, a, paced);  // a copy does not look at the format
    } else if (a.quant == 1) {
        if (fp16) {
            hipLaunchKernelGGL((dispatch_kernel<1, 1, PLAIN>), grid, block, 0, stream, a, paced);
        } else {
            hipLaunchKernelGGL((dispatch_kernel<1, 0, PLAIN>), grid, block, 0, stream, a, paced);
        }
    } else if (a.quant == 3) {  // (whole lines: never plainly)
        if (fp16) {
            hipLaunchKernelGGL((dispatch_kernel<3, 1, false>), grid, block, 0, stream, a, paced);
        } else {
            hipLaunchKernelGGL((dispatch_kernel<3, 0, false>), grid, block, 0, stream, a, paced);
        }
    } else {
        if (fp16) {
            hipLaunchKernelGGL((dispatch_kernel<2, 1, PLAIN>), grid, block, 0, stream, a, paced);
        } else {
            hipLaunchKernelGGL((dispatch_kernel<2, 0, PLAIN>), grid, block, 0, stream, a, paced);
        }
    }
}

}  // namespace

hipError_t launch_plan_dispatch(const PlanArgs &p, const DispatchArgs &a, hipStream_t stream)
{
    const long long n = (long long)p.T * p.K;
    if (n > 0 && n <= kSmallIds) {  // one launch
        if (a.H % 8 != 0 || a.H / 8 > kDispMaxChunks * kWave || (a.quant == 3 && a.H % 128 != 0) ||
            (a.smooth != nullptr && a.quant != 2) || p.K > kMaxTopk || p.E > kMaxExperts) {
            return hipErrorInvalidValue;
        }
        return p.idx_is64 ? launch_small<int64_t>(p, a, stream) : launch_small<int32_t>(p, a, stream);
    }
    const hipError_t e = launch_plan(p, stream);
    if (e != hipSuccess) {
        return e;
    }
    return launch_dispatch(a, stream);
}

hipError_t launch_dispatch(const DispatchArgs &a, hipStream_t stream)
{
    if (a.T <= 0) {
        return hipSuccess;
    }
    if (a.H % 8 != 0 || a.H / 8 > kDispMaxChunks * kWave || (a.quant == 3 && a.H % 128 != 0) || a.K > kMaxTopk) {
        return hipErrorInvalidValue;
    }
    if (a.smooth != nullptr && (a.quant != 2 || a.idx == nullptr)) {
        return hipErrorInvalidValue;
    }
    if (stores_plainly(a)) {
        launch_dispatch_as<true>(a, stream);
    } else {
        launch_dispatch_as<false>(a, stream);
    }
    return hipGetLastError();
}

}  // namespace cam
