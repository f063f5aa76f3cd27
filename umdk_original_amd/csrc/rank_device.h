// Device code shared by the routing-plan kernels: id loading, workgroup
// scans and the stable ranking of one chunk of the flat (token, k) id sequence.
#ifndef CAM_RANK_DEVICE_H_
#define CAM_RANK_DEVICE_H_

#include "cam_device.h"
#include "cam_kernels.h"

namespace cam {

constexpr int kLocalThreads = 256;  // ranking workgroup: 4 waves
constexpr int kLocalWaves = kLocalThreads / kWave;

// Ids outside [0, E) name no expert: negative ones are the reference's "dropped" marker
// (src/cam/comm_operator/pybind/moe_dispatch_prefill.cpp:106), ids >= E would index past every
// per-expert table and are treated the same way.
template <typename IdT>
__device__ __forceinline__ int load_id(const IdT *p, long long i, int E)
{
    long long v = (long long)p[i];
    return (v < 0 || v >= (long long)E) ? -1 : (int)v;
}

// Exclusive scan of one value per thread across a workgroup of NWAVES waves; returns the exclusive
// prefix and leaves the grand total in *total_out (LDS).  Uses `scratch` (>= NWAVES ints of LDS).
template <int NWAVES>
__device__ __forceinline__ int block_exclusive_scan(int v, int tid, int *scratch, int *total_out)
{
    int lane = tid & (kWave - 1);
    int w = tid >> 6;
    int inc = wave_inclusive_scan(v);
    if (lane == kWave - 1) {
        scratch[w] = inc;
    }
    __syncthreads();
    if (w == 0) {
        int t = lane < NWAVES ? scratch[lane] : 0;
        int ti = wave_inclusive_scan(t);
        if (lane < NWAVES) {
            scratch[lane] = ti - t;
        }
        if (lane == NWAVES - 1) {
            *total_out = ti;
        }
    }
    __syncthreads();
    int r = inc - v + scratch[w];
    __syncthreads();
    return r;
}

// Number of set mask entries (the active prefix of the batch); T when there is no mask.  By at least 32 threads; sixteen entries a load,
// as the quantising workgroups of a layer's plan ask for it too, every one of them.
__device__ __forceinline__ int count_active(const uint8_t *mask, int T, int tid, int nthreads, int *slot)
{
    if (mask == nullptr) {
        return T;
    }
    const int head = min((int)(-(uintptr_t)mask & 15), T);  // up to where entries are whole 16-byte words
    const int words = (T - head) >> 4;
    int c = 0;
    for (int i = tid; i < words; i += nthreads) {
        const v4u v = ((const v4u *)(mask + head))[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c += __popc((((v[j] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v[j]) & 0x80808080u);  // bytes that are not zero
        }
    }
    const int t = tid < 16 ? tid : head + 16 * words + (tid - 16);  // the entries in front of them and behind them
    if (t < (tid < 16 ? head : T) && tid < 32) {
        c += mask[t] != 0 ? 1 : 0;
    }
    c = wave_sum(c);
    if (tid == 0) {
        *slot = 0;
    }
    __syncthreads();
    if ((tid & (kWave - 1)) == 0 && c != 0) {
        atomicAdd(slot, c);
    }
    __syncthreads();
    return *slot;
}

// The per-expert counts may lie in host memory a CPU is watching (each count on its own): stored for the whole system.
__device__ __forceinline__ void store_count(int64_t *p, int v)
{
    __hip_atomic_store(p, (int64_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// (at the end of a kernel: in front of a barrier the stores would be waited for)
__device__ __forceinline__ void clear_stream_queues(const PlanArgs &a, int tid, int nthreads)
{
    if (a.stream_queues != nullptr) {
        for (int i = tid; i < 2 * kStreamQueue; i += nthreads) {
            a.stream_queues[i] = 0;
        }
    }
}

// Everything the plan says about the experts, from their complete counts cnt[0..E) (LDS), by one workgroup of NT >= 256
// threads; leaves the exclusive offsets in cnt.
template <int NT>
__device__ __forceinline__ void write_expert_outputs(const PlanArgs &a, int *cnt, int t_active, int tid, int *scan_s, int *total_s)
{
    // thread i owns experts 2i and 2i+1
    const int E = a.E;
    int c2[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        c2[h] = 2 * tid + h < E ? cnt[2 * tid + h] : 0;
    }
    const int pair_off = block_exclusive_scan<NT / kWave>(c2[0] + c2[1], tid, scan_s, total_s);
    const int total = *total_s;
    const int o2[2] = {pair_off, pair_off + c2[0]};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = 2 * tid + h;
        if (e < E) {
            cnt[e] = o2[h];
            if (a.cnt) a.cnt[e] = c2[h];
            if (a.off) a.off[e] = o2[h];
            if (a.recv_off) a.recv_off[e] = o2[h];
            if (a.recv_count) a.recv_count[e] = o2[h] + c2[h];
            if (a.tokens_per_expert) store_count(a.tokens_per_expert + e, c2[h]);
            if (a.group_list) a.group_list[e] = (int64_t)o2[h] + c2[h];
        }
    }
    if (tid == 0 && a.total) {
        a.total[0] = total;
    }
    if (tid == 0 && a.meta != nullptr) {
        a.meta[0] = 0;
        a.meta[1] = total;
        a.meta[2] = t_active;
        a.meta[3] = 0;
    }
}

// Ranks the chunk of flat entries [b*IT*256, (b+1)*IT*256) of one workgroup of 256 threads.
// Wave w owns the IT*64 entries from b*chunk + w*IT*64 and each lane keeps its IT ids in registers.
// 64 ids at a time, lanes holding the same id find each other with one ballot per id bit; the rank
// inside the wave is the wave's running count of that id (LDS) plus the number of lower lanes in the
// group, and the group's highest lane publishes the new count.  A scan over the 4 waves' histograms
// turns wave-local ranks into chunk-local ones.  Writes the chunk-local rank of every entry below
// n_all to pos_out (-1 for skipped entries and entries at or beyond n) and the chunk's per-expert
// histogram to hist_row[0..E).  `hist` is LDS, kLocalWaves * kMaxExperts ints.
template <typename IdT, int IT>
__device__ __forceinline__ void rank_chunk(const IdT *__restrict__ idx, int b, long long n, long long n_all, int E,
                                           int *hist, int32_t *pos_out, int32_t *hist_row)
{
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int w = tid >> 6;
    // the ids are requested first: their trip to memory runs while the histograms are cleared
    const long long base = (long long)b * (IT * kLocalThreads) + (long long)w * (IT * kWave);
    int e[IT], r[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const long long i = base + it * kWave + lane;
        e[it] = i < n ? load_id(idx, i, E) : -1;
    }
    for (int i = tid; i < kLocalWaves * kMaxExperts; i += kLocalThreads) {
        hist[i] = 0;
    }
    __syncthreads();
    int nbits = 0;
    while ((1 << nbits) < E) {
        ++nbits;
    }
    int *my_hist = hist + w * kMaxExperts;
    const unsigned long long lt_mask = (1ull << lane) - 1ull;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const bool act = e[it] >= 0;
        unsigned long long peers = __ballot(act);
        for (int bit_i = 0; bit_i < nbits; ++bit_i) {
            const bool bit = act && ((e[it] >> bit_i) & 1);
            const unsigned long long bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        int prior = 0;
        r[it] = -1;
        if (act) {
            prior = my_hist[e[it]];
            r[it] = prior + __popcll(peers & lt_mask);
        }
        __builtin_amdgcn_wave_barrier();
        if (act && (peers >> lane) == 1ull) {
            my_hist[e[it]] = prior + __popcll(peers);
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int ee = tid; ee < E; ee += kLocalThreads) {
        int run = 0;
#pragma unroll
        for (int ww = 0; ww < kLocalWaves; ++ww) {
            const int t = hist[ww * kMaxExperts + ee];
            hist[ww * kMaxExperts + ee] = run;
            run += t;
        }
        hist_row[ee] = run;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const long long i = base + it * kWave + lane;
        if (i < n_all) {
            const int v = e[it] >= 0 ? r[it] + my_hist[e[it]] : -1;
            pos_out[i] = v;
        }
    }
}

// What the ids say about one expert, found by one workgroup of NT threads that looks at all of them.  Wave w owns the IT * 64
// entries from w * IT * 64 on and a lane keeps its ids in registers.  The number of entries that name an earlier expert is
// the expert's offset, the number of earlier ones that name it the rank of an entry: counts of ballots, with no table and no
// atomics, so the work does not depend on how the ids are spread.  What bounds it are its instructions, about ten for 64 ids (with
// range checks and 64-bit addresses at every load it were forty).
template <int NT, int IT>
struct ExpertEntries {
    int e[IT];     // ids, none of 0 .. E - 1 where an entry names no expert
    int off, cnt;  // the expert's first row and its entries
    int prior;     // of its entries, those in front of this wave's

    static __device__ __forceinline__ int first_entry()
    {
        return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (IT * kWave);
    }

    // (n_all <= NT * IT; entries beyond it are read as zeros, see only_first)
    template <typename IdT>
    __device__ __forceinline__ void load(const IdT *idx, int n_all)
    {
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)idx, 0, n_all * (int)sizeof(IdT), 0x00020000);
        const int at = (first_entry() + (int)(threadIdx.x & (kWave - 1))) * (int)sizeof(IdT);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            if constexpr (sizeof(IdT) == 8) {
                const v2u v = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at + it * kWave * 8, 0, 0));
                e[it] = v[1] == 0u ? (int)v[0] : -1;
            } else {
                e[it] = (int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, at + it * kWave * 4, 0, 0);
            }
        }
    }

    // Entries from n on name no expert.
    __device__ __forceinline__ void only_first(int n)
    {
        if (first_entry() + IT * kWave > n) {
            const int i = first_entry() + (int)(threadIdx.x & (kWave - 1));
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                e[it] = i + it * kWave < n ? e[it] : -1;
            }
        }
    }

    // scratch: 2 * NT / 64 ints of LDS
    __device__ __forceinline__ void count(int x, int *scratch)
    {
        constexpr int kWaves = NT / kWave;
        const int lane = threadIdx.x & (kWave - 1);
        const int w = threadIdx.x >> 6;
        int below = 0, own = 0;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            below += (unsigned)e[it] < (unsigned)x ? 1 : 0;
            own += __popcll(__ballot(e[it] == x));
        }
        below = wave_sum(below);
        if (lane == 0) {
            scratch[w] = below;
            scratch[kWaves + w] = own;
        }
        __syncthreads();
        off = wave_sum(lane < kWaves ? scratch[lane] : 0);
        const int inc = wave_inclusive_scan(lane < kWaves ? scratch[kWaves + lane] : 0);
        cnt = wave_last(inc);
        prior = __shfl(inc, w, kWave) - own;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            asm volatile("" : "+v"(e[it]));  // ranks() compares anew: the masks would take two scalar registers each until then
        }
    }

    // f(entry) for every entry of none of E experts
    template <typename F>
    __device__ __forceinline__ void of_no_expert(int E, int n_all, F &&f)
    {
        const int base = first_entry() + (int)(threadIdx.x & (kWave - 1));
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            if ((unsigned)e[it] >= (unsigned)E && base + it * kWave < n_all) {
                f(base + it * kWave);
            }
        }
    }

    // f(entry, rank) for every entry of the expert
    template <typename F>
    __device__ __forceinline__ void ranks(int x, F &&f)
    {
        const int lane = threadIdx.x & (kWave - 1);
        const int base = first_entry() + lane;
        const unsigned long long lt_mask = (1ull << lane) - 1ull;
        int run = __builtin_amdgcn_readfirstlane(prior);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const unsigned long long named = __ballot(e[it] == x);
            if (named != 0) {
                if (e[it] == x) {
                    f(base + it * kWave, run + __popcll(named & lt_mask));
                }
                run += __popcll(named);
            }
        }
    }
};

}  // namespace cam

#endif  // CAM_RANK_DEVICE_H_
