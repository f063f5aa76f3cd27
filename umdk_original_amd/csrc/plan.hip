// Routing plan kernels: per-expert counts, prefix offsets, the stable within-expert rank of every
// (token, k) entry and receive bookkeeping.
//
// Reference semantics restated here (paths relative to the reference tree):
//   counts        src/cam/comm_operator/ascend_kernels/dispatch_layout/op_kernel/dispatch_layout.h:83-134
//   offsets       src/cam/comm_operator/ascend_kernels/notify_dispatch/op_kernel/notify_dispatch.h:121-152
//   ranks         src/cam/comm_operator/pybind/moe_dispatch_prefill.cpp:96-112 (a CPU loop there)
//   recv cumsum   src/cam/comm_operator/pybind/moe_dispatch_prefill.cpp:126-145
//
// Design.  The rank of an entry is its position among earlier flat (t,k) entries with the same
// expert id, i.e. a stable counting sort; atomics would make the order depend on scheduling.  Up to kExpertIds ids one
// launch, in which a workgroup per expert looks at all of them (plan_experts_kernel); beyond, two
// short launches, no atomics on results, no spinning, fully deterministic:
//   1. every workgroup ranks its own contiguous chunk of the flat id sequence (wave ballots + per-wave
//      LDS histograms) and publishes the chunk's per-expert histogram;
//   2. every workgroup sums the histograms of the chunks before it (its base), scans the per-expert
//      totals into offsets, and finishes its chunk.  The reference does this part on the CPU after a
//      device-to-host copy.
#include <algorithm>
#include <type_traits>

#include "cam_device.h"
#include "cam_kernels.h"
#include "permute_device.h"
#include "rank_device.h"
#include "sched_device.h"

namespace cam {

namespace {

constexpr int kScanThreads = 1024;  // single-workgroup scan kernel (notify)
constexpr int kGlobalThreads = 512; // phase 2: one thread per expert column
constexpr int kExpertThreads = 1024;  // of a workgroup that looks at all ids for one expert,
constexpr int kExpertIds = 16 * kExpertThreads;  // and up to how many there are such

// Phase 1.  Workgroup b ranks the flat entries [b*chunk, (b+1)*chunk), chunk = IT*256 (rank_chunk), and
// publishes the chunk's per-expert histogram in hist_out[b][*].
template <typename IdT, int IT>
__global__ __launch_bounds__(kLocalThreads) void plan_local_kernel(PlanArgs a, int32_t *hist_out)
{
    __shared__ int hist[kLocalWaves * kMaxExperts];
    __shared__ int active_s;
    const int tid = threadIdx.x;
    const int b = blockIdx.x;
    const int t_active = count_active(a.mask, a.T, tid, kLocalThreads, &active_s);
    rank_chunk<IdT, IT>((const IdT *)a.idx, b, (long long)t_active * a.K, (long long)a.T * a.K, a.E, hist, a.pos,
                        hist_out + (long long)b * a.E);
    if (b == 0 && tid == 0) {
        hist_out[(long long)gridDim.x * a.E] = t_active;
    }
}

// What phase 2 does besides in a layer: its first sched.nspec * sched.parts workgroups build the schedules of the GEMMs (from
// the counts, which they add up like all the others), and the others leave the token of every row where GMM1 gathers.
struct LayerPlan {
    int32_t *row_token;  // or null
    SchedBuild sched;
};

// A wave per token: what the workgroups of a layer's plan behind those that rank do.
constexpr int kMaskedTokens = 16384;  // up to where a workgroup looks through the whole mask, as long as its four tokens at 2048 columns
template <int CHUNKS, int QUANT, int ACT, bool PLAIN, int NT>
__device__ __forceinline__ void quantise_token(const PlanArgs &a, const DispatchArgs &d, int block, int *active_s)
{
    typedef TokenRow<CHUNKS, kWave> Row;
    const int tid = threadIdx.x;
    const int t = block * (NT / kWave) + (tid >> 6);
    const int lane = tid & (kWave - 1);
    // A token that goes nowhere, behind the active ones or without an expert, is not stored.  us, stored / not, layers of which one token
    // in sixteen goes somewhere: 8192 x 7168 to 64 experts, top-2, 229.3 / 217.0 under a mask and 240.5 / 232.0 with ids dropped, 5000 to
    // 8, top-1, 183.6 / 175.6 and 191.3 / 184.7 (when layers permuted their rows 228.6, 233.3, 179.8 and 185.3).
    Row r;
    const int at = min(t, a.T - 1);
    const int id = ((const int32_t *)a.idx)[(long long)at * a.K + min(lane, a.K - 1)];  // looked at when the row is under way
    load_token_row(d.x, at, d.H, lane, r);
    const int t_active = a.T <= kMaskedTokens ? count_active(a.mask, a.T, tid, NT, active_s) : a.T;
    if (t >= t_active || !__any(id >= 0 && id < a.E)) {
        return;
    }
    quant_token_row<QUANT, ACT>(r, WaveMax());
    const int nch = d.H >> 3;
    v2u *dst = (v2u *)((int8_t *)d.out + (long long)t * d.H);
#pragma unroll
    for (int j = 0; j < Row::kChunks; ++j) {
        const int c = j * kWave + lane;
        if (c < nch) {
            store_piece<PLAIN>(r.q[j], dst + c);
        }
    }
    if (QUANT == 3) {
        store_row_scales8(r, (uint8_t *)d.scales, t, d.H, lane);
    } else if (lane == 0) {
        d.scales[t] = r.scale_out;
    }
}

// Phase 1 of a layer whose gate/up GEMM gathers its rows: the workgroups behind the nb that rank quantise the tokens, a wave each,
// which depends on nothing that the plan finds out.  A token's row is stored once, not once per copy, and non-temporally up to 256 rows
// per expert (quantised_plainly).
// HBM bound where there are many tokens.  us, ranks + their second half + permute with schedules -> this + phase 2 with schedules
// (plain stores): 8192 tokens x 4096, top-8, int8 7.6 + 6.3 + 70.9 -> 20.9 + 15.5 (layer 1512 -> 1474); 4093 in FP8 5.5 + 5.8 + 45.0
// -> 15.5 + 13.5 (823 -> 787); 1021 x 2048, top-6, 4.8 + 4.8 + 9.1 -> 5.0 + 7.5 (160.9 -> 158.9).  With rows of 4096 columns in the
// registers for 7168, at 3 (FP8) and 4 waves a SIMD, FP8 took 19.2.
//
// Up to kWholePlanIds ids this is all of the plan (nb == 0): the schedule builders count the ids by themselves, a workgroup per expert ranks its
// entries (ExpertEntries), and the workgroups behind them quantise.  Latency bound (the builders' chain) up to some thousand tokens.
// us per layer, two launches / this; T x H, top-K of E, I: 1021 x 2048, 6 of 64, 1408 159.6 / 156.3; 700 152.2 / 148.3; 2000 x 4096, 8 of 128, 1536
// 602.5 / 597.5; 4000 x 7168, 4 of 64, 2048 940 / 933; 300 x 7168, 8 of 16, 2048 222 / 215; 16384 x 1024, 1 of 16, 512 110 / 103.5; FP8 1400 x 2048, 3 of
// 8, 1024 71.4 / 65.7, 2048 x 2048, 8 of 32, 768 141.6 / 137.2.  With 64 ids a thread for up to 32768 ids the registers of the ranking workgroups
// cost the others their waves: 4093 x 4096 in FP8, 8 of 128, 782 / 797.
constexpr int kWholeThreads = 512;
constexpr int kWholePlanIds = 32 * kWholeThreads;
template <int CHUNKS, int QUANT, int ACT, bool PLAIN>
__global__ __launch_bounds__(kWholeThreads, CHUNKS > 8 ? (QUANT == 3 ? 3 : 4) : 5) void plan_quant_kernel(PlanArgs a, DispatchArgs d,
                                                                                                         LayerPlan l, int it, int nb)
{
    extern __shared__ __attribute__((aligned(16))) int lds[];   // histograms, or what the builders need
    __shared__ int scratch[2 * kWholeThreads / kWave];
    __shared__ int active_s;
    const int tid = threadIdx.x;
    if (nb > 0) {  // kLocalThreads a workgroup
        const int b = blockIdx.x;
        if (b >= nb) {
            quantise_token<CHUNKS, QUANT, ACT, PLAIN, kLocalThreads>(a, d, b - nb, &active_s);
            return;
        }
        const int t_active = count_active(a.mask, a.T, tid, kLocalThreads, &active_s);
        auto rank = [&](auto ic) {
            rank_chunk<int32_t, decltype(ic)::value>((const int32_t *)a.idx, b, (long long)t_active * a.K, (long long)a.T * a.K,
                                                     a.E, lds, a.pos, a.hist_ws + (long long)b * a.E);
        };
        switch (it) {
            case 2: rank(std::integral_constant<int, 2>()); break;
            case 4: rank(std::integral_constant<int, 4>()); break;
            default: rank(std::integral_constant<int, 8>()); break;
        }
        if (b == 0 && tid == 0) {
            a.hist_ws[(long long)nb * a.E] = t_active;
        }
        return;
    }
    SchedShared &sched_s = *(SchedShared *)lds;
    const int builders = l.sched.nspec * l.sched.parts;
    const int x = (int)blockIdx.x - builders;
    if (x >= a.E) {
        quantise_token<CHUNKS, QUANT, ACT, PLAIN, kWholeThreads>(a, d, x - a.E, &active_s);
        return;
    }
    const int n_all = a.T * a.K;
    auto plan = [&](auto ic) {
        ExpertEntries<kWholeThreads, decltype(ic)::value> ids;
        ids.load((const int32_t *)a.idx, n_all);
        const int t_active = count_active(a.mask, a.T, tid, kWholeThreads, &active_s);
        ids.only_first(t_active * a.K);
        if (x < 0) {
            for (int e = tid; e < a.E; e += kWholeThreads) {
                sched_s.order[e] = 0;
            }
            __syncthreads();
#pragma unroll
            for (int it = 0; it < decltype(ic)::value; ++it) {
                // the lanes that name what the first one names are counted together: top-1 ids that are all the same one by one took
                // a layer of 16384 tokens x 1024 from 94.5 to 97.6 us
                const int some = __builtin_amdgcn_readfirstlane(ids.e[it]);
                const unsigned long long alike = __ballot(ids.e[it] == some);
                const bool first = (alike & ((1ull << (tid & (kWave - 1))) - 1ull)) == 0;
                if ((unsigned)ids.e[it] < (unsigned)a.E && (ids.e[it] != some || first)) {
                    atomicAdd(&sched_s.order[ids.e[it]], ids.e[it] == some ? __popcll(alike) : 1);
                }
            }
            return;
        }
        ids.count(x, scratch);
        if (tid < 2) {  // 64 bits, a word a lane
            ((int32_t *)(a.tokens_per_expert + x))[tid] = tid == 0 ? ids.cnt : 0;
        }
        if (tid == 0 && x == a.E - 1) {
            a.meta[0] = 0;
            a.meta[1] = ids.off + ids.cnt;
            a.meta[2] = t_active;
            a.meta[3] = 0;
        }
        ids.ranks(x, [&](int i, int rank) {
            a.dst_row[i] = ids.off + rank;
            l.row_token[ids.off + rank] = (int)((unsigned)i / (unsigned)a.K);
        });
        if (x == 0) {
            ids.of_no_expert(a.E, n_all, [&](int i) { a.dst_row[i] = -1; });
        }
    };
    if (n_all <= 12 * kWholeThreads) {
        plan(std::integral_constant<int, 12>());
    } else {
        plan(std::integral_constant<int, 32>());
    }
    if (x < 0) {
        __syncthreads();
        build_sched_part<kWholeThreads>(sched_s, l.sched, (int)blockIdx.x / l.sched.parts, (int)blockIdx.x % l.sched.parts, l.sched.parts);
    }
}

// Phase 2.  Every workgroup sums the histogram columns (all rows for the per-expert count, the rows
// before its own for its base), scans the counts into offsets, and finishes its own chunk:
// pos += base[e], dst_row = off[e] + pos.  Workgroup 0 also writes the per-expert outputs (counts, offsets,
// cumulative group list, receive bookkeeping), the total row count and the four words of the receive metadata.
template <typename IdT, bool LAYER>
__global__ __launch_bounds__(kGlobalThreads) void plan_global_kernel(PlanArgs a, int chunk, const int32_t *hist_in, LayerPlan l)
{
    constexpr int NW = kGlobalThreads / kWave;
    __shared__ int base_s[kMaxExperts];
    __shared__ int off_s[kMaxExperts];
    __shared__ int scan_s[NW];
    __shared__ int total_s;
    const int tid = threadIdx.x;
    const int builders = LAYER ? l.sched.nspec * l.sched.parts : 0;
    const int b = (int)blockIdx.x - builders;
    const int nb = (int)gridDim.x - builders;
    const int E = a.E;
    const IdT *__restrict__ idx = (const IdT *)a.idx;

    // This thread's first entry of the chunk is requested before the histogram columns, so that its round trip
    // to memory runs beside theirs instead of after the scan.
    const long long n_all = (long long)a.T * a.K;
    const long long lo = (long long)b * chunk;
    const long long hi = min(n_all, lo + chunk);
    const long long i0 = lo + tid;
    long long raw0 = -1;
    int pos0 = 0;
    if (b >= 0 && i0 < hi) {
        raw0 = (long long)idx[i0];
        pos0 = a.pos[i0];
    }

    int cnt = 0, base = 0;
    if (tid < E) {
        const int32_t *col = hist_in + tid;
        int bb = 0;
        for (; bb + 64 <= nb; bb += 64) {  // 64 independent loads in flight per thread: one round trip at C2
            int v[64];
#pragma unroll
            for (int j = 0; j < 64; ++j) {
                v[j] = col[(long long)(bb + j) * E];
            }
#pragma unroll
            for (int j = 0; j < 64; ++j) {
                cnt += v[j];
                base += (bb + j) < b ? v[j] : 0;
            }
        }
        if (bb < nb) {  // what is left, in one round trip as well: eight at a time as far as there are rows, the last one repeated
            int v[64];
#pragma unroll
            for (int q = 0; q < 64; q += 8) {
                if (bb + q < nb) {
#pragma unroll
                    for (int j = q; j < q + 8; ++j) {
                        v[j] = col[min(bb + j, nb - 1) * E];
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 64; q += 8) {
                if (bb + q < nb) {
#pragma unroll
                    for (int j = q; j < q + 8; ++j) {
                        cnt += bb + j < nb ? v[j] : 0;
                        base += bb + j < b ? v[j] : 0;
                    }
                }
            }
        }
    }
    if constexpr (LAYER) {
        if (b < 0) {
            __shared__ SchedShared sched_s;
            if (tid < E) {
                sched_s.order[tid] = cnt;
            }
            __syncthreads();
            build_sched_part<kGlobalThreads>(sched_s, l.sched, (int)blockIdx.x / l.sched.parts,
                                             (int)blockIdx.x % l.sched.parts, l.sched.parts);
            return;
        }
    }
    const int off = block_exclusive_scan<NW>(cnt, tid, scan_s, &total_s);
    const int total = total_s;
    base_s[tid] = base;
    off_s[tid] = off;
    __syncthreads();

    const int t_active = hist_in[(long long)nb * E];
    const long long n = (long long)t_active * a.K;
    for (long long i = i0; i < hi; i += kGlobalThreads) {
        int e, p0;
        if (i == i0) {
            e = (i < n && raw0 >= 0 && raw0 < (long long)E) ? (int)raw0 : -1;
            p0 = pos0;
        } else {
            e = i < n ? load_id(idx, i, E) : -1;
            p0 = e >= 0 ? a.pos[i] : 0;
        }
        int row = -1;
        if (e >= 0) {
            const int p = p0 + base_s[e];
            a.pos[i] = p;
            row = off_s[e] + p;
            if (LAYER && l.row_token != nullptr) {
                l.row_token[row] = (int)((unsigned)i / (unsigned)a.K);
            }
        }
        if (a.dst_row != nullptr) {
            a.dst_row[i] = row;
        }
    }
    if (b != 0) {
        return;
    }
    clear_stream_queues(a, tid, kGlobalThreads);
    if (tid < E) {
        if (a.cnt) a.cnt[tid] = cnt;
        if (a.off) a.off[tid] = off;
        if (a.recv_off) a.recv_off[tid] = off;
        if (a.recv_count) a.recv_count[tid] = off + cnt;
        if (a.tokens_per_expert) store_count(a.tokens_per_expert + tid, cnt);
        if (a.group_list) a.group_list[tid] = (int64_t)off + cnt;
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

// Both phases in one launch with a workgroup per expert, each of which looks at all ids (ExpertEntries): it finds the expert's
// offset, count and ranks by itself, so nothing passes between workgroups.  Bound by latency, and from some ten thousand ids on by
// its instructions: every workgroup goes through all ids, which is why the two launches come back beyond kExpertIds.  us, replayed
// from a graph, two launches (up to 1024 ids one workgroup) / this, ids spread over the experts: 64 ids to 8 experts 3.0 / 2.7, 1024 to 128
// 5.7 / 2.9, 2400 to 64 5.7 / 2.9, 6126 to 64 5.9 / 3.3, 11994 to 64 6.5 / 4.0, 16384 to 256 6.5 / 4.4 (all the same ids 6.4 / 4.7); with 32 and
// 64 ids a thread, 32768 to 256 7.2 / 6.7 (7.2 / 7.3), 48000 to 64 8.6 / 12.9, 64000 to 256 9.9 / 11.8, to 8 8.3 / 15.6.
template <typename IdT, int IT>
__global__ __launch_bounds__(kExpertThreads, 8) void plan_experts_kernel(PlanArgs a)
{
    __shared__ int scratch[2 * kExpertThreads / kWave];
    __shared__ int active_s;
    const int tid = threadIdx.x;
    const int x = blockIdx.x;
    const int n_all = a.T * a.K;
    ExpertEntries<kExpertThreads, IT> ids;
    ids.load((const IdT *)a.idx, n_all);
    const int t_active = count_active(a.mask, a.T, tid, kExpertThreads, &active_s);
    ids.only_first(t_active * a.K);
    ids.count(x, scratch);
    if (tid == 0) {
        const int end = ids.off + ids.cnt;
        if (a.tokens_per_expert) store_count(a.tokens_per_expert + x, ids.cnt);
        if (a.cnt) a.cnt[x] = ids.cnt;
        if (a.off) a.off[x] = ids.off;
        if (a.recv_off) a.recv_off[x] = ids.off;
        if (a.recv_count) a.recv_count[x] = end;
        if (a.group_list) a.group_list[x] = (int64_t)end;
        if (x == a.E - 1) {
            if (a.total) {
                a.total[0] = end;
            }
            if (a.meta != nullptr) {
                a.meta[0] = 0;
                a.meta[1] = end;
                a.meta[2] = t_active;
                a.meta[3] = 0;
            }
        }
    }
    ids.ranks(x, [&](int i, int rank) {
        a.pos[i] = rank;
        if (a.dst_row != nullptr) {
            a.dst_row[i] = ids.off + rank;
        }
    });
    if (x == a.E - 1) {
        clear_stream_queues(a, tid, kExpertThreads);
    }
    if (x == 0) {
        ids.of_no_expert(a.E, n_all, [&](int i) {
            a.pos[i] = -1;
            if (a.dst_row != nullptr) {
                a.dst_row[i] = -1;
            }
        });
    }
}

// The layout of up to kExpertIds ids in one launch: a workgroup per expert that looks at all ids and counts its own, and one per rank
// that marks the tokens with an id of the rank's experts in LDS, counts them and stores their flags.  Nothing passes between
// workgroups.  Latency bound: one round trip to the ids and, for a rank, one through LDS.  With very many flags a workgroup per rank
// stores too many by itself.  us, replayed from a graph, two launches (up to some hundred tokens one workgroup) / this, T tokens, top-K of E, R ranks,
// ids spread; they differ by 0.3 at most where all tokens name the same: 1, 8 of 128, 1 3.2 / 2.3; 1024, 1 of 64, 1 3.1 / 2.2; 1999, 6 of 64, 1 5.2 /
// 3.1; 2048, 8 of 512, 1 5.9 / 4.4; 16384, 1 of 128, 1 5.9 / 4.7; 2048, 8 of 256, 16 6.6 / 4.2, 64 8.1 / 4.9; 1024, 16 of 256, 128 12.9 / 4.6; 100, 2
// of 384, 384 7.0 / 3.7; 5000, 1 of 64, 64 (320000 flags) 6.4 / 5.6, but 16384, 1 of 128, 16 (262144) 6.1 / 7.2 and 8000, 2 of 384, 384 16.7 /
// 21.5.  Prefill operators, 1999 tokens x 4096, top-6 of 64: 51.9 -> 49.1.
constexpr long long kExpertFlags = 8 * kExpertIds;
template <typename IdT, typename OutT, int IT>
__global__ __launch_bounds__(kExpertThreads, 8) void layout_experts_kernel(LayoutArgs a)
{
    __shared__ __attribute__((aligned(16))) uint8_t token_s[kExpertIds];
    __shared__ int count_s[kExpertThreads / kWave];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int x = blockIdx.x;
    const int n_all = a.T * a.K;
    ExpertEntries<kExpertThreads, IT> ids;
    ids.load((const IdT *)a.idx, n_all);
    int count = 0;
    if (x < a.E) {
        ids.only_first(n_all);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            count += __popcll(__ballot(ids.e[it] == x));
        }
    } else {
        for (int i = tid; i < (a.T + 15) >> 4; i += kExpertThreads) {
            ((v4u *)token_s)[i] = v4u{0u, 0u, 0u, 0u};
        }
        __syncthreads();
        const int rank = x - a.E;
        const unsigned epr = (unsigned)(a.E / a.R);
        const float inv = 1.0f / (float)a.K;
        const int base = ids.first_entry() + lane;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int i = base + it * kWave;
            if (i < n_all && (unsigned)ids.e[it] - (unsigned)rank * epr < epr) {
                token_s[(int)(((float)i + 0.5f) * inv)] = 1;   // i / K: exact below 2^15
            }
        }
        __syncthreads();
        OutT *out = (OutT *)a.in_rank + rank;
        for (int t0 = 0; t0 < a.T; t0 += kExpertThreads) {
            const int t = t0 + tid;
            const int in = t < a.T ? token_s[t] : 0;
            if (t < a.T) {
                out[(long long)t * a.R] = (OutT)in;
            }
            count += __popcll(__ballot(in != 0));
        }
    }
    if (lane == 0) {
        count_s[tid >> 6] = count;
    }
    __syncthreads();
    if (tid < kWave) {
        count = wave_sum(lane < kExpertThreads / kWave ? count_s[lane] : 0);
        if (lane == 0) {
            (x < a.E ? a.per_expert[x] : a.per_rank[x - a.E]) = count;
        }
    }
}

// The layout (dispatch_layout.h:83-134): entries per expert, tokens per rank (a token counts once per rank) and
// isTokenInRank[t,r], of more ids or flags.  A workgroup counts the `span` tokens from its own first on in LDS and leaves its
// counts, experts then ranks, in a row of `partial`; layout_sum_kernel adds the rows up.
constexpr int kLayoutThreads = 256;
template <typename IdT, typename OutT>
__global__ __launch_bounds__(kLayoutThreads) void layout_kernel(LayoutArgs a, int span)
{
    __shared__ int count_s[kMaxExperts + kMaxRanks];
    const int tid = threadIdx.x;
    const int t0 = (int)blockIdx.x * span;
    const int t1 = min(a.T, t0 + span);
    const int E = a.E, R = a.R, K = a.K;
    const int epr = E / R;
    OutT *out = (OutT *)a.in_rank;
    for (int c = tid; c < E + R; c += kLayoutThreads) {
        count_s[c] = 0;
    }
    for (long long i = (long long)t0 * R + tid; i < (long long)t1 * R; i += kLayoutThreads) {
        out[i] = (OutT)0;
    }
    __syncthreads();
    for (int t = t0 + tid; t < t1; t += kLayoutThreads) {
        const IdT *ids = (const IdT *)a.idx + (long long)t * K;
        int e[kMaxTopk];
#pragma unroll
        for (int k = 0; k < kMaxTopk; ++k) {  // all of a token's ids in one round trip
            e[k] = k < K ? load_id(ids, k, E) : -1;
        }
#pragma unroll
        for (int k = 0; k < kMaxTopk; ++k) {
            if (e[k] < 0) {
                continue;
            }
            atomicAdd(&count_s[e[k]], 1);
            const int r = e[k] / epr;
            bool seen = false;
#pragma unroll
            for (int j = 0; j < k; ++j) {
                seen = seen || (e[j] >= r * epr && e[j] < (r + 1) * epr);
            }
            if (!seen) {
                out[(long long)t * R + r] = (OutT)1;
                atomicAdd(&count_s[E + r], 1);
            }
        }
    }
    __syncthreads();
    for (int c = tid; c < E + R; c += kLayoutThreads) {
        a.partial[(long long)blockIdx.x * (E + R) + c] = count_s[c];
    }
}

__global__ __launch_bounds__(kWave) void layout_sum_kernel(LayoutArgs a, int rows)
{
    const int c = (int)blockIdx.x * kWave + threadIdx.x;
    const int width = a.E + a.R;
    if (c >= width) {
        return;
    }
    constexpr int kAtOnce = 32;
    int sum = 0;
    for (int b = 0; b < rows; b += kAtOnce) {
        int v[kAtOnce];
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            v[j] = b + j < rows ? a.partial[(long long)(b + j) * width + c] : 0;
        }
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            sum += v[j];
        }
    }
    if (c < a.E) {
        a.per_expert[c] = sum;
    } else {
        a.per_rank[c - a.E] = sum;
    }
}

// Workgroups of a layout and tokens of each, 0 where a workgroup per expert and per rank does all of it in one launch: one round of
// tokens per workgroup up to 64 of them, whose counts are two round trips to add up.  Up to 1024 tokens it is one launch where the
// counts of the tokens beyond 256 are few, a line that one workgroup alone once set and the tests keep: beyond it two launches take 2
// to 8 us longer (1024 tokens, top-6 of 64 5.1 / 2.5).
int layout_workgroups(long long T, int K, int R, int *span)
{
    const int counts = R > 1 ? 2 * K : K;
    const bool one_launch = T <= 1024 ? T * R <= 8192 && counts <= 20 && (T - kLayoutThreads) * counts <= 1024
                                      : T * K <= kExpertIds && T * R <= kExpertFlags;
    if (one_launch || T <= kLayoutThreads) {
        return 0;
    }
    const long long rounds = std::max<long long>((T + 64 * kLayoutThreads - 1) / (64 * kLayoutThreads), 1);
    *span = (int)(rounds * kLayoutThreads);
    return (int)((T + *span - 1) / *span);
}

__global__ __launch_bounds__(kScanThreads) void notify_scan_kernel(const int32_t *cnt, int E, int num_tokens,
                                                                  int32_t *off, int32_t *send_data,
                                                                  int32_t *recv_data)
{
    __shared__ int scan_s[kScanThreads / kWave];
    __shared__ int total_s;
    const int tid = threadIdx.x;
    int c = tid < E ? cnt[tid] : 0;
    int o = block_exclusive_scan<kScanThreads / kWave>(c, tid, scan_s, &total_s);
    if (tid < E) {
        if (off) off[tid] = o;
        if (send_data) {
            send_data[3 * tid + 0] = c;
            send_data[3 * tid + 1] = o;
            send_data[3 * tid + 2] = num_tokens;
        }
        if (recv_data) {
            recv_data[3 * tid + 0] = c;
            recv_data[3 * tid + 1] = o;
            recv_data[3 * tid + 2] = num_tokens;
        }
    }
}

template <typename IdT>
hipError_t launch_plan_local(const PlanArgs &a, int it, int nb, int32_t *hist, hipStream_t stream)
{
    const dim3 grid(nb), blk(kLocalThreads);
    switch (it) {
        case 2: hipLaunchKernelGGL((plan_local_kernel<IdT, 2>), grid, blk, 0, stream, a, hist); break;
        case 4: hipLaunchKernelGGL((plan_local_kernel<IdT, 4>), grid, blk, 0, stream, a, hist); break;
        case 8: hipLaunchKernelGGL((plan_local_kernel<IdT, 8>), grid, blk, 0, stream, a, hist); break;
        default: return hipErrorInvalidValue;  // (up to kExpertIds ids come to no second launch)
    }
    return hipGetLastError();
}

// f(IT), the ids a thread of a workgroup that looks at all n keeps, n <= kExpertIds.
template <typename F>
void with_ids_per_thread(long long n, F &&f)
{
    if (n <= 4 * kExpertThreads) {
        f(std::integral_constant<int, 4>());
    } else if (n <= 8 * kExpertThreads) {
        f(std::integral_constant<int, 8>());
    } else if (n <= 12 * kExpertThreads) {
        f(std::integral_constant<int, 12>());
    } else {
        f(std::integral_constant<int, 16>());
    }
}

template <typename IdT>
hipError_t launch_plan_experts(const PlanArgs &a, hipStream_t stream)
{
    with_ids_per_thread((long long)a.T * a.K, [&](auto it) {
        hipLaunchKernelGGL((plan_experts_kernel<IdT, decltype(it)::value>), dim3(a.E), dim3(kExpertThreads), 0, stream, a);
    });
    return hipGetLastError();
}

template <typename IdT>
hipError_t launch_plan_t(const PlanArgs &a, int it, int nb, int32_t *hist, hipStream_t stream)
{
    const dim3 grid(nb), blk(kLocalThreads);
    const hipError_t e = launch_plan_local<IdT>(a, it, nb, hist, stream);
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL((plan_global_kernel<IdT, false>), grid, dim3(kGlobalThreads), 0, stream, a, it * kLocalThreads,
                       (const int32_t *)hist, LayerPlan{});
    return hipGetLastError();
}

// Whether the tokens of a layer that gathers are stored plainly: tiles of experts of few rows, which stream their weights, are slower
// behind plain stores, taller ones take as long or less.  Layers, us, plain / non-temporal, rows per expert in front: 23 3000 tokens x 4096 to 128
// experts, top-1 257.2 / 249.1; 31 2000, top-2 258.5 / 252.6; 47 3000 x 3072, top-2 224.9 / 218.6 (FP8 220.6 / 213.6); 37 1200 x 7168 to 32,
// top-1 284.3 / 278.2; 128 8192 x 2048 to 64, top-1 157.0 / 152.8; 187 4000 x 3072, top-3 232.8 / 226.9; 256 8192 x 7168, top-2 421.5 / 410.3
// and 4093 x 4096 to 128, top-8 938.6 / 932.4.  312 2500 x 4096 to 16, top-2 197.3 / 197.1; 512 8192 x 4096 to 128, top-8 1417 / 1418;
// 512 8192 x 1536 to 32, top-2 120.7 / 122.2 (FP8 113.3 / 112.9); 700 700 x 7168 to 4, top-4 257.1 / 259.2; 1024 8192 x 1024 to 16, top-2 103.6 /
// 104.8, 8192 to 32, top-4 149.3 / 152.3; 2048 8192 x 2048 to 16, top-4 220.0 / 223.0.
bool quantised_plainly(const PlanArgs &p) { return (long long)p.T * p.K > 256ll * p.E; }

template <int QUANT, int ACT, bool PLAIN>
hipError_t launch_plan_quant_as(const PlanArgs &p, const DispatchArgs &d, const LayerPlan &l, int it, int nb, hipStream_t stream)
{
    const int threads = nb > 0 ? kLocalThreads : kWholeThreads, tokens = threads / kWave;
    const int ahead = nb > 0 ? nb : l.sched.nspec * l.sched.parts + p.E;
    const size_t lds = nb > 0 ? kLocalWaves * kMaxExperts * sizeof(int) : sizeof(SchedShared);
    const dim3 grid((unsigned)(ahead + (d.T + tokens - 1) / tokens)), block((unsigned)threads);
    // rows of up to 4096 columns in registers for 4096: more waves to a SIMD
    if (d.H <= 8 * kWave * 8) {
        hipLaunchKernelGGL((plan_quant_kernel<8, QUANT, ACT, PLAIN>), grid, block, lds, stream, p, d, l, it, nb);
    } else {
        hipLaunchKernelGGL((plan_quant_kernel<kDispMaxChunks, QUANT, ACT, PLAIN>), grid, block, lds, stream, p, d, l, it, nb);
    }
    return hipGetLastError();
}

template <bool PLAIN>
hipError_t launch_plan_quant(const PlanArgs &p, const DispatchArgs &d, const LayerPlan &l, int it, int nb, hipStream_t stream)
{
    if (d.quant == 3) {
        return launch_plan_quant_as<3, 0, PLAIN>(p, d, l, it, nb, stream);
    }
    return d.x_is_fp16 ? launch_plan_quant_as<2, 1, PLAIN>(p, d, l, it, nb, stream)
                       : launch_plan_quant_as<2, 0, PLAIN>(p, d, l, it, nb, stream);
}

}  // namespace

void plan_geometry(long long n_all, int *it_out, int *nb_out)
{
    int it = 1;
    if (n_all <= 4 * kLocalThreads) {
        while ((long long)it * kLocalThreads < n_all) {
            it *= 2;
        }
    } else {
        while (it < 8 && (n_all + (long long)it * kLocalThreads - 1) / ((long long)it * kLocalThreads) > 64) {
            it *= 2;
        }
    }
    long long nb = (n_all + (long long)it * kLocalThreads - 1) / ((long long)it * kLocalThreads);
    *it_out = it;
    *nb_out = (int)(nb < 1 ? 1 : nb);
}

uint64_t plan_workspace_bytes(int64_t T, int64_t K, int E)
{
    int it, nb;
    plan_geometry(T * K, &it, &nb);
    return ((uint64_t)nb * (uint64_t)E + 4) * sizeof(int32_t);
}

hipError_t launch_plan(const PlanArgs &a, hipStream_t stream)
{
    if (a.hist_ws == nullptr) {
        return hipErrorInvalidValue;
    }
    if ((long long)a.T * a.K <= kExpertIds) {
        return a.idx_is64 ? launch_plan_experts<int64_t>(a, stream) : launch_plan_experts<int32_t>(a, stream);
    }
    int it, nb;
    plan_geometry((long long)a.T * a.K, &it, &nb);
    if (a.idx_is64) {
        return launch_plan_t<int64_t>(a, it, nb, a.hist_ws, stream);
    }
    return launch_plan_t<int32_t>(a, it, nb, a.hist_ws, stream);
}

hipError_t launch_layer_plan(const PlanArgs &p, const DispatchArgs &d, int32_t *row_token, const SchedSpec *specs,
                             hipStream_t stream)
{
    if (p.hist_ws == nullptr || p.idx_is64 || p.T <= 0 || d.T != p.T || p.E <= 0 || p.E > kMaxExperts ||
        d.H % 8 != 0 || d.H / 8 > kDispMaxChunks * kWave || (d.quant != 2 && d.quant != 3) ||
        (d.quant == 3 && (d.H % 128 != 0 || d.x_is_fp16))) {
        return hipErrorInvalidValue;
    }
    int it, nb;
    plan_geometry((long long)p.T * p.K, &it, &nb);
    LayerPlan l{};
    l.row_token = row_token;
    l.sched.G = p.E;
    l.sched.nspec = 2;
    l.sched.max_rows = (long long)p.T * p.K;
    l.sched.spec[0] = specs[0];
    l.sched.spec[1] = specs[1];
    hipError_t e = gemm_workgroups(&l.sched.queues);
    if (e != hipSuccess) {
        return e;
    }
    // a turn of items per builder workgroup where the item tables could be full: nothing else waits for the CUs, and with at
    // most 8 builders and 64-bit divisions in their turns phase 2 took 22.1 us at 8192 tokens
    const int cap = std::max(specs[0].max_items, specs[1].max_items);
    l.sched.parts = std::min(std::max((cap + kGlobalThreads - 1) / kGlobalThreads, 1), 32);
    const bool whole = row_token != nullptr && (long long)p.T * p.K <= kWholePlanIds;
    if (row_token == nullptr) {
        e = launch_plan_local<int32_t>(p, it, nb, p.hist_ws, stream);
    } else {
        const int chunks = whole ? 0 : nb;
        e = quantised_plainly(p) ? launch_plan_quant<true>(p, d, l, it, chunks, stream)
                                 : launch_plan_quant<false>(p, d, l, it, chunks, stream);
    }
    if (e != hipSuccess || whole) {
        return e;
    }
    hipLaunchKernelGGL((plan_global_kernel<int32_t, true>), dim3((unsigned)(nb + l.sched.nspec * l.sched.parts)),
                       dim3(kGlobalThreads), 0, stream, p, it * kLocalThreads, (const int32_t *)p.hist_ws, l);
    e = hipGetLastError();
    return e != hipSuccess || row_token != nullptr ? e : launch_dispatch(d, stream);
}

uint64_t layout_workspace_bytes(int64_t T, int K, int E, int R)
{
    int span;
    return (uint64_t)layout_workgroups(T, K, R, &span) * (uint64_t)(E + R) * sizeof(int32_t);
}

template <typename IdT>
void launch_layout_experts(const LayoutArgs &a, hipStream_t stream)
{
    with_ids_per_thread((long long)a.T * a.K, [&](auto it) {
        const dim3 grid((unsigned)(a.E + a.R)), block(kExpertThreads);
        if (a.in_rank_bytes == 4) {
            hipLaunchKernelGGL((layout_experts_kernel<IdT, int32_t, decltype(it)::value>), grid, block, 0, stream, a);
        } else {
            hipLaunchKernelGGL((layout_experts_kernel<IdT, uint8_t, decltype(it)::value>), grid, block, 0, stream, a);
        }
    });
}

template <typename IdT>
void launch_layout_spans(const LayoutArgs &a, int workgroups, int span, hipStream_t stream)
{
    const dim3 grid((unsigned)workgroups), block(kLayoutThreads);
    if (a.in_rank_bytes == 4) {
        hipLaunchKernelGGL((layout_kernel<IdT, int32_t>), grid, block, 0, stream, a, span);
    } else {
        hipLaunchKernelGGL((layout_kernel<IdT, uint8_t>), grid, block, 0, stream, a, span);
    }
}

hipError_t launch_layout(const LayoutArgs &a, hipStream_t stream)
{
    if (a.K > kMaxTopk || a.E > kMaxExperts || a.R > kMaxRanks) {
        return hipErrorInvalidValue;
    }
    int span = 0;
    const int n = layout_workgroups(a.T, a.K, a.R, &span);
    if (n == 0) {
        a.idx_is64 ? launch_layout_experts<int64_t>(a, stream) : launch_layout_experts<int32_t>(a, stream);
        return hipGetLastError();
    }
    if (a.partial == nullptr) {
        return hipErrorInvalidValue;
    }
    a.idx_is64 ? launch_layout_spans<int64_t>(a, n, span, stream) : launch_layout_spans<int32_t>(a, n, span, stream);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL(layout_sum_kernel, dim3((a.E + a.R + kWave - 1) / kWave), dim3(kWave), 0, stream, a, n);
    return hipGetLastError();
}

hipError_t launch_notify_scan(const int32_t *cnt, int E, int num_tokens, int32_t *off, int32_t *send_data,
                              int32_t *recv_data, hipStream_t stream)
{
    hipLaunchKernelGGL(notify_scan_kernel, dim3(1), dim3(kScanThreads), 0, stream, cnt, E, num_tokens, off,
                       send_data, recv_data);
    return hipGetLastError();
}

}  // namespace cam
