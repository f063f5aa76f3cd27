// Grouped w8a8 / FP8 GEMM for experts with few rows: a weight stream with the matrix cores beside it.
//
// Same operands, results and epilogues as gemm.hip (the reference's GMM1 / GMM2, cited there); this kernel is for
// launches whose experts have so few rows that the weights are all the time goes into.  What bounds it is the rate at
// which weight bytes arrive: HBM as a whole (7.05 TB/s for 1.5 GB of these loads with nothing else in the kernel, 6.7 for
// 240 MB), and one CU at about 50 GB/s whatever the number of loads in flight, so a launch on fewer than half the CUs is
// bound by the CUs.  The tile kernel of gemm.hip hands out 512-column panels over the whole K: 48 of them for one token
// of a 128-expert layer (H 4096, I 1536, top-8), i.e. 48 of 256 CUs at work.
//
// Measured, tile kernel -> this one: that token's GMM1 (101 MB) 55.8 -> 21 us and GMM2 24.7 -> 13 us; 16 tokens on 16
// experts (H 7168, I 2048): 123 -> 76 us (6.2 TB/s) and 41.5 -> 39 us; 512 rows over 124 experts, GMM1 248 -> 237 us
// (6.6 TB/s); 1024 rows, where both are at 6.3 TB/s, no difference.
//
// Design.
//   * An item is one row tile (32 or 128 rows) of one expert x P groups of 64 packed weight columns, chosen by the host so
//     that there are items for every CU.  The eight waves of a workgroup are P columns of S = 8 / P: the S waves of a
//     column group take every S-th 64-byte step of its K, so a workgroup always has eight streams of 4 KB steps, and
//     the sums of the S waves meet in LDS at the end (int32: exact in any order; FP8: fp32 sums added in wave order).
//   * Every weight byte is needed by exactly one wave, so it goes from memory to that wave's registers, non-temporal,
//     with no LDS and no barrier on its way.  Each wave keeps two steps (8 KB) in flight; four made no difference.  The
//     ring of two steps runs across items: while the last steps of an item are multiplied the first ones of the next are
//     already requested.
//   * The activation rows of the item lie in LDS, as much of K at a time as a buffer holds, double-buffered by
//     direct-to-LDS loads; a barrier per chunk, not per step.  Pieces of 16 bytes are placed with an XOR of the row so
//     that the fragment reads are free of bank conflicts.  The matrix cores are not what it waits for (without the
//     multiplications the decode layer's launches take the same time).
//   * No schedule: every workgroup derives the item list from the per-expert row counts by itself (a prefix sum over
//     at most 512 experts), and no builder runs before the GEMM.  All items of a launch stream the same number of bytes, but
//     workgroups do not get the same share of the memory: with all items dealt out beforehand the first was done after 172 us
//     and the last after 250, 225 on average (1.6 GB, 6 items each).  In a layer whose items make four rounds and more
//     the last quarter of the rounds is therefore taken from queues, and the items are smaller (StreamShape).
//   * In a layer whose tiles are some ten thousand products each, the GMM2 launch quantises its activations itself (PRODUCTS):
//     every workgroup reads the fp32 SwiGLU products of its tile, finds the row maxima and leaves the int8 rows in LDS while
//     its first weights are on their way.  Column blocks repeat that work, but it is a microsecond or two of latency
//     where a launch of requant_kernel takes 3.4 (layers: one token, H 4096, I 1536: 45.9 -> 44.1 us; 128 tokens on 8
//     experts, H 1024, I 512: 26.3 -> 25.1).
#include <algorithm>
#include <cmath>

#include "cam_device.h"
#include "cam_kernels.h"
#include "permute_device.h"
#include "rank_device.h"
#include "../../include/cam_expf_spec.h"

namespace cam {

namespace {

constexpr int kSThreads = 512;
constexpr int R = 2;                     // 64-byte K steps in flight per wave
constexpr int kSMaxKb = 64;              // FP8: K blocks of 128 bytes (Kd <= 8192)
constexpr int kSBuf32 = 32768;           // activation buffer of the 32-row tiles,
constexpr int kSBuf128 = 65536;          // of the 128-row tiles
constexpr int kProductQuads = 16;        // PRODUCTS: quads of products a thread holds, i.e. 32 K products a workgroup

// What the rows of a tile are padded to: the K bytes of one turn of the 8 / P waves that share the columns of an item of P groups.
constexpr int k_quantum(int P) { return 8 / P * R > 4 ? 64 * (8 / P) * R : 256; }

__device__ __forceinline__ void lds_barrier()
{
    // LDS traffic of this wave is done, weight loads stay in flight (a __syncthreads would drain them)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <typename T>
__device__ __forceinline__ unsigned lds_addr(const T *p)
{
    return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) T *)p;
}

// A wave-uniform address the compiler does not know to be one, as a scalar register pair.
__device__ __forceinline__ unsigned long long scalar_address(const void *p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Direct-to-LDS loads: lane i of the wave fetches 16 (4) bytes at base + off(i), which land at LDS byte dst + 16 i (4 i).  A
// scalar register that the vector ALU has just written (both arguments may come out of a v_readfirstlane) must not be read
// by a vector memory instruction within five wait states.  The compiler sees to that for its own instructions, not for these:
// s_mov and s_nop are the five.
__device__ __forceinline__ void load_lds16(const void *base, unsigned off, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(off), "s"(scalar_address(base))
                 : "memory", "m0");
}

__device__ __forceinline__ void load_lds4(const void *base, unsigned off, unsigned dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(off), "s"(scalar_address(base))
                 : "memory", "m0");
}

// The same value, computed anew as far as the compiler can tell: keeps loop-invariant address arithmetic out of registers.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

template <bool FP8>
struct SAcc {
    typedef v16i v16;
    typedef v4i v4;
};
template <>
struct SAcc<true> {
    typedef v16f v16;
    typedef v4f v4;
};

struct StreamItem {     // wave-uniform
    int g, row0, rows;  // expert, first row, rows of the tile (0: there is no such item)
    int blk;            // block of P column groups
    int ckb, nch;       // bytes of K per activation chunk, chunks
    const int8_t *w;    // this wave's first weight piece: expert, column group
    int wstep;          // bytes from one 64-byte K step to the next
};

// QUEUED: sa.queue is set.
template <int MF, bool FP8, int P, bool PRODUCTS, bool QUEUED>
__global__ __launch_bounds__(kSThreads, MF == 1 ? 4 : 2) void stream_gemm_kernel(StreamGemmArgs sa)
{
    typedef typename SAcc<FP8>::v16 acc16;
    typedef typename SAcc<FP8>::v4 acc4;
    constexpr int kABuf = MF == 1 ? kSBuf32 : kSBuf128;  // one of the two activation buffers
    constexpr int kSLds = 2 * kABuf;
    constexpr int NFR = MF == 1 ? 1 : 2;            // column fragments whose partial sums (32 KB each) fit a buffer
    const GemmArgs &a = sa.g;
    __shared__ __attribute__((aligned(1024))) int8_t lds[kSLds];
    __shared__ int tile_start[kMaxExperts + 1];  // row tiles of the experts before
    __shared__ int first_row[kMaxExperts + 1];
    // scales of the current and of the next item: int8 column (per group: 64, or 32 gate + 32 up) and row scales
    __shared__ __attribute__((aligned(16))) float col_scale_s[2][FP8 ? 4 : P * 64];
    __shared__ __attribute__((aligned(16))) float row_scale_s[2][FP8 ? 4 : 32 * MF];
    __shared__ __attribute__((aligned(16))) uint8_t a_scale8_s[2][FP8 ? kSMaxKb * 32 * MF : 4];
    __shared__ uint8_t w_scale8_s[FP8 ? 16 * kSMaxKb : 4];
    __shared__ int next_s;   // QUEUED: the item after the next
    __shared__ float rowmax_s[FP8 ? 8 * 32 : PRODUCTS ? 8 : 1];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = sa.G;
    constexpr int S = 8 / P;
    const int p = wave & (P - 1);      // this wave's column group of the item
    const int s = wave / P;            // and its share of K: steps s, s + S, ...
    const int Kd = a.Kd, N = a.N;
    const int KT = Kd >> 6;
    const int ngroups = N >> 6;
    const int blocks = (ngroups + P - 1) / P;
    const int turns = (KT + S * R - 1) / (S * R);   // turns of the ring per item
    constexpr int quantum = k_quantum(P);
    static_assert(NFR == 2 || S >= 4, "sums that pass one fragment at a time wait in registers for one block only");
    static_assert(32 * MF * quantum <= kABuf, "a turn of a full tile has to fit an activation buffer");
    static_assert(!PRODUCTS || !FP8, "products are quantised to int8");
    const int kpad = (Kd + quantum - 1) / quantum * quantum;
    // rows of a tile: with products no more than a workgroup can quantise
    const int lg_rows = PRODUCTS && MF == 4 ? sa.lg_tile_rows : (MF == 1 ? 5 : 7);
    const int tile_rows = 1 << lg_rows;

    // ---- the queues: one per XCD, for its eighth of the items beyond those dealt out; the count of items handed out is a device-scope
    // atomic, a round trip to the memory side.  Wave 0 asks in front of an item's epilogue, for the item after the next: asked earlier, the
    // wave's weights wait behind the answer (layer of 128 tokens 391 / 397 us).  With none left in its own, a workgroup takes from the queue
    // with most.  It ends when all are empty, or seven others were quicker in a row: these ask again after their items, so no item is left.
    // All rounds but the first from the queues instead of the last quarter: as fast or up to 2 us slower.
    const int xcd = (int)blockIdx.x & (kNumXcd - 1);
    auto ask = [&](int x) {
        return lane == 0 ? __hip_atomic_fetch_add(sa.queue + x * kStreamQueueStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    };

    // ---- the item list: every expert's first row and the row tiles before it.  Every wave works it out for itself, a lane an
    // expert, and stores it: the same values into the same places, so that no wave waits for another before it knows its first
    // weights (two block scans and five workgroup barriers until then: the layer of 128 tokens x 1024, top-2 of 8 experts,
    // 26.5 -> 25.8 us of back-to-back calls; nothing where the weights take longer).
    {
        constexpr int kChunks = kMaxExperts / kWave;
        auto listed = [&](int e) { return (int)min(max(sa.group_list[e], (int64_t)0), (int64_t)sa.max_rows); };
        int entry[kChunks], before[kChunks];
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            const int e = c * kWave + lane;
            entry[c] = 0;
            before[c] = 0;
            if (c * kWave < G) {
                entry[c] = e < G ? listed(e) : 0;
                before[c] = sa.cumulative && e > 0 && e < G ? listed(e - 1) : 0;
            }
        }
        int row = 0, tile = 0;   // of the experts before this chunk
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            const int e = c * kWave + lane;
            if (c * kWave < G) {
                int m0 = before[c], rows = max(entry[c] - m0, 0);
                if (!sa.cumulative) {
                    const int inc = wave_inclusive_scan(entry[c]);
                    m0 = min(max(row + inc - entry[c], 0), (int)sa.max_rows);
                    rows = min(entry[c], (int)sa.max_rows - m0);
                    row += wave_last(inc);
                }
                rows = e < G ? rows : 0;
                const int tiles = (rows + tile_rows - 1) >> lg_rows;
                const int inc = wave_inclusive_scan(tiles);
                if (e < G) {
                    tile_start[e] = tile + inc - tiles;
                    first_row[e] = m0;
                }
                tile += wave_last(inc);
                if (e == G - 1) {
                    tile_start[G] = tile;
                    first_row[G] = m0 + rows;   // where the last expert's rows end
                    if (sa.rows_out != nullptr && blockIdx.x == 0 && wave == 0) {
                        sa.rows_out[1] = m0 + rows;  // the rows the next kernel finds (the lists are ascending)
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // lanes read what other lanes of their wave stored
        __builtin_amdgcn_wave_barrier();
    }
    const int n_items = tile_start[G] * blocks;

    // Workgroup i runs on XCD i % 8.  Every XCD has an eighth of the list to itself and its workgroups walk through it side by
    // side: the row tiles and column blocks of an expert meet in one L2 instead of being fetched by all eight (the decode
    // layer's GMM1, 1024 rows over 128 experts: 261 -> 252 us; 512 rows over 16 experts with 32-row tiles: 110 -> 99 us).
    auto first_of = [&](int x) { return (int)((long long)n_items * x / kNumXcd); };
    const int end_item = QUEUED ? n_items : first_of(xcd + 1);
    const int item_step = (int)gridDim.x / kNumXcd;   // workgroups of an XCD
    const int dealt = max(n_items / (int)gridDim.x * 3 / 4, 1);   // rounds of items that are a workgroup's without asking
    const int dealt_items = dealt * item_step;
    auto take = [&](int asked) -> int {
        int i = first_of(xcd) + dealt_items + __builtin_amdgcn_readfirstlane(asked);
        if (i < first_of(xcd + 1)) {
            return i;
        }
        for (int tries = 0; tries < 7; ++tries) {
            int left = 0;
            if (lane < kNumXcd) {
                left = first_of(lane + 1) - first_of(lane) - dealt_items -
                       __hip_atomic_load(sa.queue + lane * kStreamQueueStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            int most = 0, x = 0;
#pragma unroll
            for (int q = 0; q < kNumXcd; ++q) {
                const int l = __builtin_amdgcn_readlane(left, q);
                x = l > most ? q : x;
                most = max(most, l);
            }
            if (most == 0) {
                break;
            }
            i = first_of(x) + dealt_items + __builtin_amdgcn_readfirstlane(ask(x));
            if (i < first_of(x + 1)) {
                return i;
            }
        }
        return n_items;
    };
    auto find_item = [&](int i) -> StreamItem {
        StreamItem it;
        it.g = 0; it.row0 = 0; it.rows = 0; it.blk = 0; it.ckb = quantum; it.nch = 1; it.w = nullptr; it.wstep = 0;
        if (i >= end_item) {
            return it;
        }
        const int q = i / blocks;      // a tile of the expert the item belongs to
        int g = 0;                     // experts whose tiles all lie before
        for (int base = 0; base < G; base += kWave) {
            const int e = base + lane;
            g += __popcll(__ballot(e < G && tile_start[min(e, G - 1) + 1] <= q));
        }
        g = __builtin_amdgcn_readfirstlane(min(g, G - 1));
        const int ts = __builtin_amdgcn_readfirstlane(tile_start[g]);
        const int tiles = __builtin_amdgcn_readfirstlane(tile_start[g + 1]) - ts;
        const int fr = __builtin_amdgcn_readfirstlane(first_row[g]);
        const int er = __builtin_amdgcn_readfirstlane(first_row[g + 1]);
        const int local = i - ts * blocks;
        int blk = local, j = 0;        // the row tiles of a column block side by side: they share its weights
        if (tiles > 1) {
            blk = local / tiles;
            j = local - blk * tiles;
        }
        it.g = g;
        it.blk = blk;
        it.row0 = fr + j * tile_rows;
        it.rows = min(er - it.row0, tile_rows);
        const int fit = kABuf / max(it.rows, 1) / quantum * quantum;
        it.ckb = min(max(fit, quantum), kpad);
        it.nch = (Kd + it.ckb - 1) / it.ckb;
        const int nw = min(blk * P + p, ngroups - 1);
        const int b8 = nw >> 3;
        it.wstep = min(8, ngroups - 8 * b8) * 4096;
        const int8_t *wg = a.per_expert ? a.list.w[g] : a.w + (long long)g * Kd * N;
        it.w = wg + (long long)b8 * 8 * Kd * 64 + (nw & 7) * 4096;
        return it;
    };

    // ---- weights: step R q + r of this wave in ring[r]
    v8i ring[R][2];  // [step][fragment]: .lo the first 32 K bytes of the step, .hi the second
    // Buffer loads, because a wave requests steps that do not exist, too: past the end of its share of K and after the
    // last item.  With zero records such a load is dropped on its way, without a branch around the requests: a branch
    // would make the compiler wait for the younger of the two steps wherever it needs the older.
    const int voff = lane * 16;
    auto issue = [&](int r, const StreamItem &it, int q) {
        const int t = s + (R * q + r) * S;
        const bool there = it.rows > 0 && t < KT;
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)it.w, 0, there ? 0x7fffffff : 0, 0x00020000);
        const int soff = there ? t * it.wstep : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4i piece = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + j * 1024, soff, 2));
            if (j < 2) {
                ring[r][j].lo = piece;
            } else {
                ring[r][j - 2].hi = piece;
            }
        }
    };

    // ---- activations: chunk c of an item straight into LDS buffer `buf`.  16-byte piece i of the chunk (row i / pieces per
    // row) lands at 16 i; which piece of its row that is follows from the XOR, so it is chosen on the global side.
    auto load_a = [&](const StreamItem &it, int c, int buf) {
        const int tid = opaque((int)threadIdx.x);
        const int slots = it.ckb >> 4;
        const float inv = 1.0f / (float)slots;
        const int8_t *base = a.a + (long long)it.row0 * Kd;
        for (int q = 0; q * kSThreads < it.rows * slots; ++q) {
            const int idx = tid + q * kSThreads;
            const int row = (int)(((float)idx + 0.5f) * inv);   // idx < 4096: exact
            const int ls = (idx - row * slots) ^ (row & 15);
            const unsigned off = (unsigned)(row * Kd + min(c * it.ckb + ls * 16, Kd - 16));
            const unsigned dst = lds_addr(lds) + (unsigned)(buf * kABuf + (q * 8 + wave) * 1024);
            if (row < it.rows) {
                load_lds16(base, off, dst);
            }
        }
    };

    // ---- scales of an item into set `set`, requested with the activations so that no epilogue waits for them.  (Loaded in
    // the epilogue they wait behind the ring, which stands still meanwhile: 12 us of a 137 us launch of 1024 items.)
    // int8: column and row scales straight to LDS.  FP8: the tile's rows of block scales as they lie in memory
    // (a_scale8_s[row * KB + kb]; whole words straight to LDS), and 2 P rows of K blocks of the weight through registers.
    constexpr int kWQ = FP8 ? 16 * kSMaxKb / kSThreads : 1;
    uint8_t wreg[kWQ];
    const int KB = Kd >> 7;
    const bool words = (KB & 3) == 0;   // a row's scales are whole words
    auto load_scales = [&](const StreamItem &it, int set) {
        const int tid = opaque((int)threadIdx.x);
        if (!FP8) {
            const float *sg = a.per_expert ? a.list.s[it.g] : a.w_scale + (long long)it.g * N;
            if (tid < P * 16) {
                const int grp = min(it.blk * P + (tid >> 4), ngroups - 1);
                const int c4 = (tid & 15) * 4;
                const int col = a.gate_up ? grp * 32 + (c4 < 32 ? c4 : c4 - 32 + (N >> 1)) : grp * 64 + c4;
                const unsigned dst = lds_addr(&col_scale_s[set][0]) + (unsigned)(wave * 1024);
                load_lds16(sg, (unsigned)(col * 4), dst);
            }
            const int r = tid - 128;        // the waves from the third on: a row each lane
            if (!PRODUCTS && r >= 0 && r < it.rows) {
                const unsigned dst = lds_addr(&row_scale_s[set][0]) + (unsigned)((wave - 2) * 256);
                load_lds4(a.a_scale + it.row0, (unsigned)(r * 4), dst);
            }
            return;
        }
        if (words) {
            const int n = it.rows * KB >> 2;
            for (int q = 0; q * kSThreads < n; ++q) {
                const int idx = tid + q * kSThreads;
                if (idx < n) {
                    const unsigned dst = lds_addr(&a_scale8_s[set][0]) + (unsigned)((q * 8 + wave) * 256);
                    load_lds4(a.a_scale8 + (long long)it.row0 * KB, (unsigned)(idx * 4), dst);
                }
            }
        }
        const int nblk = N >> 7;
        const float inv = 1.0f / (float)KB;
#pragma unroll
        for (int q = 0; q < kWQ; ++q) {
            const int idx = tid + q * kSThreads;
            const int gf = (int)(((float)idx + 0.5f) * inv);    // column group of the item * 2 + fragment
            if (gf < 2 * P) {
                const int grp = min(it.blk * P + (gf >> 1), ngroups - 1);
                const int nf = gf & 1;
                const int col = a.gate_up ? nf * (N / 2) + grp * 32 : grp * 64 + nf * 32;
                wreg[q] = a.w_scale8[((long long)it.g * KB + (idx - gf * KB)) * nblk + (col >> 7)];
            }
        }
    };
    auto store_scales = [&](const StreamItem &it, int set) {
        if (!FP8) {
            return;
        }
        const int tid = opaque((int)threadIdx.x);
        if (!words) {
            for (int idx = tid; idx < it.rows * KB; idx += kSThreads) {
                a_scale8_s[set][idx] = a.a_scale8[(long long)it.row0 * KB + idx];
            }
        }
        const float inv = 1.0f / (float)KB;
#pragma unroll
        for (int q = 0; q < kWQ; ++q) {
            const int idx = tid + q * kSThreads;
            const int gf = (int)(((float)idx + 0.5f) * inv);
            if (gf < 2 * P) {
                w_scale8_s[gf * kSMaxKb + (idx - gf * KB)] = wreg[q];
            }
        }
    };

    // ---- PRODUCTS: the tile's rows from fp32 products, all of K at once (the host has checked that it fits).  The threads
    // share the rows evenly, 512 / (rows, rounded up to a power of two) to a row, so that one round trip brings
    // everything; the arithmetic is requant_kernel's.
    v4f prod[PRODUCTS ? kProductQuads : 1];
    auto load_products = [&](const StreamItem &it) {
        const int lg = 9 - (it.rows > 1 ? 32 - __clz(it.rows - 1) : 0);   // log2 of the threads per row
        const int row = tid >> lg, l = tid & ((1 << lg) - 1);
        const v4f *src = (const v4f *)(sa.products + (long long)(it.row0 + min(row, it.rows - 1)) * Kd);
#pragma unroll
        for (int j = 0; j < (PRODUCTS ? kProductQuads : 1); ++j) {
            const int c = l + (j << lg);
            prod[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (c < Kd >> 2) {
                prod[j] = src[c];
            }
        }
    };
    auto quantise_products = [&](const StreamItem &it, int buf, int set) {
        const int lg = 9 - (it.rows > 1 ? 32 - __clz(it.rows - 1) : 0);
        const int row = tid >> lg, l = tid & ((1 << lg) - 1);
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < (PRODUCTS ? kProductQuads : 1); ++j) {
            m = fmaxf(m, fmaxf(fmaxf(fabsf(prod[j][0]), fabsf(prod[j][1])), fmaxf(fabsf(prod[j][2]), fabsf(prod[j][3]))));
        }
        m = group_max(m, min(1 << lg, kWave));
        if (lg > 6) {   // several waves to a row (all of them take this branch)
            if (lane == 0) {
                rowmax_s[wave] = m;
            }
            lds_barrier();
            const int w0 = wave & ~((1 << (lg - 6)) - 1);
            for (int i = 0; i < 1 << (lg - 6); ++i) {
                m = fmaxf(m, rowmax_s[w0 + i]);
            }
        }
        if (row < it.rows) {
            const bool zero_row = m == 0.0f;
            const float rcp = zero_row ? 0.0f : __fdiv_rn(1.0f, m);
            if (l == 0) {
                row_scale_s[set][row] = zero_row ? 0.0f : __fmul_rn(m, 1.0f / 127.0f);
            }
            int8_t *dst = lds + buf * kABuf + row * it.ckb;
#pragma unroll
            for (int j = 0; j < (PRODUCTS ? kProductQuads : 1); ++j) {
                const int c = l + (j << lg);
                if (c < Kd >> 2) {
                    int b[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        b[e] = (int)rintf(__fmul_rn(__fmul_rn(prod[j][e], 127.0f), rcp));
                    }
                    *(uint32_t *)(dst + (((c >> 2) ^ (row & 15)) << 4) + (c & 3) * 4) = pack4(b[0], b[1], b[2], b[3]);
                }
            }
        }
    };

    // The youngest requests of a wave are its ring (4 pieces a step, younger than the activations): with no more than
    // those outstanding, its share of the activations has landed.
    auto a_landed = [&]() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * R) : "memory"); };

    int set = 0;  // the set of scales in use, one per item in turn
    int buf = 0;  // the activation buffer in use; chunks take turns, across items too
    int item = first_of(xcd) + (int)blockIdx.x / kNumXcd;
    StreamItem cur = find_item(QUEUED && item >= first_of(xcd + 1) ? n_items : item);
    if (cur.rows <= 0) {
        return;
    }
    if constexpr (PRODUCTS) {
        load_products(cur);
    } else {
        load_a(cur, 0, 0);
    }
    load_scales(cur, 0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        issue(r, cur, 0);
    }
    if constexpr (PRODUCTS) {
        quantise_products(cur, 0, 0);
    }
    if (QUEUED && dealt == 1 && wave == 0) {
        const int i = take(ask(xcd));
        if (lane == 0) {
            next_s = i;
        }
    }
    store_scales(cur, 0);
    a_landed();
    lds_barrier();

    for (int turn = 0;; ++turn) {
        item = QUEUED && turn + 1 >= dealt ? __builtin_amdgcn_readfirstlane(next_s) : item + item_step;
        StreamItem nxt{};   // PRODUCTS: a workgroup has one item
        if constexpr (!PRODUCTS) {
            nxt = find_item(item);
        }
        const bool more = nxt.rows > 0;

        acc16 acc[MF][2];
#pragma unroll
        for (int mf = 0; mf < MF; ++mf) {
#pragma unroll
            for (int nf = 0; nf < 2; ++nf) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    acc[mf][nf][i] = 0;
                }
            }
        }
        int rowoff[MF];    // LDS offset of this lane's row of each fragment; rows that do not exist repeat the last
        int rowx[MF];
#pragma unroll
        for (int mf = 0; mf < MF; ++mf) {
            const int row = min(mf * 32 + (lane & 31), cur.rows - 1);
            rowoff[mf] = row * cur.ckb;
            rowx[mf] = row & 15;
        }
        const int half = lane >> 5;
        const int turns_per_chunk = cur.ckb / (64 * S * R);

        for (int c = 0; c < cur.nch; ++c) {
            const bool last_chunk = c + 1 == cur.nch;
            buf ^= c == 0 ? 0 : 1;
            if (!last_chunk) {
                load_a(cur, c + 1, buf ^ 1);
            } else if (more) {
                load_a(nxt, 0, buf ^ 1);
                load_scales(nxt, set ^ 1);
            }
            const int8_t *abuf = lds + buf * kABuf;
            const int q1 = min(turns, (c + 1) * turns_per_chunk);
            const int t0 = c * (cur.ckb >> 6);
            for (int q = c * turns_per_chunk; q < q1; ++q) {
                const bool wrap = q + 1 == turns;
                const StreamItem &src = wrap ? nxt : cur;
                const int qn = wrap ? 0 : q + 1;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int t = s + (R * q + r) * S;
                    if (t < KT) {
                        const int slot = (t - t0) * 4 + half;
                        const v8i(&bf)[2] = ring[r];
                        int sw[2] = {0, 0};
                        if (FP8) {
                            sw[0] = w_scale8_s[(p * 2 + 0) * kSMaxKb + (t >> 1)];
                            sw[1] = w_scale8_s[(p * 2 + 1) * kSMaxKb + (t >> 1)];
                        }
#pragma unroll
                        for (int mf = 0; mf < MF; ++mf) {
                            if (mf > 0 && mf * 32 >= cur.rows) {
                                continue;
                            }
                            v8i af;
                            af.lo = *(const v4i *)(abuf + rowoff[mf] + ((slot ^ rowx[mf]) << 4));
                            af.hi = *(const v4i *)(abuf + rowoff[mf] + (((slot + 2) ^ rowx[mf]) << 4));
                            if constexpr (FP8) {
                                const int sx = a_scale8_s[set][min(mf * 32 + (lane & 31), cur.rows - 1) * KB + (t >> 1)];
#pragma unroll
                                for (int nf = 0; nf < 2; ++nf) {
                                    acc[mf][nf] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[nf], af, acc[mf][nf], 0, 0,
                                                                                                  0, sw[nf], 0, sx);
                                }
                            } else {
#pragma unroll
                                for (int nf = 0; nf < 2; ++nf) {
                                    acc[mf][nf] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[nf].lo, af.lo, acc[mf][nf], 0, 0, 0);
                                }
#pragma unroll
                                for (int nf = 0; nf < 2; ++nf) {
                                    acc[mf][nf] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[nf].hi, af.hi, acc[mf][nf], 0, 0, 0);
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    issue(r, src, qn);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            a_landed();
            lds_barrier();  // the chunk has been read, and the next one has landed
        }

        // ---- the S partial sums of a column group meet in LDS, in the buffer that was read last, 32 rows at a time and
        // NFR column fragments at a time.  Register quad j of a fragment nf, lane l, is row l % 32, columns 8 j + 4 (l / 32)
        // .. + 3; it goes to a 16-byte chunk whose row is XORed so that neither the writes nor the reads below meet in
        // a bank.  Then eight lanes own a row (lane l: row l / 8 of a block of eight, piece l % 8), so that every row leaves in
        // whole 128-byte lines, and the waves of the column group share the four blocks.
        const int nw = cur.blk * P + p;
        const bool live = nw < ngroups;
        // (the compiler would keep every lane-dependent address below in registers through the whole K loop)
        const int lane = opaque(tid) & (kWave - 1);
        constexpr int BPW = S >= 4 ? 1 : 4 / S;   // blocks of eight rows per wave (the first four waves when S == 8)
        const int piece = lane & 7;
        const int I = N >> 1;
        const bool swiglu = a.epilogue != kEpiDequantBf16;
        const bool asks = QUEUED && more && wave == 0 && turn + 2 >= dealt;
        int asked = 0;
        if (asks) {
            asked = ask(xcd);
        }
#pragma unroll
        for (int mf = 0; mf < MF; ++mf) {
            if (mf > 0 && mf * 32 >= cur.rows) {   // no such rows (cur.rows is the same in every wave)
                continue;
            }
            acc4 lo, hi;   // SwiGLU: gate and up of columns 4 piece .. + 3; else columns 8 piece .. + 3 and + 4 .. + 7
            v4f keep[BPW];   // kEpiSwigluFp8: the products until their block's maximum is known
#pragma unroll
            for (int n0 = 0; n0 < 2; n0 += NFR) {
                if (mf + n0 > 0) {
                    lds_barrier();  // the sums before these have been read
                }
                acc4 *const sums = (acc4 *)(lds + buf * kABuf);
                {
                    const int row = lane & 31, half2 = lane >> 5;
                    if (mf * 32 + row < cur.rows) {
#pragma unroll
                        for (int nf = n0; nf < n0 + NFR; ++nf) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                sums[((wave * NFR + nf - n0) * 4 + j) * kWave + half2 * 32 + (row ^ ((2 * j + (half2 ^ nf)) << 1))] =
                                    acc4{acc[mf][nf][4 * j], acc[mf][nf][4 * j + 1], acc[mf][nf][4 * j + 2], acc[mf][nf][4 * j + 3]};
                            }
                        }
                    }
                }
                if (S > 1) {
                    lds_barrier();
                } else {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // a wave reads what it wrote itself
                }
                auto read_sum = [&](int nf, int j, int half2, int row) -> acc4 {
                    const acc4 *src = sums + ((p * NFR + nf - n0) * 4 + j) * kWave + half2 * 32 + (row ^ ((2 * j + (half2 ^ nf)) << 1));
                    acc4 v = src[0];
#pragma unroll
                    for (int ss = 1; ss < S; ++ss) {
                        v += src[ss * P * NFR * 4 * kWave];
                    }
                    return v;
                };
#pragma unroll
                for (int b = 0; b < BPW; ++b) {
                    const int row = (s * BPW + b) * 8 + (lane >> 3);
                    if (s < 4 && live && mf * 32 + row < cur.rows) {
                        if (swiglu) {
                            if (NFR == 2 || n0 == 0) {
                                lo = read_sum(0, piece >> 1, piece & 1, row);
                            }
                            if (NFR == 2 || n0 == 1) {
                                hi = read_sum(1, piece >> 1, piece & 1, row);
                            }
                        } else if (NFR == 2 || (piece >> 2) == n0) {
                            lo = read_sum(piece >> 2, piece & 3, 0, row);
                            hi = read_sum(piece >> 2, piece & 3, 1, row);
                        }
                    }
                    if (n0 + NFR < 2) {
                        continue;   // one fragment at a time (a wave has one block then): the other is still to come
                    }
                        const int trow = mf * 32 + row;
                        const long long grow = cur.row0 + trow;
                        const bool mine = s < 4 && live && trow < cur.rows;
                        const float xs = FP8 || !mine ? 1.0f : row_scale_s[set][trow];
                        if (swiglu) {
                            v4f y = {0.0f, 0.0f, 0.0f, 0.0f};
                            float m = 0.0f;
                            if (mine) {
                                const v4f sgate = FP8 ? v4f{} : *(const v4f *)&col_scale_s[set][FP8 ? 0 : p * 64 + piece * 4];
                                const v4f sup = FP8 ? v4f{} : *(const v4f *)&col_scale_s[set][FP8 ? 0 : p * 64 + 32 + piece * 4];
        #pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    float tg, tu;
                                    if constexpr (FP8) {
                                        tg = lo[e];
                                        tu = hi[e];
                                    } else {
                                        tg = __fmul_rn(__fmul_rn((float)lo[e], sgate[e]), xs);
                                        tu = __fmul_rn(__fmul_rn((float)hi[e], sup[e]), xs);
                                    }
                                    y[e] = __fmul_rn(cam_silu_spec(tg), tu);
                                    m = fmaxf(m, fabsf(y[e]));
                                }
                                if (a.epilogue == kEpiSwiglu) {
                                    *(v4f *)((float *)a.out + grow * I + nw * 32 + piece * 4) = y;
                                }
                            }
                            if constexpr (FP8 && P >= 4) {
                                if (a.epilogue == kEpiSwigluFp8) {
                                    keep[b] = y;
                                    m = group_max(m, 8);
                                    if (piece == 0 && s < 4) {
                                        rowmax_s[p * 32 + row] = m;
                                    }
                                }
                            }
                        } else if (mine) {
                            const int col = nw * 64 + piece * 8;
                            const v4f w0 = FP8 ? v4f{} : *(const v4f *)&col_scale_s[set][FP8 ? 0 : p * 64 + piece * 8];
                            const v4f w1 = FP8 ? v4f{} : *(const v4f *)&col_scale_s[set][FP8 ? 0 : p * 64 + piece * 8 + 4];
                            float f[8];
        #pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                if constexpr (FP8) {
                                    f[e] = lo[e];
                                    f[4 + e] = hi[e];
                                } else {
                                    f[e] = __fmul_rn(__fmul_rn((float)lo[e], w0[e]), xs);
                                    f[4 + e] = __fmul_rn(__fmul_rn((float)hi[e], w1[e]), xs);
                                }
                            }
                            v4u o;
        #pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                o[e] = a.out_fp16 ? f32_to_fp16_bits(f[2 * e]) | (f32_to_fp16_bits(f[2 * e + 1]) << 16)
                                                  : f32x2_to_bf16x2_bits(f[2 * e], f[2 * e + 1]);
                            }
                            *(v4u *)((uint16_t *)a.out + grow * N + col) = o;
                        }
                }
            }
            if constexpr (FP8 && P >= 4) {
                if (a.epilogue == kEpiSwigluFp8) {
                    // a block of 128 product columns is four neighbouring column groups (P is 4 or 8 here)
                    lds_barrier();
#pragma unroll
                    for (int b = 0; b < BPW; ++b) {
                        const int row = (s * BPW + b) * 8 + (lane >> 3);
                        const long long grow = cur.row0 + mf * 32 + row;
                        if (!live || mf * 32 + row >= cur.rows) {
                            continue;
                        }
                        const float *rm = rowmax_s + (p & 4) * 32 + row;
                        const int ex = fp8_block_scale_exp(fmaxf(fmaxf(rm[0], rm[32]), fmaxf(rm[64], rm[96])));
                        const float f1 = exp2_int(-(ex / 2)), f2 = exp2_int(-(ex - ex / 2));
                        int w = 0;
                        w = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(keep[b][0], f1), f2),
                                                            __fmul_rn(__fmul_rn(keep[b][1], f1), f2), w, false);
                        w = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(keep[b][2], f1), f2),
                                                            __fmul_rn(__fmul_rn(keep[b][3], f1), f2), w, true);
                        *(int *)((uint8_t *)a.out + grow * I + nw * 32 + piece * 4) = w;
                        if ((p & 3) == 0 && piece == 0) {
                            a.out_scale8[grow * (I >> 7) + (nw >> 2)] = (uint8_t)(ex + 127);
                        }
                    }
                    lds_barrier();  // rowmax_s is free again
                }
            }
        }
        if (!more) {
            return;
        }
        if (asks) {
            const int i = take(asked);
            if (lane == 0) {
                next_s = i;
            }
        }
        store_scales(nxt, set ^ 1);
        lds_barrier();  // the partial sums have been read, the next item's scales are in place
        buf ^= 1;
        set ^= 1;
        cur = nxt;
    }
}

template <int MF, bool FP8, int P, bool PRODUCTS = false, bool QUEUED = false>
void launch_kernel(unsigned grid, hipStream_t stream, const StreamGemmArgs &sa)
{
    hipLaunchKernelGGL((stream_gemm_kernel<MF, FP8, P, PRODUCTS, QUEUED>), dim3(grid), dim3(kSThreads), 0, stream, sa);
}

template <bool FP8>
void launch_variant(int mf, int P, bool queued, unsigned grid, hipStream_t stream, const StreamGemmArgs &sa)
{
    if (mf == 1) {
        P == 1 ? launch_kernel<1, FP8, 1>(grid, stream, sa) : launch_kernel<1, FP8, 2>(grid, stream, sa);
    } else if (queued) {
        P == 2 ? launch_kernel<4, FP8, 2, false, true>(grid, stream, sa) : launch_kernel<4, FP8, 4, false, true>(grid, stream, sa);
    } else if (P == 2) {
        launch_kernel<4, FP8, 2>(grid, stream, sa);
    } else {
        P == 4 ? launch_kernel<4, FP8, 4>(grid, stream, sa) : launch_kernel<4, FP8, 8>(grid, stream, sa);
    }
}

struct StreamShape {
    bool small;      // 32-row tiles
    int P;           // column groups per item
    long long items; // at most
    unsigned grid;
    bool queued;     // items come from queues, if there are any
};

// `products`: for a launch that takes them (an item to a workgroup).  `queues`: the launch has queues, and its sums do not depend on P.
StreamShape stream_shape(long long G, long long max_rows, int Kd, int N, bool quad, bool products, bool queues, int64_t rows_per_expert, int cus)
{
    StreamShape sh;
    // live experts at most, and the column groups they stream
    const long long live = std::min<long long>(G, max_rows);
    const long long groups = live * (N / 64);
    const bool many = groups >= 6ll * cus;
    // of items that the rows make, spread over the experts
    const double reached = many ? (double)G * (1.0 - std::pow(1.0 - 1.0 / (double)G, (double)max_rows)) : 0.0;
    auto rounds_of = [&](double tiles, int P) { return tiles * ((N / 64 + P - 1) / P) / cus; };
    auto rounds = [&](int P) { return rounds_of(reached, P); };
    // Whether the workgroup with most items, dealt out beforehand, streams fewer columns with items of P groups than of 2 P.  Skewed ids
    // (sigmoid scores with a Zipf bias) reach fewer of the experts while there are few rows, and an expert of more than 128 has two tiles:
    // then it is enough that it is so with those.  With less than a row per expert anything from half of them to all may be reached, and
    // narrower items of K from 1536 on, which gain up to a tenth where it is so and lose a thirtieth where it is not, are taken for granted:
    // 17 x 2048, 4 of 213, FP8, I 1664 77.7 / 71.7, 5 x 4608, 7 of 92, 2176 126.1 / 115.6, 16 x 5504, 3 of 81, 1408 86.0 / 88.5; of shorter K 12 x
    // 1024, 6 of 233, FP8, 2816 82.8 / 88.4, quad 8 x 1664, 2 of 70, 3072 55.2 / 59.8.
    auto fewer_of = [&](double tiles, int P) { return std::ceil(rounds_of(tiles, P)) < 2 * std::ceil(rounds_of(tiles, 2 * P)); };
    auto fewer = [&](int P) {
        const double skewed = max_rows < 4 * G ? 0.85 : max_rows < 12 * G ? 0.94 : 1.0;
        const bool two_tiles = queues && rows_per_expert > 128;
        if (!quad && Kd >= 1536 && (max_rows < G || (max_rows < 4 * G && fewer_of(0.7 * reached, P)))) {
            return true;
        }
        return fewer_of(reached, P) || (!(quad && rounds(P) >= 4) && fewer_of(skewed * reached, P)) ||
               (two_tiles && fewer_of(reached + max_rows / 256.0, P));
    };
    // 32-row tiles, two workgroups per CU, while the stream is short: few column groups and no expert with more rows, or
    // all tiles resident at once.  Otherwise 128-row tiles, so that an expert's weights are read once.
    sh.small = !quad && ((rows_per_expert <= 32 && !many) || groups + max_rows / 32 * (N / 64) <= 2ll * cus);
    // Column groups per item: as few as it takes to give every CU work, then as many as make an item of up to a megabyte of weights (its
    // sums and stores interrupt its stream for about two microseconds), or half of them where workgroups then end closer together: dealt
    // out beforehand, where the one with most items streams fewer columns (fewer); from queues.  kEpiSwigluFp8 needs the four groups of
    // a 128-column block together, and the fp32 products of kEpiSwiglu are the same sums in the same order (quad).  FP8 sums depend on P,
    // so these items are the same with queues and without.  us, twice as many groups / this; layers T x H, top-K of E, I, and
    // products alone, which have no queue, rows x K -> N of E:
    //   K over 4096, to two rounds of 4 groups (4 / 2): 30 x 5120, 6 of 44, 1536 201 / 184, 384 x 5120 -> 1024 of 96 92.0 / 84.7; as many columns, so it
    //   stays at 4: 640 x 5120 -> 2560 of 40 92.4 / 100.3, 448 x 5120 -> 1024 of 112 98.0 / 101.9; over 6144 only where the last round is
    //   not nearly full: 192 -> 2560 of 48 145.6 / 141.7, of 42 131.7 / 134.9; 40 x 6144, 4 of 40, 1280 161 / 146 with skewed ids, 168 / 175 with even ones;
    //   K over 2560, seven rounds of 2: from queues 128 x 4096, 8 of 128, 1536 393 / 388, 64 x 3072, 6 of 128, 1536 266 / 251, 48 x 7168, 8 of 64, 2048
    //   464 / 451; dealt out 384 x 3072 -> 3072 of 96 152.6 / 146.3, but as many columns 512 x 4096 -> 3072 of 128 249 / 252, x 5120 311 / 319;
    //   K to 2048 (8 / 4): 200 x 2048, 4 of 64, 1408 139 / 131 (GMM1), 192 x 2048 -> 4096 of 48 68.4 / 64.8; as many columns 560 x 2048 -> 5120 of 40 73.4 /
    //   81.0, from seven rounds of 4 on level: 512 x 1792 -> 4096 of 128 151 / 152; but experts a power of two of bytes apart, whose
    //   workgroups may meet on the same channels, 512 x 2048 -> 4096 of 128 181.9 / 169.5, FP8 -> 2048 106 / 93, not in one round: 128 -> 4096 of 32 43.8 / 45.6;
    //   K to 1536 (8 / 4): 90 x 5120, 6 of 160, 1536, ten rounds and more 519 / 512, 64 x 5120, 6 of 32, 1536, little more than one of 8 groups
    //   157 / 150, but 192 x 1408 -> 2048 of 48 27.5 / 30.1; six rounds of a dozen rows per expert (FP8, to which int8 of so many rows does not come here)
    //   256 x 4096, 8 of 128, 1536 422 / 409, 700 x 2048, 8 of 256, 1024 337 / 326; in between, 64 x 4096, 8 of 128, 1536, 359 / 363, and at K 512 116 / 119;
    //   quad (8 / 4): 200 x 1280, 6 of 96, 1536 130.4 / 117.5, 4 from queues 48 x 4096, 8 of 128, 1536 342 / 335; as many columns 128 x 1536, 8 of 128, 1536
    //   161.9 / 165.7, 768 x 1536 -> 2048 of 48 29.8 / 32.4, at K 2048, whose items are a megabyte apart, 100 x 2048, 8 of 128, 2048 300 / 273, 200, 8 of 256,
    //   1536 413 / 396.  More rows make sums that several waves share dearer: 500 x 2048, 8 of 128, 768 166 / 170.
    const long long expert = (long long)Kd * N;
    auto apart = [&] { return (expert & (expert - 1)) == 0 && rounds(8) > 1; };
    auto to2 = [&] { return fewer(2) || (Kd > 6144 && std::ceil(rounds(2)) - rounds(2) < 0.35); };
    auto to4 = [&] { return fewer(4) || rounds(4) >= 7 || apart(); };
    sh.P = 2;
    if (sh.small) {
        sh.P = 2 * groups >= 3ll * cus ? 2 : 1;
    } else if (products) {
        sh.P = 512ll * Kd <= (1 << 20) ? 8 : 4;
    } else if (quad) {
        sh.P = many && Kd <= 2048 && (max_rows > 24 * G || !(fewer(4) || apart() || (Kd == 2048 && rounds(8) > 1))) ? 8 : 4;
    } else if (many && Kd > 2560) {
        sh.P = (rounds(2) >= 7 && (queues || to2())) || (Kd > 4096 && rounds(4) < 2.2 && to2()) ? 2 : 4;
    } else if (many && Kd > 1536) {
        sh.P = Kd > 2048 || to4() ? 4 : 8;
    } else if (many) {
        sh.P = to4() && ((Kd > 1024 && rounds(8) < 1.3) || (Kd >= 1024 && (rounds(4) >= 10 || (rounds(4) >= 6 && max_rows >= 12 * G)))) ? 4 : 8;
    }
    sh.queued = many && !sh.small && !products && sh.P <= 4 && rounds(sh.P) >= 4;
    const long long tiles = live + max_rows / (sh.small ? 32 : 128);
    sh.items = tiles * ((N / 64 + sh.P - 1) / sh.P);
    // a multiple of eight workgroups: every XCD takes an eighth of the items
    sh.grid = (unsigned)((std::min<long long>(sh.items, (sh.small ? 2ll : 1ll) * cus) + kNumXcd - 1) / kNumXcd * kNumXcd);
    return sh;
}

// log2 of the rows of a tile whose products fit the registers of a workgroup, and its int8 rows, padded as the kernel pads them, an
// activation buffer; -1 where 32-row tiles are not that low.  128-row tiles are cut: tokens that name an expert once each make
// no more than one tile of it where the launch takes products, tokens that name it several times as many as their rows fill.
int lg_product_rows(const StreamShape &sh, long long max_rows, int Kd)
{
    const long long quantum = k_quantum(sh.P), kpad = (Kd + quantum - 1) / quantum * quantum;
    auto fits = [&](int lg) {
        return ((long long)Kd << lg) <= 4ll * kProductQuads * kSThreads && (kpad << lg) <= (sh.small ? kSBuf32 : kSBuf128);
    };
    if (Kd % 128 != 0 || !fits(0)) {
        return -1;
    }
    int lg = 0;
    if (sh.small) {
        while ((1ll << lg) < std::min<long long>(32, max_rows)) {
            ++lg;
        }
        return fits(lg) ? lg : -1;
    }
    while (lg < 7 && fits(lg + 1)) {
        ++lg;
    }
    return sh.P == 8 ? lg : -1;   // (four groups to an item are more items than workgroups, or 32-row tiles)
}

}  // namespace

// Rows x columns up to which the stream is the faster form: 64 rows per expert where the tile kernel has half as many
// 512-column items as CUs, 32 where it has as many, 10 where it has three times as many (measured with the shapes of
// DeepSeek-V3's, Qwen3's and smaller layers, 2 to 3072 rows; the two forms are within 5 % of each other along this line).
// FP8 goes on to three times as many while experts have no more than 32 rows on average, i.e. most of them one tile (layers,
// tile form -> this: 150 tokens on 40 experts, top-8, H 7168, I 2048: 407 -> 342 us; 1500 on 64, top-1, H 3072, I 2560: 332 ->
// 273; 512 on 128, top-8, H 4096, I 1536: 483 -> 464; with five times as many 1000 on 256, top-8, H 2048, I 1024 lost, 362 -> 367,
// and with 37 rows on average 300 on 64, H 2048, I 1408, 160 -> 162).  The tiles of the other form fetch FP8 scales item by item;
// int8 gains from 322 -> 296 to 391 -> 362 on some of these shapes and loses from 449 -> 465 to 480 -> 503 on others: rows x columns
// alone does not tell them apart, so int8 stops where it never loses.  A layer asks once, with the columns of its GMM1, and
// its GMM2 takes the same form.
bool stream_gemm_applies(int64_t rows, int64_t N, int64_t G, bool fp8)
{
    constexpr int64_t kMostRowsTimesColumns = 32ll * 512 * 256;
    return rows > 0 && (rows * N <= kMostRowsTimesColumns || (fp8 && rows <= 32 * G && rows * N <= 3 * kMostRowsTimesColumns));
}

// Where every workgroup has one item at most: with more, the quantisation of an item would interrupt the stream.  With 128-row tiles, us
// per layer, re-quantisation as a launch / here: 16 tokens x 7168, top-8 of 16, I 2048 127.7 / 126.0, 10 x 4096, 8 of 32, 1536 108.1 /
// 105.8, 16 x 7168, 2 of 16, 2048 115.7 / 113.4, 24 x 7168, 4 of 16, 1024 73.1 / 71.4.
bool stream_gemm_takes_products(int64_t max_rows, int G, int Kd, int N, int64_t rows_per_expert)
{
    int cus = 0;
    if (max_rows <= 0 || G <= 0 || gemm_workgroups(&cus) != hipSuccess) {
        return false;
    }
    const StreamShape sh = stream_shape(G, max_rows, Kd, N, false, true, false, rows_per_expert, cus);
    const int lg = lg_product_rows(sh, max_rows, Kd);
    if (lg < 0) {
        return false;
    }
    if (sh.small) {
        return sh.items <= (long long)sh.grid;
    }
    const long long experts = std::min<long long>(G, max_rows);
    return rows_per_expert <= 1ll << lg && experts * ((N / 64 + sh.P - 1) / sh.P) <= cus;
}

hipError_t launch_stream_gemm(const StreamGemmArgs &sa, int64_t rows_per_expert, hipStream_t stream)
{
    const GemmArgs &g = sa.g;
    if (sa.group_list == nullptr || sa.G <= 0 || sa.G > kMaxExperts || sa.max_rows <= 0 || g.Kd % 128 != 0 || g.Kd < 128 ||
        g.N % 64 != 0 || (g.gate_up && g.N % 128 != 0) || g.epilogue == kEpiInt32) {
        return hipErrorInvalidValue;
    }
    if (g.fp8 && (g.N % 128 != 0 || (g.gate_up && g.N % 256 != 0) || g.Kd / 128 > kSMaxKb || g.per_expert ||
                  g.a_scale8 == nullptr || g.w_scale8 == nullptr)) {
        return hipErrorInvalidValue;
    }
    if (g.epilogue == kEpiSwigluFp8 && (!g.fp8 || !g.gate_up || g.out_scale8 == nullptr)) {
        return hipErrorInvalidValue;
    }
    int cus = 0;
    const hipError_t e = gemm_workgroups(&cus);
    if (e != hipSuccess) {
        return e;
    }
    const StreamShape sh = stream_shape(sa.G, sa.max_rows, g.Kd, g.N, g.fp8 && g.gate_up, sa.products != nullptr, sa.queue != nullptr && !g.fp8,
                                        rows_per_expert, cus);
    const bool queued = sh.queued && sa.queue != nullptr;
    if (sa.products != nullptr) {
        const int lg = lg_product_rows(sh, sa.max_rows, g.Kd);
        if (g.fp8 || g.gate_up || lg < 0) {
            return hipErrorInvalidValue;
        }
        // an item to a workgroup, which is what the kernel is written for
        StreamGemmArgs sp = sa;
        sp.lg_tile_rows = lg;
        const long long items = sh.small ? sh.items
                                         : (std::min<long long>(sa.G, sa.max_rows) + (sa.max_rows >> lg)) * ((g.N / 64 + sh.P - 1) / sh.P);
        const unsigned grid = (unsigned)((items + kNumXcd - 1) / kNumXcd * kNumXcd);
        if (sh.small) {
            sh.P == 1 ? launch_kernel<1, false, 1, true>(grid, stream, sp) : launch_kernel<1, false, 2, true>(grid, stream, sp);
        } else {
            launch_kernel<4, false, 8, true>(grid, stream, sp);
        }
    } else if (g.fp8) {
        launch_variant<true>(sh.small ? 1 : 4, sh.P, queued, sh.grid, stream, sa);
    } else {
        launch_variant<false>(sh.small ? 1 : 4, sh.P, queued, sh.grid, stream, sa);
    }
    return hipGetLastError();
}

}  // namespace cam
