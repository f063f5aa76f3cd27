// Grouped w8a8 GEMM on the gfx950 matrix cores (v_mfma_i32_32x32x32_i8), with the CAM epilogues.
//
// Reference semantics (paths relative to the reference tree; FDM =
// src/cam/comm_operator/ascend_kernels/fused_deep_moe/op_kernel/fused_deep_moe):
//   GMM1 main loop  FDM/gemm/kernel/grouped_matmul_slice_m_per_token_dequant_swiglu_quant_multistage_workspace.h:490-645
//   GMM1 epilogue   FDM/epilogue/block/block_epilogue_per_token_dequant_swiglu.h:236-264
//   re-quant        the GMM1 kernel file :160-277
//   GMM2 main loop  FDM/gemm/kernel/grouped_matmul_slice_m_per_token_dequant_multistage_workspace.h:115-215
//   GMM2 epilogue   FDM/epilogue/block/block_epilogue_per_token_dequant.hpp:665-684
//
// Design (not a translation of the cube/vector split above).
//   * Persistent kernel, one workgroup of four waves per CU, one wave per SIMD with all 512 of its registers.  Work items
//     (one row tile of ONE expert x one block of packed weight columns) come from a device-built schedule
//     (sched_device.h).  Short schedules give every workgroup a queue of its own, dealt so that the queues last equally
//     long and that the workgroups of an XCD work on tiles which share operands; a workgroup whose queue runs out takes
//     from the fullest one.  Long schedules use one queue per XCD, shared by its workgroups, in which the row tiles of
//     an expert that read the same weight columns sit next to each other and big experts come first, which leaves the
//     small items for the end, where they even out the finishing times.
//   * Two tile shapes.  Tall tiles (up to 256 rows) x 256 columns: a wave owns ALL rows of the tile and 64 of its columns.
//     Flat tiles (<= 128 rows) x 512 columns, for experts that only stream weights: all rows and 128 columns (in a narrow
//     schedule, sched_device.h, x 256 like tall ones).  Either way a wave holds up to sixteen 32 x 32 sums (256 registers, all
//     of the accumulation file; a narrow item eight of them at most).  The numbers of row and column fragments are template
//     parameters, so the main loop has no control flow.
//   * A weight byte is needed by one wave only.  It goes from memory straight to that wave's registers (prepack_kernel laid
//     the weights out in the lane order the MFMA wants), a ring of four 64-byte K steps.  Only the activations go
//     through LDS: direct-to-LDS loads (16 bytes per lane, no registers) into a ring of four stages of 128 K bytes, a
//     whole line of every row, their 16-byte chunks placed with an XOR swizzle (chosen on the global side, since such a
//     load writes lane i at base + 16*i) that makes the ds_read_b128 fragment reads bank-conflict free.
//     What bounds the loop is what crosses the LDS and the clock the power limit leaves.  Per 64 bytes of K and 256 rows the
//     CU moves 16 KB of activations into LDS and 64 KB out of it, 640 of the 1024 cycles in which the matrix cores
//     multiply them.  With two teams of four waves of 128 rows, both operands in LDS and two barriers per 64 bytes of K, it
//     was 32 KB in and 96 KB out, 1024 of 1024 cycles: 1237 cycles for a step of 256 rows and 1027 for one of
//     160, now 1079 and 729 (w8a8 gate/up GEMM, 65536 rows on 128 experts, K 4096, I 1536; stamps of a --timeline build).
//     The clock falls as the matrix cores get busier (1.41 -> 1.35 GHz there), so time falls less than cycles.
//   * Between two multiplications stands at most what the wave can issue while the first is in the matrix pipe: a
//     request, or a fragment read, and a few scalar instructions.  The fragments are read six multiplications' pairs
//     ahead, across the one barrier per 128 bytes of K.  Requests past the end of K go out with an empty buffer
//     descriptor: they fetch nothing, and the counts that the waits rely on stay what they are.
//   * The loads are issued from inline assembly and the waits are written out by hand: left to itself the compiler
//     drains every outstanding load at each barrier and before LDS reads it cannot prove independent, which
//     serialises the pipeline.  The sums are named registers for a similar reason (below).
//   * The int32 accumulators stay in registers through the epilogue: dequantisation, SiLU and the
//     gate*up product are applied in place; the int32 tile never goes to memory.  The MFMAs take the
//     weights as their first operand, so a lane ends up with ONE activation row and runs of four
//     consecutive weight columns: one row scale per lane, column scales as 16-byte vectors, and each
//     32-row fragment passes through a small LDS staging slice from which whole 128-byte lines are
//     stored.  For GMM1 the prepack pairs gate column c with up column I+c inside one wave.
//   * The K order inside a 32-deep MFMA step is whatever the two operands agree on (an integer dot
//     product does not care), which is what lets both be loaded as plain 16-byte pieces.
//   * Flat items are bound by the memory; their weight panels are fetched with non-temporal loads (nobody else reads them), and so
//     are those of narrow items of up to 96 rows.
//   * Between two items.  What a workgroup has to know and to fetch before it can multiply is asked for during the item before
//     (ask_ahead, publish): from an item's start to its first multiplication it is 2 us instead of 4, of which the
//     requests for the weights take most.  Layers of 8192 / 1021 tokens 1567 -> 1535 / 181 -> 176 us, FP8 layer of 4093
//     tokens 850 -> 828.  Loading a word of every line of a flat item's first sub-steps under the epilogue as well, to have
//     them in L2, cost the layer of 1021 tokens 1 % with one sub-step, 3 % with three and 8 % with ten.
#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "cam_device.h"
#include "cam_kernels.h"
#include "rank_device.h"
#include "permute_device.h"
#include "sched_device.h"
#include "../../include/cam_expf_spec.h"

namespace cam {

namespace {

constexpr int kBK = 64;                         // K bytes per sub-step
constexpr int kThreads = 256;                   // four waves, one per SIMD
constexpr int kStageK = 128;                    // K bytes per stage of activations
constexpr int kStages = 4;
constexpr int kStage = 256 * kStageK;           // 32 KB
constexpr int kLdsBytes = kStages * kStage;     // 128 KB
constexpr int kRing = 4;                        // sub-steps of weights a wave has registers for
constexpr int kScaleKb = 64;                    // FP8: K-blocks of 128 bytes an item may span (Kd <= 8192)
constexpr int kEpiRowBytes = 144;               // epilogue staging: 128 data bytes + 16 of padding per row
constexpr int kEpiSlice = 32 * kEpiRowBytes;    // one 32-row fragment per wave

// Buffer descriptor words of `bytes` bytes at p.
__device__ __forceinline__ v4i buffer_words(const void *p, unsigned bytes)
{
    const unsigned long long v = (unsigned long long)p;
    return v4i{(int)(unsigned)v, (int)((unsigned)(v >> 32) & 0xffffu), (int)bytes, 0x00020000};
}

// Loads.  A vector memory instruction must not read a scalar register that the vector ALU wrote within five wait states, and the
// compiler does not see to that for inline assembly.  Where a scalar operand may come out of a register the compiler had
// parked in a vector lane (in front of the K loop; anywhere in the FP8 kernel, whose multiplications leave room for it),
// WAITS provides the five.  The build looks the code over that the compiler made of this (machine_code.py).

// One direct-to-LDS load: lane i of the wave fetches 16 bytes at its offset from the base, and the data lands at LDS byte
// address lds_addr + LDS_OFFSET + 16*i.  Base and offsets are scalar but for one vector register, so that issuing the load
// takes no vector ALU work.
template <int LDS_OFFSET, bool WAITS>
__device__ __forceinline__ void dma16(v4i words, unsigned voff, unsigned soff, unsigned lds_addr)
{
    if (WAITS) {
        asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(words), "s"(soff), "n"(LDS_OFFSET)
                     : "memory", "m0", "scc");
    } else {
        asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(words), "s"(soff), "n"(LDS_OFFSET)
                     : "memory", "m0", "scc");
    }
}

// A wave-uniform address the compiler does not know to be one, as a scalar register pair.
__device__ __forceinline__ unsigned long long scalar_address(const void *p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// (base and lds_addr: scalar registers already, see scalar_address)
__device__ __forceinline__ void dma16(unsigned long long base, unsigned voff, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(base)
                 : "memory", "m0");
}

__device__ __forceinline__ unsigned lds_address(const void *p)
{
    return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void *)p;
}

// The same for 4 bytes per lane.
__device__ __forceinline__ void dma4(unsigned long long base, unsigned voff, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_addr), "v"(voff), "s"(base)
                 : "memory", "m0");
}

// 16 bytes per lane to registers.  STREAM: marked non-temporal, for bytes that are read once: a stream of them moves at
// 6.6-7.1 TB/s from HBM where the plain form stays at 5.8-6.0 (measured with a bare ring of such loads, 256 workgroups).
template <int OFFSET, bool STREAM, bool WAITS>
__device__ __forceinline__ void request16(v4i &dst, v4i words, unsigned voff, unsigned soff)
{
    if (WAITS) {
        asm volatile("s_nop 4");
    }
    if (STREAM) {
        asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:%4 nt"
                     : "=v"(dst) : "v"(voff), "s"(words), "s"(soff), "n"(OFFSET) : "memory");
    } else {
        asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:%4"
                     : "=v"(dst) : "v"(voff), "s"(words), "s"(soff), "n"(OFFSET) : "memory");
    }
}

// The same value, computed anew as far as the compiler can tell: keeps loop-invariant address arithmetic out of registers.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

template <int N>
__device__ __forceinline__ void wait_loads_outstanding()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void wait_lds_reads()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// Workgroup barrier without the memory fence of __syncthreads(); the waits are explicit (above).
__device__ __forceinline__ void barrier_no_fence()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// What a wave needs to know about the item it works on (all wave-uniform).
struct ItemCtx {
    const int8_t *a_tile;   // first activation row of the tile; with a_rows, of the whole matrix
    const int8_t *wg;       // the expert's packed weights
    const float *sg;        // the expert's per-channel scales
    int g, m0, rows;        // expert, first row and rows of the tile
    int group;              // this wave's first 64-column group of the weight
    int mf;                 // row fragments the K loop runs on
    bool flat;
    int buf;                // which of the two scale buffers
    int Kd, N;
#ifdef CAM_GEMM_TIMELINE
    int *phase_s;           // LDS: wall clock at the first multiply and after the K loop (written by thread 0)
#endif
};

// f(std::integral_constant<int, I>) for I in [B, E), unrolled.
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>());
        static_for<B + 1, E>(f);
    }
}

// Accumulators.  All 256 accumulation registers of a wave hold sixteen 32 x 32 tiles, tile T in a[16 T : 16 T + 15], named here
// and not by the compiler: with that file full it spills and copies around the loop, and cannot know that no other value
// wants a place there.
#define CAM_ACC_0 "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15"
#define CAM_ACC_1 "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31"
#define CAM_ACC_2 "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47"
#define CAM_ACC_3 "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63"
#define CAM_ACC_4 "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79"
#define CAM_ACC_5 "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95"
#define CAM_ACC_6 "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111"
#define CAM_ACC_7 "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127"
#define CAM_ACC_8 "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143"
#define CAM_ACC_9 "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159"
#define CAM_ACC_10 "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175"
#define CAM_ACC_11 "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191"
#define CAM_ACC_12 "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207"
#define CAM_ACC_13 "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223"
#define CAM_ACC_14 "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239"
#define CAM_ACC_15 "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
#define CAM_ACC_TILES(X) \
    X(0, 0, 15, CAM_ACC_0) X(1, 16, 31, CAM_ACC_1) X(2, 32, 47, CAM_ACC_2) X(3, 48, 63, CAM_ACC_3) \
    X(4, 64, 79, CAM_ACC_4) X(5, 80, 95, CAM_ACC_5) X(6, 96, 111, CAM_ACC_6) X(7, 112, 127, CAM_ACC_7) \
    X(8, 128, 143, CAM_ACC_8) X(9, 144, 159, CAM_ACC_9) X(10, 160, 175, CAM_ACC_10) X(11, 176, 191, CAM_ACC_11) \
    X(12, 192, 207, CAM_ACC_12) X(13, 208, 223, CAM_ACC_13) X(14, 224, 239, CAM_ACC_14) X(15, 240, 255, CAM_ACC_15)

template <int TILE>
__device__ __forceinline__ void acc_multiply(v4i w, v4i x)
{
#define CAM_X(T, LO, HI, ...) \
    if constexpr (TILE == T) { \
        asm volatile("v_mfma_i32_32x32x32_i8 a[" #LO ":" #HI "], %0, %1, a[" #LO ":" #HI "]" ::"v"(w), "v"(x) : __VA_ARGS__); \
    }
    CAM_ACC_TILES(CAM_X)
#undef CAM_X
}

template <int TILE>
__device__ __forceinline__ void acc_multiply(v8i w, v8i x, int sw, int sx)
{
#define CAM_X(T, LO, HI, ...) \
    if constexpr (TILE == T) { \
        asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 a[" #LO ":" #HI "], %0, %1, a[" #LO ":" #HI "], %2, %3 op_sel_hi:[0,0,0]" \
                     ::"v"(w), "v"(x), "v"(sw), "v"(sx) : __VA_ARGS__); \
    }
    CAM_ACC_TILES(CAM_X)
#undef CAM_X
}

template <int TILE>
__device__ __forceinline__ void acc_clear()
{
#define CAM_X(T, LO, HI, ...) \
    if constexpr (TILE == T) { \
        asm volatile(".irp r, 0,1,2,3,4,5,6,7,8,9,10,11,12,13,14,15\n\tv_accvgpr_write_b32 a[" #LO "+\\r], 0\n\t.endr" ::: __VA_ARGS__); \
    }
    CAM_ACC_TILES(CAM_X)
#undef CAM_X
}

// Four accumulator registers from REG on.  Together, because a value that comes out of inline assembly costs a wait state if
// the next instruction uses it: read one by one as they were needed, an FP8 product cost up to two of them beside its 24
// instructions (with the one that quiet() saves: FP8 layer of 8000 tokens x 2048, top-6 of 64 experts, I 1408: 572 -> 566 us; of
// 4093 x 4096, top-8 of 128, I 1536: 832.5 -> 831; int8, where the products need no such read, within 0.3 %).
template <int REG>
__device__ __forceinline__ v4i acc_bits4()
{
    int v[4];
    asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%4+1]\n\t"
                 "v_accvgpr_read_b32 %2, a[%4+2]\n\tv_accvgpr_read_b32 %3, a[%4+3]"
                 : "=v"(v[0]), "=v"(v[1]), "=v"(v[2]), "=v"(v[3]) : "n"(REG));
    return v4i{v[0], v[1], v[2], v[3]};
}

template <int REG, bool FP8>
__device__ __forceinline__ v4f acc_values()
{
    const v4i v = acc_bits4<REG>();
    return FP8 ? __builtin_bit_cast(v4f, v) : v4f{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// A gate sum of an FP8 item: cam_silu_spec takes its minimum and its maximum, and the compiler, which does not know that the
// matrix cores make no signalling NaN, would quiet it for each of them.
__device__ __forceinline__ float quiet(float t)
{
    return __builtin_canonicalizef(t);
}

template <bool FP8>
struct FragType {
    typedef v4i type;
};
template <>
struct FragType<true> {
    typedef v8i type;
};

// The K loop, for one wave: MF row fragments x NF column fragments, sums in tiles mf * NF + nf.
//   stage s:     requests stage s + 3 of the activations (into the slot of stage s - 1, which the barrier before has set free)
//   sub-step k:  (two per stage) multiplies the weights of k with the fragments of its half of the stage, and requests the
//                weights of k + 3 into the registers that k - 1 has been multiplied from
//   slot:        (2 MF per sub-step, FP8: MF) NF multiplications with one activation fragment; reads the fragment of PD
//                slots later and sends the slot's share of the requests between the multiplications
// A stage ends with a wait and a barrier.  Fragments are read across it, i.e. stage s + 1 is read in stage s, and so has to be
// in LDS one stage early.  Loads retire in order, and the order of the requests is the same in every sub-step (activations,
// then weights), so "at most WAIT outstanding" in front of sub-step k says that its weights have come, which were the last
// requests of sub-step k - 3: since then two sub-steps have sent NB weight loads each and a stage's MF activation
// loads.  In front of a stage's first sub-step that covers the activations of stage s + 1, which are older.
// Requests past the end are for nothing (empty descriptors).
//
// FP8: v_mfma_scale_f32_32x32x64_f8f6f4 covers the 64 K bytes of a sub-step (the two 16-byte pieces a lane holds), takes the E8M0
// scale of the lane's weight column block and of its activation row for the current 128-byte K block, and accumulates in fp32.
// The scales of the rows wait in LDS (a_scale8_s), those of the wave's column fragments, one byte per fragment and K block, in a
// register each (lane kb holds K block kb).
//
// The item's first two stages and its row scales have been requested (ask_ahead in gemm_kernel).  `publish` runs between the
// requests and the wait for them.
template <int MF, int NF, bool FP8, typename Publish, typename AskRows>
__device__ __forceinline__ void k_loop(const GemmArgs &a, const ItemCtx &t, int8_t *lds, const uint8_t *a_scale8_s,
                                       const int32_t *rows_s, Publish &publish, AskRows &ask_rows)
{
    // A flat item is the only reader of its weight panel, and so is one of 256 columns and up to three row units, which only narrow
    // schedules hold.  Four units are either a narrow item of 97-128 rows, the only reader too, or the lower of the two tiles of
    // an expert of 257-288 rows, whose panel the other one shares; they run the same code and load plainly.  us, streaming items of
    // 256 columns never / up to three / up to four units: layer of 1021 fp16 tokens x 2048, top-6 of 64 experts, I 1408 166.3 /
    // 161.2 / 161.1, of 1150 tokens 176.1 / 168.7 / 167.4, FP8 layer of 1900 x 4096, top-2 of 40, I 2048 246.3 / 236.6 / 233.2; both GEMMs
    // over 272 rows on each of 128 experts, H 4096, I 1536 (three / four units) 855 / 929, on each of 32, H 7168, I 2048 604 / 564, over 288
    // on each of 8, H 4096, I 2048 112 / 123.
    constexpr bool STREAM = NF == 4 || MF < 4;
    constexpr int SLOTS = FP8 ? MF : 2 * MF;
    constexpr int AR = FP8 ? 4 : 8;                 // fragments in registers
    constexpr int PD = FP8 ? (MF == 1 ? 2 : 3) : (MF == 1 ? 4 : 6);  // (at most a stage)
    constexpr int NB = 2 * NF;                      // weight loads per sub-step
    constexpr int kHalf = (MF + 1) / 2;             // activation loads in a stage's first sub-step
    constexpr int WAIT = 2 * NB + MF;
    const int tid = threadIdx.x;
    const int lane = opaque(tid) & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ST = t.Kd / kStageK;
    const int KT = 2 * ST;
    const unsigned lds0 = lds_address(lds);

    // ---- activations: wave w brings tile rows 8 MF w .. 8 MF (w + 1) - 1, eight rows a load.  Lane i of a load brings row i / 8
    // of its eight and the 16-byte chunk whose swizzled slot is i % 8: chunk c of row r lies at slot c ^ (r / 2 % 8) of the
    // row's 128 bytes, so that sixteen neighbouring rows cover all 64 banks.  Rows beyond the tile are out of the
    // descriptor's range, which the vector offset is checked against, and come as zeros.  Gathered rows (a_rows) lie anywhere in a
    // matrix of less than 2^31 bytes.
    const bool gather = a.a_rows != nullptr;
    const v4i a_words = buffer_words(t.a_tile, (gather ? (unsigned)a.a_count : (unsigned)t.rows) * (unsigned)t.Kd);
    const unsigned a_dst = lds0 + (unsigned)(wave * (MF * 1024));
    // (one branch around all of them, so that the reads of gathered row numbers are one round trip to the LDS)
    unsigned a_voff[MF];
    const int r0 = 8 * wave * MF + (lane >> 3);
    if (gather) {
        int at[MF];
#pragma unroll
        for (int j = 0; j < MF; ++j) {
            at[j] = rows_s[r0 + 8 * j];
        }
#pragma unroll
        for (int j = 0; j < MF; ++j) {
            const int r = r0 + 8 * j;
            a_voff[j] = r < t.rows ? (unsigned)(at[j] * t.Kd + ((lane & 7) ^ ((r >> 1) & 7)) * 16) : 0x80000000u;
        }
    } else {
#pragma unroll
        for (int j = 0; j < MF; ++j) {
            const int r = r0 + 8 * j;
            a_voff[j] = (unsigned)(r * t.Kd + ((lane & 7) ^ ((r >> 1) & 7)) * 16);
        }
    }
    auto bring = [&](int s, auto jc, auto wc) {  // load j of stage s
        constexpr int j = decltype(jc)::value;
        v4i words = a_words;
        words[2] = s < ST ? words[2] : 0;
        dma16<j * 1024, decltype(wc)::value>(words, a_voff[j], (unsigned)(s * kStageK),
                                                  a_dst + (unsigned)((s & (kStages - 1)) * kStage));
    };

    // ---- weights.  Column groups lie in blocks of eight; inside a block the 4 KB of a K step of its groups lie side by
    // side, so the loads of one step of a workgroup cover one contiguous stretch of memory.
    v4i ring[kRing][NB];
    const int ngroups = t.N / 64;
    const int nw0 = min(t.group, ngroups - 1);
    const int nw1 = min(t.group + 1, ngroups - 1);
    const int b_block = nw0 >> 3;
    const int b_step = min(8, ngroups - 8 * b_block) * 4096;
    const v4i b_words = buffer_words(t.wg + (long long)b_block * 8 * t.Kd * 64 + (nw0 & 7) * 4096, 0x7fffffffu);
    const unsigned b_voff0 = (unsigned)(lane * 16);
    const unsigned b_voff1 = b_voff0 + (unsigned)((nw1 - nw0) * 4096);
    auto request = [&](v4i (&dst)[NB], int k, auto jc, auto wc) {
        constexpr int j = decltype(jc)::value;     // K half j / NF, column fragment j % NF
        constexpr int nf = j % NF, kk = j / NF;
        constexpr int off = kk * 2048 + (nf & 1) * 1024;
        v4i words = b_words;
        words[2] = k < KT ? words[2] : 0;
        request16<off, STREAM, decltype(wc)::value>(dst[j], words, nf < 2 ? b_voff0 : b_voff1, (unsigned)(k * b_step));
    };
    // The registers of a sub-step are passed through the wait for them: nothing that reads them is moved in front of it.
    // (Between the request and here nothing may read or move them at all; the build looks the code over, machine_code.py.)
    auto landed = [&](v4i (&r)[NB]) {
        if constexpr (NB == 4) {
            asm volatile("s_waitcnt vmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(WAIT) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%8)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]),
                         "+v"(r[6]), "+v"(r[7]) : "n"(WAIT) : "memory");
        }
    };

    // ---- fragments
    typename FragType<FP8>::type af[AR];
    int sa[2][MF];
    int sw[2][NF];
    const int frow = lane & 31;
    const int fbase = frow * kStageK + (((lane >> 5) ^ ((frow >> 1) & 7)) << 4);
    auto read_frag = [&](typename FragType<FP8>::type &dst, int slot, auto qc) {
        constexpr int q = decltype(qc)::value;  // slot inside the stage
        constexpr int u = q / SLOTS, i = q % SLOTS;
        if constexpr (FP8) {
            dst.lo = *(const v4i *)(lds + slot * kStage + (fbase ^ (u * 64)) + i * 4096);
            dst.hi = *(const v4i *)(lds + slot * kStage + (fbase ^ (u * 64 + 32)) + i * 4096);
        } else {
            dst = *(const v4i *)(lds + slot * kStage + (fbase ^ (u * 64 + (i / MF) * 32)) + (i % MF) * 4096);
        }
    };
    int w_scale[FP8 ? NF : 1];
    auto read_scales = [&](int b, int s) {
        if constexpr (FP8) {
            const int kb = min(s, ST - 1);
#pragma unroll
            for (int nf = 0; nf < NF; ++nf) {
                // moved here, well before the multiplication that reads it
                asm volatile("v_mov_b32 %0, %1" : "=v"(sw[b][nf]) : "s"(__builtin_amdgcn_readlane(w_scale[nf], kb)));
            }
#pragma unroll
            for (int mf = 0; mf < MF; ++mf) {
                sa[b][mf] = a_scale8_s[((kb >> 2) * 256 + mf * 32 + (lane & 31)) * 4 + (kb & 3)];
            }
        }
    };

    // ---- pipeline.  The first requests go out in the order the loop would have sent them in.
    if constexpr (FP8) {
        const int KB = t.Kd >> 7, nblk = t.N >> 7;
        const unsigned voff = (unsigned)(min(lane, KB - 1) * nblk);
#pragma unroll
        for (int nf = 0; nf < NF; ++nf) {
            const int grp = nf < 2 ? nw0 : nw1, f = nf & 1;
            // first logical column of the fragment (a paired group holds 32 gate and 32 up columns)
            const int col = a.gate_up ? f * (t.N / 2) + grp * 32 : grp * 64 + f * 32;
            const uint8_t *base = a.w_scale8 + (long long)t.g * KB * nblk + (col >> 7);
            asm volatile("s_nop 4\n\tglobal_load_ubyte %0, %1, %2"
                         : "=v"(w_scale[nf]) : "v"(voff), "s"((unsigned long long)base) : "memory");
        }
    }
    const std::true_type waits;
    static_for<0, NB>([&](auto j) { request(ring[0], 0, j, waits); });
    static_for<0, kHalf>([&](auto j) { bring(2, j, waits); });
    static_for<0, NB>([&](auto j) { request(ring[1], 1, j, waits); });
    static_for<kHalf, MF>([&](auto j) { bring(2, j, waits); });
    static_for<0, NB>([&](auto j) { request(ring[2], 2, j, waits); });
    static_for<0, MF * NF>([&](auto tc) { acc_clear<decltype(tc)::value>(); });
    publish();
    wait_lds_reads();
    landed(ring[0]);
    if constexpr (FP8) {
#pragma unroll
        for (int nf = 0; nf < NF; ++nf) {
            asm volatile("" : "+v"(w_scale[nf]));
        }
    }
    barrier_no_fence();
#ifdef CAM_GEMM_TIMELINE
    if (tid == 0) {
        t.phase_s[0] = (int)wall_clock64();
    }
#endif
    read_scales(0, 0);
    static_for<0, PD>([&](auto f) { read_frag(af[decltype(f)::value % AR], 0, f); });

    // Stage s0 + b, s0 even.  TAIL: the stage behind the last pair of an odd number of them, which requests nothing.
    auto stage = [&](int s0, auto bc, auto tc) {
        constexpr int b = decltype(bc)::value;
        constexpr bool TAIL = decltype(tc)::value;
        const int s = s0 + b;
        const int base = s0 & 2;   // slot of stage s0
        static_for<0, 2>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            constexpr int r = (2 * b + u) % kRing;
            constexpr int NA = u == 0 ? kHalf : MF / 2;
            constexpr int OPS = NA + NB;
            const std::integral_constant<bool, FP8> waits_fp8;
            if (u == 1) {
                if (TAIL) {
                    wait_loads_outstanding<0>();
                }
                landed(ring[r]);
                read_scales(b ^ 1, s + 1);
            }
            static_for<0, SLOTS>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                constexpr int f = (2 * b + u) * SLOTS + i;    // slot of the loop body
                constexpr int fn = f + PD, sn = fn / (2 * SLOTS);
                read_frag(af[fn % AR], sn == 2 ? base ^ 2 : base + sn, std::integral_constant<int, fn % (2 * SLOTS)>());
                __builtin_amdgcn_sched_barrier(0);
                // this slot's share of the sub-step's requests, spread over the gaps between its multiplications
                constexpr int o0 = i * OPS / SLOTS, on = (i + 1) * OPS / SLOTS - o0;
                static_for<0, NF>([&](auto nc) {
                    constexpr int n = decltype(nc)::value;
                    constexpr int nf = (i & 1) ? NF - 1 - n : n;  // (one operand stays from one multiplication to the next)
                    if constexpr (FP8) {
                        const v8i w = __builtin_shufflevector(ring[r][nf], ring[r][NF + nf], 0, 1, 2, 3, 4, 5, 6, 7);
                        acc_multiply<i * NF + nf>(w, af[f % AR], sw[b][nf], sa[b][i]);
                    } else {
                        acc_multiply<(i % MF) * NF + nf>(ring[r][(i / MF) * NF + nf], af[f % AR]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (n < NF - 1 && !TAIL) {
                        static_for<o0 + n * on / (NF - 1), o0 + (n + 1) * on / (NF - 1)>([&](auto oc) {
                            constexpr int o = decltype(oc)::value;
                            if constexpr (o < NA) {
                                bring(s + 3, std::integral_constant<int, u * kHalf + o>(), waits_fp8);
                            } else {
                                request(ring[(r + 3) % kRing], 2 * s + u + 3, std::integral_constant<int, o - NA>(), waits_fp8);
                            }
                        });
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
            });
        });
        if constexpr (!TAIL) {
            landed(ring[(2 * b + 2) % kRing]);
            barrier_no_fence();
        }
    };
    int s0 = 0;
    for (; s0 + 1 < ST; s0 += 2) {
        if (s0 == 2 && gather) {
            ask_rows();
        }
        stage(s0, std::integral_constant<int, 0>(), std::false_type());
        stage(s0, std::integral_constant<int, 1>(), std::false_type());
    }
    if (s0 < ST) {
        stage(s0, std::integral_constant<int, 0>(), std::true_type());
    }
    wait_loads_outstanding<0>();
#pragma unroll
    for (int j = 0; j < kRing * NB; ++j) {  // the registers of the last requests are taken until here
        asm volatile("" ::"v"(ring[j / NB][j % NB]));
    }
    wait_lds_reads();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products are in their registers
    barrier_no_fence();  // nobody reads or fills the stages any more
#ifdef CAM_GEMM_TIMELINE
    if (tid == 0) {
        t.phase_s[1] = (int)wall_clock64();
    }
#endif
}

// The epilogue of an item, for one wave: n row fragments x NF column fragments, sums in tiles mf * NF + nf.  One function for all
// numbers of row fragments: it is long straight-line code (the sums are named registers), and a copy for each of them would
// not stay in the instruction cache, which a CU shares with its neighbour.
//
// row_scale and col_scale: the item's scales in LDS, the columns by group of the item.  The stages 0 and 1 of the ring belong to the
// next item by now; what is staged here goes through the other two.
template <int NF, bool FP8>
__device__ __forceinline__ void epilogue_item(const GemmArgs &a, const ItemCtx &t, int8_t *lds, const float *row_scale,
                                              const float *col_scale)
{
    constexpr bool FLAT = NF == 4;
    constexpr int MF = FLAT ? 4 : 8;
    constexpr int NG = NF / 2;       // 64-column groups of this wave
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = opaque(tid) & (kWave - 1);
    const int row_in = lane & 31;
    const int col_half = (lane >> 5) * 4;
    const int N = t.N;
    const int ngroups = N / 64;
    const int n = (t.rows + 31) >> 5;

    // ---- epilogue, accumulators in registers.
    // Lane l holds activation row (l & 31) of each 32x32 fragment; registers 4j .. 4j+3 hold the four
    // consecutive weight columns 8j + 4*(l/32) + 0..3.  Dequantisation runs on that layout with one row scale
    // per lane and fragment and the column scales fetched as 16-byte vectors.  To store whole 128-byte lines,
    // every wave passes one 32-row block of 128 bytes at a time through its own slice of LDS: it writes the block, requests
    // it back as 16 bytes per lane and 8 rows per register, and stores it when the next block is computed, so that the
    // round trip through LDS runs under arithmetic (the wave has its SIMD to itself).  Stores past the tile's rows are out of
    // the range of their descriptor.
    int8_t *stage = lds + 2 * kStage;
    int8_t *slice = stage + wave * kEpiSlice;
    const int sub = lane >> 3;    // row inside a group of 8
    const int piece = lane & 7;   // 16-byte piece of the 128-byte row

    // compute(mf) for the n row fragments, each of which leaves a block in the slice; store(mf, v) gets it back as v[4].
    auto blocks = [&](auto &&compute, auto &&store) {
        v4u held[4];
        static_for<0, MF>([&](auto mc) {
            constexpr int mf = decltype(mc)::value;
            if (mf < n) {
                compute(mc);
                if constexpr (mf > 0) {
                    store(mf - 1, held);
                }
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    held[it] = *(const v4u *)(slice + (it * 8 + sub) * kEpiRowBytes + piece * 16);
                }
            }
        });
        store(n - 1, held);
    };
    // 128 bytes of columns from `col` on, in rows of `pitch` bytes: a descriptor for them and the offset of this lane's piece.
    // The next kernel reads these rows once; stored non-temporally (2) they do not push weight panels and activation tiles out
    // of the L2 (C3 both operators 519 -> 506 us, decode layer 427 -> 420 us).
    auto columns = [&](int col, int pitch) {
        return __builtin_amdgcn_make_buffer_rsrc((int8_t *)a.out + (long long)t.m0 * pitch + col, 0,
                                                 (unsigned)((t.rows - 1) * pitch + 128), 0x00020000);
    };
    auto store_rows = [&](__amdgpu_buffer_rsrc_t out, int pitch, int mf, const v4u (&v)[4]) {
        const unsigned at = (unsigned)((mf * 32 + sub) * pitch + piece * 16);
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            __builtin_amdgcn_raw_buffer_store_b128(v[it], out, at + (unsigned)(it * 8 * pitch), 0, 2);
        }
    };

    auto epilogue = [&]() {
        v4f csc[NG][2][4];  // column scales: [0] gate / [1] up of a paired group, or the two fragments of a plain one
        if (!FP8 && a.epilogue != kEpiInt32) {
#pragma unroll
            for (int i = 0; i < NG * 8; ++i) {
                csc[i >> 3][(i >> 2) & 1][i & 3] = *(const v4f *)(col_scale + (wave * NG + (i >> 3)) * 64 + (i & 7) * 8 + col_half);
            }
        }
        static_for<0, NG>([&](auto gc) {
            constexpr int gi = decltype(gc)::value;
            const int nw = t.group + gi;
            if (nw >= ngroups) {
                return;
            }
            if (a.epilogue == kEpiInt32) {
                static_for<0, 2>([&](auto nc) {
                    constexpr int nf = decltype(nc)::value;
                    const int col0 = a.gate_up ? (nf * (N / 2) + nw * 32) : (nw * 64 + nf * 32);
                    const __amdgpu_buffer_rsrc_t out = columns(col0 * 4, N * 4);
                    blocks([&](auto qc) {
                        static_for<0, 4>([&](auto jc) {
                            constexpr int j = decltype(jc)::value;
                            constexpr int r = (decltype(qc)::value * NF + 2 * gi + nf) * 16 + 4 * j;
                            // int32 sums, or the bits of the fp32 sums of an FP8 item
                            *(v4i *)(slice + row_in * kEpiRowBytes + (8 * j + col_half) * 4) = acc_bits4<r>();
                        });
                    }, [&](int mf, const v4u (&v)[4]) { store_rows(out, N * 4, mf, v); });
                });
            } else if (a.epilogue == kEpiSwiglu) {
                // t = (float(C) * w_scale[n]) * x_scale[m]; y = silu(t_gate) * t_up
                const __amdgpu_buffer_rsrc_t out = columns(nw * 32 * 4, N * 2);
                blocks([&](auto qc) {
                    constexpr int mf = decltype(qc)::value;
                    const float xs = FP8 ? 1.0f : row_scale[mf * 32 + row_in];
                    static_for<0, 4>([&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        constexpr int r = (mf * NF + 2 * gi) * 16 + 4 * j;
                        const v4f gate = acc_values<r, FP8>(), up = acc_values<r + 16, FP8>();
                        v4f y;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if constexpr (FP8) {  // the sums carry their scales already
                                y[e] = __fmul_rn(cam_silu_spec(quiet(gate[e])), up[e]);
                            } else {
                                const float tg = __fmul_rn(__fmul_rn(gate[e], csc[gi][0][j][e]), xs);
                                const float tu = __fmul_rn(__fmul_rn(up[e], csc[gi][1][j][e]), xs);
                                y[e] = __fmul_rn(cam_silu_spec(tg), tu);
                            }
                        }
                        *(v4f *)(slice + row_in * kEpiRowBytes + (8 * j + col_half) * 4) = y;
                    });
                }, [&](int mf, const v4u (&v)[4]) { store_rows(out, N * 2, mf, v); });
            } else {
                const __amdgpu_buffer_rsrc_t out = columns(nw * 64 * 2, N * 2);
                auto dequant = [&](auto fp16) {
                    blocks([&](auto qc) {
                        constexpr int mf = decltype(qc)::value;
                        const float xs = FP8 ? 1.0f : row_scale[mf * 32 + row_in];
                        static_for<0, 8>([&](auto jc) {
                            constexpr int nf = decltype(jc)::value / 4, j = decltype(jc)::value % 4;
                            const v4f sum = acc_values<(mf * NF + 2 * gi + nf) * 16 + 4 * j, FP8>();
                            float f[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                f[e] = FP8 ? sum[e] : __fmul_rn(__fmul_rn(sum[e], csc[gi][nf][j][e]), xs);
                            }
                            // two values per conversion instruction: with the rounding spelled out in integer
                            // arithmetic this epilogue took a quarter of a short-K tile's time in the vector ALU
                            v2u v;
                            if constexpr (decltype(fp16)::value) {
                                // each product rounded to fp32 first: the compiler would make one instruction of the
                                // multiplication and the conversion, with one rounding
                                asm("" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]));
                                v = v2u{f32_to_fp16_bits(f[0]) | (f32_to_fp16_bits(f[1]) << 16),
                                        f32_to_fp16_bits(f[2]) | (f32_to_fp16_bits(f[3]) << 16)};
                            } else {
                                v = v2u{f32x2_to_bf16x2_bits(f[0], f[1]), f32x2_to_bf16x2_bits(f[2], f[3])};
                            }
                            *(v2u *)(slice + row_in * kEpiRowBytes + (nf * 32 + 8 * j + col_half) * 2) = v;
                        });
                    }, [&](int mf, const v4u (&v)[4]) { store_rows(out, N * 2, mf, v); });
                };
                if (a.out_fp16) {
                    dequant(std::true_type());
                } else {
                    dequant(std::false_type());
                }
            }
        });
    };

    // ---- FP8 gate/up GEMM whose output feeds the next FP8 GEMM: quantise the SwiGLU product here.  A block of
    // 128 product columns is what four neighbouring column groups hold (the four waves of a tall item, two waves of a
    // flat one), so the block maximum needs one exchange through LDS; every wave of the workgroup takes part in its barrier.
    auto epilogue_quant = [&]() {
        if constexpr (FP8) {
            float *rowmax = (float *)(stage + 4 * kEpiSlice);  // [wave][tile row]
            float y[MF][NG][16];
            static_for<0, MF>([&](auto mc) {
                constexpr int mf = decltype(mc)::value;
                if (mf >= n) {
                    return;
                }
                float m = 0.0f;
                static_for<0, NG * 4>([&](auto ic) {
                    constexpr int gi = decltype(ic)::value / 4, i = decltype(ic)::value % 4 * 4;
                    constexpr int r = (mf * NF + 2 * gi) * 16 + i;
                    const v4f gate = acc_values<r, true>(), up = acc_values<r + 16, true>();
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        y[mf][gi][i + e] = __fmul_rn(cam_silu_spec(quiet(gate[e])), up[e]);
                        m = fmaxf(m, fabsf(y[mf][gi][i + e]));
                    }
                });
                m = fmaxf(m, __shfl_xor(m, 32, kWave));
                if (lane < 32) {
                    rowmax[wave * 256 + mf * 32 + lane] = m;
                }
            });
            wait_lds_reads();
            barrier_no_fence();
            if (t.group >= ngroups) {
                return;
            }
            const int I = N / 2;
            // 32 rows x 32 bytes per column group (48-byte pitch in the slice): two lanes per row store its two 16-byte halves
            const int qrow = lane >> 1, qpiece = lane & 1;
            const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
                (int8_t *)a.out + (long long)t.m0 * I + t.group * 32, 0, (unsigned)((t.rows - 1) * I + NG * 32), 0x00020000);
            v4u held[NG];
            auto store = [&](int mf) {
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
                    __builtin_amdgcn_raw_buffer_store_b128(held[gi], out, (unsigned)((mf * 32 + qrow) * I + gi * 32 + qpiece * 16),
                                                           0, 0);
                }
            };
#pragma unroll
            for (int mf = 0; mf < MF; ++mf) {
                if (mf >= n) {
                    break;
                }
                const float *pm = rowmax + (FLAT ? (wave & 2) * 256 : 0) + mf * 32 + row_in;
                const float m = FLAT ? fmaxf(pm[0], pm[256]) : fmaxf(fmaxf(pm[0], pm[256]), fmaxf(pm[512], pm[768]));
                const int ex = fp8_block_scale_exp(m);
                const float f1 = exp2_int(-(ex / 2)), f2 = exp2_int(-(ex - ex / 2));
                int w[NG][4];
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float *c = y[mf][gi] + 4 * j;
                        w[gi][j] = 0;
                        w[gi][j] = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(c[0], f1), f2),
                                                                   __fmul_rn(__fmul_rn(c[1], f1), f2), w[gi][j], false);
                        w[gi][j] = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(c[2], f1), f2),
                                                                   __fmul_rn(__fmul_rn(c[3], f1), f2), w[gi][j], true);
                    }
                }
                if (mf > 0) {
                    store(mf - 1);
                }
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
                    int8_t *part = slice + gi * (kEpiSlice / 2);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        *(int *)(part + row_in * 48 + 8 * j + col_half) = w[gi][j];
                    }
                    held[gi] = *(const v4u *)(part + qrow * 48 + qpiece * 16);
                }
                if ((FLAT ? (wave & 1) : wave) == 0 && lane < 32 && mf * 32 + lane < t.rows) {
                    const long long grow = t.m0 + mf * 32 + lane;
                    a.out_scale8[grow * (I >> 7) + (t.group >> 2)] = (uint8_t)(ex + 127);
                }
            }
            store(n - 1);
        }
    };

    if (FP8 && a.epilogue == kEpiSwigluFp8) {
        epilogue_quant();
    } else {
        epilogue();
    }
    barrier_no_fence();  // the staging slices are free again before the next item's loads land
}

template <bool FP8>
__global__ __launch_bounds__(kThreads, 1) void gemm_kernel(GemmArgs a)
{
    __shared__ __attribute__((aligned(1024))) int8_t lds[kLdsBytes];
    // int8: row scales, then column scales (64 per group), of the item at work and of the next one.  FP8: row scales of the item at
    // work, a word of four K blocks per row: [K block / 4][row].
    __shared__ __attribute__((aligned(16))) float scale_s[FP8 ? 1 : 2][FP8 ? 4 : 256 + 8 * 64];
    __shared__ __attribute__((aligned(16))) uint8_t a_scale8_s[FP8 ? kScaleKb * 256 : 4];
    __shared__ __attribute__((aligned(16))) SchedItem next_s;
    __shared__ __attribute__((aligned(16))) int32_t rows_s[256];  // with a_rows: where the rows of the item lie
    __shared__ int item_s;
#ifdef CAM_GEMM_TIMELINE
    __shared__ int phase_s[2];
    __shared__ int next_idx_s;
#endif

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int32_t *sched = a.sched;
    const int32_t *qstart = sched + kSchedQueueStart;
    int32_t *qcount = sched + kSchedQueueCount;
    const SchedItem *items = (const SchedItem *)(sched + kSchedHeader);
    const bool shared = (sched[3] & 2) != 0;   // long schedules: one queue per XCD, every item asked for
    const int me = shared ? (int)blockIdx.x % max(min(sched[2], kMaxQueues), 1) : (int)blockIdx.x;  // this workgroup's queue
    const int q0 = qstart[min(me, kMaxQueues)];
    const int qlen = me < kMaxQueues ? qstart[me + 1] - q0 : 0;
    bool own_empty = qlen <= (shared ? 0 : 1);  // an own queue's first item needs no asking; there may be nothing after it

    // Work items.  Short schedules: every workgroup has a queue of its own, built to last as long as the others
    // (sched_device.h).  Its first item is its own without asking; for the following ones it advances its queue's
    // counter with a device-scope atomic, a round trip to the memory side.  Long schedules: the workgroups of an XCD share one
    // queue and ask for every item, the first included.  Every counter has a cache line of its own.
    // The item after the current one is asked for in front of the epilogue before it, its number looked at and its
    // descriptor requested (to LDS) while the first loads of the current item are on their way, and its own first loads go
    // out between the K loop and the epilogue of the current item: no item but a workgroup's first starts with a chain of
    // round trips.
    // A workgroup whose queue has run out helps the queue with the most items left (its own XCD's first, so that
    // what it fetches is likely to be in its L2): wave 0 looks at every counter at once, one round trip, and its
    // first lane then advances the chosen one.  A counter only ever grows and every queue is finite, so every
    // workgroup leaves.
    int taken = 0;  // thread 0
    auto take_begin = [&]() {
        if (tid == 0 && !own_empty) {
            taken = atomicAdd(&qcount[me * kSchedQueueStride], 1);
        }
    };
    auto take_end = [&]() -> int {  // all threads of wave 0
        const int i = __builtin_amdgcn_readfirstlane(taken);
        if (own_empty || i >= qlen) {
            own_empty = true;
            return -1;
        }
        return q0 + i;
    };
    auto steal = [&]() -> int {  // all lanes of wave 0; the result is valid in every lane
        const int lane = tid & (kWave - 1);
        const int nq = min(sched[2], kMaxQueues);
        if ((sched[3] & 1) != 0) {  // every queue's only item is its workgroup's own: there is nothing to take over
            return -1;
        }
        for (int attempt = 0; attempt < 4; ++attempt) {
            int best = -1;  // (items left, same XCD, queue) packed so that the maximum is the choice
            for (int v = lane; v < nq; v += kWave) {
                const int len = qstart[v + 1] - qstart[v];
                const int seen = __hip_atomic_load(&qcount[v * kSchedQueueStride], __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                const int left = len - seen;
                if (left > 0 && v != me) {
                    best = max(best, (min(left, 1023) << 11) | ((v % kNumXcd == me % kNumXcd ? 1 : 0) << 10) | v);
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                best = max(best, __shfl_xor(best, off, kWave));
            }
            if (best < 0) {
                return -1;
            }
            // the queue number fits ten bits only below 1024 queues, which kMaxQueues guarantees
            const int v = best & 1023;
            int got = -1;
            if (lane == 0) {
                const int i = atomicAdd(&qcount[v * kSchedQueueStride], 1);
                got = i < qstart[v + 1] - qstart[v] ? qstart[v] + i : -1;
            }
            got = __shfl(got, 0, kWave);
            if (got >= 0) {
                return got;
            }
        }
        return -1;
    };

    auto decode = [&](const SchedItem &it, int buf) {
        ItemCtx t;
        t.g = __builtin_amdgcn_readfirstlane(it.g);
        t.m0 = __builtin_amdgcn_readfirstlane(it.m0);
        t.rows = __builtin_amdgcn_readfirstlane(it.rows);
        const int nb = __builtin_amdgcn_readfirstlane(it.nb);
        t.flat = __builtin_amdgcn_readfirstlane(it.flat) != 0;
        t.mf = (t.rows + 31) >> 5;
        t.mf = min(t.mf, t.flat ? 4 : 8);
        t.group = t.flat ? nb * 8 + 2 * wave : nb * 4 + wave;
        t.buf = buf;
        t.Kd = a.Kd;
        t.N = a.N;
        t.a_tile = a.a_rows != nullptr ? a.a : a.a + (long long)t.m0 * a.Kd;
        t.wg = a.per_expert ? a.list.w[t.g] : a.w + (long long)t.g * a.Kd * a.N;
        t.sg = a.per_expert ? a.list.s[t.g] : a.w_scale + (long long)t.g * a.N;
#ifdef CAM_GEMM_TIMELINE
        t.phase_s = phase_s;
#endif
        return t;
    };

    // The first loads of an item: stages 0 and 1 of its rows and its scales, to LDS.  Rows beyond the tile repeat its last one, what
    // lies beyond the end of K the last chunk of the row.
    auto ask_ahead = [&](const ItemCtx &t) {
        const int lane = opaque(tid) & (kWave - 1);
        const unsigned long long tile = scalar_address(t.a_tile);
        const unsigned dst = __builtin_amdgcn_readfirstlane(lds_address(lds) + (unsigned)(wave * t.mf * 1024));
        const bool gather = a.a_rows != nullptr;
        const int r0 = 8 * wave * t.mf + (lane >> 3);
        int at[8], row = min(wave * kWave + lane, t.rows - 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            at[j] = min(r0 + 8 * j, t.rows - 1);
        }
        // All of them in one round trip to the LDS, here and in the K loop.  Asked one by one, each beside its load: layer of 8192 tokens x
        // 4096 1506 us, now 1499, of 4093 in FP8 800, now 796; both GEMMs of 8192 rows x 7168, which do not gather, 453, now 446,
        // as before there was anything to gather.
        if (gather) {
            row = rows_s[row];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                at[j] = rows_s[at[j]];
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j < t.mf) {
                const int r = r0 + 8 * j;
                const int c16 = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
                dma16(tile, (unsigned)(at[j] * t.Kd + c16), dst + (unsigned)(j * 1024));
                dma16(tile, (unsigned)(at[j] * t.Kd + min(kStageK + c16, t.Kd - 16)), dst + (unsigned)(kStage + j * 1024));
            }
        }
        const long long row0 = gather ? 0 : t.m0;
        const int ngroups = t.N / 64;
        if constexpr (FP8) {
            const int KB = t.Kd >> 7;
            const uint8_t *base = a.a_scale8 + row0 * KB;
            if ((KB & 3) == 0) {
                const unsigned long long words = scalar_address(base);
                const unsigned to = __builtin_amdgcn_readfirstlane(lds_address(a_scale8_s) + (unsigned)(wave * kWave * 4));
                for (int q = 0; q < KB >> 2; ++q) {
                    dma4(words, (unsigned)(row * KB + 4 * q), to + (unsigned)(q * 1024));
                }
            } else {
                // Rows that are no whole words go through registers byte by byte, in front of the epilogue: up to 5 us of a tile.
                // FP8 GEMM of two tiles of 256 rows a workgroup, N 4096, K / 128 = 12 13 15 16: 68.5 72.4 84.0 80.0 us; 40 41 43 44: 164.9
                // 163.9 182.9 175.9.
                for (int kb = 0; kb < KB; ++kb) {
                    a_scale8_s[((kb >> 2) * 256 + wave * kWave + lane) * 4 + (kb & 3)] = base[(long long)row * KB + kb];
                }
            }
        } else if (a.epilogue != kEpiInt32) {
            const unsigned to = __builtin_amdgcn_readfirstlane(lds_address(scale_s[t.buf]));
            dma4(scalar_address(a.a_scale + row0), (unsigned)(row * 4), to + (unsigned)(wave * kWave * 4));
            const unsigned long long columns = scalar_address(t.sg);
            const int per_wave = t.flat ? 2 : 1;
            for (int gi = 0; gi < per_wave; ++gi) {
                const int nw = min(t.group + gi, ngroups - 1);
                const int col = a.gate_up ? (lane >> 5) * (t.N / 2) + nw * 32 + (lane & 31) : nw * 64 + lane;
                dma4(columns, (unsigned)(col * 4), to + (unsigned)((256 + (wave * per_wave + gi) * 64) * 4));
            }
        }
    };

#ifdef CAM_GEMM_TIMELINE
    int cur_idx = -1;
#endif
    auto first_item = [&](int buf, bool steal_only) -> ItemCtx {  // rows 0: there is none
        if (tid < kWave) {
            int idx = -1;
            if (!steal_only) {
                if (shared) {
                    take_begin();
                    idx = take_end();
                } else {
                    idx = qlen > 0 ? q0 : -1;
                }
            }
            idx = idx >= 0 ? idx : steal();
            if (tid == 0) {
                item_s = idx;
            }
        }
        __syncthreads();
        const int idx = __builtin_amdgcn_readfirstlane(item_s);
        ItemCtx t;
        t.rows = 0;
        if (idx >= 0) {
            t = decode(items[idx], buf);
            if (a.a_rows != nullptr) {
                rows_s[tid] = a.a_rows[t.m0 + min(tid, t.rows - 1)];
                __syncthreads();
            }
            ask_ahead(t);
#ifdef CAM_GEMM_TIMELINE
            cur_idx = idx;
#endif
        }
        return t;
    };
    ItemCtx t = first_item(0, false);
    take_begin();
    while (t.rows > 0) {
#ifdef CAM_GEMM_TIMELINE
        // Build option for profiling only: thread 0 leaves the item's start and end times (wall_clock64, 100 MHz)
        // and the workgroup that ran it in the item's two spare words.
        const long long timeline_t0 = wall_clock64();
#endif
        auto publish = [&]() {
            if (tid < kWave) {
                const int n = take_end();
                if (n < 0) {
                    if (tid == 0) {
                        next_s.rows = 0;
                    }
                } else if (tid < 2) {
                    dma16(scalar_address(items + n), (unsigned)(tid * 16), __builtin_amdgcn_readfirstlane(lds_address(&next_s)));
                }
#ifdef CAM_GEMM_TIMELINE
                if (tid == 0) {
                    next_idx_s = n;
                }
#endif
            }
        };
        // With a_rows: where the rows of the next item lie, asked for in the third stage of the K loop.  Its descriptor has come (wave 0
        // has waited for younger loads, and a barrier has followed), and every wave has its own item's rows in registers.  One
        // more load in flight makes the waits that count them stricter, not laxer.
        auto ask_rows = [&]() {
            const int rows = __builtin_amdgcn_readfirstlane(next_s.rows);
            if (rows > 0) {
                const int m0 = __builtin_amdgcn_readfirstlane(next_s.m0);
                const int lane = opaque(tid) & (kWave - 1);
                dma4(scalar_address(a.a_rows + m0), (unsigned)(min(wave * kWave + lane, rows - 1) * 4),
                     __builtin_amdgcn_readfirstlane(lds_address(rows_s) + (unsigned)(wave * kWave * 4)));
            }
        };
        auto run = [&](auto mc, auto nc) {
            k_loop<decltype(mc)::value, decltype(nc)::value, FP8>(a, t, lds, a_scale8_s, rows_s, publish, ask_rows);
        };
        if (t.flat) {
            const std::integral_constant<int, 4> nf;
            switch (t.mf) {
                case 1: run(std::integral_constant<int, 1>(), nf); break;
                case 2: run(std::integral_constant<int, 2>(), nf); break;
                case 3: run(std::integral_constant<int, 3>(), nf); break;
                default: run(std::integral_constant<int, 4>(), nf); break;
            }
        } else {
            const std::integral_constant<int, 2> nf;
            switch (t.mf) {
                case 1: run(std::integral_constant<int, 1>(), nf); break;
                case 2: run(std::integral_constant<int, 2>(), nf); break;
                case 3: run(std::integral_constant<int, 3>(), nf); break;
                case 5: run(std::integral_constant<int, 5>(), nf); break;
                case 6: run(std::integral_constant<int, 6>(), nf); break;
                case 7: run(std::integral_constant<int, 7>(), nf); break;
                case 8: run(std::integral_constant<int, 8>(), nf); break;
                default: run(std::integral_constant<int, 4>(), nf); break;
            }
        }
        // next_s is there: wave 0 has waited for younger loads, and a barrier ends the K loop
        const SchedItem nx = next_s;
        ItemCtx next;
        next.rows = __builtin_amdgcn_readfirstlane(nx.rows);
        if (next.rows > 0) {
            next = decode(nx, t.buf ^ 1);
            ask_ahead(next);
            take_begin();
        }
        const float *scales = scale_s[FP8 ? 0 : t.buf];
        if (t.flat) {
            epilogue_item<4, FP8>(a, t, lds, scales, scales + 256);
        } else {
            epilogue_item<2, FP8>(a, t, lds, scales, scales + 256);
        }
#ifdef CAM_GEMM_TIMELINE
        if (tid == 0) {
            int32_t *stamp = (int32_t *)&items[cur_idx];
            stamp[6] = (int32_t)timeline_t0;
            stamp[7] = (int32_t)wall_clock64();
            stamp[3] = (stamp[3] & 0xffff) | ((int)blockIdx.x << 16);  // (no kernel reads split)
            // ticks from the start of the item to its first multiply and to the end of its K loop, in the upper
            // halves of the column-block and shape words (both below 2^16 and read before an item starts)
            const int d1 = min(max(phase_s[0] - (int32_t)timeline_t0, 0), 0xffff);
            const int d2 = min(max(phase_s[1] - (int32_t)timeline_t0, 0), 0x7fff);
            stamp[4] = (stamp[4] & 0xffff) | (d1 << 16);
            stamp[5] = (stamp[5] & 0xffff) | (d2 << 16);
        }
        cur_idx = next_idx_s;
#endif
        if (next.rows == 0) {
            next = first_item(t.buf ^ 1, true);
        }
        t = next;
    }
}

__global__ __launch_bounds__(1024) void build_sched_kernel(SchedBuild sb)
{
    __shared__ SchedShared sh;
    load_group_list<1024>(sh, sb);
    build_sched_part<1024>(sh, sb, (int)blockIdx.y, (int)blockIdx.x, (int)gridDim.x);
}

// SwiGLU product rows (fp32) -> int8 rows + per-row scale:
//   m = max|y|; y_scale = m * (1/127); q = rint((y * 127) * (1/m)).   One wave per row (four rows per workgroup):
// the row waits in registers between the maximum and the scaling, the maximum needs wave shuffles only, and no
// wave waits for another.
__global__ __launch_bounds__(256) void requant_kernel(const float *__restrict__ y, int I,
                                                      const int32_t *__restrict__ sched, long long max_rows,
                                                      int8_t *__restrict__ q, float *__restrict__ scale)
{
    const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const long long valid = sched != nullptr ? min((long long)sched[1], max_rows) : max_rows;
    if (row >= valid) {
        return;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int n4 = I >> 2;
    constexpr int kMaxPer = 16;  // I <= 4096
    v4f v[kMaxPer];
    float m = 0.0f;
    const v4f *src = (const v4f *)(y + row * I);
#pragma unroll
    for (int j = 0; j < kMaxPer; ++j) {
        const int c = lane + j * kWave;
        v[j] = v4f{0.f, 0.f, 0.f, 0.f};
        if (c < n4) {
            v[j] = __builtin_nontemporal_load(src + c);
        }
    }
#pragma unroll
    for (int j = 0; j < kMaxPer; ++j) {
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[j][0]), fabsf(v[j][1])), fmaxf(fabsf(v[j][2]), fabsf(v[j][3]))));
    }
    m = wave_max(m);
    const bool zero_row = m == 0.0f;
    const float rcp = zero_row ? 0.0f : __fdiv_rn(1.0f, m);
    if (lane == 0) {
        scale[row] = zero_row ? 0.0f : __fmul_rn(m, 1.0f / 127.0f);
    }
    uint32_t *dst = (uint32_t *)(q + row * I);
#pragma unroll
    for (int j = 0; j < kMaxPer; ++j) {
        const int c = lane + j * kWave;
        if (c < n4) {
            int b[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                b[e] = (int)rintf(__fmul_rn(__fmul_rn(v[j][e], 127.0f), rcp));
            }
            dst[c] = (uint32_t)(b[0] & 0xff) | ((uint32_t)(b[1] & 0xff) << 8) | ((uint32_t)(b[2] & 0xff) << 16) |
                     ((uint32_t)(b[3] & 0xff) << 24);
        }
    }
}

// fp32 rows -> FP8 E4M3 with one E8M0 scale per row and 128 columns (include/cam_fp8_spec.h).  A wave takes 512
// columns of a row: lane l the 8 columns from 8 l, so a block of 128 columns is a quarter of the wave.
__global__ __launch_bounds__(256) void requant_fp8_kernel(const float *__restrict__ y, int I,
                                                          const int32_t *__restrict__ sched, long long max_rows,
                                                          uint8_t *__restrict__ q, uint8_t *__restrict__ scale)
{
    const long long row = blockIdx.x;
    const long long valid = sched != nullptr ? min((long long)sched[1], max_rows) : max_rows;
    if (row >= valid) {
        return;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    for (int c0 = wave * 512; c0 < I; c0 += 4 * 512) {
        const int col = c0 + lane * 8;
        const bool live = col < I;
        float x[8];
        float m = 0.0f;
        if (live) {
            const v4f lo = __builtin_nontemporal_load((const v4f *)(y + row * I + col));
            const v4f hi = __builtin_nontemporal_load((const v4f *)(y + row * I + col + 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[e] = lo[e];
                x[4 + e] = hi[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                m = fmaxf(m, fabsf(x[e]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[e] = 0.0f;
            }
        }
        m = row_max(m);
        const int ex = fp8_block_scale_exp(m);
        const float f1 = exp2_int(-(ex / 2)), f2 = exp2_int(-(ex - ex / 2));
        int lo = 0, hi = 0;
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[0], f1), f2), __fmul_rn(__fmul_rn(x[1], f1), f2), lo,
                                             false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[2], f1), f2), __fmul_rn(__fmul_rn(x[3], f1), f2), lo,
                                             true);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[4], f1), f2), __fmul_rn(__fmul_rn(x[5], f1), f2), hi,
                                             false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(__fmul_rn(x[6], f1), f2), __fmul_rn(__fmul_rn(x[7], f1), f2), hi,
                                             true);
        if (live) {
            *(v2u *)(q + row * I + col) = v2u{(uint32_t)lo, (uint32_t)hi};
            if ((lane & 15) == 0) {
                scale[row * (I >> 7) + (col >> 7)] = (uint8_t)(ex + 127);
            }
        }
    }
}

// Row-major [G,Kd,N] int8 -> MFMA operand order.  One thread writes one 16-byte piece: piece (nw, ks, nf, lane)
// holds K rows ks*32 + (lane/32)*16 + 0..15 of logical column
//   gate_up ? nf*(N/2) + nw*32 + lane%32 : nw*64 + nf*32 + lane%32.
// The NW = N/64 column groups are stored in blocks of eight (the last block may hold fewer, gw of them); a block
// starts at piece 8*(nw/8)*KS*128 of the expert and orders its pieces as [ks/2][nw%8][ks%2][nf][lane], i.e. the
// gw * 4 KB that one 64-byte K step of the block's groups needs are contiguous.
__global__ __launch_bounds__(256) void prepack_kernel(const int8_t *__restrict__ src, int8_t *__restrict__ dst,
                                                      int Kd, int N, int gate_up, long long pieces_per_expert)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int g = blockIdx.y;
    if (p >= pieces_per_expert) {
        return;
    }
    const int KS = Kd / 32;
    const int lane = (int)(p & 63);
    long long r = p >> 6;
    const int nf = (int)(r & 1);
    r >>= 1;
    const int ks = (int)(r % KS);
    const int nw = (int)(r / KS);
    const int col = gate_up ? nf * (N / 2) + nw * 32 + (lane & 31) : nw * 64 + nf * 32 + (lane & 31);
    const int k0 = ks * 32 + (lane >> 5) * 16;
    const int8_t *s = src + (long long)g * Kd * N + (long long)k0 * N + col;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t b0 = (uint8_t)s[(long long)(4 * j + 0) * N];
        uint32_t b1 = (uint8_t)s[(long long)(4 * j + 1) * N];
        uint32_t b2 = (uint8_t)s[(long long)(4 * j + 2) * N];
        uint32_t b3 = (uint8_t)s[(long long)(4 * j + 3) * N];
        w[j] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    }
    v4u o = {w[0], w[1], w[2], w[3]};
    const int NW = N / 64;
    const int block = nw >> 3;
    const int gw = min(8, NW - 8 * block);
    const long long q = (long long)block * 8 * KS * 128 + (long long)(ks >> 1) * (gw * 256) + (nw & 7) * 256 +
                        (ks & 1) * 128 + nf * 64 + lane;
    *((v4u *)(dst + (long long)g * Kd * N) + q) = o;
}

// Workgroups of the persistent kernel: one per CU of the device the launch goes to (looked up once per device).
constexpr int kMaxDevices = 64;
std::atomic<int> g_num_cus[kMaxDevices];

hipError_t cus_of_current_device(int *out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        return e;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        return hipErrorInvalidDevice;
    }
    int n = g_num_cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) {
            return e;
        }
        n = n > 0 ? n : 256;
        g_num_cus[dev].store(n, std::memory_order_relaxed);
    }
    *out = n;
    return hipSuccess;
}

}  // namespace

int sched_max_items(int64_t max_rows, int G, int N)
{
    // tall experts own at most max_rows / 129 + G row tiles between them, flat experts one each
    const int64_t tiles = max_rows / 129 + G;
    return (int)(tiles * ((N + 255) / 256));
}

uint64_t sched_bytes(int64_t max_rows, int G, int N)
{
    return (uint64_t)(kSchedHeader + (int64_t)sched_max_items(max_rows, G, N) * (int)(sizeof(SchedItem) / 4)) * 4;
}

hipError_t gemm_workgroups(int *out)
{
    int n = 0;
    const hipError_t e = cus_of_current_device(&n);
    if (e == hipSuccess) {
        *out = n < kMaxQueues ? n : kMaxQueues;
    }
    return e;
}

hipError_t launch_build_sched(const int64_t *group_list, int cumulative, int G, int64_t max_rows, int nspec,
                              const SchedSpec *specs, hipStream_t stream)
{
    if (G <= 0 || G > kMaxExperts || nspec < 1 || nspec > 2) {
        return hipErrorInvalidValue;
    }
    SchedBuild sb{};
    sb.group_list = group_list;
    sb.cumulative = cumulative;
    sb.G = G;
    sb.nspec = nspec;
    sb.max_rows = (long long)max_rows;
    sb.spec[0] = specs[0];
    sb.spec[1] = nspec > 1 ? specs[1] : specs[0];
    const hipError_t qe = gemm_workgroups(&sb.queues);
    if (qe != hipSuccess) {
        return qe;
    }
    const int cap = max(sb.spec[0].max_items, sb.spec[1].max_items);
    sb.parts = min(max(cap / 2048, 1), 4);  // long tables only: two turns of a thousand items cost no more than a second workgroup
    hipLaunchKernelGGL(build_sched_kernel, dim3((unsigned)sb.parts, (unsigned)nspec), dim3(1024), 0, stream, sb);
    return hipGetLastError();
}

// Offsets of gathered rows are 32 bits wide, half of which mean "none", and the next item's rows are asked for in the third stage of
// the K loop.
bool gemm_gathers(int64_t a_count, int64_t Kd)
{
    return a_count > 0 && Kd >= 4 * kStageK && a_count <= 0x7fffffff / Kd;
}

hipError_t launch_gemm(const GemmArgs &a, hipStream_t stream)
{
    if (a.sched == nullptr || (a.a_rows != nullptr && !gemm_gathers(a.a_count, a.Kd))) {
        return hipErrorInvalidValue;
    }
    if (a.Kd % kStageK != 0 || a.Kd < kStageK || a.N % 64 != 0 || (a.gate_up && a.N % 128 != 0)) {
        return hipErrorInvalidValue;
    }
    int num_cus = 0;
    const hipError_t ce = gemm_workgroups(&num_cus);
    if (ce != hipSuccess) {
        return ce;
    }
    if (a.fp8) {
        if (a.Kd % 128 != 0 || a.N % 128 != 0 || (a.gate_up && a.N % 256 != 0) || a.Kd / 128 > kScaleKb ||
            a.per_expert || a.a_scale8 == nullptr || a.w_scale8 == nullptr) {
            return hipErrorInvalidValue;
        }
        if (a.epilogue == kEpiSwigluFp8 && (!a.gate_up || a.out_scale8 == nullptr)) {
            return hipErrorInvalidValue;
        }
        hipLaunchKernelGGL(gemm_kernel<true>, dim3((unsigned)num_cus), dim3(kThreads), 0, stream, a);
    } else {
        if (a.epilogue == kEpiSwigluFp8) {
            return hipErrorInvalidValue;
        }
        hipLaunchKernelGGL(gemm_kernel<false>, dim3((unsigned)num_cus), dim3(kThreads), 0, stream, a);
    }
    return hipGetLastError();
}

hipError_t launch_requant(const float *y, int64_t max_rows, int I, const int32_t *sched_for_rows, int8_t *q,
                          float *scale, hipStream_t stream)
{
    if (max_rows <= 0) {
        return hipSuccess;
    }
    if (I % 4 != 0 || I > 4096) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(requant_kernel, dim3((unsigned)((max_rows + 3) / 4)), dim3(256), 0, stream, y, I, sched_for_rows,
                       (long long)max_rows, q, scale);
    return hipGetLastError();
}

hipError_t launch_requant_fp8(const float *y, int64_t max_rows, int I, const int32_t *sched_for_rows, uint8_t *q,
                              uint8_t *scale, hipStream_t stream)
{
    if (max_rows <= 0) {
        return hipSuccess;
    }
    if (I % 128 != 0) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(requant_fp8_kernel, dim3((unsigned)max_rows), dim3(256), 0, stream, y, I, sched_for_rows,
                       (long long)max_rows, q, scale);
    return hipGetLastError();
}

hipError_t launch_prepack(const int8_t *src, int8_t *dst, int G, int Kd, int N, int gate_up, hipStream_t stream)
{
    if (Kd % kBK != 0 || N % 64 != 0 || (gate_up && N % 128 != 0)) {
        return hipErrorInvalidValue;
    }
    const long long pieces = (long long)Kd * N / 16;
    dim3 grid((unsigned)((pieces + 255) / 256), (unsigned)G);
    hipLaunchKernelGGL(prepack_kernel, grid, dim3(256), 0, stream, src, dst, Kd, N, gate_up, pieces);
    return hipGetLastError();
}

}  // namespace cam
