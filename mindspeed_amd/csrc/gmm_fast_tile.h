// The tiles of the fast path of the 16-bit grouped matmul for gfx950, included by the kernels that run them (gmm_fast.hip: one
// product; gmm_pair.hip: both gradients of one): 256x256x64 macro tile per
// 256-thread workgroup (2x2 wavefronts, 128x128 per wavefront = 8x8
// v_mfma_f32_16x16x32), for problems whose pointers and strides allow 16-byte
// vector access everywhere.  All edge handling is branch-free (clamped addresses,
// zeros on the reduction tail).  The last row tile of a group may be a
// 128x256 or 64x256 tile (1x4 wavefronts of 128x64 / 64x64) so that ragged
// groups do not pay for a full 256-row tile; the tile table says which.
//
// What bounds it: with real data the board's power limit (1400 W), not the issue slots, so a
// launch's time follows its energy.  Hence the 16x16x32 matrix instruction (same rate as
// 32x32x16, 14 % less energy per product in a loop of nothing else) and operands that go from
// global memory to LDS without passing through registers.  The same tile on 32x32x16 with
// register-staged operands ran 8192 x 4096 x 28672 in 8 groups at 1189 (forward, NN) / 1231
// (dX, NT) / 1055 (dW, TN) TFLOP/s, this one at 1369 / 1454 / 1139 (bf16, random operands, one box).
//
// LDS layout per operand tile
//   * operand contiguous along the reduction dim in memory ("RED"): stored as
//     [outer][64 reduction] rows of 128 bytes with an XOR swizzle of the 16-byte
//     chunks; MFMA fragments are read with ds_read_b128 (bank-conflict free).
//   * operand contiguous along the outer dim (row of A / column of B): stored as it
//     lies in memory, [64 reduction][256 outer], so the global loads stay fully
//     coalesced (32 lanes x 16 bytes per memory row).  A lane of a 256-row tile reads
//     16 bytes = 8 outer indices of each of its 8 reduction indices (ds_read_b128, no
//     swizzle: 16 lanes read 256 consecutive bytes) and puts the MFMA fragments (8
//     consecutive reduction values of one outer index) together with v_perm_b32, one per
//     dword.  Block t then holds every eighth outer index of the wavefront from t on; the
//     epilogue undoes that.  The transposing read ds_read_b64_tr_b16, which the small
//     tiles use (their wavefronts cover 64 columns, 8 chunks, not 16), takes twice the LDS
//     instructions: 8192 x 4096 x 28672 in 8 groups with it and with this, one box, dW 1139
//     -> 1177 TFLOP/s (1326 -> 1419 on all-zero operands, where power does not limit),
//     forward 1366 -> 1389.
//
// The small tail tiles of a RED A run the same way with more stages (dma_small_k_loop below).  Those of an
// A of the other kind (the weight gradient of a width that is no multiple of 256) keep 32x32x16 and a register-staged K loop
// (the transfers' swizzle is made for 512-byte rows; whether one for shorter rows would pay there was not measured):
//   registers hold tile kt+1 (loaded one K step ago), LDS stage `cur` holds tile kt.
//   step kt, phase p = 0..3 (one 16-wide slice of the 64-wide K step each):
//       store part p of tile kt+1 from registers to LDS stage `nxt`
//       issue the global loads of part p of tile kt+2 into the same registers
//       read the MFMA fragments of slice p+1 from LDS stage `cur`
//       run the MFMAs on the fragments of slice p
//   (parts: loads 0-3 / 4-7 of A, loads 0-3 / 4-7 of B, of each lane's eight per operand)
//   in phase 3 a workgroup barrier sits between the two halves of the MFMAs; after it
//   the fragments of slice 0 of tile kt+1 are read from stage `nxt`.
#pragma once

#include <type_traits>
#include <utility>

#include "gmm_common.h"

#ifdef MS_TRACE_TILES
// Diagnostic build only (python -m mindspeed_amd.build --trace): every workgroup of the fast kernels records when it
// started, found its tile, had its first operands in LDS, left the K loop and finished (100 MHz wall clock), plus the
// compute unit it ran on, the tile's height and whether it was one of a weight gradient; ms_trace_read copies the records of
// the last launches out.  The record of workgroup b is slot b % kTraceSlots, so a launch with more workgroups than that
// overwrites its own early records.  One translation unit: gmm_fast.hip takes gmm_pair.hip in.
namespace ms {
constexpr int kTraceSlots = 16384;
__device__ long long g_tile_trace[kTraceSlots * 8];
}  // namespace ms
#define MS_TRACE(i) do { if (threadIdx.x == 0) ms::g_tile_trace[(blockIdx.x % ms::kTraceSlots) * 8 + (i)] = wall_clock64(); } while (0)
#define MS_TRACE_END(height, weight_gradient) \
    do { \
        if (threadIdx.x == 0) { \
            unsigned hw_id, xcc_id; \
            asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw_id)); \
            asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc_id)); \
            long long *rec = ms::g_tile_trace + (blockIdx.x % ms::kTraceSlots) * 8; \
            rec[0] = (static_cast<long long>(xcc_id & 0xf) << 32) | ((hw_id >> 8) & 0xff) | (1ll << 40);   /* XCC, CU/SH/SE bits, "valid" */ \
            rec[5] = wall_clock64(); \
            rec[6] = (height); \
            rec[7] = (weight_gradient) ? 1 : 0; \
        } \
    } while (0)
#else
#define MS_TRACE(i)
#define MS_TRACE_END(height, weight_gradient)
#endif

namespace ms {
namespace {

// What lanes outside the reduction range fetch instead.
__device__ __attribute__((aligned(16))) const char kZeroChunk[16] = {};

// Instruction-class masks of __builtin_amdgcn_sched_group_barrier.
constexpr int SG_MFMA = 0x008, SG_VMEM_RD = 0x020, SG_DS_RD = 0x100, SG_DS_WR = 0x200;

template <int MASK, int N, int ID>
__device__ __forceinline__ void sg() {
    if constexpr (N > 0) __builtin_amdgcn_sched_group_barrier(MASK, N, ID);
}

// Bytes of one register-staged operand tile in LDS: [64 reduction][ROWS outer] x 2 bytes with 64 bytes of padding per row.
template <int ROWS>
constexpr int tile_bytes() { return 64 * (ROWS * 2 + 64); }

constexpr int kStagePitch = 272;                          // epilogue staging: 128 x 2 bytes + 16 bytes pad
constexpr int kStagePerWave = 128 * kStagePitch;          // one 128 x 128 16-bit block per wavefront
constexpr int kStageBytes = 4 * kStagePerWave;

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint2 lds_read_tr(const char *p) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4 *)(p));
    return __builtin_bit_cast(uint2, v);
}

// One operand of a small tile of the weight gradient (ROWS outer indices x 64 reduction indices, contiguous along the
// outer dim): global -> registers -> LDS, and LDS -> MFMA fragments.
template <int ROWS>
struct Operand {
    static constexpr int NL = ROWS / 32;          // 16-byte loads per lane per K step (8, 4 or 2)
    static constexpr int PITCH = ROWS * 2 + 64;   // bytes per reduction row in LDS
    static constexpr int CP = ROWS / 8;           // 16-byte chunks per reduction row
    static constexpr int RP = 256 / CP;           // reduction rows covered by one load of the workgroup
    unsigned off[NL];   // per-lane global byte offsets of the loads, relative to the tile's base pointer
    unsigned off0;      // offset of (reduction index 0, this lane's outer chunk), always valid
    unsigned st_off;    // byte offset of this lane's first LDS store inside the tile
    unsigned frag_off;  // byte offset of this lane's fragment reads inside the tile
    v16 r[NL];

    // outer0: first outer index of the tile; outer_last: last valid start of an 8-wide chunk; wave_outer: this wavefront's
    // first outer index in the tile.
    __device__ __forceinline__ void init(int64_t stride_red, int outer0, int outer_last, int wave_outer) {
        const int tid = threadIdx.x;
        const int lane = tid & 63;
        const int chunk = tid % CP;   // 16-byte chunk along the outer dim
        const int rrow = tid / CP;    // reduction row within one load of the workgroup
        int outer = outer0 + chunk * 8;
        outer = outer > outer_last ? outer_last : outer;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            off[i] = static_cast<unsigned>((static_cast<int64_t>(i * RP + rrow) * stride_red + (outer - outer0)) * 2);
        off0 = static_cast<unsigned>((outer - outer0) * 2);
        st_off = rrow * PITCH + chunk * 16;
        // transposing read: in each group of 16 lanes, lane L supplies the 4-element segment at
        // (reduction L/4, outer 4*(L%4)) and receives reduction 0..3 of outer L.
        const int l16 = lane & 15;
        const int red = 8 * (lane >> 5) + (l16 >> 2);
        const int out = wave_outer + 16 * ((lane >> 4) & 1) + 4 * (l16 & 3);
        frag_off = red * PITCH + out * 2;
    }

    // base: pointer to element (outer0, red0) of the tile.  Loads i = h*NL/2 .. (h+1)*NL/2 - 1 of this lane.
    // TAIL: the tile may cross red_end, reduction indices >= nvalid (relative to red0) read as zero.
    template <bool TAIL>
    __device__ __forceinline__ void load_half(const char *base, int nvalid, int h) {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = h * (NL / 2); i < (h + 1) * (NL / 2); ++i) {
            if constexpr (!TAIL) {
                r[i] = *reinterpret_cast<const v16 *>(base + off[i]);
            } else {
                // one reduction index per load; masked-out lanes read a valid address (reduction index 0) instead
                const bool ok = i * RP + tid / CP < nvalid;
                const unsigned o = ok ? off[i] : off0;
                const v16 v = *reinterpret_cast<const v16 *>(base + o);
                const v16 z = {0u, 0u, 0u, 0u};
                r[i] = ok ? v : z;
            }
        }
    }

    __device__ __forceinline__ void store_half(char *tile, int h) const {
#pragma unroll
        for (int i = h * (NL / 2); i < (h + 1) * (NL / 2); ++i) *reinterpret_cast<v16 *>(tile + st_off + i * RP * PITCH) = r[i];
    }

    // Fragment t (32 outer indices) of K slice kk (16 reduction indices): 8 consecutive reduction values
    // of outer index (lane & 31), reduction half (lane >> 5).
    __device__ __forceinline__ v16 frag(const char *tile, int kk, int t) const {
        const char *p = tile + frag_off + kk * 16 * PITCH + t * 64;
        const uint2 lo = lds_read_tr(p);
        const uint2 hi = lds_read_tr(p + 4 * PITCH);
        return v16{lo.x, lo.y, hi.x, hi.y};
    }
};

// sched_group_barrier sequence for one phase: NM MFMAs with NRD LDS reads, NWR LDS writes and NLD global
// loads spread evenly between them.
constexpr int share(int total, int slots, int g) { return total * (g + 1) / slots - total * g / slots; }

template <int NM, int NRD, int NWR, int NLD, int ID, int... G>
__device__ __forceinline__ void interleave(std::integer_sequence<int, G...>) {
    ((sg<SG_DS_RD, share(NRD, NM, G), ID>(), sg<SG_DS_WR, share(NWR, NM, G), ID>(),
      sg<SG_VMEM_RD, share(NLD, NM, G), ID>(), sg<SG_MFMA, 1, ID>()),
     ...);
}

// ---- the 256-row tile: global -> LDS transfers, 16 x 16 x 32 matrix instructions ----------------------------
//
// global_load_lds_dwordx4 moves 16 bytes per lane from global memory straight into LDS, where one wavefront's 64 lanes
// fill 1 KB of consecutive bytes.  The LDS position of a lane is therefore fixed and the bank-conflict-avoiding swizzle
// is applied on the global side: the lane that owns LDS chunk c of a row fetches the memory chunk that the swizzle maps
// to c.
//   RED operand:  [256 outer][64 reduction], 128-byte rows (whole cache lines), chunk c of row r holds memory chunk
//                 c ^ (r & 7)
//   !RED operand: [64 reduction][256 outer], 512-byte rows; WIDE: as in memory; else chunk c of row r holds memory chunk
//                 c ^ ((r & 3) << 2) ^ (((r >> 3) & 1) << 1)
// (the first keeps 8 consecutive rows of one chunk column on 8 different bank groups for ds_read_b128, the last the
// rows of one ds_read_b64_tr_b16 on different 32-byte bank groups).  Whole kernels, conflict clocks per clock of LDS
// instructions (8 groups, 4096 x 14336): dW, both operands WIDE, none (0.31 with the transposing reads); forward 0.04 (0.09), dX
// 0.03 (K 28672) and 0.16 (K 4096); which of fragment reads, incoming transfers and staged epilogue was not taken apart.
constexpr int kStageTile = 256 * BK * 2;      // bytes of one operand in one stage (32 KB)
constexpr int kAStages = 2, kBStages = 3;     // 5 x 32 KB: the compute unit's whole 160 KB
constexpr int kDmaBytes = (kAStages + kBStages) * kStageTile;
constexpr int kXfers = kStageTile / 4 / 1024; // 1 KB transfers per wavefront, operand and tile (8)

constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }

using lds_ptr = char __attribute__((address_space(3))) *;

template <bool RED, int ROWS = 256, bool WIDE = false, int BLOCK_STEP = 16>
struct DmaOperand {
    static_assert(!WIDE || (!RED && ROWS == 256), "the wide form reads 256-byte pieces of 512-byte rows");
    static_assert(RED || ROWS == 256, "the swizzle of an operand that is contiguous along its outer dim is made for 512-byte rows");
    static constexpr int NX = ROWS * BK * 2 / 4 / 1024;     // 1 KB transfers per wavefront and tile (8, 4 or 2)
    unsigned off[NX];       // per-lane global byte offsets of this wavefront's transfers, relative to the tile base
    int key;                // RED: reduction index of this lane's chunk; !RED: reduction row of transfer 0
    unsigned frag_off;      // byte offset of this lane's fragment reads inside the operand tile
    unsigned tsel[8];       // !RED: swizzled 32-byte column-group offset of fragment t

    // outer0: first outer index of the tile; outer_last: clamp bound (RED: last valid outer index, !RED: last valid
    // start of an 8-wide chunk); wave_outer: this wavefront's first outer index in the tile.  The fused SwiGLU form
    // (!RED only) has gate columns c0 .. c0+127 and up columns ffn+c0 .. ffn+c0+127 in one tile, split_last = ffn.
    // WIDE: every wavefront has 64 gate columns and the up columns of the same numbers behind them, and its reads are
    // dealt so that a lane's accumulators hold both of a pair (swiglu_tile).  Else the second half of the tile's outer indices
    // lies `split` elements further on in memory than the first half's continuation would (split = ffn - 128).
    template <bool GATE_UP = false>
    __device__ __forceinline__ void init(int64_t stride_outer, int64_t stride_red, int outer0, int outer_last,
                                         int wave_outer, int wave, int split = 0, int split_last = 0) {
        const int lane = threadIdx.x & 63;
        if constexpr (RED) {
            const int cg = (lane & 7) ^ (lane >> 3);         // memory chunk of this lane: c ^ (row & 7)
            key = cg * 8;
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                int outer = outer0 + (wave * NX + i) * 8 + (lane >> 3);
                outer = outer > outer_last ? outer_last : outer;
                off[i] = static_cast<unsigned>((static_cast<int64_t>(outer - outer0) * stride_outer + cg * 8) * 2);
            }
            const int frow = lane & 15;
            frag_off = (wave_outer + frow) * 128 + (((lane >> 4) ^ (frow & 7)) << 4);
#pragma unroll
            for (int t = 0; t < 8; ++t) tsel[t] = 0;
        } else {
            key = wave * NX * 2 + (lane >> 5);
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                const int rr = key + 2 * i;
                const int cg = WIDE ? lane & 31 : (lane & 31) ^ ((rr & 3) << 2) ^ (((rr >> 3) & 1) << 1);
                const bool second = WIDE && GATE_UP ? (cg & 8) != 0 : cg >= 16;
                int outer = outer0 + (WIDE && GATE_UP ? (cg >> 4) * 64 + (cg & 7) * 8 + (second ? split_last : 0) : cg * 8 + (second ? split : 0));
                const int last = outer_last + (second ? split_last : 0);
                outer = outer > last ? last : outer;
                off[i] = static_cast<unsigned>((static_cast<int64_t>(rr) * stride_red + (outer - outer0)) * 2);
            }
            if constexpr (WIDE) {
                const int r = lane & 15;
                const int chunk = GATE_UP ? (r >> 2) * 2 + (r & 1) + (r & 2) * 4 : r;
                frag_off = 8 * (lane >> 4) * 512 + wave_outer * 2 + chunk * 16;
                return;
            }
            // transposing read: in each group of 16 lanes, lane L supplies the 4-element segment at
            // (reduction L/4, outer 4*(L%4)) and receives reduction 0..3 of outer L; lane group g covers the reduction
            // indices 8g .. 8g+7 of the 32-wide slice.
            const int l16 = lane & 15;
            const int red = 8 * (lane >> 4) + (l16 >> 2);
            const unsigned sw = ((l16 >> 2) << 6) ^ (((lane >> 4) & 1) << 5);
            frag_off = red * 512 + 8 * (l16 & 3);
#pragma unroll
            for (int t = 0; t < 8; ++t) tsel[t] = (wave_outer * 2 + (t << 5)) ^ sw;
        }
    }

    // Request transfer i of this wavefront's part of one tile.  base: pointer to element (outer0, first reduction index
    // of the tile), uniform; dst: LDS byte address of this wavefront's part of the operand's stage.
    // Written as inline assembly on purpose: the compiler then does not know that LDS is being written behind its back
    // and leaves all waiting on these transfers to the explicit s_waitcnt of the K loop (it would otherwise drain them
    // before every transposing LDS read).  M0 carries the LDS address (declared as clobbered).
    __device__ __forceinline__ void request(int i, const char *base, unsigned dst) const {
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(dst), "v"(off[i]), "s"(base), "i"(i * 1024) : "memory", "m0", "scc");
    }
    // The same for a tile that may cross the end of the group's reduction range (or lie past it altogether): nvalid is
    // the number of its reduction indices inside (<= 0 for a tile past the end), lanes whose data lies outside fetch
    // from a block of zeros, so every tile costs the same number of transfers whatever it holds.
    __device__ __forceinline__ void request_tail(int i, const char *base, unsigned dst, int nvalid, const char *zeros) const {
        const char *src = (RED ? key : key + 2 * i) < nvalid ? base + off[i] : zeros;
        asm volatile("s_add_u32 m0, %0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                     :: "s"(dst), "v"(src), "i"(i * 1024) : "memory", "m0", "scc");
    }

    // Fragment t (16 outer indices) of 32-wide slice kk of the tile at `tile`: lane l holds the reduction indices
    // 8 * (l >> 4) .. + 7 of outer index l & 15.
    __device__ __forceinline__ v16 frag(const char *tile, int kk, int t) const {
        if constexpr (RED) {
            return *reinterpret_cast<const v16 *>(tile + (frag_off ^ (kk << 6)) + t * BLOCK_STEP * 128);
        } else {
            const char *p = tile + frag_off + tsel[t] + kk * 32 * 512;
            const uint2 lo = lds_read_tr(p);
            const uint2 hi = lds_read_tr(p + 4 * 512);
            return v16{lo.x, lo.y, hi.x, hi.y};
        }
    }

    // WIDE: reduction index 8 * (lane >> 4) + s of slice kk, of the eight outer indices 8 * (lane & 15) .. + 7 of this wavefront.
    __device__ __forceinline__ v16 raw(const char *tile, int kk, int s) const {
        static_assert(WIDE, "whole rows are read of the unswizzled layout only");
        return *reinterpret_cast<const v16 *>(tile + frag_off + kk * 32 * 512 + s * 512);
    }
};

// Dword d of the fragments 2q and 2q + 1 from dword q of the raw reads 2d and 2d + 1: the reduction indices 2d and 2d + 1 of one
// outer index side by side.
__device__ __forceinline__ void take_apart(v16 (&frag)[8], int d, int q, const v16 &even, const v16 &odd) {
    frag[2 * q][d] = __builtin_amdgcn_perm(odd[q], even[q], 0x05040100u);
    frag[2 * q + 1][d] = __builtin_amdgcn_perm(odd[q], even[q], 0x07060302u);
}

// The accumulators are in their registers at this point of the program, whatever was or will be done with them.
template <int TM, int TN>
__device__ __forceinline__ void pin(f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+a"(acc[i][j]));
}

// Clears the accumulators, at this point of the program and no earlier: the 256 clearing instructions of a wavefront take
// half a microsecond, which the way of the first tiles hides once these are requested.  (Cleared ahead of the requests:
// training layers of 8 experts x 4096 x 14336 with 64 rows each 2214 us instead of 2187, with 256 rows each and a width of
// 7168 1728 instead of 1707.)
template <int TM, int TN>
__device__ __forceinline__ void clear(f32x4 (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    pin(acc);
}

// Between the clearing of the accumulators and the first mfma16x16 on them: the two instructions that it has to be away
// from an ordinary write of its operands (tests/test_matrix_instruction_hazards.py reads the built code for it).
template <int TM, int TN>
__device__ __forceinline__ void ready(f32x4 (&acc)[TM][TN]) {
    pin(acc);
    asm volatile("s_nop 1" ::: "memory");
}

// The last matrix instructions must have written their results before ordinary instructions read them (16 passes at most).
template <int TM, int TN>
__device__ __forceinline__ void settle(f32x4 (&acc)[TM][TN]) {
    pin(acc);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    pin(acc);
}

// Slots of a slice (64 products) that take raw reads apart, and how many of them lie ahead of slot u: none beside a read, none
// beside a request (slot busy of every eight) or right behind it.  (Two dwords in every slot from the twelfth on, whatever
// else is in it: dW 1150 instead of 1177 TFLOP/s, forward 1349 instead of 1389.)
constexpr bool idle_slot(int u, int busy) { return u >= 11 && u % 8 != busy && u % 8 != busy + 1 && (u >= 32 || u % 2 == 1); }
constexpr int idle_before(int u, int busy) {
    int n = 0;
    for (int w = 0; w < u; ++w) n += idle_slot(w, busy) ? 1 : 0;
    return n;
}
constexpr int kBusyB = 5, kBusyA = 1;       // slots of every eight that request a transfer of B (slice 0) and of A (slice 1)
static_assert(idle_before(64, kBusyB) >= 32 && idle_before(64, kBusyA) >= 32, "both operands' dwords find their slots");

// K loop of a 256 x 256 tile: 2 x 2 wavefronts of 128 x 128 = 8 x 8 blocks of 16 x 16, K steps of 64 = two 32-wide
// slices.  acc[i][j][e] = C[row][wn*128 + col], with r = lane & 15 and c = 4*(lane >> 4) + e: row = (2*i + wm)*16 + r (the two
// wavefronts' blocks alternate, so that both have fewer where the tile has fewer rows: RB of eight), or wm*128 + 8*r + i of
// an A that is not reduction-contiguous (its blocks hold every eighth row); col = j*16 + c, or 8*c + j likewise.
//
// Step kt multiplies slice 0 (its fragments are in registers already) while slice 1's fragments are read, then, after
// the step's only barrier, slice 1 while slice 0 of tile kt+1 is read.  At the barrier every wavefront has all of tile
// kt in registers and all its transfers of tile kt+1 have landed, so behind it tile kt's stages are free (the transfers
// of A's tile kt+2 go there at once; B, with three stages, has its tile kt+2 requested in the first half of the step
// after the one that freed it) and tile kt+1 can be read.
template <int DT, bool A_RED, bool B_RED, bool SWIGLU, int RB>
__device__ __forceinline__ void dma_k_loop(const GmmArgs &p, const TileCoord &tc, char *lds, int row0, int col0,
                                           f32x4 (&acc)[8][8]) {
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave >> 1, wn = wave & 1;
    const int red_begin = tc.e.red_begin;
    const int red_len = tc.e.red_end - red_begin;
    const int nk = (red_len + BK - 1) / BK;
    if (nk <= 0) return clear(acc);

    DmaOperand<A_RED, 256, !A_RED, A_RED ? 32 : 16> la;
    DmaOperand<B_RED, 256, !B_RED> lb;
    la.init(p.a_stride_row, p.a_stride_red, row0, A_RED ? tc.e.row_end - 1 : tc.e.row_end - 8, A_RED ? wm * 16 : wm * 128, wave);
    if constexpr (SWIGLU) {
        static_assert(!SWIGLU || !B_RED, "the fused SwiGLU form reads the weight along its columns");
        lb.template init<true>(p.b_stride_col, p.b_stride_red, col0, p.cols - 8, wn * 128, wave, 0, p.cols);
    } else {
        lb.init(p.b_stride_col, p.b_stride_red, col0, B_RED ? p.cols - 1 : p.cols - 8, wn * 128, wave);
    }
    const char *a_ptr = uniform(static_cast<const char *>(p.a) + (static_cast<int64_t>(row0) * p.a_stride_row +
                                                                  static_cast<int64_t>(red_begin) * p.a_stride_red) * 2);
    const char *b_ptr = uniform(static_cast<const char *>(p.b) + (tc.e.b_off + static_cast<int64_t>(col0) * p.b_stride_col +
                                                                  static_cast<int64_t>(red_begin) * p.b_stride_red) * 2);
    const int64_t a_step = p.a_stride_red * BK * 2;
    const int64_t b_step = p.b_stride_red * BK * 2;
    const char *zeros = kZeroChunk;

    // LDS: A stages 0, 1, then B stages 0, 1, 2.
    const unsigned lds_a = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)lds)) + wave * (kXfers * 1024);
    const unsigned lds_b = lds_a + kAStages * kStageTile;
    int a_left = red_len, b_left = red_len;     // reduction indices from the next requested tile's start to the end
    unsigned a_dst = lds_a, b_dst = lds_b;
    auto request_a = [&](auto tail_c, int i) {
        if constexpr (decltype(tail_c)::value) la.request_tail(i, a_ptr, a_dst, a_left, zeros);
        else la.request(i, a_ptr, a_dst);
    };
    auto request_b = [&](auto tail_c, int i) {
        if constexpr (decltype(tail_c)::value) lb.request_tail(i, b_ptr, b_dst, b_left, zeros);
        else lb.request(i, b_ptr, b_dst);
    };
    auto next_a = [&]() {
        a_ptr += a_step;
        a_left -= BK;
        a_dst = a_dst == lds_a ? lds_a + kStageTile : lds_a;
    };
    auto next_b = [&]() {
        b_ptr += b_step;
        b_left -= BK;
        b_dst = b_dst == lds_b + (kBStages - 1) * kStageTile ? lds_b : b_dst + kStageTile;
    };

    v16 af[2][8], bf[2][8];
    // Slot u = 0..63 of a slice: one MFMA, back and forth over the columns so that each changes one operand only (+0.4 %),
    // and at most one fragment and one request beside it: an MFMA takes 16 clocks, and everything that is issued between
    // two of them in less than that is free.  (Four MFMAs in a row and then the rest: forward 1315 instead of 1368, dX
    // 1405 instead of 1468 TFLOP/s; the requests of a slice in its first half instead of spread over all of it: 1350 and
    // 1428.  8192 x 4096 x 28672 in 8 groups.)
    auto mfma = [&](int set, int u) {
        const int i = u >> 3, j = (i & 1) ? 7 - (u & 7) : (u & 7);
        if (i < RB) mfma16x16<DT>(bf[set][j], af[set][i], acc[i][j]);
    };
    // What slot u does for the fragments of the next slice to be multiplied (slice kk of the stages a, b, into set `set`): one
    // read every other slot, B's eight and then A's; of an operand that lies along its outer dim, the pairs of raw reads are
    // taken apart in idle slots, two dwords in each.
    v16 ra[8], rb[8];
    auto next_slice = [&](int u, int set, int kk, const char *a, const char *b, int busy) {
        if (u % 2 == 0 && u < 32) {
            const int f = u / 2;
            if (f < 8) {
                if constexpr (B_RED) bf[set][f] = lb.frag(b, kk, f);
                else rb[f] = lb.raw(b, kk, f);
            } else {
                if constexpr (A_RED) { if (f - 8 < RB) af[set][f - 8] = la.frag(a, kk, f - 8); }
                else ra[f - 8] = la.raw(a, kk, f - 8);
            }
        }
        if (idle_slot(u, busy)) {
            const int v = idle_before(u, busy), d = (v >> 2) & 3, q = v & 3;
            if (v < 16) {
                if constexpr (!B_RED) take_apart(bf[set], d, q, rb[2 * d], rb[2 * d + 1]);
            } else if (v < 32) {
                if constexpr (!A_RED) take_apart(af[set], d, q, ra[2 * d], ra[2 * d + 1]);
            }
        }
    };

    // tiles 0 and 1 of both operands (the order of the steady state: B before A)
    for (int t = 0; t < nk && t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < kXfers; ++i) request_b(std::true_type{}, i);
        next_b();
#pragma unroll
        for (int i = 0; i < kXfers; ++i) request_a(std::true_type{}, i);
        next_a();
    }
    clear(acc);
    if (nk > 1) __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * kXfers, 0));
    else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    __builtin_amdgcn_s_barrier();
    MS_TRACE(3);
    const char *a_cur = lds;                                   // stages of tile kt
    const char *b_cur = lds + kAStages * kStageTile;
#pragma unroll
    for (int u = 0; u < 64; ++u) next_slice(u, 0, 0, a_cur, b_cur, kBusyA);
    ready(acc);
    __builtin_amdgcn_sched_barrier(0);

    // WHOLE, TAIL: tile kt + 2 is requested, all of it inside the range or not; DRAIN (kt = nk - 2): there is none; LAST: nor
    // a tile to read after this one.  (Two all-zero tiles of each operand requested behind every range, so that one wait
    // count served every step, are as long as a loop of two steps: a training layer of 8 experts x 4096 x 14336 with 64
    // rows each took 2248 us with them, 2214 without; 222 rows each, 4672 x 5160: 1505 and 1487.)
    enum { WHOLE, TAIL, DRAIN, LAST };
    auto k_step = [&](auto kind_c) {
        constexpr int kind = decltype(kind_c)::value;
        constexpr std::bool_constant<kind == TAIL> tail_c{};
        constexpr bool ask = kind == WHOLE || kind == TAIL;
        // slice 0; B's tile kt + 2 is requested
#pragma unroll
        for (int u = 0; u < 64; ++u) {
            mfma(0, u);
            next_slice(u, 1, 1, a_cur, b_cur, kBusyB);
            if constexpr (ask) {
                if (u % 8 == kBusyB) request_b(tail_c, u / 8);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (ask) next_b();
        if constexpr (kind != LAST) {
            a_cur = a_cur == lds ? lds + kStageTile : lds;
            b_cur = b_cur == lds + (kAStages + kBStages - 1) * kStageTile ? lds + kAStages * kStageTile : b_cur + kStageTile;
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(ask ? kXfers : 0, 0));
            __builtin_amdgcn_s_barrier();
        }
        // slice 1; A's tile kt + 2 is requested, slice 0 of tile kt + 1 is read
#pragma unroll
        for (int u = 0; u < 64; ++u) {
            mfma(1, u);
            if constexpr (kind != LAST) next_slice(u, 0, 0, a_cur, b_cur, kBusyA);
            if constexpr (ask) {
                if (u % 8 == kBusyA) request_a(tail_c, u / 8);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (ask) next_a();
    };
    int kt = 0;
    const int nk_full = red_len / BK - 2;       // steps whose requests are whole tiles inside the range
    for (; kt < nk_full; ++kt) k_step(std::integral_constant<int, WHOLE>{});
    if (kt + 2 < nk) {
        k_step(std::integral_constant<int, TAIL>{});
        ++kt;
    }
    if (kt + 1 < nk) k_step(std::integral_constant<int, DRAIN>{});
    k_step(std::integral_constant<int, LAST>{});      // (no transfer is under way any more: the stages can be reused)
    settle(acc);
}

// K loop of a small tile: TBM (128 or 64) x 256, 1 x 4 wavefronts of TBM x 64 = TBM/16 x 4 blocks of 16 x 16.  The order is
// that of the loop above, with a stage (A's and B's tile together) freed and requested again once per step, and as many
// stages as the LDS holds: four of 40 KB or three of 48 KB, so up to three of them are under way at any time.
// What bounds it: a group of few rows reads every weight for one small tile, so the loop is a stream from memory whose
// rate is the bytes in flight over the latency of a loaded memory system.  Against one K step ahead in registers (40 KB
// per compute unit under way): 24 tokens, 64 experts x 2048 x 1408, fc1 132 -> 123 us (5.7 TB/s of weights); 64 tokens,
// 8 experts x 4096 x 14336, fc1 346 -> 336 us (5.6 TB/s), fc2 204 -> 189 us (16 column tiles per expert occupy half of the
// chip).  A large copy reaches 4.9 to 5.5 TB/s on the same card.
constexpr int small_stages(int tbm) { return kDmaBytes / ((tbm + BN) * BK * 2); }

template <int DT, bool B_RED, bool SWIGLU, int TBM>
__device__ __forceinline__ void dma_small_k_loop(const GmmArgs &p, const TileCoord &tc, char *lds, int row0, int col0,
                                                 f32x4 (&acc)[TBM / 16][4]) {
    using OpA = DmaOperand<true, TBM>;
    using OpB = DmaOperand<B_RED, BN>;
    constexpr int NS = small_stages(TBM);
    constexpr int A_TILE = TBM * BK * 2, STAGE = A_TILE + BN * BK * 2;
    constexpr int NXFER = OpA::NX + OpB::NX;    // transfers per wavefront and step
    constexpr int TM = TBM / 16, NF = TM + 4, NM = TM * 4;
    static_assert(NS >= 3 && NS * STAGE <= kDmaBytes && NS * NXFER < 64 && NF <= NM, "stages, wait counts and slots");
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int red_begin = tc.e.red_begin;
    const int red_len = tc.e.red_end - red_begin;
    const int nk = (red_len + BK - 1) / BK;
    if (nk <= 0) return clear(acc);

    OpA la;
    OpB lb;
    la.init(p.a_stride_row, p.a_stride_red, row0, tc.e.row_end - 1, 0, wave);
    if constexpr (SWIGLU) lb.init(p.b_stride_col, p.b_stride_red, col0, p.cols - 8, wave * 64, wave, p.cols - BN / 2, p.cols);
    else lb.init(p.b_stride_col, p.b_stride_red, col0, B_RED ? p.cols - 1 : p.cols - 8, wave * 64, wave);
    const char *a_ptr = uniform(static_cast<const char *>(p.a) + (static_cast<int64_t>(row0) * p.a_stride_row +
                                                                  static_cast<int64_t>(red_begin) * p.a_stride_red) * 2);
    const char *b_ptr = uniform(static_cast<const char *>(p.b) + (tc.e.b_off + static_cast<int64_t>(col0) * p.b_stride_col +
                                                                  static_cast<int64_t>(red_begin) * p.b_stride_red) * 2);
    const int64_t a_step = p.a_stride_red * BK * 2;
    const int64_t b_step = p.b_stride_red * BK * 2;
    const char *zeros = kZeroChunk;

    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)lds));
    int left = red_len;                 // reduction indices from the next requested tile's start to the end
    unsigned dst = lds0;                // its stage
    auto request = [&](auto tail_c, int i) {
        constexpr bool TAIL = decltype(tail_c)::value;
        if (i < OpB::NX) {
            const unsigned at = dst + A_TILE + wave * (OpB::NX * 1024);
            if constexpr (TAIL) lb.request_tail(i, b_ptr, at, left, zeros);
            else lb.request(i, b_ptr, at);
        } else {
            const unsigned at = dst + wave * (OpA::NX * 1024);
            if constexpr (TAIL) la.request_tail(i - OpB::NX, a_ptr, at, left, zeros);
            else la.request(i - OpB::NX, a_ptr, at);
        }
    };
    auto next_tile = [&]() {
        a_ptr += a_step;
        b_ptr += b_step;
        left -= BK;
        dst = dst == lds0 + (NS - 1) * STAGE ? lds0 : dst + STAGE;
    };

    v16 af[2][TM], bf[2][4];
    const char *cur = lds;              // stage of tile kt
    auto read_frag = [&](int set, int kk, int f) {
        if (f < 4) bf[set][f] = lb.frag(cur + A_TILE, kk, f);
        else af[set][f - 4] = la.frag(cur, kk, f - 4);
    };
    auto mfma = [&](int set, int u) {
        const int i = u >> 2, j = (i & 1) ? 3 - (u & 3) : (u & 3);
        mfma16x16<DT>(bf[set][j], af[set][i], acc[i][j]);
    };

    // the first NS tiles
    for (int t = 0; t < NS; ++t) {
#pragma unroll
        for (int i = 0; i < NXFER; ++i) request(std::true_type{}, i);
        next_tile();
    }
    clear(acc);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 1) * NXFER, 0));
    __builtin_amdgcn_s_barrier();
    MS_TRACE(3);
#pragma unroll
    for (int f = 0; f < NF; ++f) read_frag(0, 0, f);
    ready(acc);
    __builtin_amdgcn_sched_barrier(0);

    auto k_step = [&](auto tail_c) {
        // slice 0 is multiplied, slice 1 read
#pragma unroll
        for (int u = 0; u < NM; ++u) {
            mfma(0, u);
            if (u < NF) read_frag(1, 1, u);
            __builtin_amdgcn_sched_barrier(0);
        }
        cur = cur == lds + (NS - 1) * STAGE ? lds : cur + STAGE;
        // all of tile kt is in registers (its stage is free behind the barrier), tile kt + 1 has landed
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * NXFER, 0));
        __builtin_amdgcn_s_barrier();
        // slice 1 is multiplied, tile kt + NS requested, slice 0 of tile kt + 1 read
#pragma unroll
        for (int u = 0; u < NM; ++u) {
            mfma(1, u);
#pragma unroll
            for (int i = u * NXFER / NM; i < (u + 1) * NXFER / NM; ++i) request(tail_c, i);
            if (u < NF) read_frag(0, 0, u);
            __builtin_amdgcn_sched_barrier(0);
        }
        next_tile();
    };
    int kt = 0;
    const int nk_full = red_len / BK - NS;      // steps whose requests are whole tiles inside the range
    for (; kt < nk_full; ++kt) k_step(std::false_type{});
    for (; kt < nk; ++kt) k_step(std::true_type{});
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    settle(acc);
}

// The accumulators of a wavefront's WR x WC block as quads of four consecutive columns of one row, whatever the
// matrix instruction that produced them.
template <int TM, int TN>
struct Acc32 {                                  // 32 x 32 blocks
    f32x16 v[TM][TN];
    static constexpr int MB = 32, ROWS = TM, QUADS = TN * 4, SIDE = 1;
    __device__ __forceinline__ static int col(int q) { return (q >> 2) * 32 + (q & 3) * 8 + 4 * ((threadIdx.x & 63) >> 5); }
    __device__ __forceinline__ f32x4 quad(int i, int q) const {
        const f32x16 &a = v[i][q >> 2];
        const int e = 4 * (q & 3);
        return f32x4{a[e], a[e + 1], a[e + 2], a[e + 3]};
    }
    __device__ __forceinline__ static int real_row(int staged) { return staged; }
    __device__ __forceinline__ static int staged_row(int row) { return row; }
};
// Quad q of block row i; staged row i * 16 + (lane & 15) of the wavefront's block is its row of that number, or, if A's outer
// indices were dealt to the blocks in turn (A_WIDE: block i holds 8 m + i), another one: real_row / staged_row.  B_WIDE the same
// for the columns: the quads 2e and 2e + 1 of a block row are then the eight columns of B's lane group, side by side.
template <int TM, int TN, bool A_WIDE = false, bool B_WIDE = false>
struct Acc16 {                                  // 16 x 16 blocks
    f32x4 v[TM][TN];
    static_assert((!A_WIDE || TM == 8) && (!B_WIDE || TN == 8), "dealing is over eight blocks");
    static constexpr int MB = 16, ROWS = TM, QUADS = TN, SIDE = B_WIDE ? 2 : 1;      // SIDE: quads that lie side by side
    __device__ __forceinline__ static int col(int q) {
        const int g = (threadIdx.x & 63) >> 4;
        return B_WIDE ? 32 * g + 4 * q : q * 16 + 4 * g;
    }
    __device__ __forceinline__ f32x4 quad(int i, int q) const {
        if constexpr (B_WIDE) {
            const int j = 4 * (q & 1), e = q >> 1;
            return f32x4{v[i][j][e], v[i][j + 1][e], v[i][j + 2][e], v[i][j + 3][e]};
        } else {
            return v[i][q];
        }
    }
    __device__ __forceinline__ static int real_row(int staged) { return A_WIDE ? 8 * (staged & 15) + (staged >> 4) : staged; }
    __device__ __forceinline__ static int staged_row(int row) { return A_WIDE ? ((row & 7) << 4) + (row >> 3) : row; }
};

// Epilogue of a 256-row tile of the fused SwiGLU form, for a wavefront's 128 rows from row0 on and its 64 activation columns from
// acol0 on: act = silu(gate) * up * prob of the rounded fc1 values, exactly what the stand-alone SwiGLU kernel computes from the
// stored fc1 output, and that output itself where it is kept (p.c).
// acc[i][j] holds, of row i * 16 + (lane & 15) and with g = lane >> 4, the gate columns 16 g + j and 16 g + 8 + j and the up
// columns of the same numbers: the activation is computed where the sums are, and only what is stored passes through LDS.
// What bounds it: 17 vector instructions per activation on compute units whose matrix cores wait.  Gate and up blocks in different
// wavefronts, both staged, read back by the partners and divided with the division's ten instructions took 8 to 12 us per tile
// beside 2.5 to 3 of the plain epilogue; us per pass with that and with this: inference, 1777 tokens over 32 experts, 2880 x 2880,
// fp16 443.5 / 438.4; 24 tokens over 64, 2048 x 1408 (small tiles, the sigmoid only) 197.5 / 196.6.  In two halves, each staged and
// written by itself, and one block of rows at a time: all of them at once cost 135 spilled registers, 470 us.
template <int DT>
__device__ __forceinline__ void swiglu_tile(const GmmArgs &p, const f32x4 (&acc)[8][8], char *lds, int row0, int row_end, int acol0,
                                            int wave) {
    using T = std::conditional_t<DT == MS_BF16, BF16, FP16>;
    const int lane = threadIdx.x & 63, qrow = lane & 15, g = lane >> 4;
    constexpr int HP = 256 + 16, AP = 128 + 16;         // LDS bytes per row of fc1 values and of activations
    constexpr int ROWS = 64;                            // staged and written at a time
    static_assert(ROWS * (HP + AP) <= kStagePerWave, "staging region too small");
    float prob[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = row0 + i * 32 + qrow;
        prob[i] = p.probs != nullptr && row < row_end ? load_scalar_as_float(p.probs, row, p.probs_dtype) : 1.f;
    }
    const bool keep = p.c != nullptr;
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();          // every wavefront is done reading the operand stages
    char *fc1 = lds + wave * kStagePerWave;             // (private to this wavefront)
    char *act = fc1 + ROWS * HP;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int m = 0; m < ROWS / 16; ++m) {
            const int i = half * (ROWS / 16) + m;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                __attribute__((aligned(16))) uint16_t gate[8], up[8], o[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    gate[j] = T::from_float(acc[i][j][e]);
                    up[j] = T::from_float(acc[i][j][e + 2]);
                    const float x = T::to_float(gate[j]);
                    o[j] = T::from_float(x * sigmoid16(x) * T::to_float(up[j]) * prob[i]);
                }
                *reinterpret_cast<v16 *>(act + (m * 16 + qrow) * AP + g * 32 + e * 16) = *reinterpret_cast<v16 *>(o);
                if (keep) {
                    char *dst = fc1 + (m * 16 + qrow) * HP + g * 32 + e * 16;
                    *reinterpret_cast<v16 *>(dst) = *reinterpret_cast<v16 *>(gate);
                    *reinterpret_cast<v16 *>(dst + 128) = *reinterpret_cast<v16 *>(up);
                }
                __builtin_amdgcn_sched_barrier(0);      // (or the sums of all rows are taken out of their registers first)
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        auto row_at = [&](int r) { return row0 + (half * (ROWS / 16) + (r >> 4)) * 32 + (r & 15); };
        {
            const int acol = acol0 + (lane & 7) * 8;
            uint16_t *dst = static_cast<uint16_t *>(p.act) + acol;
#pragma unroll
            for (int pass = 0; pass < ROWS / 8; ++pass) {
                const int r = pass * 8 + (lane >> 3);
                const v16 v = *reinterpret_cast<const v16 *>(act + r * AP + (lane & 7) * 16);
                if (acol < p.cols && row_at(r) < row_end) *reinterpret_cast<v16 *>(dst + static_cast<int64_t>(row_at(r)) * p.act_stride_row) = v;
            }
        }
        if (keep) {
            const int acol = acol0 + (lane & 7) * 8;
            uint16_t *dst = static_cast<uint16_t *>(p.c) + acol + (qrow >= 8 ? p.cols : 0);
#pragma unroll 4
            for (int pass = 0; pass < ROWS / 4; ++pass) {
                const int r = pass * 4 + g;
                const v16 v = *reinterpret_cast<const v16 *>(fc1 + r * HP + qrow * 16);
                if (acol < p.cols && row_at(r) < row_end) *reinterpret_cast<v16 *>(dst + static_cast<int64_t>(row_at(r)) * p.c_stride_row) = v;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);             // the rows have been read before the next ones overwrite them
    }
}

// One macro tile of TBM x 256 outputs.  TBM = 256: 2x2 wavefronts of 128x128, of which the first RB blocks of 16 rows are
// computed; TBM = 128 / 64: 1x4 wavefronts of 128x64 / 64x64.
template <int DT, bool A_RED, bool B_RED, int OUT, int TBM, int RB = 8>
__device__ __forceinline__ void gmm16_tile_rows(const GmmArgs &p, const TileCoord &tc, char *lds) {
    constexpr int WAVES_M = TBM == 256 ? 2 : 1;
    constexpr int WAVES_N = 4 / WAVES_M;
    constexpr int TM = TBM / WAVES_M / 32;      // 32-row MFMA blocks per wavefront
    constexpr int TN = BN / WAVES_N / 32;       // 32-column MFMA blocks per wavefront
    constexpr int A_BYTES = tile_bytes<TBM>();  // small tiles of the weight gradient only: two register-staged stages
    constexpr int STAGE = A_BYTES + tile_bytes<BN>();
    static_assert(A_RED || !B_RED, "the split on the reduction dim takes both operands along their outer dims");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    const int row0 = tc.e.row_begin + tc.row_tile * BM;   // all but the last row tile of a group are full
    const int row_end = tc.e.row_end;
    constexpr bool SWIGLU = OUT == OUT_SWIGLU;
    static_assert(A_RED || (OUT != OUT_SWIGLU && OUT != OUT_SWIGLU_GRAD), "the fused epilogues read staged rows as they are");
    constexpr int HALF = BN / 2;                          // activation columns per tile in the fused form
    const int col0 = tc.col_tile * (SWIGLU ? HALF : BN);  // fused: first activation (= gate) column
    const int col_end = p.cols;
    const int red_begin = tc.e.red_begin, red_end = tc.e.red_end;

    constexpr bool DMA = TBM == 256 || A_RED;   // operands by transfers straight to LDS
    std::conditional_t<DMA, Acc16<2 * TM, 2 * TN, TBM == 256 && !A_RED, TBM == 256 && !B_RED>, Acc32<TM, TN>> sums;
    auto &acc = sums.v;
    if constexpr (DMA) {
        if constexpr (TBM == 256) dma_k_loop<DT, A_RED, B_RED, SWIGLU, RB>(p, tc, lds, row0, col0, acc);
        else dma_small_k_loop<DT, B_RED, SWIGLU, TBM>(p, tc, lds, row0, col0, acc);
    } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
        Operand<TBM> la;
        Operand<BN> lb;
        la.init(p.a_stride_red, row0, row_end - 8, wm * TM * 32);
        lb.init(p.b_stride_red, col0, col_end - 8, wn * TN * 32);
        // uniform base pointers of element (outer0, red_begin); advanced by one K step per iteration
        const char *a_ptr = static_cast<const char *>(p.a) +
                            (static_cast<int64_t>(row0) * p.a_stride_row + static_cast<int64_t>(red_begin) * p.a_stride_red) * 2;
        const char *b_ptr = static_cast<const char *>(p.b) +
                            (tc.e.b_off + static_cast<int64_t>(col0) * p.b_stride_col +
                             static_cast<int64_t>(red_begin) * p.b_stride_red) * 2;
        const int64_t a_step = p.a_stride_red * BK * 2;
        const int64_t b_step = p.b_stride_red * BK * 2;

        const int red_len = red_end - red_begin;
        const int nk = (red_len + BK - 1) / BK;

        v16 af[2][TM], bf[2][TN];
        auto read_frags = [&](const char *stage, int set, int kk) {
#pragma unroll
            for (int t = 0; t < TM; ++t) af[set][t] = la.frag(stage, kk, t);
#pragma unroll
            for (int t = 0; t < TN; ++t) bf[set][t] = lb.frag(stage + A_BYTES, kk, t);
        };
        auto mfmas = [&](int set, int i0, int i1) {
#pragma unroll
            for (int i = i0; i < i1; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = mfma16<DT>(bf[set][j], af[set][i], acc[i][j]);
        };
        // part p of a tile: p = 0,1 -> A halves, p = 2,3 -> B halves
        auto load_part = [&](auto tail_c, int part, int nvalid) {
            constexpr bool TAIL = decltype(tail_c)::value;
            if (part < 2) la.template load_half<TAIL>(a_ptr, nvalid, part);
            else lb.template load_half<TAIL>(b_ptr, nvalid, part - 2);
        };
        auto store_part = [&](char *stage, int part) {
            if (part < 2) la.store_half(stage, part);
            else lb.store_half(stage + A_BYTES, part - 2);
        };
        auto lds_barrier = [&]() {
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0) only: global loads stay in flight
            __builtin_amdgcn_s_barrier();
        };

        if (nk > 0) {
            // tile 0 -> LDS stage 0; tile 1 -> registers.  Both use the masked loads (whose results are
            // consumed at once), so no load is outstanding when the steady-state loop is entered and the
            // loop's own issue order alone decides how long each of its waits has to be.
#pragma unroll
            for (int part = 0; part < 4; ++part) load_part(std::true_type{}, part, red_len);
#pragma unroll
            for (int part = 0; part < 4; ++part) store_part(lds, part);
            if (nk > 1) {
                a_ptr += a_step;
                b_ptr += b_step;
#pragma unroll
                for (int part = 0; part < 4; ++part) load_part(std::true_type{}, part, red_len - BK);
            }
            lds_barrier();
            MS_TRACE(3);
            read_frags(lds, 0, 0);
        }

        // instruction counts of one phase (one 16-wide K slice)
        constexpr int NM = TM * TN;                                        // MFMAs
        constexpr int NRD = 2 * TM + 2 * TN;                               // LDS fragment reads
        constexpr int NLA = Operand<TBM>::NL / 2;                          // loads / stores of an A part
        constexpr int NLB = Operand<BN>::NL / 2;                           // ... of a B part

        int kt = 0;
        // HAS1: tile kt+1 exists (it is in registers); HAS2: tile kt+2 exists; tail2_c: tile kt+2 is the last one.
        auto k_step = [&](auto has1_c, auto has2_c, auto tail2_c) {
            constexpr bool HAS1 = decltype(has1_c)::value;
            constexpr bool HAS2 = decltype(has2_c)::value;
            const char *cur = lds + (kt & 1) * STAGE;
            char *nxt = lds + ((kt + 1) & 1) * STAGE;
            if constexpr (HAS2) {
                a_ptr += a_step;
                b_ptr += b_step;
            }
            const int left2 = red_len - (kt + 2) * BK;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int set = kk & 1;
                if constexpr (HAS1) store_part(nxt, kk);
                if constexpr (HAS2) load_part(tail2_c, kk, left2);
                if (kk < 2) {
                    read_frags(cur, set ^ 1, kk + 1);
                    mfmas(set, 0, TM);
                    interleave<NM, NRD, HAS1 ? NLA : 0, HAS2 ? NLA : 0, 0>(std::make_integer_sequence<int, NM>{});
                    __builtin_amdgcn_sched_barrier(0);
                } else if (kk == 2) {
                    read_frags(cur, set ^ 1, kk + 1);
                    mfmas(set, 0, TM);
                    interleave<NM, NRD, HAS1 ? NLB : 0, HAS2 ? NLB : 0, 0>(std::make_integer_sequence<int, NM>{});
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    mfmas(set, 0, TM / 2);
                    interleave<NM / 2, 0, HAS1 ? NLB : 0, HAS2 ? NLB : 0, 0>(std::make_integer_sequence<int, NM / 2>{});
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (HAS1) {
                        lds_barrier();
                        read_frags(nxt, 0, 0);
                    }
                    mfmas(set, TM / 2, TM);
                    if constexpr (HAS1) interleave<NM / 2, NRD, 0, 0, 1>(std::make_integer_sequence<int, NM / 2>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        for (; kt + 3 < nk; ++kt) k_step(std::true_type{}, std::true_type{}, std::false_type{});
        if (kt + 3 == nk) { k_step(std::true_type{}, std::true_type{}, std::true_type{}); ++kt; }
        if (kt + 2 == nk) { k_step(std::true_type{}, std::false_type{}, std::false_type{}); ++kt; }
        if (kt + 1 == nk) { k_step(std::false_type{}, std::false_type{}, std::false_type{}); ++kt; }
    }

    // Epilogue.  sums.quad(i, q)[e] = C[row0 + wm*TM*32 + real_row(i*MB + lane % MB)][col0 + wn*TN*32 + col(q) + e]
    MS_TRACE(4);
    using Acc = decltype(sums);
    const int qrow = lane & (Acc::MB - 1);
    const int64_t ldc = p.c_stride_row;
    constexpr int WR = TM * 32, WC = TN * 32;       // this wavefront's block of the tile
    // row of the tile's row r of this wavefront's block
    auto row_at = [&](int r) { return row0 + (A_RED && TBM == 256 ? (r >> 4) * 32 + wm * 16 + (r & 15) : wm * WR + r); };
    if constexpr (SWIGLU && TBM == 256) {
        swiglu_tile<DT>(p, sums.v, lds, row0 + wm * 16, row_end, col0 + wn * (WC / 2), wave);
    } else if constexpr (OUT == OUT_SAME || OUT == OUT_SWIGLU || OUT == OUT_SWIGLU_GRAD) {
        // 16-bit output: each wavefront stages its block in its own LDS region (row pitch WC*2 + 16 bytes, so that the
        // column-slice writes of a 16 x 16 block, 8 bytes or 16 of a WIDE B, start on different banks in all its rows) and writes it out as
        // 16 bytes per lane, WC*2 contiguous bytes per row.
        constexpr int SP = WC * 2 + 16;
        static_assert(WR * SP <= kStagePerWave, "staging region too small");
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_s_barrier();          // every wavefront is done reading the operand stages
        char *stg = lds + wave * kStagePerWave;
#pragma unroll
        for (int i = 0; i < Acc::ROWS; ++i)
#pragma unroll
            for (int q = 0; q < Acc::QUADS; q += Acc::SIDE) {
                __attribute__((aligned(16))) uint16_t h[4 * Acc::SIDE];
#pragma unroll
                for (int s = 0; s < Acc::SIDE; ++s) {
                    const f32x4 v = sums.quad(i, q + s);
#pragma unroll
                    for (int e = 0; e < 4; ++e) h[4 * s + e] = DT == MS_BF16 ? BF16::from_float(v[e]) : FP16::from_float(v[e]);
                }
                using Piece = std::conditional_t<Acc::SIDE == 2, v16, uint2>;
                *reinterpret_cast<Piece *>(stg + (i * Acc::MB + qrow) * SP + Acc::col(q) * 2) = *reinterpret_cast<Piece *>(h);
            }
        __builtin_amdgcn_s_waitcnt(0xC07F);    // own writes only: the region is private to this wavefront
        constexpr int LPR = WC / 8;            // lanes per row (8 columns = 16 bytes each)
        constexpr int RPP = 64 / LPR;          // rows per pass
        const int chunk = lane % LPR;
        // Fused form: the wavefronts of the first half of the tile's columns hold gate columns, their
        // partners (same rows, other half) the matching up columns, ffn further on in the output row.
        constexpr int GATE_WAVES = WAVES_N / 2;
        const bool up_half = SWIGLU && wn >= GATE_WAVES;
        const int acol = col0 + (SWIGLU ? wn % GATE_WAVES : wn) * WC + chunk * 8;   // activation column
        const int col = SWIGLU ? acol + (up_half ? col_end : 0) : acol;
        const bool col_ok = acol < col_end;    // cols is a multiple of 8 on this path
        if constexpr (OUT == OUT_SWIGLU_GRAD) {
            // The staged block is dact = dY @ W2^T (rounded, as the stand-alone matmul would store it); what is
            // written is d_fc1 = SwiGLU backward of it on the saved fc1 output, the same arithmetic as the
            // stand-alone kernel, and per 64 columns the row sums that make up the probabilities' gradient.
            using DTT = std::conditional_t<DT == MS_BF16, BF16, FP16>;
            const uint16_t *fbase = static_cast<const uint16_t *>(p.fc1) + acol;
            uint16_t *dbase = static_cast<uint16_t *>(p.c) + acol;
#pragma unroll 2
            for (int pass = 0; pass < WR / RPP; ++pass) {
                const int r = pass * RPP + lane / LPR;
                const int row = row_at(r);
                const bool ok = col_ok && row < row_end;
                uint16_t d[8], g[8], u[8], og[8], ou[8];
                *reinterpret_cast<v16 *>(d) = *reinterpret_cast<const v16 *>(stg + r * SP + chunk * 16);
                float dot = 0.f;
                if (ok) {
                    const uint16_t *fg = fbase + static_cast<int64_t>(row) * p.fc1_stride_row;
                    *reinterpret_cast<v16 *>(g) = *reinterpret_cast<const v16 *>(fg);
                    *reinterpret_cast<v16 *>(u) = *reinterpret_cast<const v16 *>(fg + col_end);
                    const float pr = p.probs != nullptr ? load_scalar_as_float(p.probs, row, p.probs_dtype) : 1.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float gf = DTT::to_float(g[e]), uf = DTT::to_float(u[e]), df = DTT::to_float(d[e]);
                        const float sig = sigmoid16(gf);
                        const float act = gf * sig;
                        dot = fmaf(df, act * uf, dot);
                        const float dp = df * pr;
                        og[e] = DTT::from_float(dp * uf * (sig * (1.f + gf * (1.f - sig))));
                        ou[e] = DTT::from_float(dp * act);
                    }
                    uint16_t *dg = dbase + static_cast<int64_t>(row) * ldc;
                    *reinterpret_cast<v16 *>(dg) = *reinterpret_cast<v16 *>(og);
                    *reinterpret_cast<v16 *>(dg + col_end) = *reinterpret_cast<v16 *>(ou);
                }
                if (p.partials != nullptr) {
                    // 8 lanes = 64 columns: one partial sum per row and 64-column block
                    dot += __shfl_xor(dot, 1, 64);
                    dot += __shfl_xor(dot, 2, 64);
                    dot += __shfl_xor(dot, 4, 64);
                    if ((chunk & 7) == 0 && ok)
                        p.partials[static_cast<int64_t>(row) * p.partials_per_row + (acol >> 6)] = dot;
                }
            }
        } else if (!SWIGLU || p.c != nullptr) {
            uint16_t *cbase = static_cast<uint16_t *>(p.c) + tc.e.c_off + col;
#pragma unroll 4
            for (int pass = 0; pass < WR / RPP; ++pass) {
                const int r = pass * RPP + lane / LPR;
                const int row = row_at(r);
                const v16 v = *reinterpret_cast<const v16 *>(stg + Acc::staged_row(r) * SP + chunk * 16);
                if (col_ok && row < row_end) {
                    v16 *dst = reinterpret_cast<v16 *>(cbase + static_cast<int64_t>(row) * ldc);
                    // Weight gradients go past the last-level cache: nothing on the way reads them, and as ordinary
                    // stores they put out what the next kernel reads and have it wait for their write-back.  us per
                    // training pass, ordinary / non-temporal: 16 experts x 750 rows x 2048 x 1536 752 / 732, 64 of 0 to
                    // 7700 rows x 2048 x 1408 3506 / 3483, 8 x 2048 rows x 7168 x 2048 3510 / 3497, 8 x 1024 rows x 4096 x
                    // 14336 7117 / 7110.  Of any size, also where the gradient is read right behind (left alone; added to
                    // one; copied): 64 x 256 rows x 1024 x 256 (dW 64 and 32 MB) 237 294 282 / 226 297 277, 16 x 750 x 2048 x
                    // 768 (96 and 48) 467 553 528 / 454 554 519, 8 x 1024 x 4096 x 768 (96 and 48) 595 683 655 / 585 692 652, 16
                    // x 750 x 2048 x 256 (32 and 16) 253 309 290 / 246 308 282, 8 x 512 x 1024 x 1024 (32 and 16) 163 191 179 /
                    // 161 192 182; two products of 8 and 16 MB by themselves 18.3 and 28.0 / 17.2 and 27.1, with the
                    // read 23.1 and 36.2 / 22.5 and 36.3.  No line in the size has one kind on one side.
                    if constexpr (A_RED) *dst = v;
                    else MS_NT_STORE(v, dst);
                }
            }
        }
        if constexpr (SWIGLU) {
            // act = silu(gate) * up * prob from the staged (already rounded) values, exactly what the
            // stand-alone SwiGLU kernel computes from the stored fc1 output.  Each wavefront of a pair
            // takes half of the rows.
            using DTT = std::conditional_t<DT == MS_BF16, BF16, FP16>;
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __builtin_amdgcn_s_barrier();      // the partner's block is staged
            const char *gstg = lds + (wm * WAVES_N + wn % GATE_WAVES) * kStagePerWave;
            const char *ustg = gstg + GATE_WAVES * kStagePerWave;
            const int rbase = up_half ? WR / 2 : 0;
            uint16_t *abase = static_cast<uint16_t *>(p.act) + acol;
#pragma unroll 4
            for (int pass = 0; pass < WR / 2 / RPP; ++pass) {
                const int r = rbase + pass * RPP + lane / LPR;
                const int row = row_at(r);
                uint16_t g[8], u[8], o[8];
                *reinterpret_cast<v16 *>(g) = *reinterpret_cast<const v16 *>(gstg + r * SP + chunk * 16);
                *reinterpret_cast<v16 *>(u) = *reinterpret_cast<const v16 *>(ustg + r * SP + chunk * 16);
                if (col_ok && row < row_end) {
                    const float pr = p.probs != nullptr ? load_scalar_as_float(p.probs, row, p.probs_dtype) : 1.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float gf = DTT::to_float(g[e]);
                        o[e] = DTT::from_float(gf * sigmoid16(gf) * DTT::to_float(u[e]) * pr);
                    }
                    *reinterpret_cast<v16 *>(abase + static_cast<int64_t>(row) * p.act_stride_row) = *reinterpret_cast<v16 *>(o);
                }
            }
        }
    } else {
        // fp32 output or fp32 `+=`: an accumulator register holds four consecutive columns of one row, so written
        // straight from the registers one instruction would touch 32 rows with 32 bytes each.  Instead each
        // wavefront stages one 32-row strip of its block at a time in its own LDS region (row pitch WC + 4
        // floats) and moves it as whole row segments: WC * 4 contiguous bytes per row, 16 bytes per lane.
        constexpr int SPF = WC + 4;              // floats per staged row
        static_assert(32 * SPF * 4 <= kStagePerWave, "staging region too small");
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_s_barrier();          // every wavefront is done reading the operand stages
        float *stg = reinterpret_cast<float *>(lds + wave * kStagePerWave);
        constexpr int LPR = WC / 4;            // lanes per row (4 columns = 16 bytes each)
        constexpr int RPP = 64 / LPR;          // rows per pass
        const int c4 = (lane % LPR) * 4;
        const int col = col0 + wn * WC + c4;
        const bool col_ok = col < col_end;     // cols is a multiple of 4 on this path
        float *cbase = static_cast<float *>(p.c) + tc.e.c_off + col;
        const float *lbase = static_cast<const float *>(p.c) + tc.e.c_off + (col_ok ? col : col_end - 4);   // always inside the row
        constexpr int NP = 32 / RPP;           // passes per strip
        // `+=`: the old values of strip i + 1 are requested while strip i is staged and written, from clamped
        // (always valid) addresses, so that a whole strip's loads are in flight at a time
        f32x4 old[2][NP];
        auto load_old = [&](f32x4 (&dst)[NP], int i) {
#pragma unroll
            for (int pass = 0; pass < NP; ++pass) {
                int row = row_at(Acc::real_row(i * 32 + pass * RPP + lane / LPR));
                row = row < row_end ? row : row_end - 1;
                dst[pass] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(lbase + static_cast<int64_t>(row) * ldc));
            }
        };
        if constexpr (OUT == ACC_F32) load_old(old[0], 0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int b = 0; b < 32 / Acc::MB; ++b)
#pragma unroll
                for (int q = 0; q < Acc::QUADS; ++q)
                    *reinterpret_cast<f32x4 *>(stg + (b * Acc::MB + qrow) * SPF + Acc::col(q)) = sums.quad(i * (32 / Acc::MB) + b, q);
            if constexpr (OUT == ACC_F32) {
                if (i + 1 < TM) load_old(old[(i + 1) & 1], i + 1);
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);    // own writes only: the region is private to this wavefront
#pragma unroll
            for (int pass = 0; pass < NP; ++pass) {
                const int r = pass * RPP + lane / LPR;
                const int row = row_at(Acc::real_row(i * 32 + r));
                f32x4 o = *reinterpret_cast<const f32x4 *>(stg + r * SPF + c4);
                if constexpr (OUT == ACC_F32) o += old[i & 1][pass];
                if (col_ok && row < row_end) __builtin_nontemporal_store(o, reinterpret_cast<f32x4 *>(cbase + static_cast<int64_t>(row) * ldc));
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);    // the strip has been read before the next one overwrites it
        }
    }
}

// A 256-row tile of fewer rows computes them in as many blocks of 32 (16 of each of the two wavefronts of a column half) as they
// take: a group's last tile holds 129 to 256, two that share their rows (shares_last_two) 97 to 192 each.  What the rest would cost
// is energy, which bounds the long launches, and matrix
// time in the others.  All groups of so many rows, bf16, with eight blocks always and with as many as needed, us: 32 groups, 2880 x
// 5760, forward / dX 140 rows 253 / 258 -> 224 / 241, 170 rows 251 / 261 -> 232 / 248, 200 rows 256 / 260 -> 242 / 256, 250 rows 266 /
// 271 -> 265 / 271; five blocks beside six 230 -> 224 and 243 -> 241 (140 rows).  fp32 output / `+=` / SwiGLU backward in the
// epilogue, 2880 x 2880 32 of 170 rows 156 / 152 / 176 -> 144 / 146 / 172; sharing rows pays by them alone (small tiles; shared,
// eight blocks; shared): 32 of 290 rows, 2880 x 2880 217 / 234 / 286; 231 / 246 / 270; 188 / 203 / 242, 8 of 300, 4096 x 28672
// 670 / 700 / 838; 747 / 771 / 828; 599 / 628 / 713, 128 of 300, 2048 x 3072 638 / 691 / 929; 700 / 749 / 867; 587 / 644 / 802, 16 of
// 1100, 2048 x 6144 422 / 464 / 576; 441 / 489 / 618; 417 / 458 / 590 (the one of 15 sizes where a mode has small tiles 2 % faster).
// The A rows past the end are still requested (one wait count for all wavefronts).  Not for the weight gradient (its tiles' rows
// are the weight's, whole but for the last).
template <int DT, bool A_RED, bool B_RED, int OUT, int TBM>
__device__ __forceinline__ void gmm16_tile(const GmmArgs &p, const TileCoord &tc, char *lds) {
    if constexpr (A_RED && TBM == 256) {
        const int rows = tc.e.row_end - tc.e.row_begin - tc.row_tile * BM;
        if (rows > 224) gmm16_tile_rows<DT, A_RED, B_RED, OUT, TBM>(p, tc, lds);
        else if (rows > 192) gmm16_tile_rows<DT, A_RED, B_RED, OUT, TBM, 7>(p, tc, lds);
        else if (rows > 160) gmm16_tile_rows<DT, A_RED, B_RED, OUT, TBM, 6>(p, tc, lds);
        else gmm16_tile_rows<DT, A_RED, B_RED, OUT, TBM, 5>(p, tc, lds);
    } else {
        gmm16_tile_rows<DT, A_RED, B_RED, OUT, TBM>(p, tc, lds);
    }
}

// The dynamic LDS of every kernel that runs these tiles.
static_assert(kDmaBytes >= 2 * (tile_bytes<128>() + tile_bytes<BN>()) && kDmaBytes >= kStageBytes,
              "the K loop's LDS must hold the small tiles' two stages and the epilogue's staging as well");

}  // namespace
}  // namespace ms
