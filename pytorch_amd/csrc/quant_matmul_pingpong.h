// K loop of npu_quant_matmul in which the two wavefronts of a SIMD take turns: while one multiplies, the other reads its next
// fragments from LDS and requests refills.  Tiles 256x256 (2 x 4 wavefronts of 128 x 64), 128x256 and 128x320 (2 x 4 of 64 x 64 / 80).
//
// A K step of 128 bytes is two parts.  The operand of which a wavefront needs fewer rows is read whole in the first part, the other one
// half per part, so that a part is 16 to 32 MFMAs on one set of fragments beside the accumulators (64 registers; the loop has no scratch
// access.  The kernels of the 256x256 tile spill 35 to 42 registers, one store in front of the loop and the rest in the general epilogue, which
// takes what the epilogues with their parameters in LDS do not).  A part is two intervals between barriers: fragments and refills, then MFMAs.  Wavefronts w and w + 4 share a SIMD; 4 .. 7 run one interval behind 0 .. 3, so one of the two is always in its MFMAs.
//
// Slots.  Whoever reads a slot is done (lgkmcnt 0) before the barrier that ends the interval, and the wavefronts one interval behind
// before the next one; a slot is refilled two intervals after the leading wavefronts read it, i.e. never before the others are done.
// A stage is there for everybody when both groups have waited for their own loads and passed the barrier behind that wait, again one
// interval before the leading group reads it.  Every load is issued every step (past the end with an out-of-range offset), so the
// number of loads that may be outstanding at a wait is a constant.
//
// What bounds it: power.  At 4096x4096x4096 the loop runs at 2191 clocks a step where the MFMAs alone are 2048, but with operands as
// quantisation leaves them the card holds 1.65 GHz there and 2.2 with zeros, for the same cycles (55.6 and 42.4 us back to back);
// v_mfma_i32_32x32x32_i8 in the same loop needs fewer clocks (2134) and is 10 % slower (1.43 GHz).  Microseconds before (refills and
// fragment reads interleaved with the MFMAs by scheduling groups, general epilogue), with this loop and that epilogue, and with the one that has its
// parameters in LDS, on one box: 4096x4096x4096 57.3, 55.5, 52.9; 2048x14336x4096 split two ways 110.9, 105.6, 102.7 (256x256).
// 777x11008x4096 split two ways 54.8 -> 45.3 (128x256, with that epilogue).  On 256x192 and 256x224 it is level with quant_matmul_wide.h.
#pragma once
#include "common.h"
#include <type_traits>

namespace mi355 {
namespace pingpong {

typedef int32_t i32x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int BK = 128;
constexpr uint32_t kPastEnd = 0x80000000u;     // lane offset beyond every buffer: the load writes zeros

template <int WGM, int WGN, int WTM, int WTN>
struct Geometry {
    static constexpr bool SPLIT_A = WTM > WTN;               // the operand whose fragments are read in two parts
    static constexpr int UNITS_A = 2 * WGM * WTM, UNITS_B = 2 * WGN * WTN;
    static constexpr int NSA = 2, NSB = SPLIT_A ? 2 : 3;     // slots
    static constexpr int A_BYTES = UNITS_A * 1024, B_BYTES = UNITS_B * 1024;
    static constexpr int B_BASE = NSA * A_BYTES;
    static constexpr int PARAM_BASE = B_BASE + NSB * B_BYTES;
    static constexpr int LDS_BYTES = PARAM_BASE + 3072;
};

// at most VM loads outstanding and every LDS read done, as the builtin, which the compiler's own bookkeeping sees
// (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4 left at "no wait", lgkmcnt 11:8)
template <int VM>
__device__ __forceinline__ void wait_landed()
{
    static_assert(VM >= 0 && VM < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (0 << 8) | ((VM >> 4) << 14));
}
__device__ __forceinline__ void wait_reads()
{
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
}

struct LoopState {
    __amdgpu_buffer_rsrc_t rsrc_a, rsrc_b;
    uint32_t voff_a, voff_b;           // lane offsets within a unit
    int gchunk;                        // byte of the K step that the lane's 16 bytes start at
    uint32_t stride_a, stride_b;       // bytes between units (8 rows)
    uint32_t k0;                       // byte offset of the workgroup's first K step
    int KT, kbytes;                    // K steps of the workgroup; bytes of K in them
    uint32_t va, vb;                   // LDS byte offsets of the lane's first fragment rows (first 64 bytes of a K step)
    uint32_t vax, vbx;                 // ... (second 64 bytes)
};

template <int WGM, int WGN, int WTM, int WTN>
__device__ __forceinline__ void k_loop(i32x4v (&acc)[WTM][WTN], char *lds, const LoopState &st, int wave)
{
    using G = Geometry<WGM, WGN, WTM, WTN>;
    constexpr bool SA = G::SPLIT_A;
    constexpr int A_BYTES = G::A_BYTES, B_BYTES = G::B_BYTES, B_BASE = G::B_BASE, NSA = G::NSA, NSB = G::NSB;
    constexpr int W0 = SA ? WTM / 2 : (WTN + 1) / 2;          // fragments of the split operand in the first part
    constexpr int W1 = (SA ? WTM : WTN) - W0;
    constexpr int NWF = SA ? WTN : WTM;                       // fragments of the other operand
    constexpr int UA8 = G::UNITS_A / 8, UB8 = G::UNITS_B / 8; // refills of a wavefront per stage
    constexpr int YOUNG = UA8 + UB8;                          // ... and those that may be in flight when a stage has to be there
    const int KT = st.KT;

    auto load_a = [&](int kt, uint32_t slot, int u) {
        const uint32_t vo = kt * BK + st.gchunk < st.kbytes ? st.voff_a : kPastEnd;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(st.rsrc_a, (lds_void *)(lds + slot + u * 1024), 16, vo,
                                                 (uint32_t)u * st.stride_a + st.k0 + (uint32_t)kt * BK, 0, 0);
    };
    auto load_b = [&](int kt, uint32_t slot, int u) {
        const uint32_t vo = kt < KT ? st.voff_b : kPastEnd;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(st.rsrc_b, (lds_void *)(lds + B_BASE + slot + u * 1024), 16, vo,
                                                 (uint32_t)u * st.stride_b + st.k0 + (uint32_t)kt * BK, 0, 0);
    };
    // Refills.  Activations split: the first half of every wavefront's rows and all weights are free after part 0, the other half
    // after part 1.  Weights split: the activations are free after part 0, the weights after part 1.
    auto refill_b = [&](int kt, uint32_t slot) {
#pragma unroll
        for (int i = 0; i < UB8; i++) load_b(kt, slot, i * 8 + wave);
    };
    auto refill_a_part = [&](int kt, uint32_t slot, int part) {
#pragma unroll
        for (int i = 0; i < UA8 / 2; i++) load_a(kt, slot, i * 16 + part * 8 + wave);
    };
    auto refill_a = [&](int kt, uint32_t slot) {
#pragma unroll
        for (int i = 0; i < UA8; i++) load_a(kt, slot, i * 8 + wave);
    };

    i32x4v whole[2][NWF], part[2][W0];
    auto read_whole = [&](uint32_t slot) {
#pragma unroll
        for (int i = 0; i < NWF; i++) whole[0][i] = *reinterpret_cast<const i32x4v *>(lds + (SA ? st.vb : st.va) + slot + i * 2048);
#pragma unroll
        for (int i = 0; i < NWF; i++) whole[1][i] = *reinterpret_cast<const i32x4v *>(lds + (SA ? st.vbx : st.vax) + slot + i * 2048);
    };
    auto read_part = [&](uint32_t slot, auto first_c, auto n_c) {
        constexpr int F = decltype(first_c)::value, NN = decltype(n_c)::value;
#pragma unroll
        for (int i = 0; i < NN; i++) part[0][i] = *reinterpret_cast<const i32x4v *>(lds + (SA ? st.va : st.vb) + slot + (F + i) * 2048);
#pragma unroll
        for (int i = 0; i < NN; i++) part[1][i] = *reinterpret_cast<const i32x4v *>(lds + (SA ? st.vax : st.vbx) + slot + (F + i) * 2048);
    };
    auto multiply = [&](auto first_c, auto n_c) {
        constexpr int F = decltype(first_c)::value, NN = decltype(n_c)::value;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int t = 0; t < NN * NWF; t++) {
                const int i = t / NWF, j = t % NWF;
                if constexpr (SA)
                    acc[F + i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(whole[h][j], part[h][i], acc[F + i][j], 0, 0, 0);
                else
                    acc[j][F + i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(part[h][i], whole[h][j], acc[j][F + i], 0, 0, 0);
            }
        __builtin_amdgcn_s_setprio(0);
    };
    using I0 = std::integral_constant<int, 0>;
    using IW0 = std::integral_constant<int, W0>;
    using IW1 = std::integral_constant<int, W1>;
#define MI355_PP_BARRIER                 \
    __builtin_amdgcn_sched_barrier(0);   \
    __builtin_amdgcn_s_barrier();        \
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (SA) {
        refill_b(0, 0);
        refill_a_part(0, 0, 0);
        refill_a_part(0, 0, 1);
        refill_b(1, B_BYTES);
        refill_a_part(1, A_BYTES, 0);
        wait_landed<YOUNG>();
    } else {
        refill_b(0, 0);
        refill_a(0, 0);
        refill_b(1, B_BYTES);
        refill_a(1, A_BYTES);
        wait_landed<YOUNG>();
    }
    MI355_PP_BARRIER
    if (wave >= 4) { MI355_PP_BARRIER }        // wavefronts 4 .. 7 run one interval behind

    uint32_t sb = 0, sbw = (NSB - 1) * B_BYTES, sa = 0;        // slots that are read; weight slot that is refilled
    for (int kt = 0; kt < KT; kt++) {
        // ---- part 0: fragments
        read_whole(SA ? sb : sa);
        read_part(SA ? sa : sb, I0{}, IW0{});
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SA) {
            refill_a_part(kt + 1, sa ^ A_BYTES, 1);
            wait_landed<YOUNG>();    // the second activation part of this step has landed
        } else {
            refill_b(kt + NSB - 1, sbw);
            wait_reads();
        }
        MI355_PP_BARRIER
        multiply(I0{}, IW0{});
        MI355_PP_BARRIER
        // ---- part 1
        read_part(SA ? sa : sb, IW0{}, IW1{});
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SA) {
            refill_b(kt + 2, sb);
            refill_a_part(kt + 2, sa, 0);
            wait_landed<YOUNG>();    // the next step's weights and first activation part have landed
            sb ^= B_BYTES;
            sa ^= A_BYTES;
        } else {
            refill_a(kt + NSA, sa);
            wait_landed<YOUNG>();    // the next step has landed
            sa = sa == (NSA - 1) * A_BYTES ? 0u : sa + A_BYTES;
            sb = sb == (NSB - 1) * B_BYTES ? 0u : sb + B_BYTES;
            sbw = sbw == (NSB - 1) * B_BYTES ? 0u : sbw + B_BYTES;
        }
        MI355_PP_BARRIER
        multiply(IW0{}, IW1{});
        MI355_PP_BARRIER
    }
    if (wave < 4) { MI355_PP_BARRIER }         // the last interval of wavefronts 4 .. 7
#undef MI355_PP_BARRIER
    wait_landed<0>();                          // the refills past the end must not land in the epilogue's LDS
}

} // namespace pingpong
} // namespace mi355
