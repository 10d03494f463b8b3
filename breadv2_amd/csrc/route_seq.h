// route_seq.h — router logits in the reference's exact order, for the
// multi-token paths (see route.hip).  route_seq_block is the body of
// k_route_seq.
//
// The reference sums each logit sequentially (one_layer.cu:969-971):
//   logits[e] = ((0 + W[e][0] x[0]) + W[e][1] x[1]) + ... + W[e][H-1] x[H-1],
// every product rounded to fp32 and then added, never fused.  A workgroup
// of 4 waves takes 4 * NE router rows (NE a wave) and 64 tokens (one a lane);
// each lane runs its token's NE sums in that order.  A sum is one dependent
// chain, so the kernel's time is a lane's H columns of (product, add) at the
// issue rate of one wave; everything else is kept off that path.
//   - Activations travel HBM/L2 -> LDS by gfx950 direct-to-LDS loads in
//     chunks of 64 columns through a ring of four buffers, up to four chunks
//     ahead.  A buffer is a variable of its own and the loop is unrolled over
//     the ring: a read of a variable that a direct-to-LDS load may still
//     write waits for that load, and with one variable for all buffers every
//     read waited for the loads that had just gone out.  A token's chunk row
//     is 16 16-byte units stored XOR-swizzled (unit u at u ^ (token % 16)),
//     so a wave's loads write contiguous LDS and the 16-byte reads of 16
//     consecutive lanes fall in distinct banks.  Rows past the last token
//     repeat earlier ones in turn (no lane's result is stored).
//   - Router rows are the same for every lane: a row's chunk sits in one
//     register quad in each 16-lane row of the wave (lane j: columns 4j ..
//     4j+3) and each product takes its weight by DPP row_newbcast inside the
//     v_mul, with no LDS traffic and no extra instruction.
//   - The chain never drains: LDS reads run two blocks of 16 columns ahead
//     and products one, across chunk borders too; a chunk's barrier stands
//     two blocks before its end, where its last reads have returned (so its
//     buffer is free) and the next chunk's first ones go out.
// Loads past the last chunk repeat it into buffers that nothing reads, so
// the counts that the waits rely on hold to the end.
//
// Bound: one wave a SIMD issues an instruction every 2.4 ns, so 2048 columns
// of a product and an add take 10 us; where waves share a SIMD the DPP product
// takes 2.2 ns and the add 1.1.  Measured on MI355X at 256 experts, hidden
// 2048, against two 128-column buffers in one variable, a barrier and a drained
// pipeline at each chunk: 64 tokens 19.6 -> 16.3 us, 512 tokens 31.5 -> 26.7
// us, 2048 tokens 95 us both.  Weights by scalar loads two blocks ahead (a
// plain product takes half a DPP one's issue): 57 / 59 / 115 us, the loads'
// latency.
#pragma once

#include "bread_device.h"

namespace route_seq {

constexpr int RS_WAVES = 4;              // waves per workgroup
constexpr int RS_TT = WAVE;              // tokens per tile, one a lane
constexpr int RS_CJ = 64;                // columns per staged chunk
constexpr int RS_NB = 4;                 // chunk buffers, and the chunks a loop pass covers
constexpr int RS_BLK = 16;               // columns per block of the pipelined inner loop
constexpr int RS_XI = RS_TT / 4 / RS_WAVES;  // activation loads a wave issues per chunk

static_assert(RS_CJ == 64 && RS_XI == 4, "a wave instruction stages four 256-byte rows");

typedef float RsBuf[RS_TT][RS_CJ];  // a chunk of the tile's activations, units swizzled

// Native 4-float vectors (HIP's float4 struct is copied through memory).
typedef float rs_f4 __attribute__((ext_vector_type(4)));

// s_waitcnt on the vector memory counter only (gfx9 encoding: vmcnt in
// bits 3:0 and 15:14, expcnt and lgkmcnt left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Keeps the vector memory operations issued before it ahead of those issued
// after it.  The partial vmcnt waits of rs_run count on that order (gfx9
// completes a wave's vector memory operations in issue order), and nothing
// else pins it: were a chunk's weights issued ahead of its activations, a
// wait meant for those would leave part of them in flight across the barrier.
// The empty asm with a memory clobber stops the optimiser, the scheduling
// barrier the machine scheduler.
__device__ __forceinline__ void issue_order()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// A workgroup barrier without a memory fence: the direct-to-LDS data a
// barrier publishes is waited for explicitly by its issuing wave, so the
// loads running further ahead stay in flight.  The signal fences keep the
// compiler from moving LDS accesses across it.
__device__ __forceinline__ void bar()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Lane n of each 16-lane row of v, to the whole row (DPP row_newbcast; the
// compiler folds it into the consuming v_mul).
template <int N>
__device__ __forceinline__ float row_bcast(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + N, 0xF,
                                                                 0xF, false));
}

__device__ __forceinline__ float row_bcast(float v, int n)
{
    switch (n) {
    case 0: return row_bcast<0>(v);
    case 1: return row_bcast<1>(v);
    case 2: return row_bcast<2>(v);
    case 3: return row_bcast<3>(v);
    case 4: return row_bcast<4>(v);
    case 5: return row_bcast<5>(v);
    case 6: return row_bcast<6>(v);
    case 7: return row_bcast<7>(v);
    case 8: return row_bcast<8>(v);
    case 9: return row_bcast<9>(v);
    case 10: return row_bcast<10>(v);
    case 11: return row_bcast<11>(v);
    case 12: return row_bcast<12>(v);
    case 13: return row_bcast<13>(v);
    case 14: return row_bcast<14>(v);
    default: return row_bcast<15>(v);
    }
}

// Four halves widened.
__device__ __forceinline__ rs_f4 widen(uint2 g)
{
    return rs_f4{h2f(g.x), h2f(g.x >> 16), h2f(g.y), h2f(g.y >> 16)};
}

// Column col (0..63) of a row's chunk.
__device__ __forceinline__ float rs_weight(const rs_f4 &w, int col)
{
    return row_bcast(w[col & 3], col >> 2);
}

// The lane's activations of one 16-column block of a chunk.
__device__ __forceinline__ void rs_load_x(const RsBuf &buf, int lane, int blk, float (&xv)[RS_BLK])
{
#pragma unroll
    for (int q = 0; q < RS_BLK / 4; q++) {
        const rs_f4 x4 = *reinterpret_cast<const rs_f4 *>(&buf[lane][4 * ((blk * (RS_BLK / 4) + q) ^ (lane & 15))]);
        xv[4 * q] = x4[0];
        xv[4 * q + 1] = x4[1];
        xv[4 * q + 2] = x4[2];
        xv[4 * q + 3] = x4[3];
    }
}

// The sums of one wave: acc[n] += w_n[j] x[j] for j = 0 .. H - 1 in order,
// each product rounded before its add, w_n the rows from w0, or (GATE, NE 1)
// the fp16 row g.  x: the tile's first row, nt its tokens.  Every wave of the
// workgroup runs it (all of them stage), every lane too (the weights come
// from other lanes by DPP).  H % 256 == 0.
template <int NE, bool GATE>
__device__ __forceinline__ void rs_run(RsBuf &b0, RsBuf &b1, RsBuf &b2, RsBuf &b3, const float *__restrict__ x, int nt,
                                       const float *__restrict__ w0, const uint16_t *__restrict__ g, int H,
                                       float (&acc)[NE])
{
#pragma clang fp contract(off)
    static_assert(!GATE || NE == 1, "one gate row");
    constexpr int BPC = RS_CJ / RS_BLK;       // blocks a chunk
    constexpr int PER = RS_XI + NE;           // loads of a chunk: activations, then weights
    const int lane = lane_id(), wv = wave_id();
    const int nc = H / RS_CJ;
    // lane l of a load writes unit l % 16 of row l / 16 from unit (l % 16) ^
    // (row % 16) of the token's chunk
    const __amdgpu_buffer_rsrc_t xb = rsrc(x, 4u * (uint32_t)(nt * H));
    uint32_t xo[RS_XI];
#pragma unroll
    for (int i = 0; i < RS_XI; i++) {
        const int row = 4 * (wv + RS_WAVES * i) + (lane >> 4);
        xo[i] = 4u * (uint32_t)((row % nt) * H + 4 * ((lane & 15) ^ (row & 15)));
    }
    auto stage = [&](RsBuf &b, int c, int i) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, &b[4 * (wv + RS_WAVES * i)][0], 16, xo[i],
                                                 4 * RS_CJ * min(c, nc - 1), 0, 0);
    };
    // (buffer loads: plain ones from read-only arguments would not stay where
    // they are issued)
    const __amdgpu_buffer_rsrc_t wb = GATE ? rsrc(g, 2u * (uint32_t)H) : rsrc(w0, 4u * (uint32_t)(NE * H));
    rs_f4 wr[RS_NB][NE];
    uint2 gr[RS_NB];
    const uint32_t wo = (GATE ? 8 : 16) * (lane & 15);
    auto load_w = [&](int k, int c) __attribute__((always_inline)) {
        const int col = min(c, nc - 1) * RS_CJ;
        if constexpr (GATE) {
            gr[k] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(wb, wo, 2 * col, 0));
        } else {
#pragma unroll
            for (int n = 0; n < NE; n++)
                wr[k][n] = __builtin_bit_cast(rs_f4, __builtin_amdgcn_raw_buffer_load_b128(wb, wo, 4 * (n * H + col), 0));
        }
    };
    auto weight = [&](int k, int n, int col) __attribute__((always_inline)) {
        if constexpr (GATE) return rs_weight(widen(gr[k]), col);
        else return rs_weight(wr[k][n], col);
    };
    auto read = [&](int k, int blk, float (&xv)[RS_BLK]) __attribute__((always_inline)) {
        if (k == 0) rs_load_x(b0, lane, blk, xv);
        else if (k == 1) rs_load_x(b1, lane, blk, xv);
        else if (k == 2) rs_load_x(b2, lane, blk, xv);
        else rs_load_x(b3, lane, blk, xv);
    };
    auto stage_k = [&](int k, int c, int i) __attribute__((always_inline)) {
        if (k == 0) stage(b0, c, i);
        else if (k == 1) stage(b1, c, i);
        else if (k == 2) stage(b2, c, i);
        else stage(b3, c, i);
    };
    float x1[RS_BLK], x2[RS_BLK], p[NE][RS_BLK], pn[NE][RS_BLK];
#pragma unroll
    for (int k = 0; k < RS_NB; k++) {
#pragma unroll
        for (int i = 0; i < RS_XI; i++) stage_k(k, k, i);
        issue_order();
        load_w(k, k);
        issue_order();
    }
    wait_vm<NE + (RS_NB - 1) * PER>();
    bar();
    read(0, 0, x1);
#pragma unroll
    for (int j = 0; j < RS_BLK; j++)
#pragma unroll
        for (int n = 0; n < NE; n++) p[n][j] = weight(0, n, j) * x1[j];
    read(0, 1, x1);
    for (int c = 0; c < nc; c += RS_NB) {
#pragma unroll
        for (int k = 0; k < RS_NB; k++) {
#pragma unroll
            for (int bl = 0; bl < BPC; bl++) {
                const int kn = (bl + 1) / BPC ? (k + 1) % RS_NB : k, bn = (bl + 1) % BPC;  // the next block
                const int kr = (bl + 2) / BPC ? (k + 1) % RS_NB : k, br = (bl + 2) % BPC;  // the one after it
#pragma unroll
                for (int j = 0; j < RS_BLK; j++) {
#pragma unroll
                    for (int n = 0; n < NE; n++) {
                        acc[n] = acc[n] + p[n][j];
                        pn[n][j] = weight(kn, n, bn * RS_BLK + j) * x1[j];
                    }
                    if (j == 0) {
                        issue_order();
                        if (bl + 2 == BPC) {
                            // this chunk's reads have returned, and the next
                            // chunk has landed: loads issued after it stay
                            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
                            wait_vm<NE + (RS_NB - 2) * PER>();
                            bar();
                            issue_order();
                        }
                        read(kr, br, x2);
                    }
                    // the chunk four ahead into this one's buffer, its
                    // weights behind it into this one's registers
                    if (bl >= BPC - 2 && (j == 4 || j == 10)) {
                        issue_order();
                        stage_k(k, c + k + RS_NB, 2 * (bl - (BPC - 2)) + (j == 10));
                    }
                    if (bl == BPC - 1 && j == 12) {
                        issue_order();
                        load_w(k, c + k + RS_NB);
                    }
                    issue_order();
                }
#pragma unroll
                for (int j = 0; j < RS_BLK; j++) {
                    x1[j] = x2[j];
#pragma unroll
                    for (int n = 0; n < NE; n++) p[n][j] = pn[n][j];
                }
            }
        }
    }
    wait_vm<0>();  // (the loads past the end)
}

// Workgroup (bx, by) of a grid (nbx + shg_row, ceil(T / 64)) of 256
// threads, nbx = ceil(E / (4 NE)): router rows 4 NE bx .. + 4 NE - 1 (NE a
// wave) for tokens 64 by .. (one a lane); with shg_row, workgroup bx = nbx
// takes the fp16 shared gate (written to gsh by wave 0, 0 when shg is NULL).
// H % 256 == 0 and E >= NE.
template <int NE>
__device__ __forceinline__ void route_seq_block(RsBuf &b0, RsBuf &b1, RsBuf &b2, RsBuf &b3, int bx, int by,
                                                const float *__restrict__ router, const uint16_t *__restrict__ shg,
                                                const float *__restrict__ x, float *__restrict__ logits,
                                                float *__restrict__ gsh, int H, int E, int T, bool shg_row)
{
    const int lane = lane_id(), wv = wave_id();
    const int nbx = (E + RS_WAVES * NE - 1) / (RS_WAVES * NE);
    const int t0 = by * RS_TT, t = t0 + lane, nt = min(RS_TT, T - t0);
    const float *xt = x + (size_t)t0 * H;
    if (shg_row && bx == nbx) {
        float acc[1] = {0.f};
        if (shg) rs_run<1, true>(b0, b1, b2, b3, xt, nt, nullptr, shg, H, acc);
        if (wv == 0 && t < T) gsh[t] = acc[0];
        return;
    }
    // the wave stands for rows eb .. eb + NE - 1 and sums the NE consecutive
    // rows from e0 (moved back from eb so that every row read exists; rows
    // past E are not stored)
    const int eb = bx * RS_WAVES * NE + wv * NE;
    const int e0 = min(eb, E - NE);
    float acc[NE];
#pragma unroll
    for (int n = 0; n < NE; n++) acc[n] = 0.f;
    rs_run<NE, false>(b0, b1, b2, b3, xt, nt, router + (size_t)e0 * H, nullptr, H, acc);
    if (t >= T) return;
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = e0 + n;
        if (e >= eb && e < E) logits[(size_t)t * E + e] = acc[n];
    }
}

} // namespace route_seq
