// gemm1.hip -- grouped FP8 GEMM1 (7168 -> 2 x 2048) with the SwiGLU epilogue fused.
//
// Semantics: reference solution/cuda/moe.cu:222-229 on block-scaled inputs
// (moe_grouped_gemm_fp8.cu:194-264 applies the same scales inside the CUTLASS
// mainloop):
//   G1[r, n] = sum_kb sa[kb, tok(r)] * sb[e, n/128, kb] * sum_{k in kb} A[tok(r), k] W1[e, n, k]
//   C[r, i]  = silu(G1[r, 2048 + i]) * G1[r, i]        (kernel.cu:1104-1108 convention)
// C is written as one row per routed assignment for GEMM2: the fp16 form (fp16 values
// with a power-of-two exponent byte per 16-column group, nonzero only where a group
// holds a value beyond the fp16 range) by the streaming kernels, the fp8 hi/lo form by
// the prefill kernels (moe_device.h, Intermediate).
//
// Kernels: register-staged weight streaming for small T (a work item is one row tile
// of 16 or 32 rows x 16 gate + 16 up rows, its 56 K blocks split over the 4 waves of
// a workgroup and reduced through LDS in a fixed order, so results do not depend on
// scheduling), the same streaming with a 64-row tile's token rows shared by the
// workgroup for mid-size T, and MFMA-bound prefill kernels for large T (256-row tiles).
//
// MFMA: v_mfma_f32_16x16x128_f8f6f4 (e4m3 x e4m3), one instruction per 128-wide K
// block, so the per-block scales multiply a fresh fp32 partial before it joins the
// accumulator.  Weight rows feed operand A (16 n rows), gathered token rows feed
// operand B (16 tokens); lane l holds row/token l%16 and K bytes 32*(l/16)..+31 of
// the block for both operands, and receives D[n = 4*(l/16)+v][token = l%16].

#include "dispatch_rows.h"
#include "gemm1_stream.h"
#include "route_token.h"

#include <algorithm>
#include <mutex>

MOE_STAMP_TABLE(gemm1)

namespace moe {

// The streaming GEMM1 over the row tiles of a dispatch (see gemm1_rstream_item).
template <int D, int CB, int NGRP, bool TL>
__global__ __launch_bounds__(256) void gemm1_rstream_kernel(
    const uint8_t* __restrict__ hidden, TokenScales sa, int T,
    const uint8_t* __restrict__ w1, const float* __restrict__ s1,
    const int4* __restrict__ tiles, const int* __restrict__ num_tiles,
    const int* __restrict__ sorted_tok, Intermediate C, int* __restrict__ c_wide) {
    using S = Gemm1Stream<CB, NGRP, TL>;
    __shared__ __attribute__((aligned(1024))) uint8_t slot_lds[4][S::kSlot];
    __shared__ v4f red[4][2][NGRP * CB][64];
    // the first item's tile read before the tile count, both loads in flight together
    // (blockIdx.x / kItems is inside the list's capacity: the grid has at most capacity x
    // kItems workgroups; a workgroup past the count does not use what it read); each later
    // tile is read after the item before it
    const int4 tl0 = tiles[blockIdx.x / S::kItems];
    int te = __builtin_amdgcn_readfirstlane(tl0.x), tr = __builtin_amdgcn_readfirstlane(tl0.y),
        tn = __builtin_amdgcn_readfirstlane(tl0.z);
    const int nwork = (*num_tiles) * S::kItems;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int work = blockIdx.x; work < nwork; work += gridDim.x) {
        gemm1_rstream_item<D, CB, NGRP, TL>(hidden, sa, w1, s1, te, tr, tn,
                                            (work % S::kItems) * NGRP,
                                            [&](int row) { return sorted_tok[row]; }, C, c_wide,
                                            slot_lds, red, wave);
        if (work + (int)gridDim.x < nwork) {
            const int4 t = tiles[(work + gridDim.x) / S::kItems];
            te = t.x;
            tr = t.y;
            tn = t.z;
        }
    }
}

// Streaming GEMM1 with the tile's token rows shared by the workgroup.  A work item is one
// row tile of up to 64 rows x 16 NWV SwiGLU columns; each of the NWV waves streams its
// own 16 gate + 16 up weight rows over all 56 K blocks through a register ring, as the
// other streaming kernels do, while the token rows of a K block come once for the whole
// workgroup by buffer_load ... lds into a ring of LDS stages (wave w moves rows
// 64/NWV w .. 64/NWV (w + 1) - 1, wave 0 the 64 token scales).  With 8 waves the
// workgroup requests 32 KB of weights and at most 8 KB of token rows per K block for
// 64 x 128 outputs, where the 32-row kernel, whose waves split K and each load the
// tile's rows, requests 12 KB for 32 x 32; and an expert of up to 64 rows streams its
// weights once.  Each wave owns its columns over the whole K, so there is no cross-wave
// reduction; one barrier per K block hands the token stage over.
// D: register ring depth (K blocks of weights per wave); the token stages are one more,
// so that the loads of block kb + D - 1 can go out before the barrier of block kb.
template <int D, int NWV>
struct Gemm1Shared {
    static_assert(NWV == 4 || NWV == 8, "waves per workgroup");
    static constexpr int kSlot = 32 * kBlk;                 // a wave's weight transpose slot
    static constexpr int kTokStage = 64 * kBlk + 2 * 64 * 4;   // 64 token rows, their scales, zeros
    static constexpr int kStages = D + 1;
    static constexpr int kLds = NWV * kSlot + kStages * kTokStage;
    static constexpr int kItems = kI / (16 * NWV);          // work items per tile
};

// One item of gemm1_shared_kernel with CB live 16-row blocks (the tile has 16 CB - 15 ..
// 16 CB rows): wave `wave` computes SwiGLU columns 16 ng .. 16 ng + 15 of rows row0 ..
// row0 + nrows - 1.  AUX: the cache policy of the weight loads.
template <int D, int NWV, int CB, int AUX>
__device__ __forceinline__ void gemm1_shared_item(
    const uint8_t* __restrict__ hidden, const TokenScales& sa, __amdgpu_buffer_rsrc_t rs_h,
    __amdgpu_buffer_rsrc_t rs_s, const uint8_t* __restrict__ w1, const float* __restrict__ s1,
    int le, int row0, int nrows, int ng, const int* __restrict__ sorted_tok, const Intermediate& C,
    int* __restrict__ c_wide, uint8_t* lds, int wave) {
    using S = Gemm1Shared<D, NWV>;
    static_assert(kHB % D == 0, "the K loop runs in steps of the ring depth");
    const int lane = threadIdx.x & 63;
    const int r16 = lane & 15, kq = lane >> 4;
    const int drow = lane >> 3, dchunk = lane & 7;
    const int swz = swz128(r16);
    const int rd_g0 = r16 * kBlk + (((2 * kq) ^ swz) << 4);
    const int rd_g1 = r16 * kBlk + (((2 * kq + 1) ^ swz) << 4);
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    uint8_t* const slot = lds + wave * S::kSlot;
    uint8_t* const tok0 = lds + NWV * S::kSlot;

    // weight rows of this wave: slot rows 0..15 gate rows of group ng, 16..31 its up rows,
    // by buffer loads over the expert's W1 (32-bit offsets: one VGPR per load, the K block
    // in the scalar offset)
    const __amdgpu_buffer_rsrc_t rs_w = buffer_rsrc(w1 + (size_t)le * kN1 * kH, (uint32_t)kN1 * kH);
    uint32_t woff[4];
    int wr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + drow;
        const int n = (r < 16) ? ng * 16 + r : kI + ng * 16 + (r - 16);
        woff[i] = (uint32_t)n * kH + dchunk * 16;
        wr[i] = r * kBlk + ((dchunk ^ swz128(r)) << 4);
    }
    // the NWV groups of a workgroup lie in one 128-column scale block
    const float* sg = s1 + (size_t)(le * kN1B + (ng >> 3)) * kHB;
    const float* su = sg + (size_t)kIB * kHB;
    // The 2 CB loads of the token rows of the live blocks (16 CB stage rows, 8 per instruction,
    // clamped into the tile) and the load of their scales, spread over the waves: wave w issues
    // loads w, w + NWV, ...  Every wave issues the same number per K block whatever is live, so
    // that the number of loads in flight is known at compile time: past the last one it issues
    // one whose offset lies past the buffer, which moves nothing but takes its turn: with a scale
    // load from every wave, 18 experts of up to 16 rows took 92.5 instead of 88.5 us.
    constexpr int NT = (2 * CB + 1 + NWV - 1) / NWV;
    constexpr int kScaleI = 2 * CB / NWV, kScaleWave = 2 * CB % NWV;   // the scales' load
    constexpr uint32_t kNothing = 0xfffffff0u;
    uint32_t toff[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int q = wave + NWV * i;
        const int tr = 8 * q + drow;
        const uint32_t o = (uint32_t)sorted_tok[row0 + min(tr, nrows - 1)] * kH + ((dchunk ^ swz128(tr)) << 4);
        toff[i] = q < 2 * CB ? o : kNothing;
    }
    const int sr = min(lane, nrows - 1);
    const uint32_t so = (uint32_t)(sa.by_row ? row0 + sr : sorted_tok[row0 + sr]) * 4;
    if (wave == kScaleWave) toff[kScaleI] = so;
    const int sdst = 64 * kBlk + (wave == kScaleWave ? 0 : 64 * 4);   // the others' zeros land past the scales
    constexpr int kVm = 4 + NT;                              // loads per wave and K block

    // K block kb: weights in ring slot kb % D, token rows in stage kb % (D + 1)
    v4u bw[D][4];
    auto issue = [&](int kb, int ring) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            bw[ring][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, woff[i], (uint32_t)kb * kBlk, AUX);
        uint8_t* st = tok0 + (kb % S::kStages) * S::kTokStage;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if (i == kScaleI && (kScaleWave == 0 || wave >= kScaleWave))
                bdma4(rs_s, toff[i], (uint32_t)kb * sa.stride * 4, st + sdst);
            else
                bdma16(rs_h, toff[i], (uint32_t)kb * kBlk, st + 8 * (wave + NWV * i) * kBlk);
        }
    };
#pragma unroll
    for (int k = 0; k < D - 1; ++k) issue(k, k);

    v4f ag[CB], au[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) ag[c] = au[c] = zero;
    // One K block, `younger` later blocks in flight.  The loads are unconditional and the
    // last blocks peeled because the wait before a ring slot's use is counted by the
    // compiler too, as the fewest loads any path issues after it: with the token loads
    // under a wave's own branch and the last blocks' loads skipped in the loop, that count
    // was 0 in every second K block, which drained the ring there (T = 509: GEMM1 143 us).
    auto block = [&](int kb, int j, auto younger) {
        // this wave's loads of block kb are in (those of the blocks after it may stay in
        // flight); after the barrier, every wave's (the token stage)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(decltype(younger)::value * kVm));
        lds_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<v4u*>(slot + wr[i]) = bw[j][i];
        const uint8_t* st = tok0 + (kb % S::kStages) * S::kTokStage;
        const float* ssc = reinterpret_cast<const float*>(st + 64 * kBlk);
        const float wg = sg[kb], wu = su[kb];
        const v4u g0 = *reinterpret_cast<const v4u*>(slot + rd_g0);
        const v4u g1 = *reinterpret_cast<const v4u*>(slot + rd_g1);
        const v4u u0 = *reinterpret_cast<const v4u*>(slot + 16 * kBlk + rd_g0);
        const v4u u1 = *reinterpret_cast<const v4u*>(slot + 16 * kBlk + rd_g1);
        const v8i bg = {(int)g0[0], (int)g0[1], (int)g0[2], (int)g0[3], (int)g1[0], (int)g1[1], (int)g1[2], (int)g1[3]};
        const v8i bu = {(int)u0[0], (int)u0[1], (int)u0[2], (int)u0[3], (int)u1[0], (int)u1[1], (int)u1[2], (int)u1[3]};
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            __builtin_amdgcn_sched_barrier(0);   // one row block at a time: short live ranges
            const uint8_t* ts = st + 16 * c * kBlk;
            const v4u a0 = *reinterpret_cast<const v4u*>(ts + rd_g0);
            const v4u a1 = *reinterpret_cast<const v4u*>(ts + rd_g1);
            const v8i ba = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
            const float sc = ssc[16 * c + r16];
            const float fg = sc * wg, fu = sc * wu;
            const v4f tg = mfma_fp8(bg, ba, zero);
            const v4f tu = mfma_fp8(bu, ba, zero);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                ag[c][v] = __builtin_fmaf(tg[v], fg, ag[c][v]);
                au[c][v] = __builtin_fmaf(tu[v], fu, au[c][v]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int kb0 = 0; kb0 < kHB - D; kb0 += D) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            // block kb + D - 1 goes to the ring slot block kb - 1 used (written to the LDS
            // slot before) and to the stage of block kb - 2, which every wave finished
            // reading before the barrier of block kb - 1
            issue(kb0 + j + D - 1, (j + D - 1) % D);
            __builtin_amdgcn_sched_barrier(0);
            block(kb0 + j, j, IntC<D - 1>{});
        }
    }
    issue(kHB - 1, D - 1);
    __builtin_amdgcn_sched_barrier(0);
    block(kHB - D, 0, IntC<D - 1>{});
    [&]<int... J>(std::integer_sequence<int, J...>) {
        (block(kHB - D + 1 + J, 1 + J, IntC<D - 2 - J>{}), ...);
    }(std::make_integer_sequence<int, D - 1>{});
#pragma unroll
    for (int c = 0; c < CB; ++c)
        store_swiglu4(C, c_wide, row0 + 16 * c + r16, ng * 16 + kq * 4, ag[c], au[c], 16 * c + r16 < nrows);
}

// WPE: the waves per SIMD the register allocation is held to (1: the compiler's choice,
// 175 registers, two workgroups per CU; 3: 145 registers, three).
// With three per CU the kernel chooses, from the call's tile count, how many of its 768
// workgroups work: items are equal (an item streams 128 weight rows over all of K), so the
// rounds decide the time, and 768 < items <= 1024 takes two rounds either way, where two
// workgroups per CU run each item faster; then workgroups 512 .. 767 exit at once and the
// other 512 (two per CU, the workgroups being spread over the CUs in launch order) take
// the items.  Otherwise all 768 work (fewer rounds).  Which workgroup computes an item
// changes nothing in the result.
// Weights are loaded non-temporal unless their expert has kNear tiles or more (over 128 rows),
// whose tiles meet in L2.  GEMM1 us in passes over four layers' own weights and routings,
// non-temporal on every item -> by this rule: T = 509 with four experts of 509 rows 241 -> 191,
// T = 400 with eight of 400 242 -> 175, T = 600 with four of 600 265 -> 203, every route local at
// T = 509 392 -> 311; typical T = 509 133, 147, 130, 115 -> 129, 138, 135, 115.  From two tiles on
// (kNear 2) typical calls of T = 509 .. 650 are 2-3% slower, as a second tile is often a few
// rows; from four or six on, T = 509 with every route local loses 6 and 10%.  Passes that repeat one
// layer do not show this: its weights are then still in the last-level cache.
constexpr int kNear = 3;

template <int D, int NWV, int WPE>
__global__ __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm1_shared_kernel(
    const uint8_t* __restrict__ hidden, TokenScales sa, int T,
    const uint8_t* __restrict__ w1, const float* __restrict__ s1,
    const int4* __restrict__ tiles, const int* __restrict__ num_tiles,
    const int* __restrict__ sorted_tok, Intermediate C, int* __restrict__ c_wide) {
    using S = Gemm1Shared<D, NWV>;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S::kLds];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // token rows: T * 7168 < 2^32 (kMaxT); token scales: 56 x stride floats
    const __amdgpu_buffer_rsrc_t rs_h = buffer_rsrc(hidden, (uint32_t)T * kH);
    const __amdgpu_buffer_rsrc_t rs_s = buffer_rsrc(sa.p, (uint32_t)kHB * (uint32_t)sa.stride * 4);
    // the first item's tile, and the experts of the tiles around it, read before the tile count,
    // all in flight together (blockIdx.x / kItems is inside the list's capacity: the grid has
    // at most capacity x kItems workgroups, and the list's region holds twice as many 16-row
    // tiles; a workgroup past the count does not use what it read); each later tile is read
    // after the item before it
    const int lane = threadIdx.x & 63;
    auto expert_near = [&](int t) { return tiles[max(t - (kNear - 1) + min(lane, 2 * kNear - 2), 0)].x; };
    // the expert of tile t has kNear tiles or more: as many of the kNear - 1 tiles on either
    // side and itself are its own
    auto has_several = [&](int t, int e, int near, int ntiles) {
        const int i = t - (kNear - 1) + lane;
        return __popcll(__ballot(lane <= 2 * kNear - 2 && i >= 0 && i < ntiles && near == e)) >= kNear;
    };
    const int t0 = blockIdx.x / S::kItems;
    const int4 tl0 = tiles[t0];
    const int near0 = expert_near(t0);
    int te = __builtin_amdgcn_readfirstlane(tl0.x), tr = __builtin_amdgcn_readfirstlane(tl0.y),
        tn = __builtin_amdgcn_readfirstlane(tl0.z);
    const int ntiles = *num_tiles;
    const int nwork = ntiles * S::kItems;
    bool several = has_several(t0, te, near0, ntiles);
    int G = gridDim.x;
    if (WPE == 3 && G == 768 && nwork > 768 && nwork <= 1024) G = 512;
    if ((int)blockIdx.x >= G) return;   // uniform: the whole workgroup
    for (int work = blockIdx.x; work < nwork; work += G) {
        const int ng = (work % S::kItems) * NWV + wave;
        with_live_blocks(live_blocks(0, tn), [&](auto live) {
            constexpr int CB = decltype(live)::value;
            auto item = [&](auto aux) {
                gemm1_shared_item<D, NWV, CB, decltype(aux)::value>(hidden, sa, rs_h, rs_s, w1, s1, te, tr, tn,
                                                                    ng, sorted_tok, C, c_wide, lds, wave);
            };
            if constexpr (CB > 0) {
                if (several) item(IntC<0>{});
                else item(IntC<kNonTemporal>{});
            }
        });
        if (work + G < nwork) {
            const int ti = (work + G) / S::kItems;
            const int4 t = tiles[ti];
            const int near = expert_near(ti);
            te = t.x;
            tr = t.y;
            tn = t.z;
            several = has_several(ti, te, near, ntiles);
        }
        __syncthreads();   // the next item's first loads reuse the token stages
    }
}

// The streaming GEMM1 of variant 1 with the dispatch folded in, for T <= 64: every
// workgroup of a persistent grid computes the part of the call's dispatch its items need,
// into LDS.  Wave 0 takes one ballot per local expert over the tokens (lane = token),
// which gives each expert's row count, the tile list, and each row's rank among the
// expert's rows (rows follow token order); then all four waves place the tokens of the
// rows, two of each token's eight routes per wave.  The last workgroup, which has the
// fewest items (none up to T = 32), also writes the whole dispatch to the workspace
// (expert offsets, tile count and list, permutation, row weights, inverse map), where
// the GEMM2 and combine kernels after this one read it.  Workgroup b takes items b,
// b + G, ..., so the items of an expert's consecutive tiles that read the same weight
// rows (128 items apart) run on one XCD.  The dispatch launch goes away; the part of the
// dispatch before the first weight load costs a workgroup about what the separate
// kernel's two dependent loads (tile list, then permutation) cost.
//
// NRW > 0 (T <= NRW): the routing too.  Every workgroup routes the call's tokens itself
// from the logits (route_token, the route kernel's computation: wave w takes token w) into
// LDS, where the dispatch reads them; the last workgroup also writes them to the
// workspace.  NRW = 8 (5 <= T <= 8) runs workgroups of 8 waves, one per CU, so that a SIMD
// routes two tokens, not six; its waves then work as two groups of four, each taking every
// other of the workgroup's items, in step (a group without an item passes the item's two
// barriers), so a CU still streams two items at a time.  The route launch, its kernel boundary
// and the dispatch's dependent load of the routing ids go away.  Nothing clears the
// C-range flag word before this kernel: it sets the word when C goes beyond the fp16
// range, and the GEMM2 after it (variant 6) checks a nonzero word against C's group
// exponents (a stale nonzero word left by earlier calls or other data only costs that check,
// and the GEMM2 clears it).
constexpr int kDG1MaxTiles = dispatch_max_tiles(kDispatchInGemm1MaxT, 16);   // 64

template <int NRW>
__global__ __launch_bounds__(NRW == 8 ? 512 : 256) void gemm1_rstream_dispatch_kernel(
    RouteIn rin, int* __restrict__ topk_ids, float* __restrict__ topk_w, int T, int offset,
    const uint8_t* __restrict__ hidden, const float* __restrict__ hs_scale,
    const uint8_t* __restrict__ w1, const float* __restrict__ s1, int* __restrict__ meta,
    int4* __restrict__ tiles, int* __restrict__ sorted_tok, float* __restrict__ sorted_w,
    int* __restrict__ inv, Intermediate C) {
    using S = Gemm1Stream<1, 1, false>;
    constexpr int R = kDispatchInGemm1MaxT * kTopK;
    constexpr int NG = NRW == 8 ? 2 : 1;   // groups of 4 waves taking items
    __shared__ __attribute__((aligned(1024))) uint8_t slot_lds[4 * NG][S::kSlot];
    __shared__ v4f red[4 * NG][2][1][64];
    __shared__ int s_exp_off[kEL + 1];
    __shared__ int s_num_tiles;
    __shared__ int4 s_tiles[kDG1MaxTiles];
    __shared__ int s_stok[R];
    __shared__ int8_t s_lek[kDispatchInGemm1MaxT][kTopK];
    __shared__ float s_wk[kDispatchInGemm1MaxT][kTopK];
    __shared__ DispatchWaveLds s_dw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool writer = blockIdx.x == gridDim.x - 1;
    MOE_STAMP(3 * (int)blockIdx.x);
    const int* ids_src = topk_ids;
    const float* w_src = topk_w;
    if constexpr (NRW > 0) {
        static_assert(NRW == 4 || NRW == 8, "one token per wave");
        static_assert(kRouteInGemm1MaxT <= 8, "at most 8 waves route");
        __shared__ __attribute__((aligned(16))) int s_rid[NRW][kTopK];
        __shared__ __attribute__((aligned(16))) float s_rw[NRW][kTopK];
        __shared__ float s_sel[NRW][kTopK];
        __shared__ int s_sel_id[NRW][kTopK];
        const int t = wave;
        if (t < T) {   // uniform per wave
            const float4 lg = reinterpret_cast<const float4*>(rin.logits + (size_t)t * kEG)[lane];
            const uint2 bb = reinterpret_cast<const uint2*>(rin.bias)[lane];
            int id;
            float w;
            route_token(lg, bb, lane, rin.factor, s_sel[wave], s_sel_id[wave], id, w);
            if (lane < kTopK) {
                s_rid[t][lane] = id;
                s_rw[t][lane] = w;
                if (writer) {
                    topk_ids[t * kTopK + lane] = id;
                    topk_w[t * kTopK + lane] = w;
                }
            }
        }
        __syncthreads();
        ids_src = &s_rid[0][0];
        w_src = &s_rw[0][0];
    }
    if (wave == 0) {
        const TokenRoutes r = load_routes(ids_src, w_src, lane, T, offset);
        wave_ballots(r, 0, lane, s_dw.wcnt, s_dw.bal);
#pragma unroll
        for (int k = 0; k < kTopK; ++k) {
            s_lek[lane][k] = (int8_t)r.lek[k];
            s_wk[lane][k] = r.wk[k];
        }
        __builtin_amdgcn_wave_barrier();
        write_offsets_and_tiles<16, 0>(lane < kEL ? s_dw.wcnt[0][lane] : 0, lane, s_dw.off,
                                       s_exp_off, &s_num_tiles, s_tiles, nullptr, nullptr);
    }
    __syncthreads();
    const int ntiles = s_num_tiles;
    if (wave < 4 && lane < T) {   // token lane: its routes 2 wave and 2 wave + 1
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int k = 2 * wave + kk;
            const int le = s_lek[lane][k];
            int row = -1;
            if (le >= 0) {
                const uint64_t b = s_dw.bal[le];
                row = s_exp_off[le] + (int)__builtin_amdgcn_mbcnt_hi(
                                          (uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
                s_stok[row] = lane;
                if (writer) {
                    sorted_tok[row] = lane;
                    sorted_w[row] = s_wk[lane][k];
                }
            }
            if (writer) inv[lane * kTopK + k] = row;
        }
    }
    if (writer) {
        for (int i = tid; i <= kEL; i += 256) meta[i] = s_exp_off[i];
        if (tid == 0) meta[kEL + 1] = ntiles;
        for (int i = tid; i < ntiles; i += 256) tiles[i] = s_tiles[i];
    }
    __syncthreads();
    MOE_STAMP(3 * (int)blockIdx.x + 1);
    const TokenScales sa{hs_scale, T, 0};
    const int nwork = ntiles * S::kItems;
    int* const c_wide = meta + kCWideFlag;
    if constexpr (NG == 2) {
        // group g takes the workgroup's items 2 i + g (items b, b + G, b + 2 G, ...)
        const int grp = wave >> 2, w4 = wave & 3;
        const int G = gridDim.x, b = blockIdx.x;
        const int mine = b < nwork ? (nwork - b + G - 1) / G : 0;
        for (int i = 0; i < (mine + 1) / 2; ++i) {
            const int k = 2 * i + grp;
            if (k < mine) {   // uniform per wave
                const int work = b + k * G;
                const int4 tile = s_tiles[work / S::kItems];
                gemm1_rstream_item<4, 1, 1, false>(hidden, sa, w1, s1, tile.x, tile.y, tile.z,
                                                   work % S::kItems, [&](int row) { return s_stok[row]; },
                                                   C, c_wide, &slot_lds[4 * grp], &red[4 * grp], w4);
            } else {
                __syncthreads();   // the two barriers of the item the other group runs
                __syncthreads();
            }
        }
    } else {
        for (int work = blockIdx.x; work < nwork; work += gridDim.x) {
            const int4 tile = s_tiles[work / S::kItems];
            gemm1_rstream_item<4, 1, 1, false>(hidden, sa, w1, s1, tile.x, tile.y, tile.z,
                                               work % S::kItems, [&](int row) { return s_stok[row]; },
                                               C, c_wide, slot_lds, red, wave);
        }
    }
    MOE_STAMP(3 * (int)blockIdx.x + 2);
}

// Epilogue of the prefill GEMM1: SwiGLU, then the fp8 hi/lo form of C.  The wave holds 128
// rows x 32 SwiGLU columns (acc[s][i]: i < 2 gate, i >= 2 up; lane holds D[col 16 i + 4 kq
// + v][row 16 s + r16]); the waves wn = 0 .. 3 hold the 128 columns of block ng, so the row
// amax is combined across them through LDS (xch, [4][256] floats).  Per row: s = amax/448
// (1 for an all-zero row), hi = e4m3(c * 448/amax), lo = e4m3((c - hi*s) * 16*448/amax).
// A lane's 4 bytes of two rows in each of the 2 column blocks are transposed across the
// rows' 4 lanes (lanes l, l+16, l+32, l+48) with v_permlane32_swap / v_permlane16_swap,
// after which a lane holds 16 consecutive bytes of one row: one 16-byte store per form for
// two row blocks.  Row blocks past the tile (from `live` on, uniform) are skipped.
// through_f16: C is first rounded as the fp16 form holds it (moe_device.h), a 16-column group
// with a value beyond the fp16 range by its group exponent, and such a group raises *c_wide:
// the rows and the flag of a streaming GEMM1 and the conversion.
__device__ __forceinline__ void store_c_hilo(const v4f (&acc)[8][4], float* xch, int live, int wm, int wn,
                                             int kq, int r16, int row0, int nrows, int ng,
                                             const Intermediate& C, bool through_f16, int* c_wide) {
    float c[8][2][4];
    float m[8];
    // the row addresses are computed here: kept through the K loop they would spill, and a
    // reload waits for the next item's blocks
    __asm__ volatile("" : "+v"(r16));
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        m[s] = 0.f;
        if (s >= live) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) c[s][i][v] = silu_f32(acc[s][i + 2][v]) * acc[s][i][v];
            if (through_f16) {
                float mg = 0.f;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // the fp32 product first, then fp16 (fused into one rounding otherwise)
                    __asm__ volatile("" : "+v"(c[s][i][v]));
                    mg = fmaxf(mg, fabsf(c[s][i][v]));
                }
                if (!beyond_f16_in_wave(mg)) {   // the usual case: exponent 0
#pragma unroll
                    for (int v = 0; v < 4; ++v) c[s][i][v] = (float)(_Float16)c[s][i][v];
                } else {
                    const int e = group_exponent(mg);
#pragma unroll
                    for (int v = 0; v < 4; ++v) c[s][i][v] = ldexpf((float)(_Float16)ldexpf(c[s][i][v], -e), e);
                    if (e && 128 * wm + 16 * s + r16 < nrows) *c_wide = 1;   // rows past the tile hold anything
                }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) m[s] = fmaxf(m[s], fabsf(c[s][i][v]));
        }
    }
    // Row maxima of 4 row blocks across the rows' 4 lanes by lane swaps: lane kq then holds
    // those of block 4 h + kq, and computes that row's scale once for its 4 lanes.  With every
    // lane computing all 8 of its rows' scales (16 divisions a lane) an item's epilogue took
    // 6.5 us instead of 5.4, on every round of full tiles: all routes local at T = 8192, 17
    // items a workgroup, GEMM1 1754 -> 1719 us; typical T = 8192 389 -> 379.
    auto swap_max32 = [](float a, float b) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
    };
    auto swap_max16 = [](float a, float b) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
    };
#pragma unroll
    for (int h = 0; h < 2; ++h)
        xch[wn * 256 + 128 * wm + 64 * h + 16 * kq + r16] =
            swap_max16(swap_max32(m[4 * h], m[4 * h + 2]), swap_max32(m[4 * h + 1], m[4 * h + 3]));
    lds_barrier();
    // lane kq's value of x to all 4 lanes of its row, for each kq
    auto spread4 = [](float x, float* y) {
        const uint32_t u = __float_as_uint(x);
        const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        const auto q0 = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
        const auto q1 = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
        y[0] = __uint_as_float(q0[0]);
        y[1] = __uint_as_float(q1[0]);
        y[2] = __uint_as_float(q0[1]);
        y[3] = __uint_as_float(q1[1]);
    };
    float sc[8], inv[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (4 * h >= live) continue;
        const int r = 128 * wm + 64 * h + 16 * kq + r16;
        float amax = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) amax = fmaxf(amax, xch[w * 256 + r]);
        const float scr = amax > 0.f ? amax / 448.f : 1.f;
        if (wn == 0 && r < nrows) C.scales[(size_t)ng * C.rows_cap + row0 + r] = scr;
        spread4(scr, sc + 4 * h);
        spread4(amax > 0.f ? 448.f / amax : 1.f, inv + 4 * h);
    }
    // 4 x 4 transpose of 32-bit words over the 16-lane rows of the wave (word j of row kq
    // -> word kq of row j): 32-lane then 16-lane swaps
    auto transpose4 = [](uint32_t (&w)[4]) {
        auto p = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
        w[0] = p[0]; w[2] = p[1];
        p = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        w[1] = p[0]; w[3] = p[1];
        p = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
        w[0] = p[0]; w[1] = p[1];
        p = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
        w[2] = p[0]; w[3] = p[1];
    };
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        if (2 * p >= live) continue;
        uint32_t h[4], l[4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int s = 2 * p + q;
            const float inv16 = inv[s] * 16.f;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float* x = c[s][i];
                const uint32_t hw = e4m3x4_from_f32(clamp448(x[0] * inv[s]), clamp448(x[1] * inv[s]),
                                                    clamp448(x[2] * inv[s]), clamp448(x[3] * inv[s]));
                const auto h01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hw, false);
                const auto h23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hw, true);
                const float hv[4] = {h01[0], h01[1], h23[0], h23[1]};
                float lq[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) lq[v] = clamp448(__builtin_fmaf(-hv[v], sc[s], x[v]) * inv16);
                h[2 * q + i] = hw;
                l[2 * q + i] = e4m3x4_from_f32(lq[0], lq[1], lq[2], lq[3]);
            }
        }
        // every lane of the wave takes part in the swaps; lane kq then holds row block
        // 2 p + kq / 2, columns 16 (kq & 1) .. + 15 of the wave's 32
        transpose4(h);
        transpose4(l);
        const int r = 128 * wm + 16 * (2 * p + (kq >> 1)) + r16;
        if (r >= nrows) continue;
        const size_t off = (size_t)(row0 + r) * kI + ng * 128 + 32 * wn + 16 * (kq & 1);
        *reinterpret_cast<v4u*>(C.hi() + off) = v4u{h[0], h[1], h[2], h[3]};
        *reinterpret_cast<v4u*>(C.lo() + off) = v4u{l[0], l[1], l[2], l[3]};
    }
}

// ---------------------------------------------------------------------------
// Prefill GEMM1 (from a few dozen tokens per expert up): workgroup tile of up to 256
// gathered token rows x 256 weight rows (128 gate rows n0 .. n0 + 127 and the matching 128
// up rows 2048 + n0 .., i.e. 128 SwiGLU columns); waves 2 (token rows) x 4 (weight rows),
// each 128 tokens x (32 gate + 32 up) rows: per K block up to 32 MFMA 16x16x128 (a wave
// holds its 4 weight fragments and streams the token fragments past them) whose fresh
// partials are scaled by sa[token] * sb[block] into fp32 accumulators.  Two waves per SIMD,
// so registers stay <= 256 per lane.  Rows in LDS keep 16-byte chunk c at c ^ swz128(r), so
// ds_read_b128 in the MFMA layout is conflict-free.  Items (row tile, 128-column group)
// follow prefill_items_ranked, or grouped_item when that is not asked for or does not fit,
// with an XCD-contiguous mapping of each round.
//
// What bounds it.  An item of few rows is bound by its weight stream (32 KB per K block and
// CU), one of many by the matrix cores at a clock the power limit holds to 1.9 GHz; both
// lost their time waiting for operands: with two stages whatever the rows, a K block's loads
// went out after the barrier that ended the block before and had to land by its own end.
//   - The item's rows decide how many K blocks the LDS holds (Gemm1Class): the fewer rows,
//     the deeper the weight stream runs ahead.
//   - The barrier of a K block stands before its last token fragment's MFMAs, not after
//     them: every fragment has been read by then, so the next block's first fragments are
//     read under those MFMAs.
//   - With two stages the weight stage is handed over earlier still, by a barrier of its own
//     once every wave holds its weight fragments, so weight loads run 1.75 blocks ahead; the
//     loads are spread over the block's MFMAs, as a wave that issues many back to back stalls
//     on the address path (all at once: 3555 instead of 3345 cycles a K block with every
//     operand in L2).
//   - Weights that only this item's workgroup reads (the expert has one row tile) are loaded
//     non-temporal up to T = kOnceMaxT; those of an expert with more tiles are not, its tiles
//     meet in L2.
//   - Past the last K block the buffers have no bytes: the loads stay in the loop without a
//     branch, move nothing, and the counted waits hold in the last blocks too.
// Measured (GEMM1 us, two stages whatever the rows -> now): 24 experts of 16 rows 174 -> 133, of
// 48 184 -> 140, of 128 202 -> 176, of 256 237 -> 220, of 512 321 -> 304; typical routings T =
// 1024 185 -> 140, 2731 195 -> 165, 8192 356 -> 326 and 367 -> 370, 14107 439 -> 381; skewed T =
// 4096 531 -> 518 and 543 -> 550; every route local, T = 8192 1700 -> 1746, T = 27000 5459 ->
// 5673 (its K loop takes the same 96 us, the change of items 1.4 us more).  The non-temporal loads
// alone: 16 rows 147 -> 134, 128 rows 182 -> 162, 256 rows 230 -> 217, uneven T = 1024 152 ->
// 139 (on every item they cost 4% where experts have several tiles: T = 2731 215 -> 225).
// Not faster: 4 x 2 waves holding the token fragments (24 x 256 rows 236 us), 8 waves each
// with its own 32 weight rows loaded straight into registers (half-line loads: 289 us).
//
// A workgroup resolves the metadata of all its items at kernel start; an item's token ids
// and weight scales come by DMA during the item before, and its first K blocks are issued
// before the epilogue of that item and land under it.
// Token offsets are 32-bit: T * 7168 < 2^32 (T <= 2^19, checked by the host).
// ---------------------------------------------------------------------------
// Row class of an item, from its rows: how many K blocks of operands the LDS holds.
//   A  145 .. 256 rows  2 stages of 32 KB token rows + 32 KB weight rows
//   B   41 .. 144 rows  3 stages of 18 KB + 32 KB
//   C    1 ..  40 rows  4 stages of  5 KB + 32 KB
// (the rows at which the next deeper ring just fits into 160 KB beside the epilogue's and
// the items' 7 KB)
template <int NS, int ROWS, int NT>
struct Gemm1Class {
    static constexpr int kNS = NS;                     // stages
    static constexpr int kNT = NT;                     // token-row loads per wave and K block
    static constexpr int kRows = ROWS;
    static constexpr int kSlots = (ROWS + 63) / 64 + 1;   // 64-row slots of token scales, and one for zeros
    static constexpr int kTok = ROWS * kBlk;
    static constexpr int kW = 256 * kBlk;
    static constexpr int kTokBase = NS * kW;           // weight stages first
    static constexpr int kScaBase = kTokBase + NS * kTok;
    static constexpr int kBytes = kScaBase + NS * kSlots * 256;
};
// mode bits of gemm1_prefill8_kernel
constexpr int kPrefillRanked = 1, kPrefillThroughF16 = 2;
// Largest T whose weights of one-tile experts are loaded non-temporal: whole calls over four
// routings each were 6% faster for it at T = 800 .. 1400, 4% at 2000, 1% at 2731, and 0.7%
// slower at 3500, where most weights belong to experts of several tiles.  The kernel for
// larger T is compiled without the second set of K loops, which alone cost it 0.7%.
constexpr int kOnceMaxT = 2560;

using Gemm1A = Gemm1Class<2, 256, 4>;
using Gemm1B = Gemm1Class<3, 144, 3>;
using Gemm1C = Gemm1Class<4, 40, 1>;

struct Gemm1Item {   // uniform part of an item; the per-lane DMA offsets live apart
    const uint8_t* w;    // the expert's W1 from the item's first gate row on
    uint32_t wbytes;
    int row0, nrows, ng;
    bool once;           // weights loaded non-temporal: the expert has no other row tile
};

template <bool ONCE>
__global__ __launch_bounds__(512, 1) void gemm1_prefill8_kernel(
    const uint8_t* __restrict__ hidden, TokenScales sa, int T,
    const uint8_t* __restrict__ w1, const float* __restrict__ s1,
    const int4* __restrict__ tiles, const int* __restrict__ num_tiles,
    const int* __restrict__ exp_off, const int* __restrict__ sorted_tok, Intermediate C, int mode,
    int* __restrict__ c_wide) {
    constexpr int BM = 256;
    constexpr int NG = kI / 128;
    constexpr int kItemCap = 56;                // per-workgroup item table
    constexpr int kPool = std::max({Gemm1A::kBytes, Gemm1B::kBytes, Gemm1C::kBytes});
    constexpr int kXch = kPool, kTokIds = kXch + 4 * BM * 4, kWsc = kTokIds + BM * 4, kItems = kWsc + 2 * 512,
                  kRows = kItems + kItemCap * (int)sizeof(int4);
    // one LDS object: the stages, the row-maximum exchange, the next item's tokens, two
    // items' weight scales, the item table, the experts' rows
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kRows + kEL * 4];
    static_assert(sizeof(lds) <= 160 * 1024, "LDS of a CU");
    int4* const s_items = reinterpret_cast<int4*>(lds + kItems);
    const int* const s_tok = reinterpret_cast<const int*>(lds + kTokIds);
    int* const s_rows = reinterpret_cast<int*>(lds + kRows);

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int r16 = lane & 15, kq = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    const int nitems = *num_tiles * NG;
    const int G = gridDim.x;
    const int base = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);   // XCD-contiguous slot
    const int drow = lane >> 3, dchunk = lane & 7;
    const int swz = swz128(r16);
    const int c0 = r16 * kBlk + (((2 * kq) ^ swz) << 4), c1 = r16 * kBlk + (((2 * kq + 1) ^ swz) << 4);
    const __amdgpu_buffer_rsrc_t rs_ids = buffer_rsrc(sorted_tok, (uint32_t)T * kTopK * 4);
    const __amdgpu_buffer_rsrc_t rs_s1 = buffer_rsrc(s1, kEL * kN1B * kHB * 4);
    constexpr uint32_t kNothing = 0xfffffff0u;   // an offset past every buffer: moves nothing
    // wave w moves weight rows 32w..32w+31 of a stage; their lane offsets are relative to
    // the item's first gate row (the resource base), so they do not depend on the item
    uint32_t woff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 32 * wave + 8 * i + drow;
        const int n = (r < 128) ? r : kI + (r - 128);
        woff[i] = (uint32_t)n * kH + ((dchunk ^ swz128(r)) << 4);
    }

    static_assert(kRankThreads == 512 && kRankScratch <= kPool, "ranked order: threads, scratch");
    int nr = (mode & kPrefillRanked) ? prefill_items_ranked<BM>(s_items, kItemCap, NG, base, G, exp_off, lds) : -1;
    if (nr < 0) nr = prefill_items<BM>(s_items, kItemCap, nitems, NG, base, G, tiles, exp_off);
    if (nr == 0) return;   // uniform: the whole workgroup has no item
    if (ONCE && threadIdx.x < kEL) s_rows[threadIdx.x] = exp_off[threadIdx.x + 1] - exp_off[threadIdx.x];
    __syncthreads();

    // lane-dependent addresses that only the change of items needs are computed there, from a
    // lane number the compiler cannot see through: kept through the K loop they would spill,
    // and a reload waits for every DMA in flight
    auto opaque = [](int x) {
        __asm__ volatile("" : "+v"(x));
        return x;
    };
    // an item's tokens (waves 0..3, 64 each) and weight block scales (wave 4 gate, 5 up), by
    // DMA into LDS; the scales of item r in buffer r & 1
    auto fetch_side = [&](int r) {
        const int4 m = prefill_item<BM>(s_items, kItemCap, r, NG, base, G, tiles, exp_off);
        const int ln = opaque(lane);
        if (wave < 4) {
            bdma4(rs_ids, (uint32_t)(m.y + min(64 * wave + ln, m.z - 1)) * 4, 0, lds + kTokIds + wave * 256);
        } else if (wave < 6) {
            const uint32_t first = (uint32_t)(m.x * kN1B + m.w + (wave == 5 ? kIB : 0)) * kHB;
            bdma4(rs_s1, (first + min(ln, kHB - 1)) * 4, 0, lds + kWsc + (r & 1) * 512 + (wave - 4) * 256);
        }
    };
    uint32_t aoff[4], soff;   // token-row and token-scale offsets of the item being fetched
    auto make_item = [&](int r) {
        const int4 m = prefill_item<BM>(s_items, kItemCap, r, NG, base, G, tiles, exp_off);
        Gemm1Item it;
        it.row0 = m.y;
        it.nrows = m.z;
        it.ng = m.w;
        const size_t first = (size_t)m.x * kN1 + (size_t)it.ng * 128;
        it.w = w1 + first * kH;
        it.wbytes = (uint32_t)(((size_t)(m.x + 1) * kN1 - first) * kH);
        it.once = ONCE && __builtin_amdgcn_readfirstlane(s_rows[m.x]) <= BM;
        return it;
    };
    // 8-row blocks of token rows this wave moves: NT wave + i (clamped into the class's rows,
    // the clamped ones moving the last block again)
    auto tok_block = [&](auto cls, int i) {
        using Cl = decltype(cls);
        return min(Cl::kNT * wave + i, Cl::kRows / 8 - 1);
    };
    auto set_offsets = [&](auto cls, const Gemm1Item& it) {
        using Cl = decltype(cls);
        const int ln = opaque(lane);
#pragma unroll
        for (int i = 0; i < Cl::kNT; ++i) {
            const int q = tok_block(cls, i);
            const int r = 8 * q + (ln >> 3);
            // a block past the tile moves nothing
            aoff[i] = 8 * q < it.nrows ? (uint32_t)s_tok[min(r, it.nrows - 1)] * kH + (((ln & 7) ^ swz128(r)) << 4)
                                       : kNothing;
        }
        const int sr = min(64 * wave + ln, it.nrows - 1);
        soff = 64 * wave < it.nrows ? (uint32_t)(sa.by_row ? it.row0 + sr : s_tok[sr & 255]) * 4 : kNothing;
    };
    // K block kb of an item into a stage; past the last block the buffers have no bytes, so
    // that nothing moves and the number of loads in flight stays the same without a branch
    // in the K loop
    auto issue_w = [&](auto cls, auto once, const Gemm1Item& it, int kb, int stage, int i0 = 0, int i1 = 4) {
        using Cl = decltype(cls);
        const __amdgpu_buffer_rsrc_t rs_w = buffer_rsrc(it.w, kb < kHB ? it.wbytes : 0u);
#pragma unroll
        for (int i = i0; i < i1; ++i)
            bdma16<decltype(once)::value ? kNonTemporal : 0>(rs_w, woff[i], (uint32_t)kb * kBlk,
                                                             lds + stage * Cl::kW + (32 * wave + 8 * i) * kBlk);
    };
    auto issue_t = [&](auto cls, int kb, int stage, int i0 = 0, int i1 = 5) {
        using Cl = decltype(cls);
        const bool on = kb < kHB;
        const __amdgpu_buffer_rsrc_t rs_tok = buffer_rsrc(hidden, on ? (uint32_t)T * kH : 0u);
        const __amdgpu_buffer_rsrc_t rs_sca = buffer_rsrc(sa.p, on ? (uint32_t)sa.stride * kHB * 4 : 0u);
#pragma unroll
        for (int i = i0; i < i1 && i < Cl::kNT; ++i)
            bdma16(rs_tok, aoff[i], (uint32_t)kb * kBlk, lds + Cl::kTokBase + stage * Cl::kTok + 8 * tok_block(cls, i) * kBlk);
        if (i1 == 5)
        bdma4(rs_sca, soff, (uint32_t)kb * sa.stride * 4,
              lds + Cl::kScaBase + (stage * Cl::kSlots + min(wave, Cl::kSlots - 1)) * 256);
    };
    auto start = [&](auto cls, const Gemm1Item& it) {   // the item's first stages
        set_offsets(cls, it);
#pragma unroll
        for (int k = 0; k < decltype(cls)::kNS; ++k) {
            if (ONCE && it.once) issue_w(cls, BoolC<ONCE>{}, it, k, k);
            else issue_w(cls, BoolC<false>{}, it, k, k);
            if (decltype(cls)::kNS > 2 || k == 0) issue_t(cls, k, k);
            else issue_t(cls, k, k, 0, 2);   // the rest in the K loop
        }
    };
    auto with_class = [&](int nrows, auto&& f) {
        if (nrows > Gemm1B::kRows) f(Gemm1A{});
        else if (nrows > Gemm1C::kRows) f(Gemm1B{});
        else f(Gemm1C{});
    };

    fetch_side(0);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    lds_barrier();
    Gemm1Item cur = make_item(0), nxt = cur;
    with_class(cur.nrows, [&](auto cls) { start(cls, cur); });
    for (int r = 0; r < nr; ++r) {
        const bool more = r + 1 < nr;
        const float* const wsc = reinterpret_cast<const float*>(lds + kWsc + (r & 1) * 512);
        v4f acc[8][4];
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[s][i] = zero;

        // NL: row blocks 128 wm + 16 j of this wave that are computed (the live ones, rounded
        // up to the instantiated counts; padding rows are computed on whatever the LDS holds
        // and never stored)
        auto kloop_of = [&](auto cls, auto live, auto once) {
            using Cl = decltype(cls);
            constexpr int NL = decltype(live)::value;
            constexpr int NS = Cl::kNS;
            auto rd = [&](const uint8_t* rp) {
                const v4u x0 = *reinterpret_cast<const v4u*>(rp + c0);
                const v4u x1 = *reinterpret_cast<const v4u*>(rp + c1);
                return v8i{(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
            };
            auto read_t = [&](int stage, int j) {
                return rd(lds + Cl::kTokBase + stage * Cl::kTok + (128 * wm + 16 * j) * kBlk);
            };
            auto read_s = [&](int stage, int j) {
                return reinterpret_cast<const float*>(lds + Cl::kScaBase + stage * Cl::kSlots * 256)[128 * wm + 16 * j + r16];
            };
            auto read_w = [&](int stage, int i) {
                return rd(lds + stage * Cl::kW + ((i < 2 ? 0 : 128) + 32 * wn + 16 * (i & 1)) * kBlk);
            };
            // kEarly (two stages): a K block's weight stage is handed over by a barrier of its
            // own, as soon as every wave holds the block's weight fragments, and the loads are
            // spread over the block's MFMAs.  Otherwise both stages go with the barrier before
            // the last token block's MFMAs, all loads right after it.
            constexpr bool kEarly = NS == 2;
            constexpr int kFirstT = kEarly ? 2 : 5;   // token loads right after the hand-over
            // every wave holds its weight fragments of K block kb: the weight stage goes to
            // block kb + NS
            auto free_weights = [&](int kb, int stage) {
                __builtin_amdgcn_sched_barrier(0);
                lds_barrier();
                if (NL > 4) issue_w(cls, once, cur, kb + NS, stage, 0, 1);
                else issue_w(cls, once, cur, kb + NS, stage);
                __builtin_amdgcn_sched_barrier(0);
            };
            // every wave has read its last token fragment of K block kb, and block kb + 1 has
            // landed for every wave: the token stage goes to block kb + NS
            auto hand_over = [&](int kb, int stage) {
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(kEarly ? 4 : (NS - 2) * (4 + Cl::kNT + 1)));
                lds_barrier();
                if (!kEarly) issue_w(cls, once, cur, kb + NS, stage);
                issue_t(cls, kb + NS, stage, 0, kFirstT);
                __builtin_amdgcn_sched_barrier(0);
            };
            if (kEarly) __builtin_amdgcn_s_waitcnt(vmcnt_imm(4 + 2));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * (4 + Cl::kNT + 1)));
            lds_barrier();
            if (more) fetch_side(r + 1);
            int stage = 0;
            if constexpr (NL == 0) {
#pragma unroll 1
                for (int kb = 0; kb < kHB; ++kb) {
                    if (kEarly) {
                        issue_t(cls, kb - 1 + NS, stage == 0 ? NS - 1 : stage - 1, 2, 5);
                        free_weights(kb, stage);
                    }
                    hand_over(kb, stage);
                    stage = stage + 1 == NS ? 0 : stage + 1;
                }
            } else {
                int first = 0;
                __asm__ volatile("" : "+s"(first));   // as opaque()
                v8i w[4];
                v8i t = read_t(first, 0);
                float sv = read_s(first, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = read_w(first, i);
                float wg = wsc[0], wu = wsc[64];
                v4f tp[4];
                float fgp = 0.f, fup = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) tp[i] = zero;
#pragma unroll 1
                for (int kb = 0; kb < kHB; ++kb) {
                    const int nstage = stage + 1 == NS ? 0 : stage + 1;
                    const int pstage = stage == 0 ? NS - 1 : stage - 1;
                    float wgn = 0.f, wun = 0.f;
#pragma unroll
                    for (int j = 0; j < NL; ++j) {
                        if (kEarly && j == 1) free_weights(kb, stage);
                        v8i tn;
                        float svn;
                        if (j < NL - 1) {
                            tn = read_t(stage, j + 1);
                            svn = read_s(stage, j + 1);
                        } else {
                            hand_over(kb, stage);
                            tn = read_t(nstage, 0);
                            svn = read_s(nstage, 0);
                            wgn = wsc[kb + 1];
                            wun = wsc[64 + kb + 1];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            __builtin_amdgcn_sched_barrier(0);
                            const v4f tc = mfma_fp8(w[i], t, zero);
                            __builtin_amdgcn_sched_barrier(0);
                            if (j == NL - 1) w[i] = read_w(nstage, i);
                            const int jp = (j + NL - 1) % NL;
                            const float f = i < 2 ? fgp : fup;
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[jp][i][v] = __builtin_fmaf(tp[i][v], f, acc[jp][i][v]);
                            tp[i] = tc;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        if (kEarly && j == 0) issue_t(cls, kb - 1 + NS, pstage, 2, 5);
                        if (kEarly && NL > 4 && j >= 1 && j <= 3) issue_w(cls, once, cur, kb + NS, stage, j, j + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        fgp = sv * wg;
                        fup = sv * wu;
                        t = tn;
                        sv = svn;
                    }
                    wg = wgn;
                    wu = wun;
                    stage = nstage;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[NL - 1][i][v] = __builtin_fmaf(tp[i][v], i < 2 ? fgp : fup, acc[NL - 1][i][v]);
            }
        };
        const int live = min(8, max(0, (cur.nrows - 128 * wm + 15) >> 4));
        auto kloop = [&](auto cls, auto n) {
            if (ONCE && cur.once) kloop_of(cls, n, BoolC<ONCE>{});
            else kloop_of(cls, n, BoolC<false>{});
        };
        if (cur.nrows > Gemm1B::kRows) {
            if (live > 6) kloop(Gemm1A{}, IntC<8>{});
            else if (live > 4) kloop(Gemm1A{}, IntC<6>{});
            else if (live > 2) kloop(Gemm1A{}, IntC<4>{});
            else kloop(Gemm1A{}, IntC<2>{});
        } else if (cur.nrows > Gemm1C::kRows) {
            if (live > 6) kloop(Gemm1B{}, IntC<8>{});
            else if (live > 4) kloop(Gemm1B{}, IntC<6>{});
            else if (live > 1) kloop(Gemm1B{}, IntC<4>{});
            else if (live == 1) kloop(Gemm1B{}, IntC<1>{});
            else kloop(Gemm1B{}, IntC<0>{});
        } else {
            if (live > 1) kloop(Gemm1C{}, IntC<3>{});
            else if (live == 1) kloop(Gemm1C{}, IntC<1>{});
            else kloop(Gemm1C{}, IntC<0>{});
        }

        // every stage is free (each wave has passed the last block's barrier): the next
        // item's first blocks land under this item's epilogue.  The loads past the last block,
        // which still write zeros into the stages, are waited for first: the stages of an item
        // of another class overlap those of other waves.
        if (more) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            lds_barrier();
            nxt = make_item(r + 1);
            with_class(nxt.nrows, [&](auto cls) { start(cls, nxt); });
        }
        store_c_hilo(acc, reinterpret_cast<float*>(lds + kXch), live, wm, wn, kq, r16, cur.row0, cur.nrows,
                     cur.ng, C, mode & kPrefillThroughF16, c_wide);
        cur = nxt;
    }
}

static int grid_for(long long work) { return (int)(work < 4096 ? work : 4096); }

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_dg1_mu;
int g_dg1_grid[3][kMaxDevices] = {};
}  // namespace

// GEMM1 with the dispatch folded in (and with rin.logits set, T <= kRouteInGemm1MaxT, the
// routing too): a persistent grid of as many workgroups as the device holds at once
// (occupancy x CUs, looked up once per device and kernel; with the 8-wave routing of
// 5 <= T <= 8, one per CU, so that a SIMD routes two tokens, not six), capped by the most
// work items T tokens can have.  Without the routing, topk_ids / topk_w hold the routing;
// with it, the kernel writes them.  It sets the C-range flag word when C goes beyond the
// fp16 range (cleared by the route kernel, or with the routing not cleared at all).
bool launch_gemm1_dispatch(const RouteIn& rin, int* topk_ids, float* topk_w, int T, int offset,
                           const uint8_t* hidden, const float* hs_scale, const uint8_t* w1,
                           const float* s1, int* meta, int4* tiles, int* sorted_tok,
                           float* sorted_w, int* inv, const Intermediate& C,
                           hipStream_t stream) {
    const bool route = rin.logits != nullptr;
    if (T <= 0 || T > (route ? kRouteInGemm1MaxT : kDispatchInGemm1MaxT)) return false;
    if (route && rin.bias == nullptr) return false;
    const int nrw = route ? (T <= 4 ? 4 : 8) : 0;   // routing waves
    const int kind = nrw / 4;                        // 0, 1, 2
    const void* fn = nrw == 8 ? reinterpret_cast<const void*>(gemm1_rstream_dispatch_kernel<8>)
                   : nrw == 4 ? reinterpret_cast<const void*>(gemm1_rstream_dispatch_kernel<4>)
                              : reinterpret_cast<const void*>(gemm1_rstream_dispatch_kernel<0>);
    const int threads = nrw == 8 ? 512 : 256;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return false;
    int resident = 0;
    {
        std::lock_guard<std::mutex> lock(g_dg1_mu);
        int& g = g_dg1_grid[kind][dev];
        if (g == 0) {
            int per_cu = 0, cus = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0) != hipSuccess ||
                hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
                per_cu * cus <= 0)
                return false;
            g = nrw == 8 ? cus : per_cu * cus;
        }
        resident = g;
    }
    const long long items = (long long)(((long long)T * kTopK + 15) / 16 + kEL) * Gemm1Stream<1, 1, false>::kItems;
    const int grid = (int)(items < resident ? items : resident);
    if (nrw == 8)
        launch_kernel(gemm1_rstream_dispatch_kernel<8>, dim3(grid), dim3(512), 0, stream, rin,
                      topk_ids, topk_w, T, offset, hidden, hs_scale, w1, s1, meta, tiles,
                      sorted_tok, sorted_w, inv, C);
    else if (nrw == 4)
        launch_kernel(gemm1_rstream_dispatch_kernel<4>, dim3(grid), dim3(256), 0, stream, rin,
                      topk_ids, topk_w, T, offset, hidden, hs_scale, w1, s1, meta, tiles,
                      sorted_tok, sorted_w, inv, C);
    else
        launch_kernel(gemm1_rstream_dispatch_kernel<0>, dim3(grid), dim3(256), 0, stream, rin,
                      topk_ids, topk_w, T, offset, hidden, hs_scale, w1, s1, meta, tiles,
                      sorted_tok, sorted_w, inv, C);
    return true;
}

// Variants (the tile height of the dispatch they expect, and the form of C they write):
//   1  register-staged streaming, 1 row block per item    16-row tiles   fp16 (+ exponents)
//   2  register-staged, 2 row blocks x 2 column groups   32-row tiles   fp16 (+ exponents)
//   4  prefill, 8 waves, 256 x 256 workgroup tile        256-row tiles  fp8 hi/lo
//   7  register-staged weights, token rows shared in LDS  64-row tiles   fp16 (+ exponents)
//   8  variant 7 with three workgroups per CU (more loads in flight, more L2 pressure)
// (variant 5, the dispatch folded into variant 1, has its own launcher)
bool launch_gemm1(int variant, const uint8_t* hidden, const TokenScales& sa, int T,
                  const uint8_t* w1, const float* s1, const int4* tiles, const int* num_tiles,
                  const int* exp_off, int max_tiles, const int* sorted_tok, const Intermediate& C,
                  bool ranked, bool through_f16, hipStream_t stream) {
    int* c_wide = const_cast<int*>(exp_off) + kCWideFlag;   // meta word, cleared by the route kernel
    const int prefill_grid = 256;   // one resident workgroup per CU (LDS-bound)
    constexpr int G = kI / 16;      // 16-column groups
    const long long mt = max_tiles;
    switch (variant) {
        case 1:
            launch_kernel((gemm1_rstream_kernel<4, 1, 1, false>), dim3(grid_for(mt * G)), dim3(256), 0, stream,
                               hidden, sa, T, w1, s1, tiles, num_tiles, sorted_tok, C, c_wide);
            return true;
        case 2:
            launch_kernel((gemm1_rstream_kernel<2, 2, 2, true>), dim3(grid_for(mt * G / 2)), dim3(256), 0, stream,
                               hidden, sa, T, w1, s1, tiles, num_tiles, sorted_tok, C, c_wide);
            return true;
        case 7: {   // 4-wave workgroups, two resident per CU (registers)
            const long long items = mt * Gemm1Shared<2, 4>::kItems;
            launch_kernel((gemm1_shared_kernel<2, 4, 1>), dim3((int)(items < 768 ? items : 768)), dim3(256), 0,
                               stream, hidden, sa, T, w1, s1, tiles, num_tiles, sorted_tok, C, c_wide);
            return true;
        }
        case 8: {   // the same held to three resident per CU
            const long long items = mt * Gemm1Shared<2, 4>::kItems;
            launch_kernel((gemm1_shared_kernel<2, 4, 3>), dim3((int)(items < 768 ? items : 768)), dim3(256), 0,
                               stream, hidden, sa, T, w1, s1, tiles, num_tiles, sorted_tok, C, c_wide);
            return true;
        }
        case 4: {
            const int mode = (ranked ? kPrefillRanked : 0) | (through_f16 ? kPrefillThroughF16 : 0);
            if (T <= kOnceMaxT)
                launch_kernel(gemm1_prefill8_kernel<true>, dim3(prefill_grid), dim3(512), 0, stream, hidden, sa, T,
                                   w1, s1, tiles, num_tiles, exp_off, sorted_tok, C, mode, c_wide);
            else
                launch_kernel(gemm1_prefill8_kernel<false>, dim3(prefill_grid), dim3(512), 0, stream, hidden, sa, T,
                                   w1, s1, tiles, num_tiles, exp_off, sorted_tok, C, mode, c_wide);
            return true;
        }
        default: return false;
    }
}

}  // namespace moe
