// gemm2_class.hip -- prefill GEMM2 by row classes, for T <= kGemm2ClassMaxT (host_plan.h).
//
// The tiles, MFMAs and fp32 sums of gemm2_prefill8_kernel (gemm2.hip: 128 C rows x 256 columns,
// C hi and lo against W2, bit-identical rows), for calls whose experts hold few rows.  There the
// kernel is bound by the misses a CU keeps in flight, and the two-stage kernel waits each K
// block out: its stages are sized for 128 rows whatever the item has.  Three things differ:
//   - an item's rows pick its class, and with it how many K blocks of operands the LDS holds
//     (below), so an item of few rows has up to three blocks in flight behind the one in use;
//     with two stages the W2 stage is handed over as soon as every wave holds its fragments;
//   - consecutive items of one class share one ring: the last K blocks of an item load the
//     first of the next, with no drain between them;
//   - W2 rows of an expert that fits one tile are read once and loaded non-temporal, which
//     leaves L2 to C, that all column groups read.
// The K loop has no branch on what is left to load: past the end of an item's stream the
// buffers have no bytes, so the count of loads in flight, and each wait, stay constants.
// Measured (GEMM2 alone, us, before -> after): 24 experts x 16 rows 72 -> 63; T = 1024, two
// routings 101 -> 98 and 99.5 -> 94; whole calls T = 600, 800, 1024 (four routings each) 2.6,
// 2.2 and 2.6% faster (T = 1024: 239.8 -> 233.9 us), T = 1400 even, T = 2000 and 2500 1.2 and 0.4% slower (heavier items:
// more barriers per K block and the non-temporal form's second K loops), so variant 5 stays
// beyond.
#include "gemm2_rows.h"

#include <algorithm>

namespace moe {

// Row class of an item: stages of 2 C halves + 32 KB of W2 rows each.
//   A   65 .. 128 rows  2 stages, 32 KB of C rows
//   B   25 ..  64 rows  3 stages, 16 KB
//   C    1 ..  24 rows  4 stages,  6 KB
template <int NS, int ROWS, int NC>
struct Gemm2Class {
    static constexpr int kNS = NS;                     // stages
    static constexpr int kNC = NC;                     // C-row loads per wave and K block
    static constexpr int kRows = ROWS;
    static constexpr int kSlots = (ROWS + 63) / 64 + 1;   // 64-row slots of C scales, and one for zeros
    static constexpr int kC = ROWS * kBlk;             // bytes per C half
    static constexpr int kW = 256 * kBlk;
    static constexpr int kCBase = NS * kW;             // W2 stages first
    static constexpr int kScaBase = kCBase + NS * 2 * kC;
    static constexpr int kBytes = kScaBase + NS * kSlots * 256;
    static constexpr int kVmC = NC + 1;                // C loads per wave and K block
    static constexpr int kVm = 4 + kVmC;
};
using ClassA = Gemm2Class<2, 128, 4>;
using ClassB = Gemm2Class<3, 64, 2>;
using ClassC = Gemm2Class<4, 24, 1>;

struct ClassItem {   // all uniform
    const uint8_t *hi, *lo, *w;
    const float* cs;
    uint32_t csbytes;
    int le, row0, nrows, hg;
    bool once;
};

__global__ __launch_bounds__(512, 1) void gemm2_class_kernel(
    Intermediate C, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int4* __restrict__ tiles, const int* __restrict__ num_tiles,
    const int* __restrict__ exp_off, ExpertRows rows, int* __restrict__ rows_wide) {
    constexpr int BM = 128;
    constexpr int NG = kH / 256;                // 28 column groups
    constexpr int kItemCap = 32;                // per-workgroup item table (12 items at most at T = kGemm2ClassMaxT)
    constexpr int kPool = std::max({ClassA::kBytes, ClassB::kBytes, ClassC::kBytes});
    constexpr int kWsc = kPool, kItems = kWsc + 2 * 256;
    // one LDS object: the stages, two items' W2 scales, the item table
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kItems + kItemCap * sizeof(int4) + kEL * 4];
    static_assert(sizeof(lds) <= 160 * 1024, "LDS of a CU");
    int4* const s_items = reinterpret_cast<int4*>(lds + kItems);
    int* const s_rows = reinterpret_cast<int*>(s_items + kItemCap);

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
    constexpr uint32_t kNothing = 0xfffffff0u;   // an offset past every buffer: moves nothing
    const __amdgpu_buffer_rsrc_t rs_s2 = buffer_rsrc(s2, kEL * kHB * kIB * 4);
    // lane offsets of a wave's DMA, the same for every item: W2 row 32 wave + 8 i + drow of the
    // item's 256, and row drow of an 8-row block of C rows (the block's own rows added per load)
    uint32_t woff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 32 * wave + 8 * i + drow;
        woff[i] = (uint32_t)r * kI + ((dchunk ^ swz128(r)) << 4);
    }

    const int nr = prefill_items<BM>(s_items, kItemCap, nitems, NG, base, G, tiles, exp_off);
    if (nr == 0) return;   // uniform: the whole workgroup has no item
    if (threadIdx.x < kEL) s_rows[threadIdx.x] = exp_off[threadIdx.x + 1] - exp_off[threadIdx.x];
    __syncthreads();

    auto make_item = [&](int r) {
        const int4 m = prefill_item<BM>(s_items, kItemCap, r, NG, base, G, tiles, exp_off);
        ClassItem it;
        it.le = m.x;
        it.row0 = m.y;
        it.nrows = m.z;
        it.hg = m.w;
        it.once = __builtin_amdgcn_readfirstlane(s_rows[m.x]) <= BM;
        it.hi = C.hi() + (size_t)it.row0 * kI;
        it.lo = C.lo() + (size_t)it.row0 * kI;
        it.cs = C.scales + it.row0;
        it.csbytes = (uint32_t)(kIB * C.rows_cap - it.row0) * 4;
        it.w = w2 + ((size_t)it.le * kH + it.hg * 256) * kI;
        return it;
    };
    // the item's W2 block scales, 16 for each half of its columns, by DMA into buffer r & 1
    auto fetch_scales = [&](const ClassItem& it, int r) {
        if (wave == 7)
            bdma4(rs_s2, (uint32_t)((it.le * kHB + 2 * it.hg) * kIB + min(lane, 2 * kIB - 1)) * 4, 0,
                  lds + kWsc + (r & 1) * 256);
    };
    // K block f of the stream that `cur` and, where it goes on into `nxt`, its blocks make, into
    // a stage; past the stream's end the buffers have no bytes: nothing moves, and the loads in
    // flight stay the same without a branch in the K loop
    auto issue_w = [&](auto cls, auto once, const ClassItem& cur, const ClassItem& nxt, bool cont, int f, int stage, int i0 = 0, int i1 = 4) {
        using Cl = decltype(cls);
        const bool own = f < kIB;
        const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(own ? cur.w : nxt.w, own || cont ? 256 * kI : 0);
        const uint32_t k = (uint32_t)(own ? f : f - kIB) * kBlk;
#pragma unroll
        for (int i = i0; i < i1; ++i) bdma16<decltype(once)::value ? kNonTemporal : 0>(rs, woff[i], k, lds + stage * Cl::kW + (32 * wave + 8 * i) * kBlk);
    };
    auto issue_c = [&](auto cls, const ClassItem& cur, const ClassItem& nxt, bool cont, int f, int stage) {
        using Cl = decltype(cls);
        const bool own = f < kIB, on = own || cont;
        const int nrows = own ? cur.nrows : nxt.nrows;
        const uint32_t k = (uint32_t)(own ? f : f - kIB) * kBlk;
        uint8_t* const st = lds + Cl::kCBase + stage * 2 * Cl::kC;
        // 8-row blocks, hi then lo; rows past the tile lie past the buffer and move nothing
        const __amdgpu_buffer_rsrc_t rh = buffer_rsrc(own ? cur.hi : nxt.hi, on ? nrows * kI : 0);
        const __amdgpu_buffer_rsrc_t rl = buffer_rsrc(own ? cur.lo : nxt.lo, on ? nrows * kI : 0);
        auto row_off = [&](int q) { return (uint32_t)(8 * q + drow) * kI + ((dchunk ^ swz128(8 * q + drow)) << 4); };
        if constexpr (Cl::kNC >= 2) {
#pragma unroll
            for (int i = 0; i < Cl::kNC / 2; ++i) {
                const int q = Cl::kNC / 2 * wave + i;
                bdma16(rh, row_off(q), k, st + 8 * q * kBlk);
                bdma16(rl, row_off(q), k, st + Cl::kC + 8 * q * kBlk);
            }
        } else {   // waves 0 .. 2 hi, 3 .. 5 lo (6 and 7 the last block again)
            constexpr int NB = Cl::kRows / 8;
            const int q = min(wave, 2 * NB - 1) % NB;
            const bool half = wave >= NB;
            bdma16(half ? rl : rh, row_off(q), k, st + (half ? Cl::kC : 0) + 8 * q * kBlk);
        }
        const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(own ? cur.cs : nxt.cs, on ? (own ? cur.csbytes : nxt.csbytes) : 0u);
        bdma4(rs, 64 * wave < nrows && wave < Cl::kSlots - 1 ? (uint32_t)(64 * wave + min(lane, nrows - 1 - 64 * wave)) * 4 : kNothing,
              (uint32_t)(own ? f : f - kIB) * C.rows_cap * 4,
              lds + Cl::kScaBase + (stage * Cl::kSlots + min(wave, Cl::kSlots - 1)) * 256);
    };
    auto with_class = [&](int nrows, auto&& f) {
        if (nrows > ClassB::kRows) f(ClassA{});
        else if (nrows > ClassC::kRows) f(ClassB{});
        else f(ClassC{});
    };
    auto class_of = [](int nrows) { return nrows > ClassB::kRows ? 0 : nrows > ClassC::kRows ? 1 : 2; };
    auto start = [&](const ClassItem& it) {   // the item's first stages
        with_class(it.nrows, [&](auto cls) {
#pragma unroll
            for (int k = 0; k < decltype(cls)::kNS; ++k) {
                if (it.once) issue_w(cls, BoolC<true>{}, it, it, false, k, k);
                else issue_w(cls, BoolC<false>{}, it, it, false, k, k);
                issue_c(cls, it, it, false, k, k);
            }
        });
    };

    ClassItem cur = make_item(0), nxt = cur;
    fetch_scales(cur, 0);
    start(cur);
    int stage = 0;            // of the current K block
    bool fresh = true;        // the item's first blocks were issued by start()
    for (int r = 0; r < nr; ++r) {
        const bool more = r + 1 < nr;
        if (more) nxt = make_item(r + 1);
        // the stream goes on into an item of the same class
        const bool cont = more && class_of(nxt.nrows) == class_of(cur.nrows);
        const float* const wsc = reinterpret_cast<const float*>(lds + kWsc + (r & 1) * 256) + (wn >> 1) * kIB;
        v4f acc[4][4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[s][n] = zero;

        // NL: 16-row blocks of this wave that exist
        auto kloop_of = [&](auto cls, auto live, auto once) {
            using Cl = decltype(cls);
            constexpr int NL = decltype(live)::value;
            constexpr int NS = Cl::kNS;
            auto rd = [&](const uint8_t* rp) {
                const v4u x0 = *reinterpret_cast<const v4u*>(rp + c0);
                const v4u x1 = *reinterpret_cast<const v4u*>(rp + c1);
                return v8i{(int)x0[0], (int)x0[1], (int)x0[2], (int)x0[3], (int)x1[0], (int)x1[1], (int)x1[2], (int)x1[3]};
            };
            auto read_c = [&](int st, int half, int s) {
                return rd(lds + Cl::kCBase + (st * 2 + half) * Cl::kC + (64 * wm + 16 * s) * kBlk);
            };
            auto read_s = [&](int st, int s) {
                return reinterpret_cast<const float*>(lds + Cl::kScaBase + st * Cl::kSlots * 256)[64 * wm + 16 * s + r16];
            };
            auto read_w = [&](int st, int n) { return rd(lds + st * Cl::kW + (64 * wn + 16 * n) * kBlk); };
            // kEarly (two stages): the W2 stage is handed over by a barrier of its own, as soon
            // as every wave holds the block's W2 fragments
            constexpr bool kEarly = NS == 2;
            auto free_weights = [&](int kb) {
                __builtin_amdgcn_sched_barrier(0);
                lds_barrier();
                if (NL < 4) issue_w(cls, once, cur, nxt, cont, kb + NS, stage);
                __builtin_amdgcn_sched_barrier(0);
            };
            // every wave has read its last C fragments of K block kb, and block kb + 1 has landed
            // for every wave: the stage goes to block kb + NS
            auto hand_over = [&](int kb) {
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(kEarly ? 4 : (NS - 2) * Cl::kVm));
                lds_barrier();
                if (!kEarly) issue_w(cls, once, cur, nxt, cont, kb + NS, stage);
                issue_c(cls, cur, nxt, cont, kb + NS, stage);
                __builtin_amdgcn_sched_barrier(0);
            };
            if (fresh) {
                __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * Cl::kVm));
                lds_barrier();
            }
            if (more) fetch_scales(nxt, r + 1);
            if constexpr (NL == 0) {
#pragma unroll 1
                for (int kb = 0; kb < kIB; ++kb) {
                    if (kEarly) free_weights(kb);
                    hand_over(kb);
                    stage = stage + 1 == NS ? 0 : stage + 1;
                }
            } else {
                v8i w[4];
                v8i ch = read_c(stage, 0, 0), cl = read_c(stage, 1, 0);
                float sv = read_s(stage, 0);
#pragma unroll
                for (int n = 0; n < 4; ++n) w[n] = read_w(stage, n);
                float sw = wsc[0];
                v4f tp[4];
                float fp = 0.f;
#pragma unroll
                for (int n = 0; n < 4; ++n) tp[n] = zero;
#pragma unroll 1
                for (int kb = 0; kb < kIB; ++kb) {
                    const int nstage = stage + 1 == NS ? 0 : stage + 1;
                    float swn = 0.f;
#pragma unroll
                    for (int s = 0; s < NL; ++s) {
                        const bool last = s == NL - 1;
                        if (kEarly && s == (NL > 1 ? 1 : 0)) free_weights(kb);
                        v8i chn, cln;
                        float svn;
                        if (last) {
                            hand_over(kb);
                            chn = read_c(nstage, 0, 0);
                            svn = read_s(nstage, 0);
                            swn = wsc[(kb + 1) & (kIB - 1)];
                        } else {
                            chn = read_c(stage, 0, s + 1);
                            svn = read_s(stage, s + 1);
                        }
                        cln = last ? read_c(nstage, 1, 0) : read_c(stage, 1, s + 1);
                        v4f tc[4];
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            __builtin_amdgcn_sched_barrier(0);
                            tc[n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[n], ch, zero, 0, 0, 0, 0, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                            const int sp = (s + NL - 1) % NL;
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[sp][n][v] = __builtin_fmaf(tp[n][v], fp, acc[sp][n][v]);
                        }
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            __builtin_amdgcn_sched_barrier(0);
                            tc[n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[n], cl, tc[n], 0, 0, 0, 127, 0, 123);
                            __builtin_amdgcn_sched_barrier(0);
                            if (last) w[n] = read_w(nstage, n);
                            else if (kEarly && NL == 4 && s >= 1 && n < 2) issue_w(cls, once, cur, nxt, cont, kb + NS, stage, 2 * (s - 1) + n, 2 * (s - 1) + n + 1);
                        }
#pragma unroll
                        for (int n = 0; n < 4; ++n) tp[n] = tc[n];
                        fp = sv * sw;
                        ch = chn;
                        cl = cln;
                        sv = svn;
                    }
                    sw = swn;
                    stage = nstage;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[NL - 1][n][v] = __builtin_fmaf(tp[n][v], fp, acc[NL - 1][n][v]);
            }
        };
        const int live = live_blocks(64 * wm, cur.nrows);
        auto kloop = [&](auto cls, auto n) {
            if (cur.once) kloop_of(cls, n, BoolC<true>{});
            else kloop_of(cls, n, BoolC<false>{});
        };
        with_class(cur.nrows, [&](auto cls) {
            with_live_blocks(live, [&](auto n) {
                if constexpr (decltype(n)::value * 16 < decltype(cls)::kRows + 16) kloop(cls, n);
            });
        });
        // an item of another class starts a ring of its own: every stage is free (each wave has
        // passed the last block's barrier, and the loads past the stream's end, which still write
        // zeros, are waited for), and its first blocks land under this epilogue
        fresh = !cont;
        if (more && !cont) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            lds_barrier();
            start(nxt);
            stage = 0;
        }

        store_prefill_rows(acc, rows, rows_wide, cur.row0, cur.nrows, cur.hg, wm, wn, r16, kq);
        cur = nxt;
    }
}

void launch_gemm2_class(const Intermediate& C, int* flags, const uint8_t* w2, const float* s2,
                        const int4* tiles, const int* num_tiles, const int* exp_off,
                        const ExpertRows& rows, hipStream_t stream) {
    launch_kernel(gemm2_class_kernel, dim3(256), dim3(512), 0, stream, C, w2, s2, tiles, num_tiles,
                  exp_off, rows, flags + 1);
}

}  // namespace moe
