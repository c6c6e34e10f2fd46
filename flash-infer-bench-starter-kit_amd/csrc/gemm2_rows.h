// gemm2_rows.h -- the prefill GEMM2s' epilogue: a wave's 64 rows x 64 columns of fp32 sums
// to the fp16 expert rows.
#pragma once

#include "moe_device.h"

namespace moe {

// Wave (wm, wn) of the 128 x 256 tile at row0, column group hg (nrows rows exist).
__device__ __forceinline__ void store_prefill_rows(
    const v4f (&acc)[4][4], const ExpertRows& rows, int* rows_wide, int row0, int nrows, int hg,
    int wm, int wn, int r16, int kq) {
    // lane holds D[h = 64 wn + 16 n + 4 kq + v][row = 64 wm + 16 s + r16]
    float mx = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, fabsf(acc[s][n][v]));
    if (!beyond_f16_in_wave(mx)) {
        // the usual case: plain fp16, and the 4 zero exponents of a row's 64 columns
        // as one 4-byte store (lane kq = 0 of the row).  The fp16 pairs of column
        // blocks (0, 1) and (2, 3) are exchanged across the row's 4 lanes (lanes l,
        // l+16, l+32, l+48: a 32-lane then a 16-lane swap) so that lane kq holds
        // columns 8 kq .. 8 kq + 7 of the pair: one 16-byte store writes 64
        // consecutive bytes of the row.
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int rr = 64 * wm + 16 * s + r16;
            uint32_t w[4][2];
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    w[n][q] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)acc[s][n][2 * q]) |
                              ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)acc[s][n][2 * q + 1]) << 16);
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {
                const int a = 2 * pr, b = 2 * pr + 1;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const auto p = __builtin_amdgcn_permlane32_swap(w[a][q], w[b][q], false, false);
                    w[a][q] = p[0];
                    w[b][q] = p[1];
                }
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const auto p = __builtin_amdgcn_permlane16_swap(w[a][q], w[b][q], false, false);
                    w[a][q] = p[0];
                    w[b][q] = p[1];
                }
            }
            if (rr >= nrows) continue;   // after the swaps: every lane takes part
            const size_t row = (size_t)(row0 + rr);
            const int c0 = hg * 256 + 64 * wn;
#pragma unroll
            for (int pr = 0; pr < 2; ++pr)
                *reinterpret_cast<v4u*>(rows.f16 + row * kH + c0 + 32 * pr + 8 * kq) =
                    v4u{w[2 * pr][0], w[2 * pr][1], w[2 * pr + 1][0], w[2 * pr + 1][1]};
            if (kq == 0) *reinterpret_cast<uint32_t*>(rows.exp + row * (kH / kGroup16) + c0 / kGroup16) = 0u;
        }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int rr = 64 * wm + 16 * s + r16;
#pragma unroll
            for (int n = 0; n < 4; ++n)
                store_rows4(rows, rows_wide, row0 + rr, hg * 256 + 64 * wn + 16 * n + 4 * kq,
                            acc[s][n], rr < nrows);
        }
    }
}

}  // namespace moe
