// conv_tile.h - an implicit-GEMM conv launch's arguments and its split-K reduction (the
// fp32 tiles of conv_igemm.hip and the split-bf16 ones of conv_split.h), and the accumulator
// start and store of waves that hold 32x32 blocks (conv_igemm.hip).
#pragma once
#include "mfma_core.h"
#include "spinn_hip_internal.h"

namespace spinn {

struct ConvKArgs {
    const float *wpk;  // packed W^T: [group][K][ldw]
    int64_t wpk_group_stride;
    int ldw;
    int M, K;          // per group
    ConvGeom geom;
    float *__restrict__ y;
    const float *__restrict__ bias;
    const float *__restrict__ res;
    uint32_t res_bytes; // extent of res (the output's size)
    int act;
    int OC, OHW;
    float *__restrict__ ws; // split-K partials [split][OC][ntot]
    int k_chunk;       // K per split (multiple of kBK)
};

// Accumulator start values of a conv output tile: bias + residual when
// `terms` (their loads then overlap the K loop's prologue instead of arriving
// as one burst of reads after it, and the epilogue only applies the activation
// and stores; the sum is the reference's acc + bias + residual in another
// order, within fp32 rounding), else zero.
template <class WT>
__device__ __forceinline__ void conv_acc_start(const ConvKArgs &a, int group, int m0, int n0, int wm0, int wn0,
                                               int lane, bool terms, f32x16 (&c)[WT::TM][WT::TN]) {
    if (!terms) {
        ZeroAcc{}(c);
        return;
    }
    // Unconditional buffer loads: a missing bias or residual is a zero-sized
    // resource and rows or columns past the edge read at kOOB, all of which
    // return 0.
    const int h = lane >> 5;
    const int l32 = lane & 31;
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(a.bias ? a.bias + group * a.M : a.y, a.bias ? (uint32_t)a.M * 4u : 0u);
    const __amdgpu_buffer_rsrc_t rr = make_rsrc(a.res ? a.res : a.y, a.res ? a.res_bytes : 0u);
#pragma unroll
    for (int j = 0; j < WT::TN; ++j) {
        const int jcol = n0 + wn0 + j * 32 + l32;
        const bool col_ok = jcol < a.geom.ntot;
        const int img = jcol / a.OHW;
        const int p = jcol - img * a.OHW;
        const uint32_t ybase = ((uint32_t)img * a.OC + (uint32_t)(group * a.M)) * a.OHW + p;
#pragma unroll
        for (int i = 0; i < WT::TM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                const bool ok = m < a.M;
                const float bv = buf_f32(rb, ok ? (uint32_t)m * 4u : kOOB);
                const float rv = buf_f32(rr, ok && col_ok ? (ybase + (uint32_t)m * a.OHW) * 4u : kOOB);
                c[i][j][r] = bv + rv;
            }
    }
}

// Post-op and store of a finished conv output tile (accumulators already hold
// bias + residual). Lane owns columns n0 + wn0 + j*32 + lane%32 and rows
// m0 + wm0 + i*32 + 8*(r/4) + 4*(lane/32) + r%4.
template <class WT, int AC>
__device__ __forceinline__ void conv_store(const ConvKArgs &a, int group, int m0, int n0, int wm0, int wn0, int lane,
                                           const f32x16 (&acc)[WT::TM][WT::TN]) {
    const int h = lane >> 5;
    const int l32 = lane & 31;
    // A tile whose rows all exist (the usual case: OC a multiple of the tile)
    // stores without a per-element row test.
    const bool full_m = m0 + WT::WM * WT::WAVES_M <= a.M;
#pragma unroll
    for (int j = 0; j < WT::TN; ++j) {
        const int jcol = n0 + wn0 + j * 32 + l32;
        if (jcol >= a.geom.ntot) continue;
        const int img = jcol / a.OHW;
        const int p = jcol - img * a.OHW;
        float *yp = a.y + ((int64_t)img * a.OC + (int64_t)group * a.M + m0 + wm0 + 4 * h) * a.OHW + p;
        if (full_m) {
#pragma unroll
            for (int i = 0; i < WT::TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    yp[(int64_t)(i * 32 + 8 * (r >> 2) + (r & 3)) * a.OHW] = apply_act_c<AC>(acc[i][j][r]);
        } else {
#pragma unroll
            for (int i = 0; i < WT::TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int mo = i * 32 + 8 * (r >> 2) + (r & 3);
                    if (m0 + wm0 + 4 * h + mo < a.M) yp[(int64_t)mo * a.OHW] = apply_act_c<AC>(acc[i][j][r]);
                }
        }
    }
}

// Sum split-K partials in split order and apply the conv epilogue (conv_igemm.hip).
int launch_conv_splitk_reduce(int nsplit, const ConvKArgs &a, hipStream_t st);

} // namespace spinn
