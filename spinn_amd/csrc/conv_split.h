// conv_split.h - implicit-GEMM convolution on the bf16 matrix cores (split_core.h).
//
// M = output channels of a group, N = batch*OH*OW output pixels, K in (kh, kw, c)
// order with each tap's channels padded to whole octets, so the 8 values a thread
// gathers for one run of LDS share a tap.
#pragma once
#include "conv_tile.h"
#include "split_core.h"
#include "streamk.h"
#include <type_traits>

namespace spinn {

struct ConvSplitArgs {
    ConvKArgs t;
    SplitPlanes w;            // group 0
    int64_t w_group_stride;   // bytes
    int co8;                  // octets per tap
    int groups_k;             // K in groups of slices
    int chunk;                // groups per K split
    int tap_order;            // t.wpk (fp32 W^T) has K in (kh, kw, c) order, else (c, kh, kw)
};

template <int CW> struct SplitVec;
template <> struct SplitVec<1> { typedef float type; };
template <> struct SplitVec<2> { typedef f32x2 type; };
template <> struct SplitVec<4> { typedef f32x4 type; };

template <int CW>
__device__ __forceinline__ void buf_load_cw(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, float (&v)[CW]) {
    if constexpr (CW == 1) {
        v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
    } else if constexpr (CW == 2) {
        const f32x2 t = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
        v[0] = t[0];
        v[1] = t[1];
    } else {
        const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = t[i];
    }
}

// B operand loaders. fetch() loads the thread's share of the next group of slices (16
// values) into a stage, split() turns values 2q, 2q + 1 of item i into their parts, store()
// writes an item's three runs to LDS; a group has kSplitGS items per thread.

// 1x1 stride-1 unpadded conv over planes of an even pixel count, 8-byte aligned input and
// C/g a multiple of 8: 2 neighbouring pixels and 8 channels per thread, 8-byte loads.
struct SplitPw2 {
    static constexpr int CW = 2;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off; // byte offset of the thread's first pixel at channel 0; kOOB past the last
    uint32_t hw4;
    uint32_t lost = 0; // split2
    int oct;      // channel octet of the next fetch
    int co8;
    struct Stage {
        float r[8][2];
    };
    __device__ __forceinline__ void init(const ConvSplitArgs &a, int n0, int group, int tid, int g0) {
        const ConvGeom &g = a.t.geom;
        rsrc = make_rsrc(g.x, g.x_bytes);
        hw4 = (uint32_t)(g.H * g.W) * 4u;
        co8 = a.co8;
        PixelOrigin px;
        px.init(g, n0 + (tid & 31) * 2, group);
        off = px.valid ? (px.base + (uint32_t)(px.ih0 * g.W + px.iw0)) * 4u : kOOB;
        oct = g0 * (4 * kSplitGS) + (tid >> 5);
    }
    // Octets past the last read zeros (not another image's channels: those may be infinite).
    __device__ __forceinline__ void fetch(Stage &st) {
        const uint32_t v = oct < co8 ? off + (uint32_t)oct * (8u * hw4) : kOOB;
#pragma unroll
        for (int e = 0; e < 8; ++e) buf_load_cw<2>(rsrc, v, (uint32_t)e * hw4, st.r[e]);
        oct += 4 * kSplitGS;
    }
    __device__ __forceinline__ void split(const Stage &st, int i, int q, u32x4 (&p)[3]) {
        uint32_t h, m, l;
        split2(st.r[2 * q][i], st.r[2 * q + 1][i], h, m, l, lost);
        p[0][q] = h;
        p[1][q] = m;
        p[2][q] = l;
    }
    __device__ __forceinline__ void store(const u32x4 (&p)[3], int i, u32x4 *lds, int tid) const {
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) lds[split_at(pl, tid >> 5, i * 32 + (tid & 31))] = p[pl];
    }
};

// Any other conv: item i is octet wave + 4i of the group, one pixel per lane, so an octet's
// tap and channel are the same for a whole wave (scalars) and a lane keeps its window's
// byte offset. TAIL: C/g not a multiple of 8.
template <bool TAIL>
struct SplitGather {
    static constexpr int CW = 1;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off; // byte offset of (image, group channel 0, window origin)
    int ih0, iw0; // window origin; ih0 far outside the image past the last pixel
    uint32_t hw4;
    uint32_t lost = 0; // split2
    int H, W, KH, KW, Cg, co8;
    int co[kSplitGS], kh[kSplitGS], kw[kSplitGS]; // next octet to fetch
    struct Stage {
        float r[kSplitGS][8];
        int live[kSplitGS]; // channels of the octet that exist
    };
    __device__ __forceinline__ void init(const ConvSplitArgs &a, int n0, int group, int tid, int g0) {
        const ConvGeom &g = a.t.geom;
        rsrc = make_rsrc(g.x, g.x_bytes);
        H = g.H;
        W = g.W;
        KH = g.KH;
        KW = g.KW;
        Cg = g.Cg;
        co8 = a.co8;
        hw4 = (uint32_t)(g.H * g.W) * 4u;
        PixelOrigin px;
        px.init(g, n0 + (tid & 63), group);
        ih0 = px.valid ? px.ih0 : INT32_MIN / 2;
        iw0 = px.iw0;
        off = (px.base + (uint32_t)(px.ih0 * g.W + px.iw0)) * 4u;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
        for (int i = 0; i < kSplitGS; ++i) {
            const int o = (g0 * kSplitGS + i) * 4 + wave;
            const int tap = o / co8;
            co[i] = o - tap * co8;
            kh[i] = tap / KW;
            kw[i] = tap - kh[i] * KW;
        }
    }
    // Octets past the window read zeros.
    __device__ __forceinline__ void fetch(Stage &st) {
#pragma unroll
        for (int i = 0; i < kSplitGS; ++i) {
            const int ih = ih0 + kh[i], iw = iw0 + kw[i];
            const bool ok = kh[i] < KH && (unsigned)ih < (unsigned)H && (unsigned)iw < (unsigned)W;
            const uint32_t v = ok ? off + (uint32_t)(kh[i] * W + kw[i]) * 4u + (uint32_t)co[i] * (8u * hw4) : kOOB;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                st.r[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)v, (int)(e * hw4), 0));
            if constexpr (TAIL) st.live[i] = Cg - co[i] * 8;
            // at most four taps further (co8 >= 2), without a branch inside the K loop
            co[i] += 4 * kSplitGS;
#pragma unroll
            for (int t = 0; t < 2 * kSplitGS; ++t) {
                const int over = co[i] >= co8 ? 1 : 0;
                co[i] -= over ? co8 : 0;
                kw[i] += over;
                const int row = kw[i] == KW ? 1 : 0;
                kw[i] = row ? 0 : kw[i];
                kh[i] += row;
            }
        }
    }
    __device__ __forceinline__ void split(const Stage &st, int i, int q, u32x4 (&p)[3]) {
        float v0 = st.r[i][2 * q], v1 = st.r[i][2 * q + 1];
        if constexpr (TAIL) {
            v0 = 2 * q < st.live[i] ? v0 : 0.f;
            v1 = 2 * q + 1 < st.live[i] ? v1 : 0.f;
        }
        uint32_t h, m, l;
        split2(v0, v1, h, m, l, lost);
        p[0][q] = h;
        p[1][q] = m;
        p[2][q] = l;
    }
    __device__ __forceinline__ void store(const u32x4 (&p)[3], int i, u32x4 *lds, int tid) const {
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) lds[split_at(pl, (tid >> 6) + 4 * i, tid & 63)] = p[pl];
    }
};

// Accumulator start values of a wave's blocks: bias + residual when `terms`, else zero
// (their loads overlap the K loop's prologue). Missing terms are zero-sized resources,
// rows and columns past the edge read at kOOB: both give 0.
template <class T, bool RES>
__device__ __forceinline__ void split_acc_start(const ConvKArgs &a, int group, int m0, int n0, int lane, bool terms,
                                                f32x4 (&c)[T::TM][T::TN]) {
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(a.bias ? a.bias + group * a.M : a.y, a.bias && terms ? (uint32_t)a.M * 4u : 0u);
    const __amdgpu_buffer_rsrc_t rr = make_rsrc(RES ? a.res : a.y, RES && terms ? a.res_bytes : 0u);
    const int h = lane >> 4;
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + i * 16 + 4 * h + r;
            const float b = buf_f32(rb, m < a.M ? (uint32_t)m * 4u : kOOB);
#pragma unroll
            for (int j = 0; j < T::TN; ++j) c[i][j][r] = b;
        }
    if constexpr (RES) {
#pragma unroll
        for (int q = 0; q < T::NQ; ++q) {
            const int jcol = n0 + T::col0(q, lane);
            const int img = jcol / a.OHW;
            const uint32_t ybase = ((uint32_t)img * a.OC + (uint32_t)(group * a.M)) * a.OHW + (uint32_t)(jcol - img * a.OHW);
#pragma unroll
            for (int i = 0; i < T::TM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + i * 16 + 4 * h + r;
                    float v[T::CW];
                    buf_load_cw<T::CW>(rr, m < a.M && jcol < a.geom.ntot ? (ybase + (uint32_t)m * a.OHW) * 4u : kOOB, 0u, v);
#pragma unroll
                    for (int e = 0; e < T::CW; ++e) c[i][q + e * T::NQ][r] += v[e];
                }
        }
    }
}

// Post-op and store of a wave's finished blocks.
template <class T, int AC>
__device__ __forceinline__ void split_store(const ConvKArgs &a, int group, int m0, int n0, int lane,
                                            const f32x4 (&acc)[T::TM][T::TN]) {
    const int h = lane >> 4;
    const bool full_m = m0 + T::WM <= a.M; // no per-row test
    typedef typename SplitVec<T::CW>::type vec;
#pragma unroll
    for (int q = 0; q < T::NQ; ++q) {
        const int jcol = n0 + T::col0(q, lane);
        if (jcol >= a.geom.ntot) continue;
        const int img = jcol / a.OHW;
        const int p = jcol - img * a.OHW;
        float *yp = a.y + ((int64_t)img * a.OC + (int64_t)group * a.M + m0 + 4 * h) * a.OHW + p;
#pragma unroll
        for (int i = 0; i < T::TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (full_m || m0 + 4 * h + i * 16 + r < a.M) {
                    float v[T::CW];
#pragma unroll
                    for (int e = 0; e < T::CW; ++e) v[e] = apply_act_c<AC>(acc[i][q + e * T::NQ][r]);
                    *reinterpret_cast<vec *>(yp + (int64_t)(i * 16 + r) * a.OHW) = __builtin_bit_cast(vec, v);
                }
    }
}

// A wave's accumulators again on the fp32 MFMA, from the packed fp32 weights, an octet of k
// ahead of its loads' use. Where one wave of a tile has to, it takes about three times the
// time (1x1 1024 -> 256@14x14 at batch 32: 29.5 -> 97 us; with a division per element and
// no loads ahead 177); all waves at once 105 us.
template <class T, bool RES>
__device__ __forceinline__ void split_redo(const ConvSplitArgs &a, int group, int m0, int n0, int g0, int g1, bool terms,
                                           f32x4 (&acc)[T::TM][T::TN], int lane) {
    split_acc_start<T, RES>(a.t, group, m0, n0, lane, terms, acc);
    const ConvGeom &cg = a.t.geom;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(cg.x, cg.x_bytes);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.t.wpk + group * a.t.wpk_group_stride, (uint32_t)a.t.wpk_group_stride * 4u);
    const int taps = cg.KH * cg.KW;
    const uint32_t hw4 = (uint32_t)(cg.H * cg.W) * 4u;
    const int k4 = lane >> 4;
    uint32_t off[T::TN]; // byte offset of (image, group channel 0, window origin)
    int ih0[T::TN], iw0[T::TN];
#pragma unroll
    for (int j = 0; j < T::TN; ++j) {
        PixelOrigin px;
        px.init(cg, n0 + T::col0(j % T::NQ, lane) + j / T::NQ, group);
        ih0[j] = px.valid ? px.ih0 : INT32_MIN / 2;
        iw0[j] = px.iw0;
        off[j] = (px.base + (uint32_t)(px.ih0 * cg.W + px.iw0)) * 4u;
    }
    const int o0 = g0 * (4 * kSplitGS), o1 = min(g1 * (4 * kSplitGS), taps * a.co8);
    int tap = o0 / a.co8, co = o0 - tap * a.co8;
    int kh = tap / cg.KW, kw = tap - kh * cg.KW;
    // octets come in order; those past the last read zeros
    auto load = [&](int, float (&va)[2][T::TM], float (&vb)[2][T::TN]) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int c = co * 8 + 4 * s + k4;
            const bool ok = (tap < taps) & (c < cg.Cg);
            const uint32_t k = (uint32_t)(a.tap_order ? tap * cg.Cg + c : c * taps + tap);
#pragma unroll
            for (int i = 0; i < T::TM; ++i) {
                const int m = m0 + i * 16 + (lane & 15);
                va[s][i] = buf_f32(rw, (ok & (m < a.t.M)) ? (k * (uint32_t)a.t.ldw + (uint32_t)m) * 4u : kOOB);
            }
#pragma unroll
            for (int j = 0; j < T::TN; ++j) {
                const int ih = ih0[j] + kh, iw = iw0[j] + kw;
                const bool in = ok & ((unsigned)ih < (unsigned)cg.H) & ((unsigned)iw < (unsigned)cg.W);
                vb[s][j] = buf_f32(rx, in ? off[j] + (uint32_t)(kh * cg.W + kw) * 4u + (uint32_t)c * hw4 : kOOB);
            }
        }
        if (++co == a.co8) {
            co = 0;
            ++tap;
            if (++kw == cg.KW) {
                kw = 0;
                ++kh;
            }
        }
    };
    fp32_product<T::TM, T::TN>(o0, o1, acc, load);
}

// Groups [g0, g1) (of GS slices) of one output tile into acc; m0: the wave's first row,
// n0 the tile's first column. lost (LDS): the bits that each thread's activations lost.
template <class T, class BL, bool RES>
__device__ __forceinline__ void split_conv_segment(const ConvSplitArgs &a, int group, int m0, int n0, int g0, int g1,
                                                   bool terms, u32x4 (*lds)[kSplitRuns],
                                                   uint32_t *lost, f32x4 (&acc)[T::TM][T::TN], int tid, int lane) {
    constexpr int GS = kSplitGS;
    SplitPlanes w = a.w;
    w.base = (const float *)((const char *)w.base + group * a.w_group_stride);
    PlanesA<T::TM> al;
    al.init(w, m0, lane);
    BL bl;
    bl.init(a, n0, group, tid, g0);
    bf16x8 wa[2][T::TM][3];
    typename BL::Stage st[2];
    f32x4 low[T::TM][T::TN];
    u32x4 parts[3];
    bl.fetch(st[0]);
    split_acc_start<T, RES>(a.t, group, m0, n0, lane, terms, acc);
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int j = 0; j < T::TN; ++j) low[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bl.fetch(st[1]);
#pragma unroll
    for (int c = 0; c < GS; ++c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) bl.split(st[0], c, q, parts);
        bl.store(parts, c, lds[0], tid);
    }
    __builtin_amdgcn_sched_barrier(0);
    al.fetch(g0 * GS, wa[0]);
    bl.fetch(st[0]);
    al.fetch(g0 * GS + 1, wa[1]);
    __syncthreads();
    // Group g from buffer u; stage u ^ 1 holds group g + 1, which is split into the other
    // buffer, and is refilled with group g + 3. Each product's MFMAs are followed by a
    // piece of that work small enough to issue while the matrix pipe runs; the fences
    // keep the compiler from collecting the pieces.
#define SPINN_FENCE __builtin_amdgcn_sched_barrier(0)
    auto run_group = [&](int g, auto uc) {
        constexpr int u = decltype(uc)::value;
        bf16x8 b0[2][3], b1[2][3];
        read_frags<2>(lds[u], 0, 0, lane, b0);
#pragma unroll
        for (int sl = 0; sl < GS; ++sl) {
            const int w_ = sl & 1;
            read_frags<2>(lds[u], sl, 32, lane, b1);
            SPINN_FENCE;
            split_mfma<0, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            bl.split(st[u ^ 1], sl, 0, parts);
            SPINN_FENCE;
            split_mfma<1, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            bl.split(st[u ^ 1], sl, 1, parts);
            SPINN_FENCE;
            split_mfma<2, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            bl.split(st[u ^ 1], sl, 2, parts);
            SPINN_FENCE;
            split_mfma<3, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            bl.split(st[u ^ 1], sl, 3, parts);
            SPINN_FENCE;
            split_mfma<4, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            bl.store(parts, sl, lds[u ^ 1], tid);
            SPINN_FENCE;
            split_mfma<5, T::TM, T::TN, 0, 2>(wa[w_], b0, acc, low);
            SPINN_FENCE;
            if (sl + 1 < GS) read_frags<2>(lds[u], sl + 1, 0, lane, b0);
            SPINN_FENCE;
            split_mfma<0, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            if (sl == GS - 1) bl.fetch(st[u ^ 1]);
            SPINN_FENCE;
            split_mfma<1, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            split_mfma<2, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            split_mfma<3, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            split_mfma<4, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            split_mfma<5, T::TM, T::TN, 2, 2>(wa[w_], b1, acc, low);
            SPINN_FENCE;
            al.fetch(g * GS + sl + 2, wa[w_]);
            SPINN_FENCE;
        }
        lost[tid] = bl.lost; // of group g + 1 and all before it
        __syncthreads();
    };
#undef SPINN_FENCE
    int g = g0;
#pragma unroll 1
    for (; g + 2 <= g1; g += 2) {
        run_group(g, std::integral_constant<int, 0>{});
        run_group(g + 1, std::integral_constant<int, 1>{});
    }
    if (g < g1) run_group(g, std::integral_constant<int, 0>{});
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int j = 0; j < T::TN; ++j) acc[i][j] += low[i][j];
}

// Computes a finished segment again where bf16 parts could not carry it (split_core.h); lost:
// the segment's notes. `after` follows where sums were replaced. The indexes are copies that
// the compiler cannot tell from new ones: it would keep what this shares with the prologue
// in registers over the K loop.
template <class T, bool RES, class After>
__device__ __forceinline__ void split_check(const ConvSplitArgs &a, int group, int m0, int n0, int g0, int g1, bool terms,
                                            f32x4 (&acc)[T::TM][T::TN], const uint32_t *lost, int lane, const After &after) {
    if (__builtin_expect(__any(sums_suspect<T::TM, T::TN>(acc)), 0)) {
        asm volatile("" : "+v"(lane), "+s"(m0), "+s"(n0));
        const uint32_t bits = lost[lane] | lost[64 + lane] | lost[128 + lane] | lost[192 + lane];
        if (__any(sums_bad<T::TM, T::TN>(acc) | ((bits & 0xffffu) != 0u))) {
            split_redo<T, RES>(a, group, m0, n0, g0, g1, terms, acc, lane);
            after();
        }
    }
}

// One workgroup per tile and conv group, or (SPLIT) K split over blockIdx.z with raw
// partial sums to the workspace. A SIMD issues in order, so a lone wave pays for every
// load, LDS access and split operation between its MFMAs: one workgroup per CU takes 1700
// cycles per slice of a 128 x 64 tile whose MFMAs need 770, two per CU 1000 each; larger
// grids are then bound by power (1.8-2.1 GHz of 2.4). 1024 -> 1024@28x28 at batch 64
// (105 GFLOP): 534 us, 197 TFLOP/s of the 419 peak; fp32 MFMA's peak is 157.
template <class T, class BL, bool RES, int AC, bool SPLIT>
__global__ __launch_bounds__(kThreads, 2) void conv_split_kernel(ConvSplitArgs a) {
    __shared__ u32x4 lds[2][kSplitRuns];
    __shared__ uint32_t lost[kThreads];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile_m, tile_n;
    xcd_tile(gridDim.y, gridDim.x, tile_m, tile_n);
    const int m0 = tile_m * T::BM + wave * T::WM;
    const int n0 = tile_n * kSplitBN;
    const int z = blockIdx.z;
    const int group = SPLIT ? 0 : z;
    const int g0 = SPLIT ? z * a.chunk : 0;
    const int g1 = SPLIT ? min(a.groups_k, g0 + a.chunk) : a.groups_k;
    f32x4 acc[T::TM][T::TN];
    split_conv_segment<T, BL, RES>(a, group, m0, n0, g0, g1, !SPLIT, lds, lost, acc, tid, lane);
    // Opaque copies (split_check): what the store shares with the prologue, above all the
    // division of its columns, would stay in registers over the K loop, and a spilled index
    // read back there waits for every load in flight (1-pixel loads, 128 rows, up to 12 %).
    // The others do not spill, and computing it twice costs them 1-2 %.
    int ln = lane, mw = m0, nw = n0;
    if constexpr (T::BM == 128 && T::CW == 1) asm volatile("" : "+v"(ln), "+s"(mw), "+s"(nw));
    auto store = [&] {
        const int lane = ln, m0 = mw, n0 = nw;
        if constexpr (SPLIT) {
            const int ntot = a.t.geom.ntot;
#pragma unroll
            for (int j = 0; j < T::TN; ++j) {
                const int jcol = n0 + T::col0(j % T::NQ, lane) + j / T::NQ;
                if (jcol >= ntot) continue;
                float *wsz = a.t.ws + (int64_t)z * a.t.OC * ntot + jcol;
#pragma unroll
                for (int i = 0; i < T::TM; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int m = m0 + i * 16 + 4 * (lane >> 4) + r;
                        if (m < a.t.M) wsz[(int64_t)m * ntot] = acc[i][j][r];
                    }
            }
        } else {
            split_store<T, AC>(a.t, group, m0, n0, lane, acc);
        }
    };
    // Stored first, so that the check runs while the stores drain, and once more where sums
    // were replaced; not with a residual, which the output may be written over.
    if constexpr (!RES) store();
    split_check<T, RES>(a, group, m0, n0, g0, g1, !SPLIT, acc, lost, lane, [&] {
        if constexpr (!RES) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            store();
        }
    });
    if constexpr (RES) store();
}

// Data-parallel + stream-K launch (streamk.h) of a group-1 conv.
template <class T, class BL, bool RES, int AC, int SCHEME>
__global__ __launch_bounds__(kThreads, 2) void conv_split_sk_kernel(ConvSplitArgs a, SkSched s) {
    __shared__ u32x4 lds[2][kSplitRuns];
    __shared__ uint32_t lost[kThreads];
    __shared__ int sk_last;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    typedef f32x4 Acc[T::TM][T::TN];
    auto segment = [&](int t, int k0, int k1, Acc &acc) {
        // Opaque copies, so that the segments share nothing over each other's K loops.
        int ln = lane, td = tid;
        if constexpr (T::BM == 128 && T::CW == 1) asm volatile("" : "+v"(ln), "+v"(td));
        const int m0 = (t % s.tiles_m) * T::BM + wave * T::WM, n0 = (t / s.tiles_m) * kSplitBN;
        split_conv_segment<T, BL, RES>(a, 0, m0, n0, k0, k1, k0 == 0, lds, lost, acc, td, ln);
        split_check<T, RES>(a, 0, m0, n0, k0, k1, k0 == 0, acc, lost, ln, [] {});
    };
    auto store = [&](int t, const Acc &acc) {
        int ln = lane; // opaque, as in conv_split_kernel
        if constexpr (T::BM == 128 && T::CW == 1) asm volatile("" : "+v"(ln), "+s"(t));
        split_store<T, AC>(a.t, 0, (t % s.tiles_m) * T::BM + wave * T::WM, (t / s.tiles_m) * kSplitBN, ln, acc);
    };
    sk_run<SCHEME, T::TM * T::TN * 4, T::BM * kSplitBN, Acc>(s, tid, sk_last, segment, store);
}

// ---- launches ----

template <class T, class BL, bool RES, int AC>
int launch_conv_split_one(const ConvSplitArgs &a, int groups, int split, const SkSched *sk, int sk_grid,
                          hipStream_t st) {
    if (sk) {
        if (sk->scheme == kSkSplitWgs)
            hipLaunchKernelGGL((conv_split_sk_kernel<T, BL, RES, AC, kSkSplitWgs>), dim3(sk_grid), dim3(kThreads), 0,
                               st, a, *sk);
        else
            hipLaunchKernelGGL((conv_split_sk_kernel<T, BL, RES, AC, kSkPartsInDp>), dim3(sk_grid), dim3(kThreads), 0,
                               st, a, *sk);
        return check_launch();
    }
    const dim3 grid((a.t.geom.ntot + kSplitBN - 1) / kSplitBN, (a.t.M + T::BM - 1) / T::BM, split > 1 ? split : groups);
    if (split > 1) { // the post-op runs in the reduction kernel
        if constexpr (!RES && AC == 0)
            hipLaunchKernelGGL((conv_split_kernel<T, BL, false, 0, true>), grid, dim3(kThreads), 0, st, a);
        else return launch_conv_split_one<T, BL, false, 0>(a, groups, split, sk, sk_grid, st);
    } else {
        hipLaunchKernelGGL((conv_split_kernel<T, BL, RES, AC, false>), grid, dim3(kThreads), 0, st, a);
    }
    return check_launch();
}

template <int BM, class BL>
int launch_conv_split_act(const ConvSplitArgs &a, int groups, int split, const SkSched *sk, int sk_grid,
                          hipStream_t st) {
    using T = SplitTiling<BM, BL::CW>;
    const int ac = act_class(a.t.act);
    if (a.t.res) // only ADD and ADD_RELU carry a residual
        return ac == 1 ? launch_conv_split_one<T, BL, true, 1>(a, groups, split, sk, sk_grid, st)
                       : launch_conv_split_one<T, BL, true, 0>(a, groups, split, sk, sk_grid, st);
    if (ac == 1) return launch_conv_split_one<T, BL, false, 1>(a, groups, split, sk, sk_grid, st);
    if (ac == 3) return launch_conv_split_one<T, BL, false, 3>(a, groups, split, sk, sk_grid, st);
    return launch_conv_split_one<T, BL, false, 0>(a, groups, split, sk, sk_grid, st);
}

// One per loader (conv_split_*.hip), bm = 64 or 128.
int launch_conv_split_pw2(const ConvSplitArgs &a, int bm, int groups, int split, const SkSched *sk, int sk_grid, hipStream_t st);
int launch_conv_split_gather(const ConvSplitArgs &a, int bm, int groups, int split, const SkSched *sk, int sk_grid, hipStream_t st);
int launch_conv_split_gather_tail(const ConvSplitArgs &a, int bm, int groups, int split, const SkSched *sk, int sk_grid, hipStream_t st);

} // namespace spinn
